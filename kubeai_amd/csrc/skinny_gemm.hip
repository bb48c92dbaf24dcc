// Weight-streaming products for few rows: y[M,N] = x[M,K] W[N,K]^T with
// M <= 96, bf16 or fp8 e4m3 (W8A8 with row and column scales), bf16 out,
// fp32 accumulation. Decode batches and the logits of a step's last tokens.
//
// Bound by reading W once: 6.3 TB/s is what plain reads in order reach here. What it
// takes to come near that:
//  - workgroup = 4 waves x 16 rows of W. A wave's lanes read 16 rows x 64
//    contiguous bytes straight into matrix operands (no LDS for W: each byte
//    is used by one wave); two of those loads fill a 128-byte line. The steps
//    are 256 bytes of every row (step_bytes); two of them are in flight behind the one that is
//    multiplied. Loads past the end are of no bytes instead of in a branch: where
//    paths of more and of fewer loads meet, the compiler waits for all of them (one
//    row of 28672 x 4096 bf16: 46.5 us -> 43.4).
//  - x is what the CUs would re-read: with 16 rows of W per workgroup its
//    traffic is M / 16 that of W, and past M = 16 that limits (40 rows fp8:
//    54 us for 28672 x 4096 against 28 with x shared by 64 rows). It goes
//    straight to LDS (three places, one barrier a step, 16-byte units
//    XOR-swizzled by row by the choice of source) and is shared by the waves.
//  - few output columns do not fill the chip: K is cut into up to 8 parts,
//    whose fp32 sums lie in a workspace [parts, M, N]; a second
//    kernel adds them (no atomics: the order of the sum is fixed). The parts of
//    a row lie in neighbouring workgroups: what is read at a time is whole rows
//    (6144 x 4096 bf16 in 8 parts, read alone: 9.8 us apart, 9.4).
//  - uncut, the workgroups begin at columns of K apart. At the same columns of rows
//    of 2^n bytes all of them wait for the same few channels of the memory (read
//    alone, 28672 x 4096 bf16 41.9 us, 37.6 apart; multiplied, 8 waves, 51.7 / 40.2).
//  - uncut, up to 16 rows: as many waves a workgroup as share the columns evenly
//    among the CUs (waves_for).
// With N columns there are N / 64 workgroups; below 256 of them K is cut so
// that about 768 result (N = 6144, 40 rows fp8: 8.8 us with 768, 9.7 with
// 384); from 256 on the second pass costs more than the parts give (28672:
// 28.2 us whole, 29.8 in two parts).
// Where a consumer can add the parts itself (skinny_sums; the norm after an
// attention or feed-forward block, the rotation of q and k) that second pass,
// about 5 us of launch and drain, is gone; so is the activation's launch behind gate
// and up (skinny_gated).
// W out of cache, us, with branches and the same first columns -> now:
//   bf16, 1 row   4096 -> 28672  47.4 -> 41.2 (5.7 TB/s), with silu 49.6 -> 42.0
//                 4096 -> 6144   12.1 -> 11.5; 4096 -> 4096 9.2 -> 8.6
//                 14336 -> 4096  24.4 -> 22.5; 2304 -> 18432 23.4 -> 20.3
//                 4096 -> 128256 200 -> 176
//   bf16, 96 rows 4096 -> 4096 14.3 -> 14.3; 14336 -> 4096 35.3 -> 35.2
//   fp8, 8 rows   4096 -> 28672 29.0 -> 24.8; 4096 -> 6144 7.7 -> 7.3; 4096 -> 4096
//                 5.3 -> 5.4; 14336 -> 4096 15.4 -> 13.4; 2304 -> 18432 16.3 -> 12.5
//   fp8, 40 rows  4096 -> 6144 9.9 -> 9.8; 4096 -> 4096 7.2 -> 6.7
// The grouped form multiplies every expert's rows of a mixture in one launch,
// x rows gathered by index, its columns in order (below). 8 experts, 80 rows, 28672 x 4096
// and 4096 x 14336: fp8 183 + 93 us -> 177 + 89, bf16 353 + 198 -> 354 + 194. The experts
// that have rows are counted off by the workgroups: with a place for every expert, and
// all workgroups in place at once, some CUs had two to four of them and others none (16
// experts of 4096 x 6400, bf16, 4 rows 88 -> 44 us, 16 rows 136 -> 115; 32 of 2816 x 2048 16
// rows 53 -> 41).
#include <torch/extension.h>

#include <cmath>
#include <type_traits>

#include "common.h"

namespace {

constexpr int kNW = 4;         // waves per workgroup (waves_for: of uncut few rows)
constexpr int kMaxRows = 96;
constexpr int kMaxParts = 8;
// Bytes of K a step. Experts of many fp8 rows: x of three steps of 256 in passes of 96 rows
// would leave a CU two workgroups (7168 x 1024, 4 experts, 391 rows 23.8 us, 21.4). Passes of
// 64 rows lose by the shorter steps (28672 x 4096, 8 experts, 3 to 5 %), and so does bf16
// (4096 x 14336, 8 experts, 206 rows 197 us, 204).
constexpr int step_bytes(bool fp8, int mt, bool grouped) {
  return fp8 && grouped && mt > 4 ? 128 : 256;
}
constexpr int kAhead = 3;      // steps of x in LDS and of w in registers
constexpr int64_t kFarRows = (int64_t)1 << 23;  // bytes

typedef __attribute__((ext_vector_type(8))) short bf16x8;
typedef __attribute__((ext_vector_type(4))) float f32x4;
typedef __attribute__((ext_vector_type(4))) int i32x4;
typedef __attribute__((ext_vector_type(2))) long i64x2;

// 64 bytes of K per row: one step of bf16, two of fp8. Both operands take
// their K in the same order (lane group kg holds bytes [16 kg, 16 kg + 16)),
// so any order will do.
template <bool FP8>
DEV_INLINE f32x4 mfma_64b(i32x4 a, i32x4 b, f32x4 c) {
  if constexpr (FP8) {
    const i64x2 x = __builtin_bit_cast(i64x2, a);
    const i64x2 y = __builtin_bit_cast(i64x2, b);
    c = __builtin_amdgcn_mfma_f32_16x16x32_fp8_fp8(x[0], y[0], c, 0, 0, 0);
    return __builtin_amdgcn_mfma_f32_16x16x32_fp8_fp8(x[1], y[1], c, 0, 0, 0);
  } else {
    return __builtin_amdgcn_mfma_f32_16x16x32_bf16(
        __builtin_bit_cast(bf16x8, a), __builtin_bit_cast(bf16x8, b), c, 0, 0, 0);
  }
}

// rows of a product over experts: expert e owns rows [begin[e], begin[e + 1])
// of the result; row i reads row src[i] of x (i itself without src) and its
// scale. W and sw are stacked by expert.
struct Groups {
  const int32_t* begin;
  const int32_t* src;
};

// four neighbouring columns of a row, scaled, biased and rounded
DEV_INLINE void store4(ushort* y, f32x4 v, const float* sx, const float* sw,
                       const ushort* bias, int m, int n) {
  const float s = sx ? sx[m] : 1.0f;
  ushort4_t o;
#pragma unroll
  for (int e = 0; e < 4; ++e) {
    float f = v[e];
    if (sw) f = f * s * sw[n + e];
    if (bias) f += bf16_to_f32(bias[n + e]);
    o[e] = f32_to_bf16(f);
  }
  *reinterpret_cast<ushort4_t*>(y) = o;
}

// 16 bytes a lane from base + voff + soff, zeros past `size` bytes; to registers or
// to l + 16 * lane in LDS
DEV_INLINE i32x4 load16(const char* base, int size, int voff, int soff) {
#ifdef __HIP_DEVICE_COMPILE__
  const auto r = __builtin_amdgcn_make_buffer_rsrc((void*)base, 0, size, 0x00020000);
  return __builtin_bit_cast(i32x4, __builtin_amdgcn_raw_buffer_load_b128(r, voff, soff, 0));
#else
  return i32x4{};
#endif
}
DEV_INLINE void load_lds16(const char* base, int size, char* l, int voff, int soff) {
#ifdef __HIP_DEVICE_COMPILE__
  const auto r = __builtin_amdgcn_make_buffer_rsrc((void*)base, 0, size, 0x00020000);
  __builtin_amdgcn_raw_ptr_buffer_load_lds(
      r, (__attribute__((address_space(3))) uint32_t*)l, 16, voff, soff, 0, 0);
#endif
}
constexpr int kNowhere = 0x7fffffff;  // past the end of every buffer

// own LDS reads are done, all but the last N loads have landed
template <int N>
DEV_INLINE void wait_loads() {
  static_assert(N < 64);
  __builtin_amdgcn_s_waitcnt((N & 15) | ((N >> 4) << 14) | 0x70);
}

// Nothing moves over it, loads neither: x and w are not __restrict__, so the
// compiler takes the asm to write what they point to. (wait_loads counts them.)
DEV_INLINE void in_order() {
  __builtin_amdgcn_sched_barrier(0);
  asm volatile("" ::: "memory");
  __builtin_amdgcn_sched_barrier(0);
}
DEV_INLINE void barrier() {
  in_order();
  __builtin_amdgcn_s_barrier();
  in_order();
}

// the n-th of the experts that have rows, -1 if there are fewer
DEV_INLINE int expert_with_rows(const int32_t* begin, int experts, int n, int lane) {
  for (int at = 0; at < experts; at += WAVE_SIZE) {
    const int i = min(at + lane, experts - 1);
    const bool has = at + lane < experts && begin[i + 1] > begin[i];
    const uint64_t mask = __builtin_amdgcn_ballot_w64(has);
    const int count = __builtin_popcountll(mask);
    if (n < count) {
      const int before = __builtin_amdgcn_mbcnt_hi(
          (uint32_t)(mask >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)mask, 0u));
      return at + __builtin_ctzll(__builtin_amdgcn_ballot_w64(has && before == n));
    }
    n -= count;
  }
  return -1;
}

// MT: 16-row tiles of x. part != null: raw sums of this K range.
// GROUPED: blockIdx.z is the place among the experts with rows; an expert's rows are
// taken MT * 16 at a time (W is read again for each such pass: the host picks MT so
// that one is usual).
// ACT (bf16): silu (1) or tanh-gelu (2) of column n times column n + N / 2, in fp32,
// rounded once; a wave has 8 columns of either half.
template <bool FP8, int MT, bool GROUPED, int ACT, int NW>
__launch_bounds__(NW * WAVE_SIZE) __global__ void skinny_kernel(
    ushort* y,         // [M, N], ACT: [M, N / 2]
    float* part,       // [parts, M, N]
    const char* x,     // M rows of KB bytes, ldx apart
    const char* w,     // N rows of KB bytes
    const float* sx, const float* sw, const ushort* bias, const int M_all,
    const int N, const int KB, const int ldx, const int xbytes, const int k_part,
    const int parts, const Groups grp) {
  constexpr int kStep = step_bytes(FP8, MT, GROUPED), CH = kStep / 64, UPR = kStep / 16;
  constexpr int RW = ACT ? 8 : 16;             // columns of the result a wave
  constexpr int NX = (MT * 16 * UPR - 1) / (NW * WAVE_SIZE) + 1, L = NX + CH;  // loads a step
  constexpr int PLACE = NX * NW * WAVE_SIZE * 16;  // x of a step in LDS
  static_assert(!GROUPED || PLACE == MT * 16 * kStep);  // (else M <= 16 MT)
  __shared__ __attribute__((aligned(16))) char xs[kAhead * PLACE];

  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / WAVE_SIZE);
  const int lane = threadIdx.x % WAVE_SIZE, r = lane & 15, kg = lane >> 4;
  const int tile = blockIdx.x / parts, of = blockIdx.x % parts;
  const int cols = ACT ? N / 2 : N;  // of the result
  const int n0 = (tile * NW + wave) * RW;
  const int k0 = of * k_part, k1 = min(KB, k0 + k_part);
  const int steps = (k1 - k0 + kStep - 1) / kStep;
  // whole rows of 2^n bytes: workgroups that read the same columns of K at a time
  // wait for the same few of the memory's channels. Not those of experts: in a routed
  // model a sum in another order moves tokens whose scores all but tie.
  const int first =
      !GROUPED && parts == 1 ? __builtin_amdgcn_readfirstlane((blockIdx.x >> 3) * 3u % (uint32_t)steps) : 0;
  int m0 = 0, M = M_all;  // this pass's first row and the rows from it on
  int m_end = M_all;
  if constexpr (GROUPED) {
    const int e = expert_with_rows(grp.begin, gridDim.z, blockIdx.z, lane);
    if (e < 0) return;  // whole workgroup
    m0 = grp.begin[e];
    m_end = grp.begin[e + 1];
    w += (int64_t)e * N * KB;
    if (sw) sw += (int64_t)e * N;
    M = m_end - m0;
  }
  const char* wb = w + (int64_t)n0 * KB;
  const int left = max(0, min(cols - n0, RW));  // rows of w
  const int wbytes = left == 0 ? 0 : (ACT ? cols + left : left) * KB;
  // lane's offsets; xk: within a row's step
  const int wo = (ACT ? (r & 7) + (r >> 3) * cols : r) * KB + kg * 16;
  int xo[NX], xk[NX];

  f32x4 acc[MT];
  i32x4 wf[kAhead][CH];
  do {
#pragma unroll
    for (int j = 0; j < MT; ++j) acc[j] = f32x4{0.f, 0.f, 0.f, 0.f};
    // offsets are 32 bits: where experts' rows lie in order, from this pass's first on
    const bool in_rows = GROUPED && !grp.src;
    const char* xb = in_rows ? x + (int64_t)m0 * ldx : x;
    const int xn = in_rows ? (min(M, MT * 16) - 1) * ldx + KB : xbytes;
#pragma unroll
    for (int i = 0; i < NX; ++i) {
      // 16-byte unit u of row r lies at u ^ (r & 7): made by the choice of source
      const int at = (wave * NX + i) * WAVE_SIZE + lane, row = at / UPR;
      xk[i] = ((at % UPR) ^ (row & 7)) * 16;
      xo[i] = kNowhere;
      if (row < M) {
        int from = row;
        if constexpr (GROUPED) {
          if (!in_rows) from = grp.src[m0 + row];
        }
        xo[i] = from * ldx + xk[i];
      }
    }
    int next = first, ahead = 0;  // the step to load and the number loaded
    auto load = [&](auto place) {
      constexpr int P = decltype(place)::value;
      const int k = k0 + next * kStep, on = ahead < steps;
#pragma unroll
      for (int i = 0; i < NX; ++i)
        load_lds16(xb, on ? xn : 0, xs + P * PLACE + (wave * NX + i) * 1024,
                   xk[i] < k1 - k ? xo[i] : kNowhere, k);
#pragma unroll
      for (int c = 0; c < CH; ++c)
        wf[P][c] = load16(wb, on && k + c * 64 < k1 ? wbytes : 0, wo + c * 64, k);
      next = next + 1 == steps ? 0 : next + 1;
      ++ahead;
    };
    // one step: its loads have landed everywhere, and everyone is done with the
    // step before it, whose place the next loads take
    auto step = [&](auto place, auto behind, auto more) {
      constexpr int P = decltype(place)::value;
      in_order();
      wait_loads<decltype(behind)::value * L>();  // so many steps are loaded behind this one
      barrier();
      if constexpr (decltype(more)::value) {
        load(std::integral_constant<int, (P + kAhead - 1) % kAhead>{});
        in_order();
      }
#pragma unroll
      for (int c = 0; c < CH; ++c)
#pragma unroll
        for (int j = 0; j < MT; ++j) {
          if (GROUPED && j * 16 >= M) break;  // the same in every lane
          const i32x4 xf = *reinterpret_cast<const i32x4*>(
              xs + P * PLACE + (j * 16 + r) * kStep + (((c * 4 + kg) ^ (r & 7)) << 4));
          acc[j] = mfma_64b<FP8>(wf[P][c], xf, acc[j]);
        }
    };
    static_assert(kAhead == 3);
    constexpr std::integral_constant<int, 0> zero;
    constexpr std::integral_constant<int, 1> one;
    constexpr std::integral_constant<int, 2> two;
    in_order();
    load(zero);
    in_order();  // wait_loads counts on it
    load(one);
    // (a loop that is left in its middle has the compiler wait for all loads)
    for (int s = steps; s >= kAhead; s -= kAhead) {
      step(zero, one, one);
      step(one, one, one);
      step(two, one, one);
    }
    if (steps % kAhead > 0) step(zero, one, zero);
    if (steps % kAhead > 1) step(one, zero, zero);
    wait_loads<0>();  // (the last ones, of nothing, write LDS too)

    // accumulator: row (W) 4 kg + e, column (x) r; with ACT the lanes from 32 on have
    // the other half's
    const int n = n0 + kg * 4;
#pragma unroll
    for (int j = 0; j < MT; ++j) {
      f32x4 v = acc[j];
      if constexpr (ACT != 0) {
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          const float up = __shfl_xor(v[e], 32);
          float z = v[e];  // gelu: 0.5 (1 + tanh y) = 1 / (1 + e^-2y)
          if constexpr (ACT == 2) z = 1.5957691216057308f * (z + 0.044715f * z * z * z);
          v[e] = v[e] / (1.0f + __expf(-z)) * up;
        }
        if (kg >= 2) continue;
      }
      const int m = j * 16 + r;
      if (m >= M || n >= cols) continue;  // (cols: a multiple of 4)
      if (part)
        *reinterpret_cast<f32x4*>(part + ((int64_t)of * M_all + m) * N + n) = v;
      else
        store4(y + (int64_t)(m0 + m) * cols + n, v, sx, sw, bias,
               GROUPED && grp.src ? grp.src[m0 + m] : m0 + m, n);
    }
    if constexpr (GROUPED) {
      m0 += MT * 16;
      M = m_end - m0;
      if (M > 0) barrier();  // everyone has read the last step
    }
  } while (GROUPED && M > 0);
}

__launch_bounds__(256) __global__ void skinny_sum_kernel(
    ushort* __restrict__ y, const float* __restrict__ part,
    const float* __restrict__ sx, const float* __restrict__ sw,
    const ushort* __restrict__ bias, const int M, const int N,
    const int parts) {
  const int i = blockIdx.x * 256 + threadIdx.x;  // M * N / 4 < 2^31
  if (i >= M * (N / 4)) return;
  const int m = i / (N / 4), n = i % (N / 4) * 4;
  const float* p = part + (int64_t)m * N + n;
  f32x4 v = *reinterpret_cast<const f32x4*>(p);
  for (int s = 1; s < parts; ++s)
    v += *reinterpret_cast<const f32x4*>(p + (int64_t)s * M * N);
  store4(y + (int64_t)m * N + n, v, sx, sw, bias, m, n);
}

// how K is cut: no part is empty
struct Cut {
  int parts, k_part;
};
Cut cut_for(int N, int KB) {
  const int wgs = (N + kNW * 16 - 1) / (kNW * 16);
  int parts = 1;
  if (wgs < 256)
    parts = std::max(1, std::min({kMaxParts, (768 + wgs - 1) / wgs, KB / 512}));
  const int k_part = (KB / 64 + parts - 1) / parts * 64;
  return {(KB + k_part - 1) / k_part, k_part};
}

struct Shape {
  int M, N, KB;
  bool fp8;
};

// Offsets are 32 bits: rows under 8 MB apart (others are copied).
torch::Tensor near_rows(const torch::Tensor& x) {
  return x.dim() == 2 && x.stride(0) * x.element_size() >= kFarRows ? x.contiguous() : x;
}

Shape check(const torch::Tensor& x, const torch::Tensor& w,
            const c10::optional<torch::Tensor>& sx,
            const c10::optional<torch::Tensor>& sw,
            const c10::optional<torch::Tensor>& bias, bool raw = false) {
  const bool fp8 = w.scalar_type() == torch::kFloat8_e4m3fn;
  TORCH_CHECK(fp8 || w.scalar_type() == torch::kBFloat16,
              "bf16 or fp8 e4m3 weights");
  TORCH_CHECK(x.scalar_type() == w.scalar_type() && x.is_cuda() && w.is_cuda());
  TORCH_CHECK(x.dim() == 2 && w.dim() == 2 && x.size(1) == w.size(1));
  TORCH_CHECK(x.stride(1) == 1 && w.is_contiguous());
  const int es = fp8 ? 1 : 2;
  const Shape s{(int)x.size(0), (int)w.size(0), (int)w.size(1) * es, fp8};
  TORCH_CHECK(s.M >= 1 && s.M <= kMaxRows, "1 to 96 rows");
  TORCH_CHECK(s.KB >= 64 && s.KB % 64 == 0 && s.KB < kFarRows && s.N % 4 == 0 &&
              (int64_t)s.M * s.N < (1ll << 31));
  TORCH_CHECK(x.stride(0) * es % 16 == 0 && x.stride(0) >= x.size(1) &&
              ((uintptr_t)x.data_ptr() & 15) == 0 &&
              ((uintptr_t)w.data_ptr() & 15) == 0,
              "16-byte aligned rows");
  TORCH_CHECK(raw || fp8 == (sx.has_value() && sw.has_value()),
              "fp8 operands come with their scales, bf16 ones without");
  if (fp8 && !raw) {
    TORCH_CHECK(sx->scalar_type() == torch::kFloat32 && sx->is_contiguous() &&
                sx->is_cuda() && sx->numel() == s.M &&
                sw->scalar_type() == torch::kFloat32 && sw->is_contiguous() &&
                sw->is_cuda() && sw->numel() == s.N);
  }
  if (bias.has_value())
    TORCH_CHECK(bias->scalar_type() == torch::kBFloat16 && bias->is_cuda() &&
                bias->is_contiguous() && bias->numel() == s.N);
  return s;
}

// Waves of a workgroup of a whole product of up to 16 rows: those with which the CUs
// have the most even share of the columns' tiles, as many as possible, which share
// x. us at one row, bf16, 2 / 4 / 8 waves: 28672 x 4096
// 45.6 / 43.1 / 41.1, 24576 x 4096 35.7 / 42.1 / 37.9, 18432 x 2304 20.3 / 24.5 / 22.5,
// 16384 x 4096 25.3 / 25.0 / 40.0, 53248 x 4096 83.1 / 87.8 / 86.9.
int waves_for(int N) {
  int best = 8, most = 1 << 30;
  for (int nw = 8; nw >= 2; nw /= 2) {
    const int wgs = (N + nw * 16 - 1) / (nw * 16), on_one = (wgs + 255) / 256 * nw;
    if (on_one < most) {
      best = nw;
      most = on_one;
    }
  }
  return best;
}

void launch(ushort* y, float* part, const torch::Tensor& x,
            const torch::Tensor& w, const float* sx, const float* sw,
            const ushort* bias, const Shape& s, const Cut& cut, int act = 0) {
  const int nw = s.M <= 16 && cut.parts == 1 ? waves_for(s.N) : kNW;
  const dim3 grid((s.N + nw * 16 - 1) / (nw * 16) * cut.parts);
  const int ldx = x.stride(0) * x.element_size();
  const int xbytes = (s.M - 1) * ldx + s.KB;
  auto stream = c10::hip::getCurrentHIPStream().stream();
  auto go = [&](auto fp8, auto mt, auto a, auto waves) {
    constexpr int NW = decltype(waves)::value;
    hipLaunchKernelGGL((skinny_kernel<decltype(fp8)::value, decltype(mt)::value, false,
                                      decltype(a)::value, NW>),
                       grid, dim3(NW * WAVE_SIZE), 0, stream, y, part,
                       (const char*)x.data_ptr(), (const char*)w.data_ptr(),
                       sx, sw, bias, s.M, s.N, s.KB, ldx, xbytes, cut.k_part, cut.parts,
                       Groups{});
  };
  constexpr std::integral_constant<int, 0> none;
  constexpr std::integral_constant<int, 1> one;
  constexpr std::integral_constant<int, 2> two;
  constexpr std::integral_constant<int, kNW> four;
  constexpr std::integral_constant<int, 8> eight;
  auto few = [&](auto fp8, auto a) {
    if (nw == 8) go(fp8, one, a, eight);
    else if (nw == 4) go(fp8, one, a, four);
    else go(fp8, one, a, two);
  };
  if (act) {
    if (act == 1) few(std::false_type{}, one);
    else few(std::false_type{}, two);
    HIP_CHECK_KERNEL();
    return;
  }
  auto tiles = [&](auto fp8) {
    switch ((s.M + 15) / 16) {
      case 1: few(fp8, none); break;
      case 2: go(fp8, two, none, four); break;
      case 3: go(fp8, std::integral_constant<int, 3>{}, none, four); break;
      case 4: go(fp8, four, none, four); break;
      case 5: go(fp8, std::integral_constant<int, 5>{}, none, four); break;
      default: go(fp8, std::integral_constant<int, 6>{}, none, four); break;
    }
  };
  if (s.fp8) tiles(std::true_type{});
  else tiles(std::false_type{});
  HIP_CHECK_KERNEL();
}

}  // namespace

// y = x w^T (x, w bf16), or (x * sx) (w * sw)^T (fp8 with scales), + bias
void skinny_linear(torch::Tensor y, torch::Tensor x, torch::Tensor w,
                   c10::optional<torch::Tensor> sx,
                   c10::optional<torch::Tensor> sw,
                   c10::optional<torch::Tensor> bias) {
  x = near_rows(x);
  const Shape s = check(x, w, sx, sw, bias);
  TORCH_CHECK(y.scalar_type() == torch::kBFloat16 && y.is_contiguous() &&
              y.is_cuda() && y.dim() == 2 && y.size(0) == s.M && y.size(1) == s.N);
  const float* sxp = s.fp8 ? sx->data_ptr<float>() : nullptr;
  const float* swp = s.fp8 ? sw->data_ptr<float>() : nullptr;
  const ushort* bp = bias.has_value() ? (const ushort*)bias->data_ptr() : nullptr;
  auto* yp = (ushort*)y.data_ptr();
  const Cut cut = cut_for(s.N, s.KB);
  if (cut.parts == 1) {
    launch(yp, nullptr, x, w, sxp, swp, bp, s, cut);
    return;
  }
  auto part = torch::empty({cut.parts, s.M, s.N}, x.options().dtype(torch::kFloat32));
  launch(nullptr, part.data_ptr<float>(), x, w, nullptr, nullptr, nullptr, s, cut);
  hipLaunchKernelGGL(skinny_sum_kernel, dim3((s.M * (s.N / 4) + 255) / 256),
                     dim3(256), 0, c10::hip::getCurrentHIPStream().stream(), yp,
                     part.data_ptr<float>(), sxp, swp, bp, s.M, s.N, cut.parts);
  HIP_CHECK_KERNEL();
}

// the fp32 sums of x w^T alone, [parts, M, N], for a consumer that adds the
// parts itself (and applies an fp8 product's scales)
torch::Tensor skinny_sums(torch::Tensor x, torch::Tensor w) {
  c10::optional<torch::Tensor> none;
  x = near_rows(x);
  const Shape s = check(x, w, none, none, none, true);
  const Cut cut = cut_for(s.N, s.KB);
  auto part = torch::empty({cut.parts, s.M, s.N}, x.options().dtype(torch::kFloat32));
  launch(nullptr, part.data_ptr<float>(), x, w, nullptr, nullptr, nullptr, s, cut);
  return part;
}

// y [M, N / 2] = silu (act 1) or tanh-gelu (act 2) of the first N / 2 columns of x w^T
// times the others; bf16, up to 16 rows
void skinny_gated(torch::Tensor y, torch::Tensor x, torch::Tensor w, int64_t act) {
  c10::optional<torch::Tensor> none;
  x = near_rows(x);
  const Shape s = check(x, w, none, none, none);
  TORCH_CHECK(!s.fp8 && s.M <= 16 && s.N % 8 == 0 && (act == 1 || act == 2));
  TORCH_CHECK((int64_t)s.N * s.KB < (1ll << 31), "gate and up columns");
  TORCH_CHECK(y.scalar_type() == torch::kBFloat16 && y.is_contiguous() &&
              y.is_cuda() && y.dim() == 2 && y.size(0) == s.M && y.size(1) == s.N / 2);
  launch((ushort*)y.data_ptr(), nullptr, x, w, nullptr, nullptr, nullptr, s, {1, s.KB},
         (int)act);
}

// y[i] = x[src[i]] w[e]^T for the rows i of expert e, scaled as above; w
// [E, N, K] (sw [E, N]), begin int32 [E + 1] ascending with begin[E] <= rows
// of y, src int32 (entries are rows of x) or none
void skinny_experts(torch::Tensor y, torch::Tensor x, torch::Tensor w,
                    c10::optional<torch::Tensor> sx,
                    c10::optional<torch::Tensor> sw, torch::Tensor begin,
                    c10::optional<torch::Tensor> src) {
  const bool fp8 = w.scalar_type() == torch::kFloat8_e4m3fn;
  TORCH_CHECK(fp8 || w.scalar_type() == torch::kBFloat16);
  TORCH_CHECK(x.scalar_type() == w.scalar_type() && x.is_cuda() && w.is_cuda());
  TORCH_CHECK(x.dim() == 2 && w.dim() == 3 && x.size(1) == w.size(2));
  TORCH_CHECK(x.stride(1) == 1 && w.is_contiguous());
  const int es = fp8 ? 1 : 2;
  const int E = w.size(0), N = w.size(1), KB = (int)w.size(2) * es;
  TORCH_CHECK(KB >= 64 && KB % 64 == 0 && KB < kFarRows && N % 4 == 0 && E >= 1 &&
              E <= 65535);
  TORCH_CHECK(x.stride(0) * es % 16 == 0 && x.stride(0) >= x.size(1) &&
              ((uintptr_t)x.data_ptr() & 15) == 0 &&
              ((uintptr_t)w.data_ptr() & 15) == 0,
              "16-byte aligned rows");
  TORCH_CHECK(fp8 == (sx.has_value() && sw.has_value()));
  TORCH_CHECK(begin.scalar_type() == torch::kInt32 && begin.is_contiguous() &&
              begin.is_cuda() && begin.numel() == E + 1);
  TORCH_CHECK(y.scalar_type() == torch::kBFloat16 && y.is_contiguous() &&
              y.is_cuda() && y.dim() == 2 && y.size(1) == N);
  if (src.has_value()) {
    TORCH_CHECK(src->scalar_type() == torch::kInt32 && src->is_contiguous() &&
                src->is_cuda() && src->numel() == y.size(0));
  } else {
    TORCH_CHECK(x.size(0) == y.size(0));
  }
  if (fp8) {
    TORCH_CHECK(sx->scalar_type() == torch::kFloat32 && sx->is_contiguous() &&
                sx->is_cuda() && sx->numel() == x.size(0) &&
                sw->scalar_type() == torch::kFloat32 && sw->is_contiguous() &&
                sw->is_cuda() && sw->numel() == (int64_t)E * N);
  }
  const int R = y.size(0);
  if (R == 0) return;
  if (src.has_value() && x.size(0) * x.stride(0) * es >= (1ll << 31)) {
    // offsets are 32 bits: the rows in the order of the experts
    if (fp8) sx = sx->reshape(-1).index_select(0, *src);
    x = x.view(torch::kUInt8).index_select(0, *src).view(x.scalar_type());
    src = c10::nullopt;
  }
  if (!src.has_value()) x = near_rows(x);
  const float* sxp = fp8 ? sx->data_ptr<float>() : nullptr;
  const float* swp = fp8 ? sw->data_ptr<float>() : nullptr;
  const Groups g{begin.data_ptr<int32_t>(),
                 src.has_value() ? src->data_ptr<int32_t>() : nullptr};
  const int ldx = x.stride(0) * es;
  const int xbytes = src.has_value() ? (x.size(0) - 1) * ldx + KB : 0;  // (else by the pass)
  auto stream = c10::hip::getCurrentHIPStream().stream();
  auto go = [&](auto f, auto mt, auto waves) {
    constexpr int NW = decltype(waves)::value;
    const dim3 grid((N + NW * 16 - 1) / (NW * 16), 1, E);
    hipLaunchKernelGGL((skinny_kernel<decltype(f)::value, decltype(mt)::value, true, 0, NW>),
                       grid, dim3(NW * WAVE_SIZE), 0, stream,
                       (ushort*)y.data_ptr(), nullptr, (const char*)x.data_ptr(),
                       (const char*)w.data_ptr(), sxp, swp, nullptr, R, N, KB,
                       ldx, xbytes, KB, 1, g);
  };
  // rows per expert if they are spread evenly; half as many again fit a pass
  const int mean = (R + E - 1) / E;
  // Few rows whose experts (as many as R rows at random reach) have fewer than four
  // workgroups a CU: two waves each, so that the CUs' shares are more even. us, with
  // branches in the loop and four waves / four / two: 8 of 4096 x 14336 bf16 8 rows 134 /
  // 164 / 132, 16 rows 171 / 189 / 176, fp8 8 rows 68 / 78 / 65; but 8 of 28672 x 4096
  // bf16 16 rows 350 / 348 / 359. Over 883 products (up to 64 experts) of under four a
  // CU 1.27 times as fast as with branches, 0.88 at worst (four waves 1.16), over 342 of
  // more 1.02 (four 1.04).
  const double reached = E * (1.0 - std::pow(1.0 - 1.0 / E, R));
  const bool thin = reached * ((N + kNW * 16 - 1) / (kNW * 16)) < 4 * 256;
  // Many bf16 rows, of which a workgroup reads as many bytes as of the weights: eight waves
  // where those are just one workgroup a CU (us, four / eight: 8 of 4096 x 14336 206 rows 198
  // / 178, 376 rows 216 / 196; but 16 of 12800 x 4096 416 rows 336 / 356, more than one a CU.
  // Where half the rows are one expert's, its passes lie on fewer CUs: both products of a
  // mixture of 128 tokens 788 / 802, 224 899 / 910; spread evenly 647 / 643, 689 / 681).
  const double eights = reached * ((N + 127) / 128);
  const bool one_each = eights > 192 && eights <= 256;
  constexpr std::integral_constant<int, 2> two;
  constexpr std::integral_constant<int, kNW> four;
  auto tiles = [&](auto f) {
    constexpr std::integral_constant<int, 1> one;
    if constexpr (!decltype(f)::value) {
      constexpr std::integral_constant<int, 8> eight;
      if (mean > 44 && one_each) return go(f, std::integral_constant<int, 6>{}, eight);
      if (mean > 22 && one_each) return go(f, four, eight);
    }
    if (mean <= 8 && thin) go(f, one, two);
    else if (mean <= 8) go(f, one, four);
    else if (mean <= 22) go(f, two, four);
    else if (mean <= 44) go(f, four, four);
    else go(f, std::integral_constant<int, 6>{}, four);
  };
  if (fp8) tiles(std::true_type{});
  else tiles(std::false_type{});
  HIP_CHECK_KERNEL();
}

void skinny_gemm(torch::Tensor y, torch::Tensor x, torch::Tensor w) {
  skinny_linear(y, x, w, c10::nullopt, c10::nullopt, c10::nullopt);
}
