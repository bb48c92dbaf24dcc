// Products of a mixture's large steps: y[i] = x[src[i]] w[e]^T for the rows i
// of every expert e, in one launch, bf16 or fp8 e4m3 (W8A8 with row and column
// scales), bf16 out, fp32 accumulation. The row counts stay on the device:
// the grid covers the most row tiles any split over the experts can have
// (rows / tile + experts) and what is left over ends at once, so a step needs
// no look at its routing from the host.
//
// Bound by the matrix cores and by LDS, which feeds them at most of its rate:
//  - 512 threads, tiles of 128, 192 or 256 rows x 256 columns with K in steps of
//    128 bytes. A wave multiplies half the rows x 64 in 32 x 32 matrix
//    instructions; the taller, the fewer LDS bytes per product.
//  - both operands go straight to LDS (16 bytes a lane), the next step's while
//    this one's are multiplied. Such a load writes 64 lanes in a row, so the
//    swizzle that keeps the reads free of bank conflicts (16-byte unit u of
//    row r lies at u ^ (r & 7)) is made by the lane's choice of source.
//  - at 192 and 256 rows the two waves of a SIMD take turns at LDS and at the
//    matrix cores (8 experts of 2048 rows, 28672 x 4096 bf16: 987 -> 1095
//    TFLOP/s; at 128 rows all waves read and multiply together, which is 3 to
//    8 % faster there).
//  - an XCD's tiles are consecutive: an expert's row tiles down one column, then
//    the next column, so they read the same rows of w from its L2.
// One workgroup per CU, so a grid takes whole passes of 256 and an expert's last
// tile is half empty on average: the tile height is the one with the least
// passes x cost of a pass (bf16 40 : 50 : 61, fp8 40 : 46 : 53, as measured). With
// few rows the product streams the weights, and empty rows cost the least in
// the smallest tile (16 rows per expert, 28672 x 4096 fp8: 194 us, 253 with
// tiles of 256).
// A layer of 8 experts of 3584 x 2048 (squared ReLU, 2 of 8), us, a library
// product per expert -> this: 300 tokens 484 -> 174, 3072 tokens 625 -> 390,
// 8192 tokens 1063 -> 880.
// Where the next operation is relu(y)^2 times a weight per row it is done on
// the rounded product before it is stored.
#include <torch/extension.h>

#include <type_traits>

#include "common.h"

namespace {

constexpr int kThreads = 512;
constexpr int kStep = 128;  // bytes of K per step

typedef __attribute__((ext_vector_type(8))) short bf16x8;
typedef __attribute__((ext_vector_type(16))) float f32x16;
typedef __attribute__((ext_vector_type(4))) int i32x4;
typedef __attribute__((ext_vector_type(8))) int i32x8;
typedef __attribute__((ext_vector_type(4))) __bf16 bf4;
typedef __attribute__((ext_vector_type(4))) float f32x4;

DEV_INLINE void load_lds16(const char* g, char* l) {
  __builtin_amdgcn_global_load_lds(
      (const __attribute__((address_space(1))) uint32_t*)g,
      (__attribute__((address_space(3))) uint32_t*)l, 16, 0, 0);
}

struct Work {
  int expert, row, rows, col;  // rows == 0: nothing to do
};

// Sums over the lanes up to this one.
DEV_INLINE int lane_sums(int v) {
#pragma unroll
  for (int d = 1; d < 64; d *= 2) {
    const int a = __shfl_up(v, d);
    if ((int)(threadIdx.x & 63) >= d) v += a;
  }
  return v;
}

// What this workgroup does, from the experts' row counts (or offsets).
template <int BM>
DEV_INLINE Work find_tile(const int* bounds, bool offsets, int E, int R, int nt) {
  const int lane = threadIdx.x & 63;
  auto count = [&](int e) {
    return e >= E ? 0 : offsets ? bounds[e + 1] - bounds[e] : bounds[e];
  };
  int total = 0;  // row tiles
  for (int base = 0; base < E; base += 64) {
    total += __shfl(lane_sums((count(base + lane) + BM - 1) / BM), 63);
  }
  // workgroups go to the XCDs in turn: each XCD gets consecutive tiles
  const int all = total * nt, per = all / 8, rem = all % 8;
  const int xcd = blockIdx.x % 8, seq = blockIdx.x / 8;
  if (seq >= per + (xcd < rem)) return {0, 0, 0, 0};
  const int id = xcd * per + min(xcd, rem) + seq;
  int tiles0 = 0, rows0 = 0;
  for (int base = 0; base < E; base += 64) {
    const int c = count(base + lane), t = (c + BM - 1) / BM;
    const int tiles = lane_sums(t), rows = lane_sums(c);
    const uint64_t past = __ballot(id < (tiles0 + tiles) * nt);
    if (past) {
      const int f = __ffsll((unsigned long long)past) - 1;
      const int mine = __shfl(t, f), first = rows0 + __shfl(rows - c, f);
      const int end = min(rows0 + __shfl(rows, f), R);
      // within the expert: bands of up to 8 row tiles, down each column
      int at = id - (tiles0 + __shfl(tiles - t, f)) * nt;
      const int band = at / (8 * nt);
      at -= band * 8 * nt;
      const int high = min(8, mine - band * 8);
      const int row = first + (band * 8 + at % high) * BM;
      return {__builtin_amdgcn_readfirstlane(base + f),
              __builtin_amdgcn_readfirstlane(row),
              __builtin_amdgcn_readfirstlane(max(0, min(BM, end - row))),
              __builtin_amdgcn_readfirstlane(at / high)};
    }
    tiles0 += __shfl(tiles, 63);
    rows0 += __shfl(rows, 63);
  }
  return {0, 0, 0, 0};
}

template <bool FP8, int WM, bool SQUARE>
__global__ __launch_bounds__(kThreads, 2) void grouped_kernel(
    ushort* __restrict__ y, const char* __restrict__ x,
    const char* __restrict__ w, const float* __restrict__ sx,
    const float* __restrict__ sw, const float* __restrict__ row_weight,
    const int* __restrict__ bounds, const int* __restrict__ src, bool offsets,
    int E, int R, int N, int KB, int64_t ldx, int64_t ldw, int64_t ew) {
  // waves 2 x 4, each WM x 2 tiles of 32 x 32
  constexpr int WN = 2, BM = 2 * WM * 32, BN = 4 * WN * 32;
  constexpr int AC = BM / 64, BC = BN / 64;  // loads of 8 rows per wave and step
  constexpr int kStage = (BM + BN) * kStep;
  __shared__ __attribute__((aligned(16))) char lds[2 * kStage];

  const Work work = find_tile<BM>(bounds, offsets, E, R, (N + BN - 1) / BN);
  if (work.rows == 0) return;
  const int m0 = work.row, rows = work.rows, n0 = work.col * BN;
  w += work.expert * ew;

  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int lane = threadIdx.x & 63, l31 = lane & 31, hi = lane >> 5;
  const int wm = wave % 2, wn = wave / 2;
  const int unit = ((lane & 7) ^ (lane >> 3)) * 16;
  const char *ap[AC], *bp[BC];
#pragma unroll
  for (int i = 0; i < AC; i++) {
    const int m = m0 + min((wave * AC + i) * 8 + (lane >> 3), rows - 1);
    ap[i] = x + (int64_t)(src ? src[m] : m) * ldx + unit;
  }
#pragma unroll
  for (int i = 0; i < BC; i++) {
    bp[i] = w + (int64_t)min(n0 + (wave * BC + i) * 8 + (lane >> 3), N - 1) * ldw + unit;
  }
  auto load = [&](int stage, int kb) {
    char* to = lds + stage * kStage;
#pragma unroll
    for (int i = 0; i < AC; i++) load_lds16(ap[i] + kb, to + (wave * AC + i) * 1024);
#pragma unroll
    for (int i = 0; i < BC; i++) {
      load_lds16(bp[i] + kb, to + BM * kStep + (wave * BC + i) * 1024);
    }
  };

  f32x16 acc[WN][WM];
#pragma unroll
  for (int i = 0; i < WN; i++) {
#pragma unroll
    for (int j = 0; j < WM; j++) {
#pragma unroll
      for (int r = 0; r < 16; r++) acc[i][j][r] = 0.f;
    }
  }
  // Large tiles: the two waves of a SIMD take turns, one reads its operands
  // from LDS while the other multiplies; waves 4 to 7 are one barrier behind.
  constexpr bool kTurns = WM > 2;
  constexpr int kChunks = FP8 ? 2 : 4;
  auto barrier = [] {
    __builtin_amdgcn_sched_barrier(0);
    asm volatile("" ::: "memory");
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
    __builtin_amdgcn_sched_barrier(0);
  };
  const int steps = KB / kStep;
  load(0, 0);
  if constexpr (kTurns) {
    __builtin_amdgcn_s_waitcnt(0x0070);
    barrier();
    if (wave >= 4) barrier();
  }
  for (int s = 0; s < steps; s++) {
    const char* A = lds + (s & 1) * kStage + (wm * WM * 32 + l31) * kStep;
    const char* B = lds + (s & 1) * kStage + (BM + wn * WN * 32 + l31) * kStep;
    if constexpr (!kTurns) {
      // own loads have landed and own reads are done; behind the barrier that
      // holds for everyone, so the other stage can be written
      __builtin_amdgcn_sched_barrier(0);
      __builtin_amdgcn_s_waitcnt(0x0070);
      barrier();
      if (s + 1 < steps) load((s + 1) & 1, (s + 1) * kStep);
    }
#pragma unroll
    for (int c = 0; c < kChunks; c++) {
      typename std::conditional<FP8, i32x8, bf16x8>::type a[WM], b[WN];
      if constexpr (FP8) {
        const int u0 = ((4 * c + 2 * hi) ^ (l31 & 7)) << 4;
        const int u1 = ((4 * c + 2 * hi + 1) ^ (l31 & 7)) << 4;
        auto read = [&](const char* p) {
          const i32x4 lo = *(const i32x4*)(p + u0), up = *(const i32x4*)(p + u1);
          return __builtin_shufflevector(lo, up, 0, 1, 2, 3, 4, 5, 6, 7);
        };
#pragma unroll
        for (int j = 0; j < WM; j++) a[j] = read(A + j * 32 * kStep);
#pragma unroll
        for (int i = 0; i < WN; i++) b[i] = read(B + i * 32 * kStep);
      } else {
        const int u = ((2 * c + hi) ^ (l31 & 7)) << 4;
#pragma unroll
        for (int j = 0; j < WM; j++) a[j] = *(const bf16x8*)(A + j * 32 * kStep + u);
#pragma unroll
        for (int i = 0; i < WN; i++) b[i] = *(const bf16x8*)(B + i * 32 * kStep + u);
      }
      if constexpr (kTurns) {
        // Everyone's reads of the other stage ended before a barrier that lies
        // behind: it can be written. Its loads have landed, each wave's own,
        // before the barrier at the end of the last reads of this stage.
        if (c == 0 && s + 1 < steps) load((s + 1) & 1, (s + 1) * kStep);
        __builtin_amdgcn_sched_barrier(0);
        if (c == kChunks - 1) __builtin_amdgcn_s_waitcnt(0x0070);
        else __builtin_amdgcn_s_waitcnt(0xc07f);
        barrier();
        __builtin_amdgcn_s_setprio(1);
      }
#pragma unroll
      for (int i = 0; i < WN; i++) {
#pragma unroll
        for (int j = 0; j < WM; j++) {
          if constexpr (FP8) {  // block scales of 1
            acc[i][j] = __builtin_amdgcn_mfma_scale_f32_32x32x64_f8f6f4(
                b[i], a[j], acc[i][j], 0, 0, 0, 0x7f7f7f7f, 0, 0x7f7f7f7f);
          } else {
            acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(b[i], a[j], acc[i][j], 0, 0, 0);
          }
        }
      }
      if constexpr (kTurns) {
        __builtin_amdgcn_s_setprio(0);
        barrier();
      }
    }
  }
  if (kTurns && wave < 4) barrier();

  // a lane holds row l31 of x and, four at a time, columns 8 q + 4 hi
#pragma unroll
  for (int j = 0; j < WM; j++) {
    const int m = wm * WM * 32 + j * 32 + l31;
    if (m >= rows) continue;
    const float s = FP8 ? sx[src ? src[m0 + m] : m0 + m] : 1.f;
    const float rw = SQUARE ? row_weight[m0 + m] : 1.f;
    ushort* out = y + (int64_t)(m0 + m) * N;
#pragma unroll
    for (int i = 0; i < WN; i++) {
#pragma unroll
      for (int q = 0; q < 4; q++) {
        const int n = n0 + (wn * WN + i) * 32 + 8 * q + 4 * hi;
        if (n >= N) continue;
        f32x4 v;
#pragma unroll
        for (int t = 0; t < 4; t++) v[t] = acc[i][j][q * 4 + t];
        if constexpr (FP8) {
          const f32x4 c = *(const f32x4*)(sw + (int64_t)work.expert * N + n);
#pragma unroll
          for (int t = 0; t < 4; t++) v[t] = v[t] * s * c[t];
        }
        bf4 o = __builtin_convertvector(v, bf4);
        if constexpr (SQUARE) {
#pragma unroll
          for (int t = 0; t < 4; t++) {
            const float r = fmaxf((float)o[t], 0.f);
            v[t] = r * r * rw;
          }
          o = __builtin_convertvector(v, bf4);
        }
        *(bf4*)(out + n) = o;
      }
    }
  }
}

}  // namespace

// y [R, N] = rows of x [*, K] times w[e]^T, w [E, N, K] with any strides of e
// and n; bounds int32: E row counts or E + 1 offsets; src int32 [R] the rows
// of x, or none; fp8: sx fp32 [rows of x], sw fp32 [E, N]; square fp32 [R]:
// y = relu(product)^2 * square
void grouped_linear(torch::Tensor y, torch::Tensor x, torch::Tensor w,
                    c10::optional<torch::Tensor> sx,
                    c10::optional<torch::Tensor> sw, torch::Tensor bounds,
                    c10::optional<torch::Tensor> src,
                    c10::optional<torch::Tensor> square) {
  const bool fp8 = w.scalar_type() == torch::kFloat8_e4m3fn;
  TORCH_CHECK(fp8 || w.scalar_type() == torch::kBFloat16);
  TORCH_CHECK(x.scalar_type() == w.scalar_type() && x.is_cuda() && w.is_cuda());
  TORCH_CHECK(x.dim() == 2 && w.dim() == 3 && x.size(1) == w.size(2));
  TORCH_CHECK(x.stride(1) == 1 && w.stride(2) == 1);
  const int es = fp8 ? 1 : 2;
  const int64_t E = w.size(0), N = w.size(1), KB = w.size(2) * es;
  const int64_t ldx = x.stride(0) * es, ldw = w.stride(1) * es, ew = w.stride(0) * es;
  TORCH_CHECK(KB >= kStep && KB % kStep == 0 && KB < (int64_t)1 << 30);
  TORCH_CHECK(N >= 4 && N % 4 == 0 && N < (int64_t)1 << 30 && E >= 1 && E < 65536);
  TORCH_CHECK(ldx >= KB && ldx % 16 == 0 && ldw >= KB && ldw % 16 == 0 && ew >= 0 &&
                  ew % 16 == 0 && ((uintptr_t)x.data_ptr() & 15) == 0 &&
                  ((uintptr_t)w.data_ptr() & 15) == 0,
              "16-byte aligned rows");
  TORCH_CHECK(fp8 == (sx.has_value() && sw.has_value()));
  TORCH_CHECK(bounds.scalar_type() == torch::kInt32 && bounds.is_contiguous() &&
              bounds.is_cuda() && (bounds.numel() == E || bounds.numel() == E + 1));
  TORCH_CHECK(y.scalar_type() == torch::kBFloat16 && y.is_contiguous() &&
              y.is_cuda() && y.dim() == 2 && y.size(1) == N &&
              y.size(0) < (int64_t)1 << 30);
  const int64_t R = y.size(0);
  if (src.has_value()) {
    TORCH_CHECK(src->scalar_type() == torch::kInt32 && src->is_contiguous() &&
                src->is_cuda() && src->numel() == R);
  } else {
    TORCH_CHECK(x.size(0) == R);
  }
  if (fp8) {
    TORCH_CHECK(sx->scalar_type() == torch::kFloat32 && sx->is_contiguous() &&
                sx->is_cuda() && sx->numel() == x.size(0) &&
                sw->scalar_type() == torch::kFloat32 && sw->is_contiguous() &&
                sw->is_cuda() && sw->numel() == E * N &&
                ((uintptr_t)sw->data_ptr() & 15) == 0);
  }
  if (square.has_value()) {
    TORCH_CHECK(!fp8 && square->scalar_type() == torch::kFloat32 &&
                square->is_contiguous() && square->is_cuda() && square->numel() == R);
  }
  if (R == 0) return;
  const int64_t nt = (N + 255) / 256;
  // passes over the CUs of the likely number of tiles, times a pass's cost
  auto cost = [&](int64_t bm, int64_t c) {
    return c * (((R + std::min(E, R) * bm / 2) * nt + 256 * bm - 1) / (256 * bm));
  };
  const int64_t c2 = cost(128, 40), c3 = cost(192, fp8 ? 46 : 50),
                c4 = cost(256, fp8 ? 53 : 61);
  const int wm = R <= 96 * E || (c2 <= c3 && c2 <= c4) ? 2 : c3 < c4 ? 3 : 4;
  const int64_t row_tiles = R / (64 * wm) + std::min(E, R);
  TORCH_CHECK(row_tiles * nt < (int64_t)1 << 30);
  auto stream = c10::hip::getCurrentHIPStream().stream();
  auto go = [&](auto f, auto tile, auto sq) {
    hipLaunchKernelGGL(
        (grouped_kernel<decltype(f)::value, decltype(tile)::value, decltype(sq)::value>),
        dim3(row_tiles * nt), dim3(kThreads), 0, stream, (ushort*)y.data_ptr(),
        (const char*)x.data_ptr(), (const char*)w.data_ptr(),
        fp8 ? sx->data_ptr<float>() : nullptr, fp8 ? sw->data_ptr<float>() : nullptr,
        square.has_value() ? square->data_ptr<float>() : nullptr,
        bounds.data_ptr<int32_t>(), src.has_value() ? src->data_ptr<int32_t>() : nullptr,
        bounds.numel() == E + 1, (int)E, (int)R, (int)N, (int)KB, ldx, ldw, ew);
  };
  auto tiles = [&](auto f, auto sq) {
    if (wm == 4) go(f, std::integral_constant<int, 4>{}, sq);
    else if (wm == 3) go(f, std::integral_constant<int, 3>{}, sq);
    else go(f, std::integral_constant<int, 2>{}, sq);
  };
  if (fp8) tiles(std::true_type{}, std::false_type{});
  else if (square.has_value()) tiles(std::false_type{}, std::true_type{});
  else tiles(std::false_type{}, std::false_type{});
  HIP_CHECK_KERNEL();
}
