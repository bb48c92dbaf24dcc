// Multi-LoRA batched apply.
//
//   y[t] += B_a (A_a x[t]) * scale_a        a = the adapter of token t
//
// Shapes: A [R, H] (shrink), B [out, R] (expand), LoRA rank R <= 64.
//
// lora_apply takes the whole batch: every token's adapter id and a table of
// the loaded adapters (pointers, rank, id, scale), all on the device. Two
// launches, no host knowledge of which adapters are present:
//  - lora_shrink: workgroup = 16 tokens x 1024 inputs. x is read once into
//    matrix-core operands (16x16x32); for each adapter among the 16 tokens
//    its A rows are multiplied against all of them and the rows of its own
//    tokens are kept, as fp32 partial sums per input range. 16 tokens share
//    each A byte; splitting the inputs gives 14336-wide inputs 14 workgroups
//    per 16 tokens.
//  - lora_expand: workgroup = 16 tokens x 256 outputs, on the matrix cores:
//    B rows are bf16 as they are, v (fp32) is cut into three bf16 parts that
//    add up to it exactly, and a token keeps its own adapter's result. A lane
//    holds 16 neighbouring outputs of one token (32: 27 us for 28672 outputs
//    instead of 22, too few waves in flight). Into bf16 rows; into the fp32 sums
//    that a product is handed on as, which its reader adds and rounds once; or,
//    for gate and up, with the activation behind it.
// All are bound by latency: a few dependent loads (ids and table, entry, v, B)
// and a launch each. So the table is searched in registers, one load for all
// its ids, x, y and the first adapter's B are asked for before v is there, the
// next adapter's weights while one is multiplied, and no load stands in a branch
// that waits for it (the shrink's loads of x and A are in one each, for inputs past the
// last, with no wait between them).
// 4 adapters of rank 16, 28 decode rows and 304 prompt tokens (384 padded), us:
// shrink 8.5; expand 4096 -> 4096 and 6144 8.0, 14336 -> 4096 into sums 9.9, 4096 ->
// 28672 with the activation 22.0. With v cut at every product, loads one behind
// the other and the activation in a launch of its own 9.2; 8.5, 12.8 and 30. One
// launch per adapter took 4 x 59 each, and finding the adapters present four
// synchronisations.
//
// sgmv applies one adapter to the rows that `idx` names (the form for
// adapters that the table does not take, see engine/lora.py). Design:
// workgroup per gathered token; phase 1 computes the R-vector
// v = A x (wave-split rows, lane-split H, butterfly reduce) into LDS;
// phase 2 streams B once per token with y[t, o] += dot(B[o, :], v)
// (v broadcast from LDS). A and B are small (<= ~350 KB combined) and
// stay L2-resident across the segment's workgroups.
#include <torch/extension.h>

#include "common.h"

namespace {

constexpr int kBlock = 256;
constexpr int kMaxR = 64;

__global__ void sgmv_kernel(
    ushort* __restrict__ y,        // [T, out] bf16 (+=)
    const ushort* __restrict__ x,  // [T, H] bf16
    const ushort* __restrict__ A,  // [R, H] bf16
    const ushort* __restrict__ B,  // [out, R] bf16
    const int64_t* __restrict__ idx,  // [n] gathered token rows
    const float scale, const int H, const int R, const int out,
    const int64_t x_stride, const int64_t y_stride) {
  const int64_t t = idx[blockIdx.x];
  const int wave = threadIdx.x / WAVE_SIZE;
  const int lane = threadIdx.x % WAVE_SIZE;
  const ushort8* xrow =
      reinterpret_cast<const ushort8*>(x + t * x_stride);

  __shared__ float v[kMaxR];

  // phase 1: v[r] = dot(A[r], x[t]) — waves split rows, lanes split H
  for (int r = wave; r < R; r += kBlock / WAVE_SIZE) {
    const ushort8* arow = reinterpret_cast<const ushort8*>(A + (int64_t)r * H);
    float acc = 0.f;
    for (int i = lane; i < H / 8; i += WAVE_SIZE) {
      const ushort8 xa = xrow[i];
      const ushort8 aa = arow[i];
#pragma unroll
      for (int j = 0; j < 8; ++j)
        acc = fmaf(bf16_to_f32(xa[j]), bf16_to_f32(aa[j]), acc);
    }
    acc = wave_reduce_sum(acc);
    if (lane == 0) v[r] = acc * scale;
  }
  __syncthreads();

  // phase 2: y[t, o] += dot(B[o, :R], v) — threads stride output features
  ushort* yrow = y + t * y_stride;
  for (int o = threadIdx.x; o < out; o += kBlock) {
    const ushort* brow = B + (int64_t)o * R;
    float acc = 0.f;
    for (int r = 0; r < R; ++r)
      acc = fmaf(bf16_to_f32(brow[r]), v[r], acc);
    yrow[o] = f32_to_bf16(bf16_to_f32(yrow[o]) + acc);
  }
}

// ---- the whole batch ---------------------------------------------------
constexpr int kTok = 16;      // tokens per workgroup
constexpr int kShrinkK = 1024;  // inputs per shrink workgroup
constexpr int kLaneOut = 16;    // outputs per expand lane

typedef __attribute__((ext_vector_type(8))) short bf16x8;
typedef __attribute__((ext_vector_type(4))) float f32x4;

// one row of the table: 4 x int64
struct LoraEntry {
  const ushort* A;   // [rank, H]
  const ushort* B;   // [out, rank]
  int32_t rank, id;
  float scale;
  int32_t pad;
};
static_assert(sizeof(LoraEntry) == 32, "the host builds rows of 4 int64");

// table row of the adapter id of every lane (-1: base model or not loaded);
// all lanes take part
DEV_INLINE int lora_slot(const LoraEntry* tab, int n, int id) {
  const int lane = threadIdx.x % WAVE_SIZE;
  int slot = -1;
  for (int base = 0; base < n; base += WAVE_SIZE) {
    const int here = base + lane < n ? tab[base + lane].id : 0;
    for (int i = 0; i < min(n - base, WAVE_SIZE); ++i)
      if (__builtin_amdgcn_readlane(here, i) == id && slot < 0) slot = base + i;
  }
  return id == 0 ? -1 : slot;
}

// Weights whose address was put together from lanes: said to be in device memory,
// or the loads are flat ones, which wait for the LDS too.
typedef const __attribute__((address_space(1))) ushort* Weights;
typedef const __attribute__((address_space(1))) bf16x8* Weights8;

// The adapters of a wave's tokens, one after the other. Every lane has its own
// token's at hand, so the next one's weights are asked for without a look at the
// table, and while the rows before are multiplied.
struct Walk {
  uint64_t todo;        // tokens whose adapters are still to come
  int slot, rank;       // the lane's own
  uint64_t weights;
  int cur, R;           // the adapter at hand
  Weights W;

  DEV_INLINE void next() {
    const int tok = __builtin_ctzll(todo);
    cur = __builtin_amdgcn_readlane(slot, tok);
    R = __builtin_amdgcn_readlane(rank, tok);
    W = (Weights)(
        (uint64_t)(uint32_t)__builtin_amdgcn_readlane((int)weights, tok) |
        (uint64_t)(uint32_t)__builtin_amdgcn_readlane((int)(weights >> 32), tok) << 32);
    todo &= (todo - 1) & ~__ballot(slot == cur);  // shrinks in any case
  }
};

__global__ __launch_bounds__(kBlock) void lora_shrink_kernel(
    float* __restrict__ part,        // [splits, T, r_pad]
    const ushort* __restrict__ x,    // [T, H], rows strided
    const LoraEntry* __restrict__ tab, const int n,
    const int32_t* __restrict__ ids, const int64_t T, const int H,
    const int64_t x_stride, const int r_pad) {
  constexpr int NW = kBlock / WAVE_SIZE;
  constexpr int STEPS = kShrinkK / NW / 32;
  const int64_t t0 = (int64_t)blockIdx.x * kTok;
  const int split = blockIdx.y;
  const int wave = threadIdx.x / WAVE_SIZE, lane = threadIdx.x % WAVE_SIZE;
  const int m = lane & 15, kg = lane >> 4;
  __shared__ float red[2][NW][kTok][kTok + 1];

  const int id = t0 + m < T ? ids[t0 + m] : 0;
  const int k0 = split * kShrinkK + wave * (kShrinkK / NW) + kg * 8;
  const ushort* xr = x + min(t0 + m, T - 1) * x_stride;
  bf16x8 xf[STEPS];
#pragma unroll
  for (int i = 0; i < STEPS; ++i) {
    const int k = k0 + i * 32;  // H is a multiple of 8
    xf[i] = k < H ? *reinterpret_cast<const bf16x8*>(xr + k) : bf16x8{};
  }
  const int slot = lora_slot(tab, n, id);
  const uint64_t todo = __ballot(slot >= 0) & 0xffffull;
  if (todo == 0) return;  // the same in every wave
  const LoraEntry* own_entry = tab + max(slot, 0);
  Walk walk{todo, slot, own_entry->rank, (uint64_t)own_entry->A};
  int r0 = 0;
  bf16x8 af[STEPS];
  const auto load = [&] {
    const Weights ar = walk.W + (int64_t)min(r0 + m, walk.R - 1) * H;
#pragma unroll
    for (int i = 0; i < STEPS; ++i) {
      const int k = k0 + i * 32;
      af[i] = k < H ? *(Weights8)(ar + k) : bf16x8{};
    }
  };
  walk.next();
  load();
  for (int turn = 0;; turn ^= 1) {
    f32x4 acc = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int i = 0; i < STEPS; ++i)
      acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(xf[i], af[i], acc, 0, 0, 0);
    const int done = walk.cur, done_r0 = r0, done_R = walk.R;
    r0 += kTok;
    const bool more = r0 < walk.R || walk.todo != 0;
    if (more) {
      if (r0 >= walk.R) {
        walk.next();
        r0 = 0;
      }
      load();
    }
    // (two places, so the threads that read one are past it when it is written again)
#pragma unroll
    for (int i = 0; i < 4; ++i) red[turn][wave][kg * 4 + i][m] = acc[i];
    __syncthreads();
    const int tok = threadIdx.x / kTok, r = threadIdx.x % kTok;
    float v = 0.f;
#pragma unroll
    for (int w = 0; w < NW; ++w) v += red[turn][w][tok][r];
    // lane tok of any wave holds that token's slot
    const int own = __shfl(slot, tok, WAVE_SIZE);
    if (own == done && done_r0 + r < done_R)
      part[((int64_t)split * T + t0 + tok) * r_pad + done_r0 + r] = v;
    if (!more) break;
  }
}

// v of a workgroup's tokens: the partial sums added and scaled, 0 above a rank, in
// three bf16 parts of 8 bits each, cut off: their sum is v. A part that would be 0
// is 2^-100 with v's sign (or v, if that is less): 0 times an infinite B would be
// NaN. Nothing else is left of infinities and NaN. Cut once for all adapters and
// outputs of the workgroup (cut again at every product: gated 27 us instead of 22).
struct Ranks {
  // rows of whole 16-byte units, on other banks than the rows beside them
  short part[3][kTok][kMaxR + 8];
};

DEV_INLINE void lora_ranks(Ranks& v, const float* part, int rank, float scale,
                           int64_t t0, int64_t T, int r_pad, int splits) {
  const int cols = r_pad <= 32 ? 32 : kMaxR;  // whole steps of K
  for (int i = threadIdx.x; i < kTok * cols; i += kBlock) {
    const int tok = i / cols, r = i % cols;
    const bool own = r < __shfl(rank, tok);
    // loaded in any case, from a place that is there: no branch, no wait for each
    const float* from = part + min(t0 + tok, T - 1) * r_pad + min(r, r_pad - 1);
    float s = 0.f;
    for (int k0 = 0; k0 < splits; k0 += 8) {
      float some[8];
#pragma unroll
      for (int k = 0; k < 8; ++k)
        some[k] = from[(int64_t)min(k0 + k, splits - 1) * T * r_pad];
#pragma unroll
      for (int k = 0; k < 8; ++k) s += own && k0 + k < splits ? some[k] : 0.f;
    }
    float rest = s * __shfl(scale, tok);
    const uint32_t sign = __float_as_uint(rest) & 0x80000000u;
    const float least = fminf(fabsf(rest), 0x1p-100f);
#pragma unroll
    for (int p = 0; p < 3; ++p) {
      const uint32_t top = __float_as_uint(rest) & 0xffff0000u;
      v.part[p][tok][r] = (short)(top >> 16);
      // (inf - inf is NaN, which the maximum passes over)
      const float left = fmaxf(fabsf(rest - __uint_as_float(top)), least);
      rest = __uint_as_float(__float_as_uint(left) | sign);
    }
  }
  __syncthreads();
}

// The rows of B that make 16 outputs of every lane's token, from output wave_out +
// 16 kg on, at ranks k0 to k0 + 31. Ranks of 8, 16, .. are asked for without a
// branch, so that all of them are on their way at once; what is above the rank
// holds something else then, which masked() takes out when it is used. Other ranks
// come a value at a time, and only below the rank: what lanes sit out costs the
// address unit nothing (rank 4 of 20 adapters, 5504 -> 27776, 61 rows: shrink and
// expand 42 us, 111 with every lane's values asked for).
DEV_INLINE void lora_rows(bf16x8 (&b)[kLaneOut / 4], Weights B, int R, int k0,
                          int wave_out, int out) {
  const int lane = threadIdx.x % WAVE_SIZE;
  const int m = lane & 15, k = k0 + (lane >> 4) * 8;
  // row m of tile j: outputs 4 j .. 4 j + 3 of every lane's 16
  const int o0 = wave_out + (m >> 2) * kLaneOut + (m & 3);
  if ((R & 7) == 0) {
#pragma unroll
    for (int j = 0; j < kLaneOut / 4; ++j)
      b[j] = *(Weights8)(B + (int64_t)min(o0 + j * 4, out - 1) * R + min(k, R - 8));
  } else {
#pragma unroll
    for (int j = 0; j < kLaneOut / 4; ++j) {
      const Weights row = B + (int64_t)min(o0 + j * 4, out - 1) * R + k;
      b[j] = bf16x8{};
#pragma unroll
      for (int e = 0; e < 8; ++e)
        if (k + e < R) b[j][e] = (short)row[e];
    }
  }
}

DEV_INLINE bf16x8 masked(bf16x8 b, bool keep) { return keep ? b : bf16x8{}; }

// acc: what the adapters add to 16 outputs of every lane's token, from wave_out +
// 16 kg on. b holds the first adapter's rows at ranks 0 to 31.
DEV_INLINE void lora_outputs(f32x4 (&acc)[kLaneOut / 4], const Ranks& v, Walk walk,
                             bf16x8 (&b)[kLaneOut / 4], int wave_out, int out) {
  constexpr int kTiles = kLaneOut / 4;
  const int lane = threadIdx.x % WAVE_SIZE;
  const int m = lane & 15, kg = lane >> 4;
  f32x4 sum[kTiles];  // of all tokens; kept for the adapter's own
#pragma unroll
  for (int j = 0; j < kTiles; ++j) sum[j] = acc[j] = f32x4{0.f, 0.f, 0.f, 0.f};
  for (int k0 = 0;;) {
    bf16x8 part3[3];
#pragma unroll
    for (int p = 0; p < 3; ++p)
      part3[p] = *reinterpret_cast<const bf16x8*>(&v.part[p][m][k0 + kg * 8]);
    const bool keep = k0 + kg * 8 < walk.R;
#pragma unroll
    for (int j = 0; j < kTiles; ++j) {
      const bf16x8 rows = masked(b[j], keep);
#pragma unroll
      for (int p = 2; p >= 0; --p)
        sum[j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(rows, part3[p], sum[j], 0, 0, 0);
    }
    const int cur = walk.cur;
    k0 += 32;
    const bool last = k0 >= walk.R;  // of this adapter
    const bool more = !last || walk.todo != 0;
    if (more) {
      if (last) {
        walk.next();
        k0 = 0;
      }
      lora_rows(b, walk.W, walk.R, k0, wave_out, out);
    }
    if (last) {
#pragma unroll
      for (int j = 0; j < kTiles; ++j)
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          acc[j][e] = walk.slot == cur ? sum[j][e] : acc[j][e];
          sum[j][e] = 0.f;
        }
    }
    if (!more) break;
  }
}

// VEC: rows of y are whole 16-byte units. Y: bf16, or fp32 where y is the first
// part of a product's sums (384 rows x 4096 x 14336 in bf16: the library's product 77
// us, 52 as sums and 3 more in the norm that adds them).
template <bool VEC, typename Y>
__global__ __launch_bounds__(kBlock) void lora_expand_kernel(
    Y* __restrict__ y,               // [T, out] +=, rows strided
    const float* __restrict__ part,  // [splits, T, r_pad]
    const LoraEntry* __restrict__ tab, const int n,
    const int32_t* __restrict__ ids, const int64_t T, const int out,
    const int64_t y_stride, const int r_pad, const int splits) {
  const int64_t t0 = (int64_t)blockIdx.x * kTok;
  const int wave = threadIdx.x / WAVE_SIZE, lane = threadIdx.x % WAVE_SIZE;
  const int m = lane & 15, kg = lane >> 4;
  __shared__ __attribute__((aligned(16))) Ranks v;

  const int id = t0 + m < T ? ids[t0 + m] : 0;
  // this lane's outputs of token m
  const int wave_out = (blockIdx.y * (kBlock / WAVE_SIZE) + wave) * 4 * kLaneOut;
  const int o0 = wave_out + kg * kLaneOut;
  constexpr int VN = 16 / sizeof(Y);
  typedef __attribute__((ext_vector_type(VN))) Y Unit;
  Y* yr = y + min(t0 + m, T - 1) * y_stride + o0;
  Unit old[kLaneOut / VN];
  if constexpr (VEC) {
#pragma unroll
    for (int q = 0; q < kLaneOut / VN; ++q) {
      old[q] = Unit{};
      if (id != 0 && o0 + VN * q < out) old[q] = *reinterpret_cast<Unit*>(yr + VN * q);
    }
  }
  const int slot = lora_slot(tab, n, id);
  const uint64_t todo = __ballot(slot >= 0) & 0xffffull;
  if (todo == 0) return;  // the same in every wave
  const LoraEntry* own = tab + max(slot, 0);
  const float scale = slot >= 0 ? own->scale : 0.f;
  Walk walk{todo, slot, slot >= 0 ? own->rank : 0, (uint64_t)own->B};
  walk.next();
  bf16x8 b[kLaneOut / 4];
  lora_rows(b, walk.W, walk.R, 0, wave_out, out);
  lora_ranks(v, part, walk.rank, scale, t0, T, r_pad, splits);
  f32x4 acc[kLaneOut / 4];
  lora_outputs(acc, v, walk, b, wave_out, out);
  if (slot < 0) return;
  const auto added = [&](Y was, int j) -> Y {
    const float a = acc[j / 4][j % 4];
    if constexpr (sizeof(Y) == 4) return was + a;
    else return f32_to_bf16(bf16_to_f32(was) + a);
  };
#pragma unroll
  for (int q = 0; q < kLaneOut / VN; ++q) {
    if constexpr (VEC) {
      if (o0 + VN * q >= out) continue;
      Unit to;
#pragma unroll
      for (int e = 0; e < VN; ++e) to[e] = added(old[q][e], VN * q + e);
      *reinterpret_cast<Unit*>(yr + VN * q) = to;
    } else {
#pragma unroll
      for (int e = 0; e < VN; ++e)
        if (o0 + VN * q + e < out) yr[VN * q + e] = added(yr[VN * q + e], VN * q + e);
    }
  }
}

// z = silu(gate) * up of y's rows (gate columns, then up columns) and the adapters'
// products: y is read once and not written. I % 8 == 0, rows of 16-byte units. (Both
// sets of outputs in one pass over the adapters take 131 registers: 22.7 us; held
// to 128 33.)
__global__ __launch_bounds__(kBlock) void lora_expand_gated_kernel(
    ushort* __restrict__ z,          // [T, I] dense
    const ushort* __restrict__ y,    // [T, 2 I], rows strided
    const float* __restrict__ part,  // [splits, T, r_pad]
    const LoraEntry* __restrict__ tab, const int n,
    const int32_t* __restrict__ ids, const int64_t T, const int I,
    const int64_t y_stride, const int r_pad, const int splits) {
  const int64_t t0 = (int64_t)blockIdx.x * kTok;
  const int wave = threadIdx.x / WAVE_SIZE, lane = threadIdx.x % WAVE_SIZE;
  const int m = lane & 15, kg = lane >> 4;
  __shared__ __attribute__((aligned(16))) Ranks v;

  const int id = t0 + m < T ? ids[t0 + m] : 0;
  const int wave_out = (blockIdx.y * (kBlock / WAVE_SIZE) + wave) * 4 * kLaneOut;
  const int o0 = wave_out + kg * kLaneOut;
  const ushort* yr = y + min(t0 + m, T - 1) * y_stride + o0;
  ushort8 gate[kLaneOut / 8], up[kLaneOut / 8];
#pragma unroll
  for (int q = 0; q < kLaneOut / 8; ++q) {
    gate[q] = up[q] = ushort8{};
    if (o0 + 8 * q < I) {
      gate[q] = *reinterpret_cast<const ushort8*>(yr + 8 * q);
      up[q] = *reinterpret_cast<const ushort8*>(yr + I + 8 * q);
    }
  }
  const int slot = lora_slot(tab, n, id);
  const uint64_t todo = __ballot(slot >= 0) & 0xffffull;
  f32x4 add[2][kLaneOut / 4];
#pragma unroll
  for (int j = 0; j < kLaneOut / 4; ++j) add[0][j] = add[1][j] = f32x4{0.f, 0.f, 0.f, 0.f};
  if (todo) {  // the same in every wave
    const LoraEntry* own = tab + max(slot, 0);
    const float scale = slot >= 0 ? own->scale : 0.f;
    Walk walk{todo, slot, slot >= 0 ? own->rank : 0, (uint64_t)own->B};
    walk.next();
    bf16x8 gate_rows[kLaneOut / 4], up_rows[kLaneOut / 4];
    lora_rows(gate_rows, walk.W, walk.R, 0, wave_out, 2 * I);
    lora_rows(up_rows, walk.W, walk.R, 0, I + wave_out, 2 * I);
    lora_ranks(v, part, walk.rank, scale, t0, T, r_pad, splits);
    lora_outputs(add[0], v, walk, gate_rows, wave_out, 2 * I);
    lora_outputs(add[1], v, walk, up_rows, I + wave_out, 2 * I);
  }
  if (t0 + m >= T) return;
  ushort* zr = z + (t0 + m) * I + o0;
#pragma unroll
  for (int q = 0; q < kLaneOut / 8; ++q) {
    if (o0 + 8 * q >= I) continue;
    ushort8 to;
#pragma unroll
    for (int e = 0; e < 8; ++e) {
      const float g = bf16_to_f32(gate[q][e]) + add[0][2 * q + e / 4][e % 4];
      const float u = bf16_to_f32(up[q][e]) + add[1][2 * q + e / 4][e % 4];
      to[e] = f32_to_bf16(g / (1.f + __expf(-g)) * u);
    }
    *reinterpret_cast<ushort8*>(zr + 8 * q) = to;
  }
}

}  // namespace

// y: bf16 rows, or fp32 ones (the first part of a product's sums);
// table: int64 [n, 4] rows of LoraEntry; ids: int32 [T]; max_rank: of the
// table's adapters. The caller keeps the tensors that the table points to.
// z: if given, y is left and z takes silu(gate) * up of the result
void lora_apply(torch::Tensor y, torch::Tensor x, torch::Tensor table,
                torch::Tensor ids, int64_t max_rank,
                std::optional<torch::Tensor> z) {
  const bool sums = y.scalar_type() == torch::kFloat32;
  TORCH_CHECK(x.scalar_type() == torch::kBFloat16 &&
              (sums || y.scalar_type() == torch::kBFloat16));
  TORCH_CHECK(x.dim() == 2 && y.dim() == 2 && x.size(0) == y.size(0));
  TORCH_CHECK(x.stride(1) == 1 && y.stride(1) == 1);
  TORCH_CHECK(ids.scalar_type() == torch::kInt32 && ids.is_contiguous() &&
              ids.numel() == x.size(0));
  TORCH_CHECK(table.scalar_type() == torch::kInt64 && table.is_contiguous() &&
              table.dim() == 2 && table.size(1) == 4);
  TORCH_CHECK(table.is_cuda() && ids.is_cuda() && x.is_cuda() && y.is_cuda());
  // its rows are read 16 bytes at a time
  if ((x.stride(0) % 8 != 0 && x.size(0) > 1) || ((uintptr_t)x.data_ptr() & 15) != 0)
    x = x.clone(at::MemoryFormat::Contiguous);
  TORCH_CHECK(max_rank >= 1 && max_rank <= kMaxR);
  const int64_t T = x.size(0);
  const int H = x.size(1), out = y.size(1), n = table.size(0);
  TORCH_CHECK(H % 8 == 0);
  if (z) {
    TORCH_CHECK(!sums && z->is_cuda() && z->scalar_type() == torch::kBFloat16 &&
                z->is_contiguous() && z->dim() == 2 && z->size(0) == T &&
                out == 2 * z->size(1) && out % 16 == 0 && n > 0);
    TORCH_CHECK((y.stride(0) % 8 == 0 || T <= 1) && ((uintptr_t)y.data_ptr() & 15) == 0 &&
                ((uintptr_t)z->data_ptr() & 15) == 0);
  }
  if (T == 0 || n == 0) return;
  const int r_pad = ((int)max_rank + 7) / 8 * 8;
  const int splits = (H + kShrinkK - 1) / kShrinkK;
  auto part = torch::empty({splits, T, r_pad}, x.options().dtype(torch::kFloat32));
  auto stream = c10::hip::getCurrentHIPStream().stream();
  const auto* tab = (const LoraEntry*)table.data_ptr();
  const uint32_t tiles = (uint32_t)((T + kTok - 1) / kTok);
  hipLaunchKernelGGL(lora_shrink_kernel, dim3(tiles, splits), dim3(kBlock), 0,
                     stream, part.data_ptr<float>(),
                     (const ushort*)x.data_ptr(), tab, n,
                     ids.data_ptr<int32_t>(), T, H, x.stride(0), r_pad);
  HIP_CHECK_KERNEL();
  constexpr int kOut = kBlock / 16 * kLaneOut;  // outputs per workgroup
  if (z) {
    const int I = out / 2;
    hipLaunchKernelGGL(lora_expand_gated_kernel, dim3(tiles, (I + kOut - 1) / kOut),
                       dim3(kBlock), 0, stream, (ushort*)z->data_ptr(),
                       (const ushort*)y.data_ptr(), part.data_ptr<float>(), tab, n,
                       ids.data_ptr<int32_t>(), T, I, y.stride(0), r_pad, splits);
    HIP_CHECK_KERNEL();
    return;
  }
  const dim3 grid(tiles, (out + kOut - 1) / kOut);
  auto expand = [&](auto kernel, auto* to) {
    hipLaunchKernelGGL(kernel, grid, dim3(kBlock), 0, stream,
                       to, part.data_ptr<float>(), tab, n,
                       ids.data_ptr<int32_t>(), T, out, y.stride(0), r_pad,
                       splits);
  };
  const int unit = sums ? 4 : 8;
  const bool vec = out % unit == 0 && y.stride(0) % unit == 0 &&
                   ((uintptr_t)y.data_ptr() & 15) == 0;
  if (sums) {
    auto* to = y.data_ptr<float>();
    vec ? expand(lora_expand_kernel<true, float>, to)
        : expand(lora_expand_kernel<false, float>, to);
  } else {
    auto* to = (ushort*)y.data_ptr();
    vec ? expand(lora_expand_kernel<true, ushort>, to)
        : expand(lora_expand_kernel<false, ushort>, to);
  }
  HIP_CHECK_KERNEL();
}

void sgmv(torch::Tensor y, torch::Tensor x, torch::Tensor A, torch::Tensor B,
          torch::Tensor idx, double scale) {
  TORCH_CHECK(x.scalar_type() == torch::kBFloat16);
  TORCH_CHECK(A.is_contiguous() && B.is_contiguous());
  TORCH_CHECK(idx.scalar_type() == torch::kInt64);
  const int H = x.size(1), R = A.size(0), out = B.size(0);
  TORCH_CHECK(A.size(1) == H && B.size(1) == R && R <= kMaxR);
  TORCH_CHECK(H % 8 == 0);
  TORCH_CHECK(x.stride(1) == 1 && y.stride(1) == 1);
  const int n = idx.size(0);
  if (n == 0) return;
  hipLaunchKernelGGL(sgmv_kernel, dim3(n), dim3(kBlock), 0,
                     c10::hip::getCurrentHIPStream().stream(),
                     (ushort*)y.data_ptr(), (const ushort*)x.data_ptr(),
                     (const ushort*)A.data_ptr(), (const ushort*)B.data_ptr(),
                     idx.data_ptr<int64_t>(), (float)scale, H, R, out,
                     x.stride(0), y.stride(0));
  HIP_CHECK_KERNEL();
}
