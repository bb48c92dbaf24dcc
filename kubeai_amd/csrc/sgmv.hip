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
//    instead of 22, too few waves in flight).
// Both are bound by latency: a few dependent loads (ids and table, entry, v, B)
// and a launch each. So the table is searched in registers, one load for all
// its ids, and x and y are asked for before anything is known about them.
// 4 adapters of rank 16, 28 decode rows and 304 prompt tokens (384 padded),
// us for shrink + expand: 4096 -> 4096 9 + 9.5, 4096 -> 28672 9 + 22, 14336 ->
// 4096 10 + 9 (expand 16, 22 and 16 with a search per thread, the vector ALUs
// and y read last); one launch per adapter took 4 x 59 each, and finding the adapters
// present four synchronisations.
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
  __shared__ float red[NW][kTok][kTok + 1];

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
  uint64_t todo = __ballot(slot >= 0) & 0xffffull;
  if (todo == 0) return;  // the same in every wave
  while (todo) {
    const int cur = __builtin_amdgcn_readlane(slot, __builtin_ctzll(todo));
    todo &= (todo - 1) & ~__ballot(slot == cur);  // shrinks in any case
    const ushort* A = tab[cur].A;
    const int R = tab[cur].rank;
    for (int r0 = 0; r0 < R; r0 += kTok) {
      const ushort* ar = A + (int64_t)min(r0 + m, R - 1) * H;
      f32x4 acc = {0.f, 0.f, 0.f, 0.f};
      bf16x8 af[STEPS];
#pragma unroll
      for (int i = 0; i < STEPS; ++i) {
        const int k = k0 + i * 32;
        af[i] = k < H ? *reinterpret_cast<const bf16x8*>(ar + k) : bf16x8{};
      }
#pragma unroll
      for (int i = 0; i < STEPS; ++i)
        acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(xf[i], af[i], acc, 0, 0, 0);
#pragma unroll
      for (int i = 0; i < 4; ++i) red[wave][kg * 4 + i][m] = acc[i];
      __syncthreads();
      {
        const int tok = threadIdx.x / kTok, r = threadIdx.x % kTok;
        float v = 0.f;
#pragma unroll
        for (int w = 0; w < NW; ++w) v += red[w][tok][r];
        // lane tok of any wave holds that token's slot
        const int own = __shfl(slot, tok, WAVE_SIZE);
        if (own == cur && r0 + r < R)
          part[((int64_t)split * T + t0 + tok) * r_pad + r0 + r] = v;
      }
      __syncthreads();
    }
  }
}

// VEC: rows of y are whole 16-byte units
template <bool VEC>
__global__ __launch_bounds__(kBlock) void lora_expand_kernel(
    ushort* __restrict__ y,          // [T, out] +=, rows strided
    const float* __restrict__ part,  // [splits, T, r_pad]
    const LoraEntry* __restrict__ tab, const int n,
    const int32_t* __restrict__ ids, const int64_t T, const int out,
    const int64_t y_stride, const int r_pad, const int splits) {
  constexpr int kTiles = kLaneOut / 4;
  const int64_t t0 = (int64_t)blockIdx.x * kTok;
  const int wave = threadIdx.x / WAVE_SIZE, lane = threadIdx.x % WAVE_SIZE;
  const int m = lane & 15, kg = lane >> 4;
  __shared__ __attribute__((aligned(16))) float v[kTok][kMaxR + 4];

  const int id = t0 + m < T ? ids[t0 + m] : 0;
  // this lane's outputs of token m
  const int wave_out = (blockIdx.y * (kBlock / WAVE_SIZE) + wave) * 4 * kLaneOut;
  const int o0 = wave_out + kg * kLaneOut;
  ushort* yr = y + min(t0 + m, T - 1) * y_stride + o0;
  ushort8 old[kLaneOut / 8];
  if constexpr (VEC) {
#pragma unroll
    for (int q = 0; q < kLaneOut / 8; ++q) {
      old[q] = ushort8{};
      if (id != 0 && o0 + 8 * q < out) old[q] = *reinterpret_cast<ushort8*>(yr + 8 * q);
    }
  }
  const int slot = lora_slot(tab, n, id);
  uint64_t todo = __ballot(slot >= 0) & 0xffffull;
  if (todo == 0) return;  // the same in every wave
  const int rank = slot >= 0 ? tab[slot].rank : 0;
  const float scale = slot >= 0 ? tab[slot].scale : 0.f;

  const int cols = r_pad <= 32 ? 32 : kMaxR;  // whole steps of K
  for (int i = threadIdx.x; i < kTok * cols; i += kBlock) {
    const int tok = i / cols, r = i % cols;
    const bool own = r < __shfl(rank, tok);
    const float* from = part + (t0 + tok) * r_pad + r;
    float s = 0.f;
#pragma unroll 4
    for (int k = 0; k < splits; ++k)
      s += own ? from[(int64_t)k * T * r_pad] : 0.f;
    v[tok][r] = s * __shfl(scale, tok);
  }
  __syncthreads();

  f32x4 acc[kTiles];
#pragma unroll
  for (int j = 0; j < kTiles; ++j) acc[j] = f32x4{0.f, 0.f, 0.f, 0.f};
  while (todo) {
    const int cur = __builtin_amdgcn_readlane(slot, __builtin_ctzll(todo));
    todo &= (todo - 1) & ~__ballot(slot == cur);  // shrinks in any case
    const ushort* B = tab[cur].B;
    const int R = tab[cur].rank;
    f32x4 sum[kTiles];  // of all tokens; kept for the adapter's own
#pragma unroll
    for (int j = 0; j < kTiles; ++j) sum[j] = f32x4{0.f, 0.f, 0.f, 0.f};
    for (int k0 = 0; k0 < R; k0 += 32) {
      const int k = k0 + kg * 8;
      bf16x8 b[kTiles];
#pragma unroll
      for (int j = 0; j < kTiles; ++j) {
        // row m of tile j: outputs 4 j .. 4 j + 3 of every lane's 16
        const int o = wave_out + (m >> 2) * kLaneOut + j * 4 + (m & 3);
        const ushort* br = B + (int64_t)min(o, out - 1) * R + k;
        b[j] = bf16x8{};
        if ((R & 7) == 0) {
          if (k < R) b[j] = *reinterpret_cast<const bf16x8*>(br);
        } else {
#pragma unroll
          for (int e = 0; e < 8; ++e)
            if (k + e < R) b[j][e] = (short)br[e];
        }
      }
      // v in three parts of 8 bits each, cut off: their sum is v. A part that
      // would be 0 is 2^-100 with v's sign (or v, if that is less): 0 times an
      // infinite B would be NaN. Nothing else is left of infinities and NaN.
      bf16x8 part3[3];
#pragma unroll
      for (int e = 0; e < 8; ++e) {
        float rest = v[m][k + e];
        const uint32_t sign = __float_as_uint(rest) & 0x80000000u;
        const float least = fminf(fabsf(rest), 0x1p-100f);
#pragma unroll
        for (int p = 0; p < 3; ++p) {
          const uint32_t top = __float_as_uint(rest) & 0xffff0000u;
          part3[p][e] = (short)(top >> 16);
          // (inf - inf is NaN, which the maximum passes over)
          const float left = fmaxf(fabsf(rest - __uint_as_float(top)), least);
          rest = __uint_as_float(__float_as_uint(left) | sign);
        }
      }
#pragma unroll
      for (int j = 0; j < kTiles; ++j)
#pragma unroll
        for (int p = 2; p >= 0; --p)
          sum[j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(b[j], part3[p], sum[j], 0, 0, 0);
    }
#pragma unroll
    for (int j = 0; j < kTiles; ++j)
#pragma unroll
      for (int e = 0; e < 4; ++e) acc[j][e] = slot == cur ? sum[j][e] : acc[j][e];
  }
  if (slot < 0) return;
#pragma unroll
  for (int q = 0; q < kLaneOut / 8; ++q) {
    if constexpr (VEC) {
      if (o0 + 8 * q >= out) continue;
      ushort8 to;
#pragma unroll
      for (int e = 0; e < 8; ++e)
        to[e] = f32_to_bf16(bf16_to_f32(old[q][e]) + acc[2 * q + e / 4][e % 4]);
      *reinterpret_cast<ushort8*>(yr + 8 * q) = to;
    } else {
#pragma unroll
      for (int e = 0; e < 8; ++e)
        if (o0 + 8 * q + e < out)
          yr[8 * q + e] =
              f32_to_bf16(bf16_to_f32(yr[8 * q + e]) + acc[2 * q + e / 4][e % 4]);
    }
  }
}

}  // namespace

// table: int64 [n, 4] rows of LoraEntry; ids: int32 [T]; max_rank: of the
// table's adapters. The caller keeps the tensors that the table points to.
void lora_apply(torch::Tensor y, torch::Tensor x, torch::Tensor table,
                torch::Tensor ids, int64_t max_rank) {
  TORCH_CHECK(x.scalar_type() == torch::kBFloat16 &&
              y.scalar_type() == torch::kBFloat16);
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
  const dim3 grid(tiles, (out + kOut - 1) / kOut);
  auto expand = [&](auto kernel) {
    hipLaunchKernelGGL(kernel, grid, dim3(kBlock), 0, stream,
                       (ushort*)y.data_ptr(), part.data_ptr<float>(), tab, n,
                       ids.data_ptr<int32_t>(), T, out, y.stride(0), r_pad,
                       splits);
  };
  if (out % 8 == 0 && y.stride(0) % 8 == 0 && ((uintptr_t)y.data_ptr() & 15) == 0)
    expand(lora_expand_kernel<true>);
  else
    expand(lora_expand_kernel<false>);
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
