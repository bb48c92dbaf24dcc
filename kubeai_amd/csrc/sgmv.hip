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
//  - lora_expand: workgroup = 16 tokens x 512 outputs (2 a thread). B rows
//    are held in registers and used for the adapter's tokens; the products
//    stay fp32 x fp32 on the vector ALUs (v is not rounded; 2 R flops per
//    element of y, which is read and written once, is below the memory time).
// It is bound by reading and writing y, and at decode sizes by the launches.
// 4 adapters of rank 16, 28 decode rows and 304 prompt tokens (384 padded),
// us for shrink + expand: 4096 -> 4096 9 + 16, 4096 -> 28672 9 + 22, 14336 ->
// 4096 11 + 16; one launch per adapter took 4 x 59 each, and finding the
// adapters present four synchronisations.
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

// table row of every token's adapter (-1: base model or not loaded)
DEV_INLINE int lora_slot(const LoraEntry* tab, int n, const int32_t* ids,
                         int64_t t, int64_t T) {
  if (t >= T) return -1;
  const int id = ids[t];
  if (id == 0) return -1;
  for (int i = 0; i < n; ++i)
    if (tab[i].id == id) return i;
  return -1;
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

  const int slot = lora_slot(tab, n, ids, t0 + m, T);
  uint64_t todo = __ballot(slot >= 0) & 0xffffull;
  if (todo == 0) return;  // the same in every wave

  const int k0 = split * kShrinkK + wave * (kShrinkK / NW) + kg * 8;
  const ushort* xr = x + min(t0 + m, T - 1) * x_stride;
  bf16x8 xf[STEPS];
#pragma unroll
  for (int i = 0; i < STEPS; ++i) {
    const int k = k0 + i * 32;  // H is a multiple of 8
    xf[i] = k < H ? *reinterpret_cast<const bf16x8*>(xr + k) : bf16x8{};
  }
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

// COLS: outputs per thread (2 where rows of y are 4-byte aligned)
template <int COLS>
__global__ __launch_bounds__(kBlock) void lora_expand_kernel(
    ushort* __restrict__ y,          // [T, out] +=, rows strided
    const float* __restrict__ part,  // [splits, T, r_pad]
    const LoraEntry* __restrict__ tab, const int n,
    const int32_t* __restrict__ ids, const int64_t T, const int out,
    const int64_t y_stride, const int r_pad, const int splits) {
  const int64_t t0 = (int64_t)blockIdx.x * kTok;
  const int lane = threadIdx.x % WAVE_SIZE;
  __shared__ float v[kTok][kMaxR];

  const int slot = lora_slot(tab, n, ids, t0 + (lane & 15), T);
  uint64_t todo = __ballot(slot >= 0) & 0xffffull;
  const uint32_t active = (uint32_t)todo;
  if (todo == 0) return;

  for (int i = threadIdx.x; i < kTok * r_pad; i += kBlock) {
    const int tok = i / r_pad, r = i % r_pad;
    const int own = lora_slot(tab, n, ids, t0 + tok, T);
    float s = 0.f;
    if (own >= 0 && r < tab[own].rank) {
      for (int k = 0; k < splits; ++k)
        s += part[((int64_t)k * T + t0 + tok) * r_pad + r];
      s *= tab[own].scale;
    }
    v[tok][r] = s;
  }
  __syncthreads();

  // lanes past the last output stay: the ballots below need every token's lane
  const int o_own = (blockIdx.y * kBlock + threadIdx.x) * COLS;
  const bool live = o_own < out;
  const int o = live ? o_own : 0;
  float acc[kTok][COLS];
#pragma unroll
  for (int i = 0; i < kTok; ++i)
#pragma unroll
    for (int c = 0; c < COLS; ++c) acc[i][c] = 0.f;
  while (todo) {
    const int cur = __builtin_amdgcn_readlane(slot, __builtin_ctzll(todo));
    const uint32_t mine = (uint32_t)(__ballot(slot == cur) & todo);
    todo &= (todo - 1) & ~(uint64_t)mine;  // shrinks in any case
    const ushort* B = tab[cur].B;
    const int R = tab[cur].rank;
    for (int r0 = 0; r0 < R; r0 += 8) {
      float b[COLS][8];
#pragma unroll
      for (int c = 0; c < COLS; ++c) {
        const ushort* br = B + (int64_t)(o + c) * R + r0;
        if ((R & 7) == 0) {
          const ushort8 bv = *reinterpret_cast<const ushort8*>(br);
#pragma unroll
          for (int j = 0; j < 8; ++j) b[c][j] = bf16_to_f32(bv[j]);
        } else {
#pragma unroll
          for (int j = 0; j < 8; ++j)
            b[c][j] = r0 + j < R ? bf16_to_f32(br[j]) : 0.f;
        }
      }
#pragma unroll
      for (int i = 0; i < kTok; ++i) {
        if (!(mine >> i & 1)) continue;  // the same in every lane
#pragma unroll
        for (int j = 0; j < 8; ++j) {
          const float vj = v[i][r0 + j];
#pragma unroll
          for (int c = 0; c < COLS; ++c) acc[i][c] = fmaf(b[c][j], vj, acc[i][c]);
        }
      }
    }
  }
#pragma unroll
  for (int i = 0; i < kTok; ++i) {
    if (!live || !(active >> i & 1)) continue;
    ushort* yp = y + (t0 + i) * y_stride + o;
    if constexpr (COLS == 2) {
      const uint32_t old = *reinterpret_cast<uint32_t*>(yp);
      const uint32_t lo = f32_to_bf16(bf16_to_f32((ushort)old) + acc[i][0]);
      const uint32_t hi = f32_to_bf16(bf16_to_f32((ushort)(old >> 16)) + acc[i][1]);
      *reinterpret_cast<uint32_t*>(yp) = lo | (hi << 16);
    } else {
      *yp = f32_to_bf16(bf16_to_f32(*yp) + acc[i][0]);
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
  TORCH_CHECK(table.is_cuda() && ids.is_cuda());
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
  const bool pair = out % 2 == 0 && y.stride(0) % 2 == 0 &&
                    ((uintptr_t)y.data_ptr() & 3) == 0;
  const int cols = pair ? 2 : 1;
  const dim3 grid(tiles, (out + kBlock * cols - 1) / (kBlock * cols));
  if (pair)
    hipLaunchKernelGGL((lora_expand_kernel<2>), grid, dim3(kBlock), 0, stream,
                       (ushort*)y.data_ptr(), part.data_ptr<float>(), tab, n,
                       ids.data_ptr<int32_t>(), T, out, y.stride(0), r_pad,
                       splits);
  else
    hipLaunchKernelGGL((lora_expand_kernel<1>), grid, dim3(kBlock), 0, stream,
                       (ushort*)y.data_ptr(), part.data_ptr<float>(), tab, n,
                       ids.data_ptr<int32_t>(), T, out, y.stride(0), r_pad,
                       splits);
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
