// Row kernels of the decoder layers for gfx950: RMSNorm (with the residual
// add) in bf16 or straight to fp8 (OCP e4m3) with a scale per row, SwiGLU to
// fp8, and plain fp8 row quantization.
//
// Semantics: kubeai_amd/ops/ref.py (fp32 inside, bf16 in). fp8: per row,
// scale = max|v| / 448, out = v / scale rounded to nearest even — what
// torch._scaled_mm's rowwise scale_a expects.
//
// One workgroup per row, bound by reading and writing the rows. A row stays
// in registers between the passes over it (sum of squares, maximum, output):
// the values per thread are a template parameter, since a register array
// that is indexed by a runtime trip count lives in scratch memory. With many
// rows 256 threads each hold more of a row; with few rows as many threads as
// the row has 16-byte units (up to 1024) shorten the chain of loads.
// Measured, us (runtime trip count, 256 threads -> this):
//   8192 rows: residual add + norm to fp8, 4096 wide     116 ->  39 (5.9 TB/s)
//              SwiGLU to fp8, 14336 wide                 229 -> 124 (4.7 TB/s)
//              quantization, 4096 wide                    61 ->  18
//   2048 rows: residual add + norm, 4096 wide              25 ->  11
//   40 rows:   SwiGLU to fp8                               11 ->   5
//              residual add + norm to fp8                   6 ->   5
// With few rows what is left is the launch.
#include <torch/extension.h>

#include <type_traits>

#include "common.h"

namespace {

constexpr int kCUs = 256;
constexpr int kMaxH = 16384;     // bf16 norms
constexpr int kMaxHFp8 = 32768;  // fp8 outputs

typedef __attribute__((ext_vector_type(2))) uint32_t u32x2;

DEV_INLINE float block_max(float v, float* smem) {
  const int wave = threadIdx.x / WAVE_SIZE, lane = threadIdx.x % WAVE_SIZE;
  const int n_waves = blockDim.x / WAVE_SIZE;
  v = wave_reduce_max(v);
  if (lane == 0) smem[wave] = v;
  __syncthreads();
  float m = 0.f;
#pragma unroll
  for (int w = 0; w < 16; ++w)
    if (w < n_waves) m = fmaxf(m, smem[w]);
  return m;
}

// 8 values -> 8 bytes of e4m3, round to nearest even; |v| <= 448 up to
// rounding, so nothing overflows
DEV_INLINE u32x2 to_fp8x8(const float* v, float inv_scale) {
  u32x2 o;
#pragma unroll
  for (int h = 0; h < 2; ++h) {
    int w = __builtin_amdgcn_cvt_pk_fp8_f32(v[4 * h] * inv_scale,
                                            v[4 * h + 1] * inv_scale, 0, false);
    w = __builtin_amdgcn_cvt_pk_fp8_f32(v[4 * h + 2] * inv_scale,
                                        v[4 * h + 3] * inv_scale, w, true);
    o[h] = (uint32_t)w;
  }
  return o;
}

// scale a row held in registers (VPT units of 8 per thread) to fp8
template <int VPT>
DEV_INLINE void write_fp8_row(unsigned char* out, float* out_scale, int64_t row,
                              const float (&vals)[VPT][8], float amax, int H,
                              float* smem) {
  const float gmax = fmaxf(block_max(amax, smem), 1e-6f);
  if (threadIdx.x == 0) out_scale[row] = gmax / 448.0f;
  const float inv_scale = 448.0f / gmax;
#pragma unroll
  for (int k = 0; k < VPT; ++k) {
    const int i = threadIdx.x + k * blockDim.x;
    if (i < H / 8)
      *reinterpret_cast<u32x2*>(out + row * H + i * 8) =
          to_fp8x8(vals[k], inv_scale);
  }
}

// one unit of a product's sums
DEV_INLINE ushort8 sums_unit(const ProductSums& p, int64_t row, int n,
                             const SumScales<1>& by) {
  ushort8 o[1];
  read_sums8<1>(p, row, {n}, by, o);
  return o[0];
}

// ADD: residual += x, norm of the sum. FP8: fp8 output with a row scale. SUMS:
// x is a product's parts (added here instead of in a launch of their own).
template <bool ADD, bool FP8, bool SUMS, int VPT>
__launch_bounds__(VPT == 8 ? 512 : 1024) __global__ void rmsnorm_kernel(
    void* __restrict__ out, float* __restrict__ out_scale,
    const ushort* x,        // [T, H]; may be `out`
    ushort* __restrict__ residual,
    const ushort* __restrict__ w, const float eps, const int H,
    const ProductSums sums) {
  const int64_t row = blockIdx.x;
  const int nvec = H / 8;
  __shared__ float red[2][16];
  float vals[VPT][8];
  float ssum = 0.f;
  // Out of sums: bound by one latency after the other, so what does not wait for
  // anything is asked for before the parts. us, 40 rows of 4096 into fp8 7.1 -> 5.1, 560
  // rows 13.8 -> 10.0. (Not of a bf16 row: it would wait for the weights too. Rows in cache,
  // weights out of it, 40 x 2048 2.8 us with, 2.6 without.)
  ushort8 early_r[SUMS ? VPT : 1], early_w[SUMS ? VPT : 1];
  if constexpr (SUMS) {
#pragma unroll
    for (int k = 0; k < VPT; ++k) {
      const int i = min((int)(threadIdx.x + k * blockDim.x), nvec - 1);
      if constexpr (ADD)
        early_r[k] = reinterpret_cast<const ushort8*>(residual + row * H)[i];
      early_w[k] = reinterpret_cast<const ushort8*>(w)[i];
    }
    asm volatile("" ::: "memory");  // (or the loads move to where they are used)
  }
#pragma unroll
  for (int k = 0; k < VPT; ++k) {
    const int i = threadIdx.x + k * blockDim.x;
    if (i < nvec) {
      ushort8 xv;
      if constexpr (SUMS) {
        const SumScales<1> by(sums, row, {i * 8});
        asm volatile("" ::: "memory");  // (or the loads move behind the parts')
        xv = sums_unit(sums, row, i * 8, by);
        if constexpr (ADD) asm volatile("" : "+v"(early_r[k]));
      } else {
        xv = reinterpret_cast<const ushort8*>(x + row * H)[i];
      }
      if constexpr (ADD) {
        ushort8* rp = reinterpret_cast<ushort8*>(residual + row * H) + i;
        ushort8 rin;
        if constexpr (SUMS) rin = early_r[k];
        else rin = *rp;
        ushort8 rv;
#pragma unroll
        for (int j = 0; j < 8; ++j) {
          vals[k][j] = bf16_to_f32(xv[j]) + bf16_to_f32(rin[j]);
          rv[j] = f32_to_bf16(vals[k][j]);
        }
        *rp = rv;
      } else {
#pragma unroll
        for (int j = 0; j < 8; ++j) vals[k][j] = bf16_to_f32(xv[j]);
      }
#pragma unroll
      for (int j = 0; j < 8; ++j) ssum += vals[k][j] * vals[k][j];
    }
    if constexpr (SUMS) asm volatile("" : "+v"(early_w[k]));
  }
  const float total = block_reduce_sum(ssum, red[0]);
  const float inv_rms = rsqrtf(total / (float)H + eps);
  float amax = 0.f;
#pragma unroll
  for (int k = 0; k < VPT; ++k) {
    const int i = threadIdx.x + k * blockDim.x;
    if (i < nvec) {
      ushort8 wv;
      if constexpr (SUMS) wv = early_w[k];
      else wv = reinterpret_cast<const ushort8*>(w)[i];
      if constexpr (FP8) {
#pragma unroll
        for (int j = 0; j < 8; ++j) {
          vals[k][j] *= inv_rms * bf16_to_f32(wv[j]);
          amax = fmaxf(amax, fabsf(vals[k][j]));
        }
      } else {
        ushort8 o;
#pragma unroll
        for (int j = 0; j < 8; ++j)
          o[j] = f32_to_bf16(vals[k][j] * inv_rms * bf16_to_f32(wv[j]));
        reinterpret_cast<ushort8*>((ushort*)out + row * H)[i] = o;
      }
    }
  }
  if constexpr (FP8)
    write_fp8_row<VPT>((unsigned char*)out, out_scale, row, vals, amax, H, red[1]);
}

// hidden = residual + branch, out = norm of hidden, where branch is x or (FIRST)
// the norm of x: what lies between two sublayers whose outputs are normed too.
// Every step rounds to bf16 as the launches that it replaces did, so the bits
// are the same (but for 257 to 1023 rows of more than 4096 values out of sums: the last
// norm by itself adds its squares over more threads there). SUMS as above.
// A row is read once, in place of two passes over it (norm; add and norm); us in a
// model, separate launches / this: 5376 x 2304 35.1 / 20.9 (weights
// asked for behind the sums 22.3).
// EARLY: the weights are asked for before the branch.
template <bool FIRST, bool SUMS, int VPT, bool EARLY>
__launch_bounds__(VPT == 8 ? 512 : 1024) __global__ void norm_add_norm_kernel(
    ushort* __restrict__ out, ushort* __restrict__ hidden,
    const ushort* __restrict__ x, const ushort* __restrict__ residual,
    const ushort* __restrict__ w1, const ushort* __restrict__ w2,
    const float eps, const int H, const ProductSums sums) {
  const int64_t row = blockIdx.x;
  const int nvec = H / 8;
  __shared__ float red[2][16];
  float vals[VPT][8];
  ushort8 res[VPT];
  float ssum = 0.f;
  constexpr bool kEarly = EARLY && VPT <= 2;
  ushort8 early1[kEarly && FIRST ? VPT : 1], early2[kEarly ? VPT : 1];
#pragma unroll
  for (int k = 0; k < VPT; ++k) {
    const int i = min((int)(threadIdx.x + k * blockDim.x), nvec - 1);
    res[k] = reinterpret_cast<const ushort8*>(residual + row * H)[i];
    if constexpr (kEarly && FIRST) early1[k] = reinterpret_cast<const ushort8*>(w1)[i];
    if constexpr (kEarly) early2[k] = reinterpret_cast<const ushort8*>(w2)[i];
  }
  asm volatile("" ::: "memory");
#pragma unroll
  for (int k = 0; k < VPT; ++k) {
    const int i = threadIdx.x + k * blockDim.x;
    if (i < nvec) {
      ushort8 xv;
      if constexpr (SUMS) xv = sums_unit(sums, row, i * 8, {sums, row, {i * 8}});
      else xv = reinterpret_cast<const ushort8*>(x + row * H)[i];
#pragma unroll
      for (int j = 0; j < 8; ++j) {
        vals[k][j] = bf16_to_f32(xv[j]);
        ssum += vals[k][j] * vals[k][j];
      }
    }
    asm volatile("" : "+v"(res[k]));
    if constexpr (kEarly && FIRST) asm volatile("" : "+v"(early1[k]));
    if constexpr (kEarly) asm volatile("" : "+v"(early2[k]));
  }
  float inv = 1.f;
  if constexpr (FIRST)
    inv = rsqrtf(block_reduce_sum(ssum, red[0]) / (float)H + eps);
  ssum = 0.f;
#pragma unroll
  for (int k = 0; k < VPT; ++k) {
    const int i = threadIdx.x + k * blockDim.x;
    if (i < nvec) {
      ushort8 wv;
      if constexpr (FIRST && kEarly) wv = early1[k];
      else if constexpr (FIRST) wv = reinterpret_cast<const ushort8*>(w1)[i];
      ushort8 hv;
#pragma unroll
      for (int j = 0; j < 8; ++j) {
        float a = vals[k][j];
        if constexpr (FIRST)
          a = bf16_to_f32(f32_to_bf16(a * inv * bf16_to_f32(wv[j])));
        hv[j] = f32_to_bf16(bf16_to_f32(res[k][j]) + a);
        vals[k][j] = bf16_to_f32(hv[j]);
        ssum += vals[k][j] * vals[k][j];
      }
      reinterpret_cast<ushort8*>(hidden + row * H)[i] = hv;
    }
  }
  inv = rsqrtf(block_reduce_sum(ssum, red[1]) / (float)H + eps);
#pragma unroll
  for (int k = 0; k < VPT; ++k) {
    const int i = threadIdx.x + k * blockDim.x;
    if (i < nvec) {
      ushort8 wv;
      if constexpr (kEarly) wv = early2[k];
      else wv = reinterpret_cast<const ushort8*>(w2)[i];
      ushort8 o;
#pragma unroll
      for (int j = 0; j < 8; ++j)
        o[j] = f32_to_bf16(vals[k][j] * inv * bf16_to_f32(wv[j]));
      reinterpret_cast<ushort8*>(out + row * H)[i] = o;
    }
  }
}

// SILU: silu(gate) * up of packed [T, 2H] rows, else the rows as they are.
// src: row i is row src[i] of the input.
template <bool SILU, int VPT>
__launch_bounds__(VPT == 8 ? 512 : 1024) __global__ void to_fp8_kernel(
    unsigned char* __restrict__ out, float* __restrict__ out_scale,
    const ushort* __restrict__ xin, const int32_t* __restrict__ src,
    const int H) {
  const int64_t row = blockIdx.x;
  const int nvec = H / 8;
  const int64_t from = src ? src[row] : row;
  const ushort8* xr =
      reinterpret_cast<const ushort8*>(xin + from * (SILU ? 2 : 1) * H);
  __shared__ float red[16];
  float vals[VPT][8];
  float amax = 0.f;
#pragma unroll
  for (int k = 0; k < VPT; ++k) {
    const int i = threadIdx.x + k * blockDim.x;
    if (i < nvec) {
      const ushort8 g = xr[i];
      if constexpr (SILU) {
        const ushort8 u = xr[nvec + i];
#pragma unroll
        for (int j = 0; j < 8; ++j) {
          const float gf = bf16_to_f32(g[j]);
          vals[k][j] = gf / (1.0f + __expf(-gf)) * bf16_to_f32(u[j]);
        }
      } else {
#pragma unroll
        for (int j = 0; j < 8; ++j) vals[k][j] = bf16_to_f32(g[j]);
      }
#pragma unroll
      for (int j = 0; j < 8; ++j) amax = fmaxf(amax, fabsf(vals[k][j]));
    }
  }
  write_fp8_row<VPT>(out, out_scale, row, vals, amax, H, red);
}

// threads per row and units per thread for T rows of H values
struct Split {
  int threads, vpt;
};
Split split_for(int64_t T, int H, bool sums = false) {
  const int nvec = H / 8;
  // from about four rows a CU on the chip is full with 256 threads a row;
  // longer rows take 512, so that a thread's registers do not limit the waves.
  // Out of sums, whose threads have about 100 registers, two rows of more than 512
  // threads do not fit a CU (us, 1024 / 512 threads: 370 rows of 8192, one part, 9.0 / 7.1,
  // 849 of two 22.9 / 16.9; norm, sum and norm, 789 of six, 37.9 / 30.4).
  const int most = sums && T > kCUs ? 512 : 1024;
  const int threads = T >= 1024 ? (nvec <= 1024 ? 256 : 512)
                                : std::min(most, (nvec + 63) / 64 * 64);
  return {threads, (nvec + threads - 1) / threads};
}

// call f with the smallest instantiated number of units; 8 units come with at
// most 512 threads (32768 values: 8 x 512 or 4 x 1024)
template <typename F>
void with_vpt(int vpt, F&& f) {
  if (vpt <= 1) f(std::integral_constant<int, 1>{});
  else if (vpt <= 2) f(std::integral_constant<int, 2>{});
  else if (vpt <= 4) f(std::integral_constant<int, 4>{});
  else f(std::integral_constant<int, 8>{});
}

void check_row_op(const torch::Tensor& x, int max_h) {
  TORCH_CHECK(x.is_contiguous());
  TORCH_CHECK(x.scalar_type() == torch::kBFloat16);
  TORCH_CHECK(x.size(-1) % 8 == 0 && x.size(-1) <= max_h);
}

template <bool ADD, bool FP8, bool SUMS = false>
void launch_norm(void* out, float* out_scale, const ushort* x, int64_t T, int H,
                 ushort* residual, const torch::Tensor& weight, double eps,
                 const ProductSums& sums = {}) {
  const Split s = split_for(T, H, SUMS);
  with_vpt(s.vpt, [&](auto vpt) {
    hipLaunchKernelGGL((rmsnorm_kernel<ADD, FP8, SUMS, decltype(vpt)::value>),
                       dim3((uint32_t)T), dim3(s.threads), 0,
                       c10::hip::getCurrentHIPStream().stream(), out, out_scale,
                       x, residual, (const ushort*)weight.data_ptr(), (float)eps,
                       H, sums);
  });
  HIP_CHECK_KERNEL();
}

template <bool SILU>
void launch_to_fp8(torch::Tensor& out, torch::Tensor& out_scale,
                   const torch::Tensor& x, int64_t T, int H,
                   const int32_t* src = nullptr) {
  if (T == 0) return;
  const Split s = split_for(T, H);
  with_vpt(s.vpt, [&](auto vpt) {
    hipLaunchKernelGGL((to_fp8_kernel<SILU, decltype(vpt)::value>),
                       dim3((uint32_t)T), dim3(s.threads), 0,
                       c10::hip::getCurrentHIPStream().stream(),
                       (unsigned char*)out.data_ptr(),
                       out_scale.data_ptr<float>(),
                       (const ushort*)x.data_ptr(), src, H);
  });
  HIP_CHECK_KERNEL();
}

// a product's parts fp32 [parts, T, H], with sx [T] and sw [H] of fp8 operands
ProductSums sums_of(const torch::Tensor& part, const c10::optional<torch::Tensor>& sx,
                    const c10::optional<torch::Tensor>& sw, int max_h) {
  TORCH_CHECK(part.scalar_type() == torch::kFloat32 && part.is_contiguous() &&
              part.is_cuda() && part.dim() == 3);
  const int64_t T = part.size(1);
  const int H = part.size(2);
  TORCH_CHECK(H % 8 == 0 && H <= max_h);
  TORCH_CHECK(sx.has_value() == sw.has_value());
  if (sx.has_value())
    TORCH_CHECK(sx->scalar_type() == torch::kFloat32 && sx->is_contiguous() &&
                sx->numel() == T && sw->scalar_type() == torch::kFloat32 &&
                sw->is_contiguous() && sw->numel() == H);
  return {part.data_ptr<float>(), sx.has_value() ? sx->data_ptr<float>() : nullptr,
          sw.has_value() ? sw->data_ptr<float>() : nullptr, (int)part.size(0), T * H, H};
}

}  // namespace

void rmsnorm(torch::Tensor out, torch::Tensor x, torch::Tensor weight,
             double eps) {
  check_row_op(x, kMaxH);
  TORCH_CHECK(out.is_contiguous());
  launch_norm<false, false>(out.data_ptr(), nullptr, (const ushort*)x.data_ptr(),
      x.numel() / x.size(-1), x.size(-1), nullptr, weight, eps);
}

void fused_add_rmsnorm(torch::Tensor x, torch::Tensor residual,
                       torch::Tensor weight, double eps) {
  check_row_op(x, kMaxH);
  TORCH_CHECK(residual.is_contiguous());
  launch_norm<true, false>(x.data_ptr(), nullptr, (const ushort*)x.data_ptr(),
      x.numel() / x.size(-1), x.size(-1), (ushort*)residual.data_ptr(), weight, eps);
}

void rmsnorm_fp8(torch::Tensor out, torch::Tensor out_scale, torch::Tensor x,
                 torch::Tensor weight, double eps) {
  check_row_op(x, kMaxHFp8);
  launch_norm<false, true>(out.data_ptr(), out_scale.data_ptr<float>(), (const ushort*)x.data_ptr(),
      x.numel() / x.size(-1), x.size(-1), nullptr, weight, eps);
}

void fused_add_rmsnorm_fp8(torch::Tensor out, torch::Tensor out_scale,
                           torch::Tensor x, torch::Tensor residual,
                           torch::Tensor weight, double eps) {
  check_row_op(x, kMaxHFp8);
  TORCH_CHECK(residual.is_contiguous());
  launch_norm<true, true>(out.data_ptr(), out_scale.data_ptr<float>(), (const ushort*)x.data_ptr(),
      x.numel() / x.size(-1), x.size(-1), (ushort*)residual.data_ptr(), weight, eps);
}

void silu_and_mul_fp8(torch::Tensor out, torch::Tensor out_scale,
                      torch::Tensor x) {
  check_row_op(x, 2 * kMaxHFp8);
  const int I = x.size(1) / 2;
  TORCH_CHECK(I % 8 == 0 && I <= kMaxHFp8);
  launch_to_fp8<true>(out, out_scale, x, x.size(0), I);
}

void quant_fp8(torch::Tensor out, torch::Tensor out_scale, torch::Tensor x) {
  check_row_op(x, kMaxHFp8);
  const int H = x.size(-1);
  launch_to_fp8<false>(out, out_scale, x, x.numel() / H, H);
}

// rows of x in the order of src (int32, entries are rows of x), quantized
void quant_fp8_rows(torch::Tensor out, torch::Tensor out_scale, torch::Tensor x,
                    torch::Tensor src) {
  check_row_op(x, kMaxHFp8);
  TORCH_CHECK(x.dim() == 2 && src.scalar_type() == torch::kInt32 &&
              src.is_contiguous() && src.is_cuda());
  const int64_t n = src.numel();
  TORCH_CHECK(out.is_contiguous() && out.numel() == n * x.size(1) &&
              out.element_size() == 1 && out_scale.is_contiguous() &&
              out_scale.numel() == n);
  launch_to_fp8<false>(out, out_scale, x, n, x.size(1), src.data_ptr<int32_t>());
}

// the norms of a row that is still a product's parts: part fp32 [parts, T, H],
// sx [T] and sw [H] for fp8 operands. residual: added and updated, or none.
// out_scale given: out is fp8, else bf16.
void rmsnorm_sums(torch::Tensor out, c10::optional<torch::Tensor> out_scale,
                  torch::Tensor part, c10::optional<torch::Tensor> sx,
                  c10::optional<torch::Tensor> sw,
                  c10::optional<torch::Tensor> residual, torch::Tensor weight,
                  double eps) {
  const ProductSums p = sums_of(part, sx, sw, out_scale.has_value() ? kMaxHFp8 : kMaxH);
  const int64_t T = part.size(1);
  const int H = part.size(2);
  TORCH_CHECK(out.is_contiguous() && out.numel() == T * H &&
              out.element_size() == (out_scale.has_value() ? 1 : 2));
  TORCH_CHECK(weight.scalar_type() == torch::kBFloat16 && weight.numel() == H);
  ushort* res = nullptr;
  if (residual.has_value()) {
    TORCH_CHECK(residual->is_contiguous() && residual->numel() == T * H &&
                residual->scalar_type() == torch::kBFloat16);
    res = (ushort*)residual->data_ptr();
  }
  float* scale = nullptr;
  if (out_scale.has_value()) {
    TORCH_CHECK(out_scale->scalar_type() == torch::kFloat32 &&
                out_scale->is_contiguous() && out_scale->numel() == T);
    scale = out_scale->data_ptr<float>();
  }
  void* o = out.data_ptr();
  if (res && scale) launch_norm<true, true, true>(o, scale, nullptr, T, H, res, weight, eps, p);
  else if (res) launch_norm<true, false, true>(o, nullptr, nullptr, T, H, res, weight, eps, p);
  else if (scale) launch_norm<false, true, true>(o, scale, nullptr, T, H, nullptr, weight, eps, p);
  else launch_norm<false, false, true>(o, nullptr, nullptr, T, H, nullptr, weight, eps, p);
}

// hidden = residual + branch, out = norm(hidden, w2), where branch is x [T, H] or with
// w1 the norm of x (or, with part, of a product's sums)
void norm_add_norm(torch::Tensor out, torch::Tensor hidden,
                   c10::optional<torch::Tensor> x, c10::optional<torch::Tensor> part,
                   c10::optional<torch::Tensor> sx, c10::optional<torch::Tensor> sw,
                   torch::Tensor residual, c10::optional<torch::Tensor> w1,
                   torch::Tensor w2, double eps) {
  TORCH_CHECK(x.has_value() != part.has_value() && (w1.has_value() || x.has_value()));
  check_row_op(residual, kMaxH);
  const int H = residual.size(-1);
  const int64_t T = residual.numel() / H;
  ProductSums p{};
  if (part.has_value()) {
    p = sums_of(*part, sx, sw, kMaxH);
    TORCH_CHECK(part->size(1) == T && part->size(2) == H);
  } else {
    check_row_op(*x, kMaxH);
    TORCH_CHECK(x->numel() == T * H && x->size(-1) == H);
  }
  for (const auto& t : {out, hidden})
    TORCH_CHECK(t.is_contiguous() && t.numel() == T * H &&
                t.scalar_type() == torch::kBFloat16);
  for (const auto& w : {w1.has_value() ? *w1 : w2, w2})
    TORCH_CHECK(w.scalar_type() == torch::kBFloat16 && w.numel() == H && w.is_contiguous());
  if (T == 0) return;
  const Split s = split_for(T, H, part.has_value());
  auto launch = [&](auto first, auto sums, auto vpt, auto early) {
    hipLaunchKernelGGL((norm_add_norm_kernel<decltype(first)::value, decltype(sums)::value,
                                             decltype(vpt)::value, decltype(early)::value>),
                       dim3((uint32_t)T), dim3(s.threads), 0,
                       c10::hip::getCurrentHIPStream().stream(), (ushort*)out.data_ptr(),
                       (ushort*)hidden.data_ptr(),
                       x.has_value() ? (const ushort*)x->data_ptr() : nullptr,
                       (const ushort*)residual.data_ptr(),
                       w1.has_value() ? (const ushort*)w1->data_ptr() : nullptr,
                       (const ushort*)w2.data_ptr(), (float)eps, H, p);
  };
  using Yes = std::true_type;
  using No = std::false_type;
  // Registers for the weights: not in rows of 1024 threads, of which two share a CU then
  // (1000 x 16384 33 us with, 27 without; 8 x 8192 4.7 / 4.6; 40 x 2304 gains as above).
  auto go = [&](auto first, auto sums, auto vpt) {
    if (decltype(sums)::value || s.threads < 1024) launch(first, sums, vpt, Yes{});
    else launch(first, sums, vpt, No{});
  };
  with_vpt(s.vpt, [&](auto vpt) {
    if (part.has_value()) go(Yes{}, Yes{}, vpt);
    else if (w1.has_value()) go(Yes{}, No{}, vpt);
    else go(No{}, No{}, vpt);
  });
  HIP_CHECK_KERNEL();
}
