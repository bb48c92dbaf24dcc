// Routing of a sparse mixture-of-experts block for gfx950: which experts a
// token takes and with what weight, the tokens in expert order, and the
// weighted sum of what the experts returned. All of it on the device, with
// shapes that do not depend on the routing, so that a step can be recorded.
//
//  - moe_route: workgroup = token; a wave per expert (up to 16, then in turn), the products
//    of the bf16 hidden row and router rows summed in fp32. A chain of loads: the kernel
//    has 40 registers, and a unit of either row is waited for before the next ones'
//    products (with the order, us, four waves / a wave an expert: 40 x 4096 8 experts 9.1 / 7.9,
//    32 experts 21.2 / 13.4, 40 x 2048 16 experts 10.7 / 8.6); the largest top_k
//    (ties: the lower expert) and the softmax over them in fp32. NaN is the
//    largest score, and infinite scores make the weights NaN, as in the library
//    calls that this stands for: a token whose scores are not finite shows it.
//  - moe_order: one workgroup sorts the T * top_k (token, choice) pairs by
//    expert, tokens ascending: every thread counts a run of pairs per expert
//    (LDS [expert][thread]), the counts are scanned, every thread places its
//    run. No atomics: the order is fixed.
//  - moe_combine: workgroup = token; sum over its choices of weight * row in
//    fp32, rounded once.
// Bound by launches at decode sizes; they take the place of about 60 of them
// (fp32 copies of the router, a library top-k, and per expert two library
// products, an activation, a scaling and an addition).
#include <torch/extension.h>

#include <algorithm>

#include "common.h"

namespace {

constexpr int kMaxExperts = 32;
constexpr int kMaxTop = 8;
constexpr int kOrderThreads = 256;
constexpr int kMostRouteWaves = 16;

__launch_bounds__(kMostRouteWaves * WAVE_SIZE) __global__ void moe_route_kernel(
    int32_t* __restrict__ index,   // [T, top]
    float* __restrict__ weight,    // [T, top]
    const ushort* __restrict__ x,  // [T, H]
    const ushort* __restrict__ w,  // [E, H]
    const int H, const int E, const int top) {
  const int64_t t = blockIdx.x;
  const int wave = threadIdx.x / WAVE_SIZE, lane = threadIdx.x % WAVE_SIZE;
  __shared__ float logit[kMaxExperts];
  const ushort8* xr = reinterpret_cast<const ushort8*>(x + t * H);
  for (int e = wave; e < E; e += blockDim.x / WAVE_SIZE) {
    const ushort8* wr = reinterpret_cast<const ushort8*>(w + (int64_t)e * H);
    float acc = 0.f;
#pragma unroll 4
    for (int i = lane; i < H / 8; i += WAVE_SIZE) {
      const ushort8 a = xr[i], b = wr[i];
#pragma unroll
      for (int j = 0; j < 8; ++j)
        acc = fmaf(bf16_to_f32(a[j]), bf16_to_f32(b[j]), acc);
    }
    acc = wave_reduce_sum(acc);
    if (lane == 0) logit[e] = acc;
  }
  __syncthreads();
  if (wave != 0) return;
  // lane e holds expert e; the order of the scores, lanes past E below all
  const float v = lane < E ? logit[lane] : -INFINITY;
  const bool nan = v != v;
  bool taken = lane >= E;
  float first = 0.f, total = 0.f, mine = 0.f;
  for (int k = 0; k < top; ++k) {
    float best = taken ? -INFINITY : nan ? INFINITY : v;
    // among equals: NaN, then the lower expert; one that is left before the rest
    int at = lane + (taken ? 2 * WAVE_SIZE : nan ? 0 : WAVE_SIZE);
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) {
      const float ov = __shfl_xor(best, off, 64);
      const int oa = __shfl_xor(at, off, 64);
      if (ov > best || (ov == best && oa < at)) {
        best = ov;
        at = oa;
      }
    }
    if (at < WAVE_SIZE) best = NAN;
    at %= WAVE_SIZE;
    if (k == 0) first = best;
    const float p = __expf(best - first);
    total += p;
    if (lane == k) {
      mine = p;
      index[t * top + k] = at;
    }
    if (lane == at) taken = true;
  }
  if (lane < top) weight[t * top + lane] = mine / total;
}

__launch_bounds__(kOrderThreads) __global__ void moe_order_kernel(
    int32_t* __restrict__ begin,  // [E + 1]
    int32_t* __restrict__ src,    // [n] token of every sorted row
    int32_t* __restrict__ place,  // [n] sorted row of every pair
    const int32_t* __restrict__ index, const int n, const int E,
    const int top) {
  extern __shared__ int32_t cnt[];  // [E][threads], then the experts' starts
  int32_t* start = cnt + E * kOrderThreads;
  const int tid = threadIdx.x;
  const int per = (n + kOrderThreads - 1) / kOrderThreads;
  const int lo = min(n, tid * per), hi = min(n, lo + per);
  for (int e = 0; e < E; ++e) cnt[e * kOrderThreads + tid] = 0;
  for (int i = lo; i < hi; ++i) ++cnt[index[i] * kOrderThreads + tid];
  __syncthreads();
  // exclusive scan of every expert's counts, a wave per expert
  const int wave = tid / WAVE_SIZE, lane = tid % WAVE_SIZE;
  for (int e = wave; e < E; e += kOrderThreads / WAVE_SIZE) {
    int base = 0;
    for (int c = 0; c < kOrderThreads; c += WAVE_SIZE) {
      const int v = cnt[e * kOrderThreads + c + lane];
      int s = v;
#pragma unroll
      for (int off = 1; off < 64; off <<= 1) {
        const int o = __shfl_up(s, off, 64);
        if (lane >= off) s += o;
      }
      cnt[e * kOrderThreads + c + lane] = base + s - v;
      base += __shfl(s, 63, 64);
    }
    if (lane == 0) start[e + 1] = base;
  }
  __syncthreads();
  if (tid == 0) {
    int sum = 0;
    start[0] = 0;
    for (int e = 0; e < E; ++e) {
      sum += start[e + 1];
      start[e + 1] = sum;
    }
  }
  __syncthreads();
  if (tid <= E) begin[tid] = start[tid];
  for (int i = lo; i < hi; ++i) {
    const int e = index[i];
    const int at = start[e] + cnt[e * kOrderThreads + tid]++;
    src[at] = i / top;
    place[i] = at;
  }
}

__launch_bounds__(256) __global__ void moe_combine_kernel(
    ushort* __restrict__ out,          // [T, H]
    const ushort* __restrict__ y,      // [T * top, H], expert order
    const int32_t* __restrict__ place, const float* __restrict__ weight,
    const int H, const int top) {
  const int64_t t = blockIdx.x;
  int32_t at[kMaxTop];
  float w[kMaxTop];
#pragma unroll
  for (int k = 0; k < kMaxTop; ++k)
    if (k < top) {
      at[k] = place[t * top + k];
      w[k] = weight[t * top + k];
    }
  for (int i = threadIdx.x; i < H / 8; i += 256) {
    float acc[8];
#pragma unroll
    for (int j = 0; j < 8; ++j) acc[j] = 0.f;
#pragma unroll
    for (int k = 0; k < kMaxTop; ++k)
      if (k < top) {
        const ushort8 v =
            reinterpret_cast<const ushort8*>(y + (int64_t)at[k] * H)[i];
#pragma unroll
        for (int j = 0; j < 8; ++j) acc[j] = fmaf(w[k], bf16_to_f32(v[j]), acc[j]);
      }
    ushort8 o;
#pragma unroll
    for (int j = 0; j < 8; ++j) o[j] = f32_to_bf16(acc[j]);
    reinterpret_cast<ushort8*>(out + t * H)[i] = o;
  }
}

}  // namespace

// index int32 [T, top], weight fp32 [T, top], begin int32 [E + 1], src and
// place int32 [T * top] of hidden x [T, H] and router w [E, H], both bf16
void moe_route(torch::Tensor index, torch::Tensor weight, torch::Tensor begin,
               torch::Tensor src, torch::Tensor place, torch::Tensor x,
               torch::Tensor w) {
  const int64_t T = x.size(0);
  const int H = x.size(1), E = w.size(0), top = index.size(1);
  TORCH_CHECK(x.scalar_type() == torch::kBFloat16 && x.is_contiguous() &&
              x.is_cuda() && w.scalar_type() == torch::kBFloat16 &&
              w.is_contiguous() && w.is_cuda() && w.size(1) == H && H % 8 == 0);
  TORCH_CHECK(E >= 1 && E <= kMaxExperts && top >= 1 && top <= kMaxTop && top <= E);
  const int64_t n = T * top;
  auto i32 = [&](const torch::Tensor& t, int64_t k) {
    TORCH_CHECK(t.scalar_type() == torch::kInt32 && t.is_contiguous() &&
                t.is_cuda() && t.numel() == k);
  };
  i32(index, n);
  i32(begin, E + 1);
  i32(src, n);
  i32(place, n);
  TORCH_CHECK(weight.scalar_type() == torch::kFloat32 && weight.is_contiguous() &&
              weight.is_cuda() && weight.numel() == n && n < (1ll << 30));
  if (T == 0) return;
  auto stream = c10::hip::getCurrentHIPStream().stream();
  // more tokens than two a CU fill the chip with four waves each (us, 16 / 4 waves: 20
  // experts of 4096 500 tokens 15.0 / 17.0, 600 19.2 / 17.6; 16 of 1024 800 13.6 / 12.2)
  const int waves = T > 512 ? 4 : std::min(kMostRouteWaves, std::max(4, E));
  hipLaunchKernelGGL(moe_route_kernel, dim3((uint32_t)T), dim3(waves * WAVE_SIZE), 0, stream,
                     index.data_ptr<int32_t>(), weight.data_ptr<float>(),
                     (const ushort*)x.data_ptr(), (const ushort*)w.data_ptr(),
                     H, E, top);
  HIP_CHECK_KERNEL();
  // at most 33 KB
  const size_t smem = sizeof(int32_t) * ((size_t)E * kOrderThreads + E + 1);
  hipLaunchKernelGGL(moe_order_kernel, dim3(1), dim3(kOrderThreads), smem, stream,
                     begin.data_ptr<int32_t>(), src.data_ptr<int32_t>(),
                     place.data_ptr<int32_t>(), index.data_ptr<int32_t>(),
                     (int)n, E, top);
  HIP_CHECK_KERNEL();
}

void moe_combine(torch::Tensor out, torch::Tensor y, torch::Tensor place,
                 torch::Tensor weight) {
  const int64_t T = out.size(0);
  const int H = out.size(1), top = weight.size(1);
  TORCH_CHECK(out.scalar_type() == torch::kBFloat16 && out.is_contiguous() &&
              y.scalar_type() == torch::kBFloat16 && y.is_contiguous() &&
              y.size(0) == T * top && y.size(1) == H && H % 8 == 0);
  TORCH_CHECK(place.scalar_type() == torch::kInt32 && place.is_contiguous() &&
              place.numel() == T * top);
  TORCH_CHECK(weight.scalar_type() == torch::kFloat32 && weight.is_contiguous() &&
              weight.size(0) == T && top >= 1 && top <= kMaxTop);
  if (T == 0) return;
  hipLaunchKernelGGL(moe_combine_kernel, dim3((uint32_t)T), dim3(256), 0,
                     c10::hip::getCurrentHIPStream().stream(),
                     (ushort*)out.data_ptr(), (const ushort*)y.data_ptr(),
                     place.data_ptr<int32_t>(), weight.data_ptr<float>(), H, top);
  HIP_CHECK_KERNEL();
}
