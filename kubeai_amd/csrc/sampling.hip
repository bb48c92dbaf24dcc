// Token sampling kernels (two-stage argmax reduction).
//
// greedy_sample:  argmax over the vocab row.
// gumbel_sample:  argmax(logits/T + Gumbel noise) — exact temperature
//   sampling without softmax or sort. RNG = counter-based splitmix64 hash
//   (common.h), spec-identical to ops/ref.py.
// Tie-break: lowest index wins (matches torch.argmax).
//
// Stage 1 splits each vocab row into kSplits chunks (B*kSplits workgroups
// keep all 256 CUs busy even at decode batch ~32); stage 2 is one wave per
// row reducing the partials.
//
// With log-probabilities the same pass has the sum of exp(x - max) as well: a thread
// holds 16 values at a time, their maximum moves its sum once, so a value costs one
// exponential. Bound by reading the logits once and by two launches: 40 rows of 128256
// 11.6 us (the greedy tokens alone 7.4; torch's logsumexp, gather and difference behind
// that 72), one row 7.6 (5.7 and 49), 96 rows 22.5 (15.2 and 89).
#include <torch/extension.h>

#include <type_traits>

#include "common.h"

namespace {

constexpr int kBlock = 256;
constexpr int kSplits = 32;
constexpr int kUnits = 4;  // of 4 values, a thread at a time

// a chunk's best value (with its noise) and where, and with log-probabilities that
// place's logit, the largest logit and the sum of exp(logit - it)
template <bool kLogprob>
struct Part {
  float best;
  int32_t idx;
};
template <>
struct Part<true> {
  float best;
  int32_t idx;
  float raw, m, z;
};
template <bool kLogprob>
DEV_INLINE Part<kLogprob> none(int32_t idx) {
  if constexpr (kLogprob) return {-INFINITY, idx, -INFINITY, -INFINITY, 0.f};
  else return {-INFINITY, idx};
}

template <bool kLogprob>
DEV_INLINE void keep_best(Part<kLogprob>& p, float v, int32_t i, float raw) {
  if (v > p.best || (v == p.best && i < p.idx)) {
    p.best = v;
    p.idx = i;
    if constexpr (kLogprob) p.raw = raw;
  }
}
// (a maximum of -inf has only zeros behind it)
DEV_INLINE float finite_or_0(float m) { return m == -INFINITY ? 0.f : m; }
DEV_INLINE void keep_sum(Part<true>& p, float m, float z) {
  const float most = fmaxf(p.m, m), use = finite_or_0(most);
  p.z = p.z * expf(p.m - use) + z * expf(m - use);
  p.m = most;
}
template <bool kLogprob>
DEV_INLINE void over_lanes(Part<kLogprob>& p) {
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) {
    const float v = __shfl_xor(p.best, off);
    const int32_t i = __shfl_xor(p.idx, off);
    if constexpr (kLogprob) {
      const float raw = __shfl_xor(p.raw, off), m = __shfl_xor(p.m, off),
                  z = __shfl_xor(p.z, off);
      keep_best(p, v, i, raw);
      keep_sum(p, m, z);
    } else {
      keep_best(p, v, i, 0.f);
    }
  }
}

// kMany: a thread takes 16 values at a time, else one
template <bool kGumbel, bool kLogprob, bool kMany>
__launch_bounds__(kBlock) __global__ void sample_stage1(
    Part<kLogprob>* __restrict__ part,     // [B, kSplits]
    const float* __restrict__ logits,      // [B, V]
    const float* __restrict__ temperature,  // [B]
    const int64_t* __restrict__ seeds,      // [B]
    const int64_t step, const int V, const bool wide) {
  const int b = blockIdx.x;
  const int split = blockIdx.y;
  const int chunk = ((V + kSplits - 1) / kSplits + 3) / 4 * 4;
  const int lo = min(V, split * chunk);
  const int hi = min(V, lo + chunk);
  const float* row = logits + (int64_t)b * V;
  float temp = 1.0f;
  uint64_t key = 0;
  bool greedy = !kGumbel;
  if constexpr (kGumbel) {
    temp = temperature[b];
    if (temp <= 0.f) greedy = true;
    key = (uint64_t)seeds[b] * 1000003ull + (uint64_t)step;
  }

  auto noisy = [&](float val, int v) {
    if (!greedy) {
      const float u = hash_uniform(key, (uint64_t)v);
      val = val / temp + (-__logf(-__logf(u)));
    }
    return val;
  };
  static_assert(kMany || !kLogprob);
  Part<kLogprob> p = none<kLogprob>(V);
  if constexpr (!kMany) {
    for (int v = lo + threadIdx.x; v < hi; v += kBlock) keep_best(p, noisy(row[v], v), v, 0.f);
  }
  for (int base = lo; kMany && base < hi; base += kBlock * 4 * kUnits) {
    float4_t x[kUnits];
#pragma unroll
    for (int j = 0; j < kUnits; ++j) {
      const int v = base + (j * kBlock + threadIdx.x) * 4;
      x[j] = float4_t{-INFINITY, -INFINITY, -INFINITY, -INFINITY};
      if (wide) {  // (then hi is a multiple of 4 too)
        if (v < hi) x[j] = *reinterpret_cast<const float4_t*>(row + v);
      } else {
#pragma unroll
        for (int k = 0; k < 4; ++k)
          if (v + k < hi) x[j][k] = row[v + k];
      }
    }
    float most = -INFINITY;
#pragma unroll
    for (int j = 0; j < kUnits; ++j) {
#pragma unroll
      for (int k = 0; k < 4; ++k) {
        const int v = base + (j * kBlock + threadIdx.x) * 4 + k;
        if (v < hi) keep_best(p, noisy(x[j][k], v), v, x[j][k]);
        if constexpr (kLogprob) most = fmaxf(most, x[j][k]);
      }
    }
    if constexpr (kLogprob) {
      most = fmaxf(most, p.m);
      const float use = finite_or_0(most);
      float z = p.z * expf(p.m - use);
#pragma unroll
      for (int j = 0; j < kUnits; ++j) {
#pragma unroll
        for (int k = 0; k < 4; ++k) z += expf(x[j][k] - use);
      }
      p.m = most;
      p.z = z;
    }
  }
  over_lanes<kLogprob>(p);
  __shared__ Part<kLogprob> waves[kBlock / WAVE_SIZE];
  const int wave = threadIdx.x / WAVE_SIZE;
  if (threadIdx.x % WAVE_SIZE == 0) waves[wave] = p;
  __syncthreads();
  if (threadIdx.x == 0) {
#pragma unroll
    for (int w = 1; w < kBlock / WAVE_SIZE; ++w) {
      const Part<kLogprob> o = waves[w];
      if constexpr (kLogprob) {
        keep_best(p, o.best, o.idx, o.raw);
        keep_sum(p, o.m, o.z);
      } else {
        keep_best(p, o.best, o.idx, 0.f);
      }
    }
    part[b * kSplits + split] = p;
  }
}

template <bool kLogprob>
__global__ void sample_stage2(int64_t* __restrict__ out, float* __restrict__ logprob,
                              const Part<kLogprob>* __restrict__ part) {
  const int b = blockIdx.x;
  const int lane = threadIdx.x;
  Part<kLogprob> p = none<kLogprob>(INT32_MAX);
  if (lane < kSplits) p = part[b * kSplits + lane];
  over_lanes<kLogprob>(p);
  if (lane == 0) {
    out[b] = p.idx;
    if constexpr (kLogprob) logprob[b] = p.raw - (finite_or_0(p.m) + logf(p.z));
  }
}

template <bool kGumbel, bool kLogprob>
void launch_sample(torch::Tensor out, float* logprob, torch::Tensor logits,
                   const float* temp_ptr, const int64_t* seed_ptr,
                   int64_t step) {
  const int B = logits.size(0), V = logits.size(1);
  if (B == 0) return;
  auto part = torch::empty({B, kSplits, (int64_t)sizeof(Part<kLogprob>)},
                           torch::TensorOptions().device(logits.device()).dtype(torch::kUInt8));
  auto* pp = reinterpret_cast<Part<kLogprob>*>(part.data_ptr());
  const bool wide = V % 4 == 0 && ((uintptr_t)logits.data_ptr() & 15) == 0;
  auto stream = c10::hip::getCurrentHIPStream().stream();
  auto stage1 = [&](auto many) {
    hipLaunchKernelGGL((sample_stage1<kGumbel, kLogprob, decltype(many)::value>),
                       dim3(B, kSplits), dim3(kBlock), 0, stream, pp, logits.data_ptr<float>(),
                       temp_ptr, seed_ptr, step, V, wide);
  };
  // Tokens alone take a value at a time: the noise hides the loads, and a chunk of a small
  // vocabulary has no 16 values for each thread (us, at a time one / 16: 278 rows of 3954
  // greedy 11.2 / 17.2, noise 12.5 / 20.9; 144 of 27950 11.4 / 11.9, 14.4 / 16.7; 109 of 77195
  // 14.5 / 14.2, 22.3 / 24.6; 198 of 91860 31.4 / 21.4, 41.3 / 41.5; 22 of 188508 14.0 / 9.8,
  // 17.8 / 17.1).
  if constexpr (kLogprob) stage1(std::true_type{});
  else if (!kGumbel && V >= 65536) stage1(std::true_type{});
  else stage1(std::false_type{});
  HIP_CHECK_KERNEL();
  hipLaunchKernelGGL((sample_stage2<kLogprob>), dim3(B), dim3(WAVE_SIZE), 0, stream,
                     out.data_ptr<int64_t>(), logprob, pp);
  HIP_CHECK_KERNEL();
}

template <bool kGumbel>
void launch_sample(torch::Tensor out, const c10::optional<torch::Tensor>& logprob,
                   torch::Tensor logits, const float* temp_ptr, const int64_t* seed_ptr,
                   int64_t step) {
  if (!logprob.has_value()) {
    launch_sample<kGumbel, false>(out, nullptr, logits, temp_ptr, seed_ptr, step);
    return;
  }
  TORCH_CHECK(logprob->scalar_type() == torch::kFloat32 && logprob->is_contiguous() &&
              logprob->is_cuda() && logprob->numel() == logits.size(0));
  launch_sample<kGumbel, true>(out, logprob->data_ptr<float>(), logits, temp_ptr, seed_ptr,
                               step);
}

}  // namespace

// logprob (fp32 [B], or none): the sampled token's logit - log(sum(exp(row)))
void greedy_sample(torch::Tensor out, torch::Tensor logits,
                   c10::optional<torch::Tensor> logprob) {
  TORCH_CHECK(logits.is_contiguous());
  TORCH_CHECK(logits.scalar_type() == torch::kFloat32,
              "sampling expects fp32 logits");
  launch_sample<false>(out, logprob, logits, nullptr, nullptr, 0);
}

void gumbel_sample(torch::Tensor out, torch::Tensor logits,
                   torch::Tensor temperature, torch::Tensor seeds,
                   int64_t step, c10::optional<torch::Tensor> logprob) {
  TORCH_CHECK(logits.is_contiguous());
  TORCH_CHECK(logits.scalar_type() == torch::kFloat32);
  TORCH_CHECK(temperature.scalar_type() == torch::kFloat32);
  TORCH_CHECK(seeds.scalar_type() == torch::kInt64);
  launch_sample<true>(out, logprob, logits, temperature.data_ptr<float>(),
                      seeds.data_ptr<int64_t>(), step);
}

// ---------------------------------------------------------------------
// Rejection-based nucleus sampling support (runner._sample_topk_topp):
// one pass computes per-row softmax stats; per candidate draw another
// single pass decides membership (probability mass strictly above the
// sampled logit < top_p, and rank < top_k) — no [S,V] intermediates.

namespace {

__global__ void nucleus_stats_kernel(
    float* __restrict__ m_out, float* __restrict__ z_out,
    const float* __restrict__ logits, const float* __restrict__ temps,
    const int V) {
  const int row = blockIdx.x;
  const float* x = logits + (int64_t)row * V;
  const float t = fmaxf(temps[row], 1e-6f);
  __shared__ float red[16];
  float m = -INFINITY;
  for (int i = threadIdx.x; i < V; i += blockDim.x) m = fmaxf(m, x[i]);
  m = wave_reduce_max(m);
  const int wave = threadIdx.x / WAVE_SIZE, lane = threadIdx.x % WAVE_SIZE;
  const int nw = blockDim.x / WAVE_SIZE;
  if (lane == 0) red[wave] = m;
  __syncthreads();
  float mm = -INFINITY;
  for (int w = 0; w < nw; ++w) mm = fmaxf(mm, red[w]);
  __syncthreads();
  float z = 0.f;
  for (int i = threadIdx.x; i < V; i += blockDim.x)
    z += __expf((x[i] - mm) / t);
  z = block_reduce_sum(z, red);
  if (threadIdx.x == 0) {
    m_out[row] = mm;
    z_out[row] = z;
  }
}

__global__ void nucleus_accept_kernel(
    unsigned char* __restrict__ ok,      // [S]
    const float* __restrict__ logits,    // [S, V]
    const int64_t* __restrict__ cand,    // [S]
    const float* __restrict__ m_in, const float* __restrict__ z_in,
    const float* __restrict__ temps, const float* __restrict__ top_ps,
    const int32_t* __restrict__ top_ks, const int V) {
  const int row = blockIdx.x;
  const float t0 = temps[row];
  if (t0 <= 0.f) {  // greedy rows: argmax is always in the nucleus
    if (threadIdx.x == 0) ok[row] = 1;
    return;
  }
  const float* x = logits + (int64_t)row * V;
  const int64_t c = cand[row];
  if (c < 0 || c >= V) {  // (what the sampler gives for a row in which no value compares)
    if (threadIdx.x == 0) ok[row] = 0;
    return;
  }
  const float lt = x[c];
  const float t = fmaxf(t0, 1e-6f);
  const float m = m_in[row], z = z_in[row];
  __shared__ float red[16];
  float mass = 0.f;
  int cnt = 0;
  for (int i = threadIdx.x; i < V; i += blockDim.x) {
    const float xi = x[i];
    if (xi > lt) {
      mass += __expf((xi - m) / t);
      ++cnt;
    }
  }
  mass = block_reduce_sum(mass, red);
  __syncthreads();
  float cntf = block_reduce_sum((float)cnt, red);
  if (threadIdx.x == 0) {
    const float mass_above = mass / z;
    const int k = top_ks[row];
    ok[row] = (mass_above < top_ps[row] && (k <= 0 || (int)cntf < k)) ? 1 : 0;
  }
}

}  // namespace

void nucleus_stats(torch::Tensor m, torch::Tensor z, torch::Tensor logits,
                   torch::Tensor temps) {
  TORCH_CHECK(logits.is_contiguous() &&
              logits.scalar_type() == torch::kFloat32);
  const int S = logits.size(0), V = logits.size(1);
  auto stream = c10::hip::getCurrentHIPStream().stream();
  hipLaunchKernelGGL(nucleus_stats_kernel, dim3(S), dim3(512), 0, stream,
                     m.data_ptr<float>(), z.data_ptr<float>(),
                     logits.data_ptr<float>(), temps.data_ptr<float>(), V);
  HIP_CHECK_KERNEL();
}

void nucleus_accept(torch::Tensor ok, torch::Tensor logits,
                    torch::Tensor cand, torch::Tensor m, torch::Tensor z,
                    torch::Tensor temps, torch::Tensor top_ps,
                    torch::Tensor top_ks) {
  TORCH_CHECK(logits.is_contiguous() &&
              logits.scalar_type() == torch::kFloat32);
  TORCH_CHECK(cand.scalar_type() == torch::kInt64);
  TORCH_CHECK(top_ks.scalar_type() == torch::kInt32);
  const int S = logits.size(0), V = logits.size(1);
  auto stream = c10::hip::getCurrentHIPStream().stream();
  hipLaunchKernelGGL(nucleus_accept_kernel, dim3(S), dim3(512), 0, stream,
                     ok.data_ptr<unsigned char>(),
                     logits.data_ptr<float>(), cand.data_ptr<int64_t>(),
                     m.data_ptr<float>(), z.data_ptr<float>(),
                     temps.data_ptr<float>(), top_ps.data_ptr<float>(),
                     top_ks.data_ptr<int32_t>(), V);
  HIP_CHECK_KERNEL();
}
