// NeoX rotary embedding, in-place over q and k, one launch.
//
// Semantics: kubeai_amd/ops/ref.py::rope. cos/sin are precomputed on host
// ([max_pos, head_dim] fp32, cos | sin halves) — on-device trig would turn
// this memory-bound op VALU-bound (guide Appendix B).
//
// Grid: one wave per (token, head); lane i handles the rotation pair
// (i, i + hd/2) for hd=128 (one pair per lane), generic loop otherwise.
#include <torch/extension.h>

#include <type_traits>

#include "common.h"

namespace {

__global__ void rope_kernel(
    ushort* __restrict__ q,        // [T, n_q, hd]
    ushort* __restrict__ k,        // [T, n_kv, hd]
    const int32_t* __restrict__ positions,  // [T]
    const float* __restrict__ cos_sin,      // [max_pos, hd]
    const int n_q, const int n_kv, const int hd, const int64_t n_tok,
    const int64_t q_stride, const int64_t k_stride) {
  const int n_heads = n_q + n_kv;
  const int64_t flat = (int64_t)blockIdx.x * (blockDim.x / WAVE_SIZE) +
                       threadIdx.x / WAVE_SIZE;
  const int64_t tok = flat / n_heads;
  if (tok >= n_tok) return;
  const int head = (int)(flat % n_heads);
  const int lane = threadIdx.x % WAVE_SIZE;
  const int half = hd / 2;

  const int pos = positions[tok];
  const float* cs = cos_sin + (int64_t)pos * hd;
  ushort* base = (head < n_q)
                     ? q + tok * q_stride + (int64_t)head * hd
                     : k + tok * k_stride + (int64_t)(head - n_q) * hd;

  for (int i = lane; i < half; i += WAVE_SIZE) {
    const float c = cs[i];
    const float s = cs[half + i];
    const float x1 = bf16_to_f32(base[i]);
    const float x2 = bf16_to_f32(base[half + i]);
    base[i] = f32_to_bf16(x1 * c - x2 * s);
    base[half + i] = f32_to_bf16(x2 * c + x1 * s);
  }
}

// Rotation and cache write in one pass over the qkv projection: q is rotated
// in place, k is rotated into its cache row, v is copied into its own. A
// thread takes 8 rotation pairs (two 16-byte units, half a head apart) or 8
// values of v. Replaces two launches, and k's round trip between them.
// 8192 tokens, 32/8 heads of 128: 39 us (4.3 TB/s), before 71 + 21; 40 tokens:
// 4.9 us, before 4.7 + 4.7.
template <typename CT>
DEV_INLINE void put_row8(CT* dst, const ushort8& v) {
  if constexpr (sizeof(CT) == 2) {
    *reinterpret_cast<ushort8*>(dst) = v;
  } else {
    uint64_t o = 0;
#pragma unroll
    for (int j = 0; j < 8; ++j)
      o |= (uint64_t)f32_to_e5m2(bf16_to_f32((ushort)v[j])) << (8 * j);
    *reinterpret_cast<uint64_t*>(dst) = o;
  }
}

// SUMS: the projection is a product's parts; q goes to its own rows.
// A chain of latencies at few tokens: slot and position at once, then angles, scales
// and the parts of both halves at once; no division in 64 bits where 32 will do. 40
// tokens, 32/8 heads of 128: 6.4 us with each behind the one before, now 4.7.
template <typename CT, bool SUMS>
__launch_bounds__(256) __global__ void rope_cache_kernel(
    ushort* __restrict__ qkv,  // [T, (n_q + 2 n_kv) hd], rows strided; SUMS:
                               // q out [T, n_q hd]
    const ProductSums sums,
    const int32_t* __restrict__ positions,
    const float* __restrict__ cos_sin,   // [max_pos, hd]
    CT* __restrict__ k_cache,            // [nb, n_kv, bs, hd]
    CT* __restrict__ v_cache,
    const int64_t* __restrict__ slot_mapping, const int n_q, const int n_kv,
    const int hd, const int bs, const int64_t n_tok, const int64_t stride) {
  const int half = hd / 2;
  const int ppu = half / 8;                        // pair units per head
  const int n_rot = (n_q + n_kv) * ppu;
  const int n_item = n_rot + n_kv * (hd / 8);
  const int64_t flat = (int64_t)blockIdx.x * 256 + threadIdx.x;
  // (a division in 64 bits takes longer than the whole item)
  const bool small = n_tok * n_item + 256 <= UINT32_MAX;
  const int64_t tok = small ? (uint32_t)flat / (uint32_t)n_item : flat / n_item;
  if (tok >= n_tok) return;
  const int item = (int)(flat - tok * n_item);
  ushort* row = qkv + tok * stride;
  if (item < n_rot) {
    const int head = item / ppu, p = item % ppu * 8;
    ushort* base = row + (int64_t)head * hd + p;
    int64_t slot = slot_mapping[tok];
    int pos = positions[tok];
    asm volatile("" : "+v"(slot), "+v"(pos));  // both on their way before either is used
    if (head < n_q) slot = 0;
    if (slot < 0) return;  // a padding token's key goes nowhere
    const float* cs = cos_sin + (int64_t)pos * hd + p;
    float cv[8], sv[8];
#pragma unroll
    for (int j = 0; j < 8; ++j) {
      cv[j] = cs[j];
      sv[j] = cs[half + j];
    }
    ushort8 a, b;
    if constexpr (SUMS) {
      // both halves' parts at once
      const int cols[2] = {head * hd + p, head * hd + p + half};
      const SumScales<2> by(sums, tok, cols);
      asm volatile("" ::: "memory");  // (or the angles' loads move behind the parts')
      ushort8 ab[2];
      read_sums8<2>(sums, tok, cols, by, ab);
#pragma unroll
      for (int j = 0; j < 8; ++j) asm volatile("" : "+v"(cv[j]), "+v"(sv[j]));
      a = ab[0];
      b = ab[1];
    } else {
      a = *reinterpret_cast<const ushort8*>(base);
      b = *reinterpret_cast<const ushort8*>(base + half);
    }
    ushort8 oa, ob;
#pragma unroll
    for (int j = 0; j < 8; ++j) {
      const float c = cv[j], s = sv[j];
      const float x1 = bf16_to_f32(a[j]), x2 = bf16_to_f32(b[j]);
      oa[j] = f32_to_bf16(x1 * c - x2 * s);
      ob[j] = f32_to_bf16(x2 * c + x1 * s);
    }
    if (head < n_q) {
      *reinterpret_cast<ushort8*>(base) = oa;
      *reinterpret_cast<ushort8*>(base + half) = ob;
    } else {
      CT* dst = k_cache +
                (((slot / bs) * n_kv + head - n_q) * bs + slot % bs) * hd + p;
      put_row8(dst, oa);
      put_row8(dst + half, ob);
    }
  } else {
    const int64_t slot = slot_mapping[tok];
    if (slot < 0) return;
    const int upr = hd / 8;
    const int head = (item - n_rot) / upr, u = (item - n_rot) % upr * 8;
    ushort8 v;
    if constexpr (SUMS) {
      const int cols[1] = {(n_q + n_kv + head) * hd + u};
      const SumScales<1> by(sums, tok, cols);
      ushort8 one[1];
      read_sums8<1>(sums, tok, cols, by, one);
      v = one[0];
    } else {
      v = *reinterpret_cast<const ushort8*>(
          row + (int64_t)(n_q + n_kv + head) * hd + u);
    }
    put_row8(v_cache + (((slot / bs) * n_kv + head) * bs + slot % bs) * hd + u, v);
  }
}

}  // namespace

// qkv: the bf16 projection (q is rotated in place), or with `part` its sums
// (fp32 [parts, T, width], sx and sw for fp8 operands), and q's rows out
void rope_cache(torch::Tensor qkv, torch::Tensor positions,
                torch::Tensor cos_sin, torch::Tensor k_cache,
                torch::Tensor v_cache, torch::Tensor slot_mapping, int64_t n_q,
                c10::optional<torch::Tensor> part,
                c10::optional<torch::Tensor> sx,
                c10::optional<torch::Tensor> sw) {
  TORCH_CHECK(qkv.scalar_type() == torch::kBFloat16 && qkv.dim() == 2 &&
              qkv.stride(1) == 1 && qkv.stride(0) % 8 == 0 &&
              ((uintptr_t)qkv.data_ptr() & 15) == 0);
  TORCH_CHECK(positions.scalar_type() == torch::kInt32);
  TORCH_CHECK(cos_sin.scalar_type() == torch::kFloat32);
  TORCH_CHECK(slot_mapping.scalar_type() == torch::kInt64);
  TORCH_CHECK(k_cache.is_contiguous() && v_cache.is_contiguous());
  TORCH_CHECK(k_cache.scalar_type() == v_cache.scalar_type() &&
              (k_cache.scalar_type() == torch::kBFloat16 ||
               k_cache.scalar_type() == torch::kFloat8_e5m2));
  const int n_kv = k_cache.size(1), bs = k_cache.size(2), hd = k_cache.size(3);
  const int64_t T = qkv.size(0);
  const int width = (int)(n_q + 2 * n_kv) * hd;
  TORCH_CHECK(hd % 16 == 0 && cos_sin.size(1) == hd &&
              v_cache.sizes() == k_cache.sizes() &&
              qkv.size(1) == (part.has_value() ? n_q * hd : width));
  TORCH_CHECK(positions.numel() >= T && slot_mapping.numel() >= T);
  ProductSums p{};
  if (part.has_value()) {
    TORCH_CHECK(part->scalar_type() == torch::kFloat32 && part->is_contiguous() &&
                part->dim() == 3 && part->size(1) == T && part->size(2) == width);
    TORCH_CHECK(sx.has_value() == sw.has_value());
    p = {part->data_ptr<float>(), nullptr, nullptr, (int)part->size(0), T * width,
         width};
    if (sx.has_value()) {
      TORCH_CHECK(sx->scalar_type() == torch::kFloat32 && sx->is_contiguous() &&
                  sx->numel() == T && sw->scalar_type() == torch::kFloat32 &&
                  sw->is_contiguous() && sw->numel() == width);
      p.sx = sx->data_ptr<float>();
      p.sw = sw->data_ptr<float>();
    }
  }
  if (T == 0) return;
  const int64_t items = T * ((n_q + n_kv) * (hd / 16) + n_kv * (hd / 8));
  const dim3 grid((uint32_t)((items + 255) / 256));
  auto go = [&](auto ct, auto sums) {
    using CT = decltype(ct);
    hipLaunchKernelGGL((rope_cache_kernel<CT, decltype(sums)::value>), grid,
                       dim3(256), 0, c10::hip::getCurrentHIPStream().stream(),
                       (ushort*)qkv.data_ptr(), p,
                       positions.data_ptr<int32_t>(),
                       cos_sin.data_ptr<float>(), (CT*)k_cache.data_ptr(),
                       (CT*)v_cache.data_ptr(),
                       slot_mapping.data_ptr<int64_t>(), (int)n_q, n_kv, hd, bs,
                       T, qkv.stride(0));
  };
  auto with_ct = [&](auto sums) {
    if (k_cache.scalar_type() == torch::kBFloat16) go((ushort)0, sums);
    else go((unsigned char)0, sums);
  };
  if (part.has_value()) with_ct(std::true_type{});
  else with_ct(std::false_type{});
  HIP_CHECK_KERNEL();
}

void rope(torch::Tensor q, torch::Tensor k, torch::Tensor positions,
          torch::Tensor cos_sin) {
  // q/k may be row-strided views into the fused qkv projection output
  TORCH_CHECK(q.stride(2) == 1 && q.stride(1) == q.size(2));
  TORCH_CHECK(k.stride(2) == 1 && k.stride(1) == k.size(2));
  TORCH_CHECK(q.scalar_type() == torch::kBFloat16);
  TORCH_CHECK(positions.scalar_type() == torch::kInt32);
  TORCH_CHECK(cos_sin.scalar_type() == torch::kFloat32);
  const int T = q.size(0);
  const int n_q = q.size(1), n_kv = k.size(1), hd = q.size(2);
  TORCH_CHECK(hd % 2 == 0 && cos_sin.size(1) == hd);
  const int64_t total_waves = (int64_t)T * (n_q + n_kv);
  const int waves_per_block = 4;  // 256 threads
  const int64_t blocks = (total_waves + waves_per_block - 1) / waves_per_block;
  // guard tail waves: launch exact multiple; tail handled by tok bound check
  hipLaunchKernelGGL(rope_kernel, dim3((uint32_t)blocks),
                     dim3(waves_per_block * WAVE_SIZE), 0,
                     c10::hip::getCurrentHIPStream().stream(), (ushort*)q.data_ptr(),
                     (ushort*)k.data_ptr(),
                     positions.data_ptr<int32_t>(),
                     cos_sin.data_ptr<float>(), n_q, n_kv, hd, (int64_t)T,
                     q.stride(0), k.stride(0));
  HIP_CHECK_KERNEL();
}
