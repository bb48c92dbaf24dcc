// Common helpers for kubeai_amd gfx950 (CDNA4) kernels.
//
// Conventions (see /opt/skills/guides/cdna_hip_programming.md):
//  - wave = 64 lanes, hard-coded.
//  - bf16 global loads are vectorized as ushort4/ushort8 (hipcc does not
//    auto-vectorize scalar bf16 loads).
//  - fp32 accumulation everywhere.
#pragma once

#include <hip/hip_runtime.h>
#include <hip/hip_bf16.h>
#include <hip/hip_fp16.h>
#include <hip/hip_fp8.h>
#include <stdint.h>
#include <c10/hip/HIPStream.h>

#define WAVE_SIZE 64
#define DEV_INLINE __device__ __forceinline__

typedef __hip_bfloat16 bf16_t;

// 16-byte vector of 8 bf16 values (one coalesced lane-load).
typedef ushort __attribute__((ext_vector_type(8))) ushort8;
typedef ushort __attribute__((ext_vector_type(4))) ushort4_t;
typedef float __attribute__((ext_vector_type(4))) float4_t;

DEV_INLINE float bf16_to_f32(ushort u) {
  union {
    uint32_t i;
    float f;
  } c;
  c.i = ((uint32_t)u) << 16;
  return c.f;
}

DEV_INLINE ushort f32_to_bf16(float f) {
  // round-to-nearest-even, matching PyTorch's bf16 cast
  union {
    float f;
    uint32_t i;
  } c;
  c.f = f;
  uint32_t x = c.i;
  uint32_t rb = ((x >> 16) & 1u) + 0x7fffu;
  x += rb;
  return (ushort)(x >> 16);
}

// ---------------- fp8 e5m2 KV-cache element (OCP bf8) ----------------
// e5m2 [s eeeee mm] -> f32 by bit widening: bias 15 -> 127. Matches
// torch.float8_e5m2 exactly incl. subnormals/inf/nan (pure exponent
// remap; subnormals handled by normalizing the 2-bit mantissa).

DEV_INLINE float e5m2_to_f32(unsigned char b) {
  const uint32_t s = ((uint32_t)b & 0x80u) << 24;
  uint32_t e = (b >> 2) & 0x1fu;
  uint32_t m = b & 0x3u;
  uint32_t out;
  if (e == 0) {
    if (m == 0) {
      out = s;  // +-0
    } else {
      // subnormal: value = m * 2^-16; normalize
      int shift = (m & 2u) ? 0 : 1;  // m=2,3 -> msb at bit1; m=1 -> bit0
      e = 127 - 15 + 1 - 1 - shift;  // 2^-15 / 2^-16
      m = (m << (shift + 1)) & 0x3u;  // drop the implicit leading 1
      out = s | (e << 23) | (m << 21);
    }
  } else if (e == 0x1fu) {
    out = s | 0x7f800000u | (m << 21);  // inf / nan
  } else {
    out = s | ((e - 15u + 127u) << 23) | (m << 21);
  }
  union { uint32_t i; float f; } c;
  c.i = out;
  return c.f;
}

// 8 packed e5m2 bytes -> 8 bf16 values (one staging unit).
//
// Route: e5m2 is bit-identical to the TOP BYTE of an IEEE fp16, so
// fp16 = byte<<8 (pure integer move); fp16 -> f32 is one hardware cvt;
// f32 -> bf16 truncates losslessly (every e5m2 value, subnormals and
// inf/nan included, is exactly representable in bf16).
//
// Deliberately NOT via __builtin_amdgcn_cvt_pk_f32_bf8 + bit-level
// truncation: this toolchain mis-simplifies bit manipulation of that
// intrinsic's result (low mantissa bit folded to zero — 129/256 byte
// values corrupt, device-verified in scripts/dbg_cvt.hip; an opaque
// asm barrier does not stop it).
DEV_INLINE ushort8 e5m2x8_to_bf16x8(uint64_t raw) {
  ushort8 out;
#pragma unroll
  for (int j = 0; j < 8; ++j) {
    const ushort h = (ushort)((raw >> (8 * j)) << 8);
    const float f = __half2float(__builtin_bit_cast(__half, h));
    out[j] = (ushort)(__builtin_bit_cast(uint32_t, f) >> 16);
  }
  return out;
}

DEV_INLINE unsigned char f32_to_e5m2(float x) {
  // RNE with saturation to max finite (K/V magnitudes stay far below
  // e5m2's 57344 ceiling in practice)
  return (unsigned char)__hip_cvt_float_to_fp8(x, __HIP_SATFINITE, __HIP_E5M2);
}

constexpr float kLog2e = 1.4426950408889634f;

// cap * tanh(x / cap) of attention scores. With u = (x / cap)^2, where it is
// less than 0.49: x (1 + u q(u)), q fitted to (tanh(y) / y - 1) / y^2 for the
// least largest error (6.3e-10 of the result; the rounding of u counts only in
// the correction). Beyond: cap - 2 cap / (1 + 2^z), z = 2 log2(e) x / cap, with the
// rounding of z brought back into the power. Against 64 bits, largest and mean
// error at a cap of 50: 1.8e-6 and 3.4e-7 below, 4.1e-6 and 9.6e-7 above, where
// the library's tanh has 5.8e-6, 5.7e-7, 5.8e-6 and 1.2e-6. (That one beyond
// the edge costs prompt attention registers: 3029 + 2145, heads 8/4 x 256, scores of
// standard deviation 1, 10 and 32: 284, 368, 415 us, this 268, 280, 316; heads 8/4 x
// 128, 0.7, 7 and 23: 172, 236, 306, this 115, 115, 159. An exponential and reciprocal
// without corrections, 1.3e-5 off: 258 and 124 whatever the scores.)
struct SoftCap {
  float cap, inv, edge, k, k_lo;

  // nothing but the edge is used where there is no cap
  DEV_INLINE explicit SoftCap(float c)
      : cap(c), inv(scalar(1.0f / c)), edge(scalar(0.7f * c)) {
    constexpr double both = 2.0 * 1.4426950408889634;
    constexpr float hi = (float)both, lo = (float)(both - (double)hi);
    k = scalar(hi * inv);
    k_lo = scalar((fmaf(-k, c, hi) + lo) * inv);
  }
  // the same in every lane: kept in a scalar register
  DEV_INLINE static float scalar(float v) {
    return __uint_as_float(__builtin_amdgcn_readfirstlane(__float_as_uint(v)));
  }
  DEV_INLINE float small(float x) const {
    const float y = x * inv, u = y * y;
    float q = fmaf(u, 0.001901791315f, -0.007892170921f);
    q = fmaf(u, q, 0.02157583274f);
    q = fmaf(u, q, -0.05392212048f);
    q = fmaf(u, q, 0.1333299577f);
    q = fmaf(u, q, -0.3333332539f);
    return fmaf(x * u, q, x);
  }
  DEV_INLINE float large(float x) const {
    const float ax = fminf(fabsf(x), 20.f * cap);  // there 2^z is e^40
    const float z = ax * k;
    const float rest = fmaf(ax, k_lo, fmaf(ax, k, -z));
    float e = __builtin_amdgcn_exp2f(z);
    e = fmaf(e, rest * 0.6931471806f, e);
    const float r = __builtin_amdgcn_rcpf(1.0f + e);
    return __builtin_copysignf(fmaf(-2.0f * cap, r, cap), x);
  }
  // A wave's scores, times scale, capped. The second form is passed over where
  // no lane needs it; what a value becomes does not depend on the others. NaN
  // stays NaN (no comparison with it holds).
  template <typename V, int M>
  DEV_INLINE void apply(V (&s)[M], float scale) const {
    constexpr int n = sizeof(V) / sizeof(float);
    float amax = 0.f;
#pragma unroll
    for (int m = 0; m < M; ++m)
#pragma unroll
      for (int i = 0; i < n; ++i) {
        s[m][i] *= scale;
        amax = fmaxf(amax, fabsf(s[m][i]));
      }
    V t[M];
#pragma unroll
    for (int m = 0; m < M; ++m)
#pragma unroll
      for (int i = 0; i < n; ++i) t[m][i] = small(s[m][i]);
    if (__builtin_expect(__any(amax >= edge), 0)) {
#pragma unroll
      for (int m = 0; m < M; ++m)
#pragma unroll
        for (int i = 0; i < n; ++i) {
          float l = large(s[m][i]);
          asm volatile("" : "+v"(l));  // a selection, not a branch per value
          t[m][i] = fabsf(s[m][i]) >= edge ? l : t[m][i];
        }
    }
#pragma unroll
    for (int m = 0; m < M; ++m) s[m] = t[m];
  }
};

// The result of a matrix product that was cut along K: fp32 sums of every
// part, [parts, M, N], to be added, scaled (fp8 operands) and rounded to bf16
// by whoever reads it.
struct ProductSums {
  const float* part;
  const float* sx;  // per row, or null
  const float* sw;  // per column
  int parts;
  int64_t stride;   // M * N
  int N;
};

// The scales of N times 8 neighbouring columns n[i].. of row m, asked for before the
// parts: loads in any case (of something else without sx, and not used then), since
// a load under a branch is waited for by itself.
template <int N>
struct SumScales {
  float sx, sw[N][8];
  DEV_INLINE SumScales(const ProductSums& p, int64_t m, const int (&n)[N]) {
    const float* rows = p.sx ? p.sx + m : p.part;
    const float* cols = p.sx ? p.sw : p.part;
    sx = *rows;
#pragma unroll
    for (int i = 0; i < N; ++i)
#pragma unroll
      for (int j = 0; j < 8; ++j) sw[i][j] = cols[n[i] + j];
  }
};

// Sum of PARTS parts of N times 8 neighbouring columns; every load is issued before
// the first addition (a chain of eight would cost eight latencies).
template <int PARTS, int N>
DEV_INLINE void add_parts8(const float* const (&a)[N], int64_t first, int64_t stride,
                           float4_t (&v)[N][2]) {
  float4_t t[PARTS][N][2];
#pragma unroll
  for (int s = 0; s < PARTS; ++s)
#pragma unroll
    for (int i = 0; i < N; ++i) {
      const float4_t* b = reinterpret_cast<const float4_t*>(a[i] + (first + s) * stride);
      t[s][i][0] = b[0];
      t[s][i][1] = b[1];
    }
#pragma unroll
  for (int s = 0; s < PARTS; ++s)
#pragma unroll
    for (int i = 0; i < N; ++i) {
      v[i][0] += t[s][i][0];
      v[i][1] += t[s][i][1];
    }
}

// N times 8 neighbouring columns n[i].. of row m, as the bf16 values a stored product
// would have (the parts are added in order, whatever their number; what is left of
// the eights at once too: 7 parts one by one cost four latencies)
template <int N>
DEV_INLINE void read_sums8(const ProductSums& p, int64_t m, const int (&n)[N],
                           const SumScales<N>& by, ushort8 (&o)[N]) {
  const float* a[N];
  float4_t v[N][2];
#pragma unroll
  for (int i = 0; i < N; ++i) {
    a[i] = p.part + m * p.N + n[i];
    v[i][0] = v[i][1] = float4_t{0.f, 0.f, 0.f, 0.f};
  }
  // (16 at once are more than the compiler gives registers to)
  constexpr int kAtOnce = N > 1 ? 4 : 8;
  int s = 0;
  for (; s + kAtOnce <= p.parts; s += kAtOnce) add_parts8<kAtOnce>(a, s, p.stride, v);
  switch (p.parts - s) {
    case 1: add_parts8<1>(a, s, p.stride, v); break;
    case 2: add_parts8<2>(a, s, p.stride, v); break;
    case 3: add_parts8<3>(a, s, p.stride, v); break;
    case 4: add_parts8<4>(a, s, p.stride, v); break;
    case 5: add_parts8<5>(a, s, p.stride, v); break;
    case 6: add_parts8<6>(a, s, p.stride, v); break;
    case 7: add_parts8<7>(a, s, p.stride, v); break;
  }
#pragma unroll
  for (int i = 0; i < N; ++i)
#pragma unroll
    for (int j = 0; j < 8; ++j) {
      float f = v[i][j / 4][j % 4];
      if (p.sx) f = f * by.sx * by.sw[i][j];
      o[i][j] = f32_to_bf16(f);
    }
}

// ---------------- wave reductions (64-wide) ----------------

DEV_INLINE float wave_reduce_sum(float v) {
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) v += __shfl_xor(v, off, 64);
  return v;
}

DEV_INLINE float wave_reduce_max(float v) {
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) v = fmaxf(v, __shfl_xor(v, off, 64));
  return v;
}

// Block-level sum reduce across up to 16 waves; `smem` must hold >= 16 floats.
// Every thread returns the total.
DEV_INLINE float block_reduce_sum(float v, float* smem) {
  const int wave = threadIdx.x / WAVE_SIZE;
  const int lane = threadIdx.x % WAVE_SIZE;
  const int n_waves = (blockDim.x + WAVE_SIZE - 1) / WAVE_SIZE;
  v = wave_reduce_sum(v);
  if (lane == 0) smem[wave] = v;
  __syncthreads();
  float total = 0.f;
#pragma unroll
  for (int w = 0; w < 16; ++w)
    if (w < n_waves) total += smem[w];
  return total;
}

// ---------------- hash RNG (kernel/ref-identical spec) ----------------
//
// Sampling uses a counter-based hash RNG so the HIP kernel and the PyTorch
// reference produce bit-identical streams: u64 = splitmix64(key*M ^ idx).
DEV_INLINE uint64_t splitmix64(uint64_t z) {
  z += 0x9e3779b97f4a7c15ull;
  z = (z ^ (z >> 30)) * 0xbf58476d1ce4e5b9ull;
  z = (z ^ (z >> 27)) * 0x94d049bb133111ebull;
  return z ^ (z >> 31);
}

// uniform in (0, 1]
DEV_INLINE float hash_uniform(uint64_t key, uint64_t idx) {
  uint64_t h = splitmix64(key ^ (idx * 0xd1342543de82ef95ull));
  // take top 24 bits -> (0,1] to keep -log well-defined
  uint32_t m = (uint32_t)(h >> 40);
  return ((float)m + 1.0f) * (1.0f / 16777216.0f);
}

#define HIP_CHECK_KERNEL()                                    \
  do {                                                        \
    hipError_t e = hipGetLastError();                         \
    if (e != hipSuccess) {                                    \
      TORCH_CHECK(false, "HIP kernel launch failed: ",        \
                  hipGetErrorString(e));                      \
    }                                                         \
  } while (0)
