// Weight-streaming products for few rows: y[M,N] = x[M,K] W[N,K]^T with
// M <= 96, bf16 or fp8 e4m3 (W8A8 with row and column scales), bf16 out,
// fp32 accumulation. Decode batches and the logits of a step's last tokens.
//
// Bound by reading W once. What it takes to read it at the card's rate:
//  - workgroup = 4 waves x 16 rows of W. A wave's lanes read 16 rows x 64
//    contiguous bytes straight into matrix operands (no LDS for W: each byte
//    is used by one wave); two of those loads fill a 128-byte line. The next
//    256 (M <= 32: 512) bytes of every row are in flight while the current
//    ones are multiplied.
//  - x is what the CUs would re-read: with 16 rows of W per workgroup its
//    traffic is M / 16 that of W, and past M = 16 that limits (40 rows fp8:
//    54 us for 28672 x 4096 against 28 with x shared by 64 rows). It is
//    staged through LDS (double-buffered, one barrier a step, 16-byte units
//    XOR-swizzled by row) and shared by the four waves.
//  - few output columns do not fill the chip: K is cut into up to 8 parts
//    (blockIdx.y), whose fp32 sums lie in a workspace [parts, M, N]; a second
//    kernel adds them (no atomics: the order of the sum is fixed).
// With N columns there are N / 64 workgroups; below 256 of them K is cut so
// that about 768 result (N = 6144, 40 rows fp8: 8.8 us with 768, 9.7 with
// 384); from 256 on the second pass costs more than the parts give (28672:
// 28.2 us whole, 29.8 in two parts).
// Where a consumer can add the parts itself (skinny_sums; the norm after an
// attention or feed-forward block, the rotation of q and k) that second pass,
// about 5 us of launch and drain, is gone.
// Measured in the decode step, W out of cache, us (library product + what
// reads it -> this + that):
//   fp8, 40 rows  4096 -> 6144 and rotation   13.5 + 4.9 ->  9.6 + 6.9
//                 14336 -> 4096 and norm      23.0 + 5.1 -> 16.4 + 7.4
//                 4096 -> 4096 and norm       11.8 + 5.1 ->  8.0 + 7.4
//   bf16, 8 rows  4096 -> 6144 and rotation   15.5 + 4.9 -> 12.1 + 4.8
//                 14336 -> 4096 and norm      25.6 + 5.2 -> 23.0 + 4.8
//                 4096 -> 28672               62.9       -> 49.6 (4.7 TB/s)
//   bf16, 96 rows 14336 -> 4096 and norm      54.1 + 5.5 -> 36.0 + 5.8
// The grouped form multiplies every expert's rows of a mixture in one launch,
// x rows gathered by index. 8 experts of 4096 x 14336, 40 tokens of 2 experts
// each, both products with routing and activation: fp8 297 us (4.8 TB/s over
// the weights), 542 with a library product per expert; bf16 561 and 822.
#include <torch/extension.h>

#include <type_traits>

#include "common.h"

namespace {

constexpr int kNW = 4;         // waves per workgroup
constexpr int kMaxRows = 96;
constexpr int kMaxParts = 8;

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

// MT: 16-row tiles of x. part != null: raw sums of this K range.
// GROUPED: blockIdx.z is the expert; its rows are taken MT * 16 at a time (W
// is read again for each such pass: the host picks MT so that one is usual).
template <bool FP8, int MT, bool GROUPED>
__launch_bounds__(kNW * WAVE_SIZE) __global__ void skinny_kernel(
    ushort* __restrict__ y,         // [M, N]
    float* __restrict__ part,       // [parts, M, N]
    const char* __restrict__ x,     // M rows of KB bytes, ldx apart
    const char* __restrict__ w,     // N rows of KB bytes
    const float* __restrict__ sx, const float* __restrict__ sw,
    const ushort* __restrict__ bias, const int M_all, const int N, const int KB,
    const int64_t ldx, const int k_part, const Groups grp) {
  constexpr int KC = MT <= 2 ? 512 : 256;  // bytes of K per step
  constexpr int CH = KC / 64;
  constexpr int UPR = KC / 16;
  constexpr int XU = MT * 16 * UPR;
  constexpr int NX = XU / (kNW * WAVE_SIZE);  // staged units per thread
  static_assert(XU % (kNW * WAVE_SIZE) == 0, "whole units per thread");
  __shared__ __attribute__((aligned(16))) char xs[2][MT * 16 * KC];

  const int wave = threadIdx.x / WAVE_SIZE, lane = threadIdx.x % WAVE_SIZE;
  const int r = lane & 15, kg = lane >> 4;
  const int n0 = (blockIdx.x * kNW + wave) * 16;
  const int k0 = blockIdx.y * k_part, k1 = min(KB, k0 + k_part);
  const int steps = (k1 - k0 + KC - 1) / KC;
  int m0 = 0, M = M_all;  // this pass's first row and the rows from it on
  int m_end = M_all;
  if constexpr (GROUPED) {
    m0 = grp.begin[blockIdx.z];
    m_end = grp.begin[blockIdx.z + 1];
    w += (int64_t)blockIdx.z * N * KB;
    if (sw) sw += (int64_t)blockIdx.z * N;
    M = m_end - m0;
    if (M <= 0) return;  // whole workgroup
  }
  const char* wp = w + (int64_t)min(n0 + r, N - 1) * KB + kg * 16;

  f32x4 acc[MT];
  i32x4 wf[2][CH], xr[NX];
  int64_t x_off[NX];  // of the staged units' rows

  // loads past the end of the range read its last bytes again; their
  // products are skipped
  auto load_w = [&](int b, int s) {
#pragma unroll
    for (int c = 0; c < CH; ++c)
      wf[b][c] = *reinterpret_cast<const i32x4*>(
          wp + min(k0 + s * KC + c * 64, k1 - 64));
  };
  auto load_x = [&](int s) {
#pragma unroll
    for (int i = 0; i < NX; ++i) {
      const int u = threadIdx.x + i * kNW * WAVE_SIZE;
      xr[i] = *reinterpret_cast<const i32x4*>(
          x + x_off[i] + min(k0 + s * KC + u % UPR * 16, k1 - 16));
    }
  };
  auto put_x = [&](int b) {
#pragma unroll
    for (int i = 0; i < NX; ++i) {
      const int u = threadIdx.x + i * kNW * WAVE_SIZE;
      const int row = u / UPR;
      *reinterpret_cast<i32x4*>(
          &xs[b][row * KC + (((u % UPR) ^ (row & 7)) << 4)]) = xr[i];
    }
  };
  auto multiply = [&](int b, int s) {
#pragma unroll
    for (int c = 0; c < CH; ++c)
      if (k0 + s * KC + c * 64 < k1)
#pragma unroll
        for (int j = 0; j < MT; ++j) {
          if (GROUPED && j * 16 >= M) break;  // the same in every lane
          const i32x4 xf = *reinterpret_cast<const i32x4*>(
              &xs[b][(j * 16 + r) * KC + (((c * 4 + kg) ^ (r & 7)) << 4)]);
          acc[j] = mfma_64b<FP8>(wf[b][c], xf, acc[j]);
        }
  };

  do {
#pragma unroll
    for (int j = 0; j < MT; ++j) acc[j] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int i = 0; i < NX; ++i) {
      int row = min((threadIdx.x + i * kNW * WAVE_SIZE) / UPR, (unsigned)M - 1);
      if constexpr (GROUPED) {
        row += m0;
        if (grp.src) row = grp.src[row];
      }
      x_off[i] = (int64_t)row * ldx;
    }
    load_x(0);
    load_w(0, 0);
    put_x(0);
    if (steps > 1) load_x(1);
    __syncthreads();
    for (int s = 0; s < steps; s += 2) {
      if (s + 1 < steps) {
        load_w(1, s + 1);
        put_x(1);
        if (s + 2 < steps) load_x(s + 2);
      }
      multiply(0, s);
      __syncthreads();
      if (s + 1 < steps) {
        if (s + 2 < steps) {
          load_w(0, s + 2);
          put_x(0);
          if (s + 3 < steps) load_x(s + 3);
        }
        multiply(1, s + 1);
        __syncthreads();
      }
    }

    // accumulator: row (W) 4 kg + e, column (x) r
    const int n = n0 + kg * 4;
    if (n < N) {  // N is a multiple of 4
#pragma unroll
      for (int j = 0; j < MT; ++j) {
        const int m = j * 16 + r;
        if (m >= M) continue;
        if (part)
          *reinterpret_cast<f32x4*>(
              part + ((int64_t)blockIdx.y * M_all + m) * N + n) = acc[j];
        else
          store4(y + (int64_t)(m0 + m) * N + n, acc[j], sx, sw, bias,
                 GROUPED && grp.src ? grp.src[m0 + m] : m0 + m, n);
      }
    }
    if constexpr (GROUPED) {
      m0 += MT * 16;
      M = m_end - m0;
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
  TORCH_CHECK(s.KB >= 64 && s.KB % 64 == 0 && s.N % 4 == 0 &&
              (int64_t)s.M * s.N < (1ll << 31));
  TORCH_CHECK(x.stride(0) * es % 16 == 0 && x.stride(0) >= x.size(1) &&
              ((uintptr_t)x.data_ptr() & 15) == 0 &&
              ((uintptr_t)w.data_ptr() & 15) == 0,
              "16-byte aligned rows");
  TORCH_CHECK(raw || fp8 == (sx.has_value() && sw.has_value()),
              "fp8 operands come with their scales, bf16 ones without");
  if (fp8 && !raw) {
    TORCH_CHECK(sx->scalar_type() == torch::kFloat32 && sx->is_contiguous() &&
                sx->numel() == s.M && sw->scalar_type() == torch::kFloat32 &&
                sw->is_contiguous() && sw->numel() == s.N);
  }
  if (bias.has_value())
    TORCH_CHECK(bias->scalar_type() == torch::kBFloat16 &&
                bias->is_contiguous() && bias->numel() == s.N);
  return s;
}

void launch(ushort* y, float* part, const torch::Tensor& x,
            const torch::Tensor& w, const float* sx, const float* sw,
            const ushort* bias, const Shape& s, const Cut& cut) {
  const dim3 grid((s.N + kNW * 16 - 1) / (kNW * 16), cut.parts);
  const int64_t ldx = x.stride(0) * x.element_size();
  auto stream = c10::hip::getCurrentHIPStream().stream();
  auto go = [&](auto fp8, auto mt) {
    hipLaunchKernelGGL((skinny_kernel<decltype(fp8)::value, decltype(mt)::value, false>),
                       grid, dim3(kNW * WAVE_SIZE), 0, stream, y, part,
                       (const char*)x.data_ptr(), (const char*)w.data_ptr(),
                       sx, sw, bias, s.M, s.N, s.KB, ldx, cut.k_part, Groups{});
  };
  auto tiles = [&](auto fp8) {
    switch ((s.M + 15) / 16) {
      case 1: go(fp8, std::integral_constant<int, 1>{}); break;
      case 2: go(fp8, std::integral_constant<int, 2>{}); break;
      case 3: go(fp8, std::integral_constant<int, 3>{}); break;
      case 4: go(fp8, std::integral_constant<int, 4>{}); break;
      case 5: go(fp8, std::integral_constant<int, 5>{}); break;
      default: go(fp8, std::integral_constant<int, 6>{}); break;
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
  const Shape s = check(x, w, none, none, none, true);
  const Cut cut = cut_for(s.N, s.KB);
  auto part = torch::empty({cut.parts, s.M, s.N}, x.options().dtype(torch::kFloat32));
  launch(nullptr, part.data_ptr<float>(), x, w, nullptr, nullptr, nullptr, s, cut);
  return part;
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
  TORCH_CHECK(KB >= 64 && KB % 64 == 0 && N % 4 == 0 && E >= 1 && E <= 65535);
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
                sx->numel() == x.size(0) &&
                sw->scalar_type() == torch::kFloat32 && sw->is_contiguous() &&
                sw->numel() == (int64_t)E * N);
  }
  const int R = y.size(0);
  if (R == 0) return;
  const float* sxp = fp8 ? sx->data_ptr<float>() : nullptr;
  const float* swp = fp8 ? sw->data_ptr<float>() : nullptr;
  const Groups g{begin.data_ptr<int32_t>(),
                 src.has_value() ? src->data_ptr<int32_t>() : nullptr};
  const dim3 grid((N + kNW * 16 - 1) / (kNW * 16), 1, E);
  const int64_t ldx = x.stride(0) * es;
  auto stream = c10::hip::getCurrentHIPStream().stream();
  auto go = [&](auto f, auto mt) {
    hipLaunchKernelGGL((skinny_kernel<decltype(f)::value, decltype(mt)::value, true>),
                       grid, dim3(kNW * WAVE_SIZE), 0, stream,
                       (ushort*)y.data_ptr(), nullptr, (const char*)x.data_ptr(),
                       (const char*)w.data_ptr(), sxp, swp, nullptr, R, N, KB,
                       ldx, KB, g);
  };
  // rows per expert if they are spread evenly; half as many again fit a pass
  const int mean = (R + E - 1) / E;
  auto tiles = [&](auto f) {
    if (mean <= 8) go(f, std::integral_constant<int, 1>{});
    else if (mean <= 22) go(f, std::integral_constant<int, 2>{});
    else if (mean <= 44) go(f, std::integral_constant<int, 4>{});
    else go(f, std::integral_constant<int, 6>{});
  };
  if (fp8) tiles(std::true_type{});
  else tiles(std::false_type{});
  HIP_CHECK_KERNEL();
}

void skinny_gemm(torch::Tensor y, torch::Tensor x, torch::Tensor w) {
  skinny_linear(y, x, w, c10::nullopt, c10::nullopt, c10::nullopt);
}
