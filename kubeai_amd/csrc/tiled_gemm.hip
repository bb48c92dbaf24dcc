// What the tiled products (tiled_gemm.h) are given: checks, the tile shape, the
// parts of K.
#include <torch/extension.h>

#include <cmath>

#include "tiled_gemm.h"

namespace tiled {
namespace {

// A launch takes passes over the CUs x (steps x step + tile) + rest us, and mb us
// for each MB of sums. One matrix: fitted to 225 products of each shape and type (40
// to 8192 rows, 1024 to 32000 columns, K 512 to 14336, weights out of cache), 8 to 15 %
// off in the mean; the shape with the least is 0.1 % slower than the best one in
// the mean, 15 % at worst. Sums: the same products in 1 to 8 parts; what reads
// them adds their bytes at 4.5 TB/s (0.9 %, 20 %). Experts cost what one matrix does:
// over 578 mixtures (2 to 64 experts, 256 to 30000 columns, K 256 to 14336, 1 to 5000
// rows each, evenly and not) the shape chosen is 4 % slower than the best one in the
// mean, 14 % in nine of ten. Costs of their own, fitted to 8 large experts with even
// rows, were right for those alone (17 % in the mean): 8 of 4096 x 2560, 4176 rows, fp8
// 81 us, now 60; 64 of 1280 x 512, 636 rows 23.3, now 16.6.
struct Cost {
  float step, tile, rest, mb;
};
constexpr Cost kOne[2][kNarrow] = {
    {{1.083f, 8.7f, 0.f}, {0.869f, 6.7f, 0.f}, {0.878f, 7.1f, 0.f}, {0.724f, 5.5f, 0.f},
     {0.752f, 4.1f, 0.f}, {0.577f, 3.7f, 0.f}, {0.484f, 2.6f, 0.f}, {0.357f, 1.3f, 1.1f}},
    {{1.058f, 10.8f, 0.f}, {0.874f, 9.1f, 0.f}, {0.877f, 10.9f, 0.f}, {0.710f, 9.0f, 0.f},
     {0.676f, 6.7f, 0.f}, {0.518f, 5.6f, 0.f}, {0.404f, 4.4f, 0.f}, {0.292f, 2.5f, 1.2f}}};
constexpr Cost kParts[2][kNarrow] = {
    {{1.081f, 2.5f, 5.2f, 0.21f}, {0.857f, 0.8f, 5.3f, 0.25f}, {0.869f, 1.3f, 5.1f, 0.23f},
     {0.701f, 1.0f, 4.3f, 0.25f}, {0.742f, 0.f, 4.4f, 0.27f},  {0.568f, 0.6f, 3.3f, 0.28f},
     {0.480f, 0.4f, 2.6f, 0.31f}, {0.365f, 1.0f, 1.9f, 0.27f}},
    {{1.036f, 2.7f, 5.4f, 0.20f}, {0.835f, 1.5f, 5.5f, 0.23f}, {0.852f, 2.7f, 4.5f, 0.20f},
     {0.662f, 2.3f, 4.0f, 0.22f}, {0.660f, 0.8f, 4.6f, 0.24f}, {0.475f, 0.7f, 3.7f, 0.27f},
     {0.379f, 0.9f, 3.1f, 0.28f}, {0.277f, 1.2f, 2.3f, 0.28f}}};
constexpr double kReadMb = 1. / 4.5;
constexpr int kMaxParts = 8;

struct Plan {
  int shape, parts;
  double us;
};

// R rows of E experts against cols columns of the result (halves: a tile has
// half as many)
Plan plan(bool fp8, int64_t R, int64_t E, int64_t cols, int64_t KB, bool halves, bool sums) {
  Plan best{-1, 1, 0.};
  for (int i = 0; i < kNarrow; i++) {
    const Shape s = kShapes[i];
    if (halves && s.wn % 2) continue;
    const Cost c = (sums ? kParts : kOne)[fp8][i];
    const int64_t bn = s.cols() / (halves ? 2 : 1), nt = (cols + bn - 1) / bn;
    double row_tiles = (R + s.rows() - 1) / s.rows();
    if (E > 1) {  // the mean over row counts within 30 % of an even split
      row_tiles = 0.;
      for (int k = -3; k <= 3; k++) {
        row_tiles += std::ceil((double)R / E * (1. + 0.1 * k) / s.rows()) * E / 7.;
      }
    }
    for (int parts = 1; parts <= (sums ? kMaxParts : 1); parts++) {
      const int64_t all = KB / kStep, steps = (all + parts - 1) / parts;
      if (parts > 1 && (steps < 4 || (all + steps - 1) / steps != parts)) continue;
      const double full = row_tiles * nt * parts / 256;
      double passes = std::ceil(full);
      if (E > 1) {  // a few tiles more may begin another pass
        passes = 0.;
        for (int k = -2; k <= 2; k++) passes += std::ceil(full * (1. + 0.05 * k)) / 5.;
      }
      const double us = passes * (steps * c.step + c.tile) + c.rest +
                        (sums ? parts * R * cols * 4e-6 * (c.mb + kReadMb) : 0.);
      if (best.shape < 0 || us < best.us) best = {i, parts, us};
    }
  }
  return best;
}

struct Operands {
  bool fp8;
  torch::Tensor x, w;  // x [*, K], w [E, N, K]
  Args a;
};

// Offsets within a tile are 32 bits: rows under 8 MB apart (others are copied).
torch::Tensor near_rows(const torch::Tensor& t) {
  const int64_t es = t.element_size(), far = (int64_t)1 << 23;
  const int d = t.dim() - 2;
  return t.stride(d) * es < far ? t : t.contiguous();
}

Operands operands(const torch::Tensor& x0, const torch::Tensor& w0,
                  const c10::optional<torch::Tensor>& sx,
                  const c10::optional<torch::Tensor>& sw, bool raw) {
  const bool fp8 = w0.scalar_type() == torch::kFloat8_e4m3fn;
  TORCH_CHECK(fp8 || w0.scalar_type() == torch::kBFloat16);
  TORCH_CHECK(x0.scalar_type() == w0.scalar_type() && x0.is_cuda() && w0.is_cuda());
  TORCH_CHECK(x0.dim() == 2 && w0.dim() == 3 && x0.size(1) == w0.size(2));
  TORCH_CHECK(x0.stride(1) == 1 && w0.stride(2) == 1);
  Operands o{fp8, near_rows(x0), near_rows(w0), {}};
  const auto &x = o.x, &w = o.w;
  const int es = fp8 ? 1 : 2;
  const int64_t E = w.size(0), N = w.size(1), KB = w.size(2) * es;
  const int64_t ldx = x.stride(0) * es, ldw = w.stride(1) * es, ew = w.stride(0) * es;
  TORCH_CHECK(KB >= kStep && KB % kStep == 0 && KB < (int64_t)1 << 23);
  TORCH_CHECK(N >= 4 && N % 4 == 0 && N < (int64_t)1 << 30 && E >= 1 && E < 65536);
  TORCH_CHECK((x.size(0) < 2 || ldx >= KB) && ldx % 16 == 0 && ldw >= KB && ldw % 16 == 0 &&
                  ew >= 0 && ew % 16 == 0 && ((uintptr_t)x.data_ptr() & 15) == 0 &&
                  ((uintptr_t)w.data_ptr() & 15) == 0,
              "16-byte aligned rows");
  TORCH_CHECK(raw || fp8 == (sx.has_value() && sw.has_value()));
  Args& a = o.a;
  if (fp8 && !raw) {
    TORCH_CHECK(sx->scalar_type() == torch::kFloat32 && sx->is_contiguous() &&
                sx->is_cuda() && sx->numel() == x.size(0) &&
                sw->scalar_type() == torch::kFloat32 && sw->is_contiguous() &&
                sw->is_cuda() && sw->numel() == E * N &&
                ((uintptr_t)sw->data_ptr() & 15) == 0);
    a.sx = sx->data_ptr<float>();
    a.sw = sw->data_ptr<float>();
  }
  a.x = (const char*)x.data_ptr();
  a.w = (const char*)w.data_ptr();
  a.E = (int)E;
  a.N = (int)N;
  a.KB = a.k_part = (int)KB;
  a.ldx = ldx;
  a.ldw = ldw;
  a.ew = ew;
  return o;
}

void check_result(const torch::Tensor& y, int64_t cols, Args& a) {
  TORCH_CHECK(y.scalar_type() == torch::kBFloat16 && y.is_contiguous() && y.is_cuda() &&
              y.dim() == 2 && y.size(1) == cols && y.size(0) < (int64_t)1 << 30);
  a.R = (int)y.size(0);
  a.y = (ushort*)y.data_ptr();
  a.wide = cols % 8 == 0 && ((uintptr_t)y.data_ptr() & 15) == 0;
}

Epilogue epilogue_of(int64_t act, const Operands& o) {
  TORCH_CHECK(act >= 0 && act <= 2, "0: none, 1: silu, 2: gelu");
  if (act == 0) return kRows;
  TORCH_CHECK(o.a.N % 16 == 0 && o.a.N * o.a.ldw < (int64_t)1 << 31, "gate and up columns");
  TORCH_CHECK(!o.fp8, "activations: bf16");
  return act == 1 ? kSilu : kGelu;
}

void run(const Operands& o, Epilogue epi, int shape, int64_t grid) {
  TORCH_CHECK(grid < (int64_t)1 << 30);
  if (o.fp8) launch_fp8(shape, epi, o.a, (int)grid);
  else launch_bf16(shape, epi, o.a, (int)grid);
}

}  // namespace
}  // namespace tiled

using namespace tiled;

// y [R, N] = rows of x [*, K] times w[e]^T, w [E, N, K] with any strides of e
// and n; bounds int32: E row counts or E + 1 offsets; src int32 [R] the rows
// of x, or none; fp8: sx fp32 [rows of x], sw fp32 [E, N]; square fp32 [R]:
// y = relu(product)^2 * square. act 1 or 2: y [R, N / 2] = silu or tanh-gelu of the
// first N / 2 columns times the others.
void grouped_linear(torch::Tensor y, torch::Tensor x, torch::Tensor w,
                    c10::optional<torch::Tensor> sx,
                    c10::optional<torch::Tensor> sw, torch::Tensor bounds,
                    c10::optional<torch::Tensor> src,
                    c10::optional<torch::Tensor> square, int64_t act) {
  const int64_t R = y.size(0);
  if (src.has_value()) {
    TORCH_CHECK(src->scalar_type() == torch::kInt32 && src->is_contiguous() &&
                src->is_cuda() && src->numel() == R);
    if (x.dim() == 2 && x.size(0) * x.stride(0) * x.element_size() >= (int64_t)1 << 31) {
      // offsets of gathered rows are 32 bits
      if (sx.has_value()) sx = sx->reshape(-1).index_select(0, *src);
      x = x.view(torch::kUInt8).index_select(0, *src).view(x.scalar_type());
      src = c10::nullopt;
    }
  }
  Operands o = operands(x, w, sx, sw, false);
  Args& a = o.a;
  const int64_t E = a.E;
  TORCH_CHECK(bounds.scalar_type() == torch::kInt32 && bounds.is_contiguous() &&
              bounds.is_cuda() && (bounds.numel() == E || bounds.numel() == E + 1));
  Epilogue epi = epilogue_of(act, o);
  const int64_t cols = act ? a.N / 2 : a.N;
  check_result(y, cols, a);
  if (!src.has_value()) TORCH_CHECK(o.x.size(0) == R);
  if (square.has_value()) {
    TORCH_CHECK(!o.fp8 && act == 0 && square->scalar_type() == torch::kFloat32 &&
                square->is_contiguous() && square->is_cuda() && square->numel() == R);
    a.row_weight = square->data_ptr<float>();
    epi = kSquare;
  }
  if (R == 0) return;
  a.bounds = bounds.data_ptr<int32_t>();
  a.offsets = bounds.numel() == E + 1;
  a.src = src.has_value() ? src->data_ptr<int32_t>() : nullptr;
  a.xbytes = (o.x.size(0) - 1) * a.ldx + a.KB;
  const Plan p = plan(o.fp8, R, E, cols, a.KB, act != 0, false);
  const Shape s = kShapes[p.shape];
  const int64_t bn = s.cols() / (act ? 2 : 1);
  run(o, epi, p.shape, (R / s.rows() + std::min(E, R)) * ((cols + bn - 1) / bn));
}

// y [M, N] = x [M, K] w [N, K]^T with the operands, scales and act of
// grouped_linear
void tiled_linear(torch::Tensor y, torch::Tensor x, torch::Tensor w,
                  c10::optional<torch::Tensor> sx, c10::optional<torch::Tensor> sw,
                  int64_t act) {
  Operands o = operands(x, w.unsqueeze(0), sx, sw, false);
  Args& a = o.a;
  const Epilogue epi = epilogue_of(act, o);
  const int64_t cols = act ? a.N / 2 : a.N;
  check_result(y, cols, a);
  TORCH_CHECK(o.x.size(0) == a.R);
  if (a.R == 0) return;
  const Plan p = plan(o.fp8, a.R, 1, cols, a.KB, act != 0, false);
  const Shape s = kShapes[p.shape];
  const int64_t bn = s.cols() / (act ? 2 : 1);
  run(o, epi, p.shape, (a.R + s.rows() - 1) / s.rows() * ((cols + bn - 1) / bn));
}

// x w^T as `parts` sums (none of them empty) in tiles of a shape
static torch::Tensor sums_of(Operands& o, int shape, int parts) {
  Args& a = o.a;
  auto part = torch::empty({parts, a.R, a.N}, o.x.options().dtype(torch::kFloat32));
  if (a.R == 0) return part;
  a.k_part = (a.KB / kStep + parts - 1) / parts * kStep;
  a.part = part.data_ptr<float>();
  const Shape s = kShapes[shape];
  run(o, kSums, shape,
      (int64_t)(a.R + s.rows() - 1) / s.rows() * ((a.N + s.cols() - 1) / s.cols()) * parts);
  return part;
}

// the fp32 sums of x w^T alone, [parts, M, N], for a consumer that adds the
// parts itself (and applies an fp8 product's scales)
torch::Tensor tiled_sums(torch::Tensor x, torch::Tensor w) {
  Operands o = operands(x, w.unsqueeze(0), c10::nullopt, c10::nullopt, true);
  TORCH_CHECK(o.x.size(0) < (int64_t)1 << 30);
  o.a.R = (int)o.x.size(0);
  const Plan p = plan(o.fp8, o.a.R, 1, o.a.N, o.a.KB, false, true);
  return sums_of(o, p.shape, p.parts);
}

// The same of up to 64 rows in tiles of 64 columns, whose workgroups are at most one a
// CU: half the parts that tiles of 128 columns need to fill the chip, which half the
// bytes are written and read again by (40 rows of 4096 columns in 8 parts: 5.2 MB, where
// the fp8 weights of K 4096 are 16.8), and five steps of 16 KB on their way to each CU.
// us with the norm, weights out of cache, the streaming or wider tiles' sums / these: fp8
// 4096 x 4096 1 row 10.4 / 10.3, 24 rows 12.2 / 11.4, 40 rows 13.5 / 12.2, 64 rows 14.4 /
// 13.3; 6144 x 4096 1 row 12.9 / 12.4, 40 rows 15.2 / 14.4; 4096 x 14336 40 rows 20.5 / 19.1;
// bf16 4096 x 4096 1 row 13.0 / 13.0, 40 rows 15.8 / 14.0; 4096 x 14336 1 row 29.1 / 29.3, 40
// rows 31.1 / 29.2; 2304 x 9216 40 rows 19.6 / 15.9. With four places instead of six 0.3 to 0.9 less gain where K is long,
// with eight where it is short.
torch::Tensor narrow_sums(torch::Tensor x, torch::Tensor w) {
  Operands o = operands(x, w.unsqueeze(0), c10::nullopt, c10::nullopt, true);
  constexpr Shape s = kShapes[kNarrow];
  TORCH_CHECK(o.x.size(0) <= s.rows(), "up to 64 rows");
  o.a.R = (int)o.x.size(0);
  const int tiles = (o.a.N + s.cols() - 1) / s.cols(), steps = o.a.KB / kStep;
  const int most = std::max(1, std::min({kMaxParts, 256 / tiles, steps}));
  const int per = (steps + most - 1) / most;
  return sums_of(o, kNarrow, (steps + per - 1) / per);
}

// How a product (or M rows of that many experts' products) is planned, whole or as
// its sums: tile shape, parts of K, us (with the reading of the sums)
std::tuple<int64_t, int64_t, double> tiled_plan(int64_t M, int64_t N, int64_t KB, bool fp8,
                                                bool sums, int64_t experts) {
  TORCH_CHECK(M >= 1 && N >= 1 && KB >= kStep && KB % kStep == 0 && experts >= 1);
  const Plan p = plan(fp8, M, experts, N, KB, false, sums);
  return {p.shape, p.parts, p.us};
}
