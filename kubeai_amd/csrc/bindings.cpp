// Python bindings for the kubeai_amd gfx950 HIP kernels.
#include <torch/extension.h>

#include <algorithm>

void rmsnorm(torch::Tensor out, torch::Tensor x, torch::Tensor weight,
             double eps);
void fused_add_rmsnorm(torch::Tensor x, torch::Tensor residual,
                       torch::Tensor weight, double eps);
void rope(torch::Tensor q, torch::Tensor k, torch::Tensor positions,
          torch::Tensor cos_sin);
void rope_cache(torch::Tensor qkv, torch::Tensor positions,
                torch::Tensor cos_sin, torch::Tensor k_cache,
                torch::Tensor v_cache, torch::Tensor slot_mapping, int64_t n_q,
                c10::optional<torch::Tensor> part,
                c10::optional<torch::Tensor> sx,
                c10::optional<torch::Tensor> sw);
torch::Tensor skinny_sums(torch::Tensor x, torch::Tensor w);
void skinny_gated(torch::Tensor y, torch::Tensor x, torch::Tensor w, int64_t act);
void quant_fp8_rows(torch::Tensor out, torch::Tensor out_scale, torch::Tensor x,
                    torch::Tensor src);
void rmsnorm_sums(torch::Tensor out, c10::optional<torch::Tensor> out_scale,
                  torch::Tensor part, c10::optional<torch::Tensor> sx,
                  c10::optional<torch::Tensor> sw,
                  c10::optional<torch::Tensor> residual, torch::Tensor weight,
                  double eps);
void norm_add_norm(torch::Tensor out, torch::Tensor hidden,
                   c10::optional<torch::Tensor> x, c10::optional<torch::Tensor> part,
                   c10::optional<torch::Tensor> sx, c10::optional<torch::Tensor> sw,
                   torch::Tensor residual, c10::optional<torch::Tensor> w1,
                   torch::Tensor w2, double eps);
void reshape_and_cache_fp8(torch::Tensor k, torch::Tensor v,
                           torch::Tensor k_cache, torch::Tensor v_cache,
                           torch::Tensor slot_mapping);
void reshape_and_cache(torch::Tensor k, torch::Tensor v, torch::Tensor k_cache,
                       torch::Tensor v_cache, torch::Tensor slot_mapping);
void paged_attention_decode(torch::Tensor out, torch::Tensor q,
                            torch::Tensor k_cache, torch::Tensor v_cache,
                            torch::Tensor block_tables, torch::Tensor seq_lens,
                            double scale, int64_t window, double softcap,
                            c10::optional<torch::Tensor> out_scale,
                            c10::optional<torch::Tensor> plan);
void paged_attention_step(torch::Tensor out, c10::optional<torch::Tensor> out_scale,
                          torch::Tensor q, int64_t n_decode, torch::Tensor k_cache,
                          torch::Tensor v_cache, torch::Tensor decode_tables,
                          torch::Tensor decode_lens, torch::Tensor plan,
                          torch::Tensor prompt_tables, torch::Tensor query_start_loc,
                          torch::Tensor prompt_lens, double scale, int64_t window,
                          double softcap);
void paged_attention_decode_sums(torch::Tensor out, torch::Tensor part,
                                 c10::optional<torch::Tensor> sx,
                                 c10::optional<torch::Tensor> sw, int64_t n_q,
                                 torch::Tensor positions, torch::Tensor cos_sin,
                                 torch::Tensor slots, torch::Tensor k_cache,
                                 torch::Tensor v_cache, torch::Tensor block_tables,
                                 torch::Tensor seq_lens, double scale, int64_t window,
                                 double softcap, c10::optional<torch::Tensor> out_scale,
                                 c10::optional<torch::Tensor> plan);
torch::Tensor paged_decode_plan(torch::Tensor seq_lens, int64_t n_kv, int64_t hd,
                                int64_t element_size, int64_t window);
int paged_decode_splits(int rows, int n_kv, int hd, int max_blocks);
void paged_attention_prefill(torch::Tensor out, torch::Tensor q,
                             torch::Tensor k_cache, torch::Tensor v_cache,
                             torch::Tensor block_tables,
                             torch::Tensor query_start_loc,
                             torch::Tensor seq_lens, double scale,
                             int64_t window, double softcap);
void silu_and_mul(torch::Tensor out, torch::Tensor x);
void gelu_and_mul(torch::Tensor out, torch::Tensor x);
void skinny_linear(torch::Tensor y, torch::Tensor x, torch::Tensor w,
                   c10::optional<torch::Tensor> sx,
                   c10::optional<torch::Tensor> sw,
                   c10::optional<torch::Tensor> bias);
void skinny_experts(torch::Tensor y, torch::Tensor x, torch::Tensor w,
                    c10::optional<torch::Tensor> sx,
                    c10::optional<torch::Tensor> sw, torch::Tensor begin,
                    c10::optional<torch::Tensor> src);
void grouped_linear(torch::Tensor y, torch::Tensor x, torch::Tensor w,
                    c10::optional<torch::Tensor> sx,
                    c10::optional<torch::Tensor> sw, torch::Tensor bounds,
                    c10::optional<torch::Tensor> src,
                    c10::optional<torch::Tensor> square, int64_t act);
void tiled_linear(torch::Tensor y, torch::Tensor x, torch::Tensor w,
                  c10::optional<torch::Tensor> sx,
                  c10::optional<torch::Tensor> sw, int64_t act);
torch::Tensor tiled_sums(torch::Tensor x, torch::Tensor w);
torch::Tensor narrow_sums(torch::Tensor x, torch::Tensor w);
std::tuple<int64_t, int64_t, double> tiled_plan(int64_t M, int64_t N, int64_t KB,
                                                bool fp8, bool sums, int64_t experts);
void moe_route(torch::Tensor index, torch::Tensor weight, torch::Tensor begin,
               torch::Tensor src, torch::Tensor place, torch::Tensor x,
               torch::Tensor w);
void moe_combine(torch::Tensor out, torch::Tensor y, torch::Tensor place,
                 torch::Tensor weight);
void skinny_gemm(torch::Tensor y, torch::Tensor x, torch::Tensor w);
void greedy_sample(torch::Tensor out, torch::Tensor logits,
                   c10::optional<torch::Tensor> logprob);
void gumbel_sample(torch::Tensor out, torch::Tensor logits, torch::Tensor temperature,
                   torch::Tensor seeds, int64_t step, c10::optional<torch::Tensor> logprob);
void sgmv(torch::Tensor y, torch::Tensor x, torch::Tensor A, torch::Tensor B,
          torch::Tensor idx, double scale);
void lora_apply(torch::Tensor y, torch::Tensor x, torch::Tensor table,
                torch::Tensor ids, int64_t max_rank,
                std::optional<torch::Tensor> z);
void register_chwbl(pybind11::module_& m);
// one-shot fused all-reduce over xGMI (allreduce.hip)
pybind11::bytes xgmi_alloc();
void xgmi_connect(int64_t rank, int64_t world,
                  const std::vector<pybind11::bytes>& handles);
void xgmi_fused_allreduce_add_rmsnorm(torch::Tensor x, torch::Tensor residual,
                                      torch::Tensor weight, double eps);
int64_t xgmi_error_count();
int64_t xgmi_max_elems();
void xgmi_shutdown();
void rmsnorm_fp8(torch::Tensor out, torch::Tensor out_scale, torch::Tensor x,
                 torch::Tensor weight, double eps);
void fused_add_rmsnorm_fp8(torch::Tensor out, torch::Tensor out_scale,
                           torch::Tensor x, torch::Tensor residual,
                           torch::Tensor weight, double eps);
void silu_and_mul_fp8(torch::Tensor out, torch::Tensor out_scale,
                      torch::Tensor x);
void quant_fp8(torch::Tensor out, torch::Tensor out_scale, torch::Tensor x);
void nucleus_stats(torch::Tensor m, torch::Tensor z, torch::Tensor logits,
                   torch::Tensor temps);
void nucleus_accept(torch::Tensor ok, torch::Tensor logits,
                    torch::Tensor cand, torch::Tensor m, torch::Tensor z,
                    torch::Tensor temps, torch::Tensor top_ps,
                    torch::Tensor top_ks);

// out [R, C] int32 on the host: row i takes rows[i], zeros elsewhere
static void fill_rows(torch::Tensor out, const py::list& rows) {
  TORCH_CHECK(out.device().is_cpu() && out.scalar_type() == torch::kInt32 &&
              out.dim() == 2 && out.is_contiguous());
  const int64_t R = out.size(0), C = out.size(1), n = (int64_t)rows.size();
  TORCH_CHECK(n <= R, n, " lists for ", R, " rows");
  int32_t* to = out.data_ptr<int32_t>();
  std::fill(to, to + R * C, 0);
  for (int64_t i = 0; i < n; ++i, to += C) {
    PyObject* row = PyList_GET_ITEM(rows.ptr(), i);
    TORCH_CHECK(PyList_Check(row), "rows are lists");
    const int64_t k = PyList_GET_SIZE(row);
    TORCH_CHECK(k <= C, "a list of ", k, " for a row of ", C);
    for (int64_t j = 0; j < k; ++j) {
      const long v = PyLong_AsLong(PyList_GET_ITEM(row, j));
      if (v == -1 && PyErr_Occurred()) throw py::error_already_set();
      TORCH_CHECK(v >= INT32_MIN && v <= INT32_MAX, "32-bit values");
      to[j] = (int32_t)v;
    }
  }
}

PYBIND11_MODULE(TORCH_EXTENSION_NAME, m) {
  m.def("rmsnorm", &rmsnorm, "RMSNorm (bf16, fp32 accum)");
  m.def("fused_add_rmsnorm", &fused_add_rmsnorm,
        "in-place residual add + RMSNorm");
  m.def("rope", &rope, "NeoX rotary embedding, in-place q/k");
  m.def("rope_cache", &rope_cache,
        "rotary embedding of q in place, rotated k and v into the paged cache");
  m.def("reshape_and_cache", &reshape_and_cache, "paged KV cache write");
  m.def("reshape_and_cache_fp8", &reshape_and_cache_fp8,
        "paged KV cache write, fp8 e5m2 cache");
  m.def("paged_attention_decode", &paged_attention_decode,
        "paged attention, one query token per seq", py::arg("out"), py::arg("q"),
        py::arg("k_cache"), py::arg("v_cache"), py::arg("block_tables"),
        py::arg("seq_lens"), py::arg("scale"), py::arg("window"), py::arg("softcap"),
        py::arg("out_scale") = py::none(), py::arg("plan") = py::none());
  m.def("paged_attention_step", &paged_attention_step,
        "a step's prompt portions and decode rows in one launch");
  m.def("paged_attention_decode_sums", &paged_attention_decode_sums,
        "paged decode attention of rows that are a product's sums");
  m.def("paged_decode_plan", &paged_decode_plan,
        "splits of all rows of a decode step (lengths, kv heads, head size, bytes of an "
        "element, window)");
  m.def("paged_decode_splits", &paged_decode_splits,
        "splits of a decode row's keys (rows, kv heads, head size, table width)");
  m.def("paged_attention_prefill", &paged_attention_prefill,
        "paged causal flash attention over cached KV");
  m.def("gelu_and_mul", &gelu_and_mul, "GeGLU tanh-gelu(gate)*up");
  m.def("silu_and_mul", &silu_and_mul, "SwiGLU activation");
  m.def("skinny_gemm", &skinny_gemm, "weight-streaming product, bf16");
  m.def("skinny_experts", &skinny_experts,
        "weight-streaming product of each expert's rows");
  m.def("grouped_linear", &grouped_linear,
        "all experts' products of a large step, bf16 or fp8 e4m3", py::arg("y"),
        py::arg("x"), py::arg("w"), py::arg("sx"), py::arg("sw"), py::arg("bounds"),
        py::arg("src"), py::arg("square"), py::arg("act") = 0);
  m.def("tiled_linear", &tiled_linear, "product of many rows, bf16 or scaled fp8");
  m.def("tiled_plan", &tiled_plan,
        "tile shape, parts and us of a tiled product, whole or as sums",
        py::arg("M"), py::arg("N"), py::arg("KB"), py::arg("fp8"), py::arg("sums"),
        py::arg("experts") = 1);
  m.def("narrow_sums", &narrow_sums, "sums of up to 64 rows, tiles of 64 columns");
  m.def("tiled_sums", &tiled_sums, "fp32 part sums of a product of many rows");
  m.def("skinny_sums", &skinny_sums, "fp32 part sums of a skinny product");
  m.def("skinny_gated", &skinny_gated, "weight-streaming gate and up, activated");
  m.def("quant_fp8_rows", &quant_fp8_rows, "gathered bf16 rows -> fp8");
  m.def("rmsnorm_sums", &rmsnorm_sums, "norm of a product's part sums");
  m.def("norm_add_norm", &norm_add_norm,
        "norm of a branch, residual add and the next norm, or the last two");
  m.def("moe_route", &moe_route,
        "router scores, top-k weights and tokens in expert order");
  m.def("moe_combine", &moe_combine, "weighted sum of the experts' rows");
  m.def("skinny_linear", &skinny_linear,
        "weight-streaming product of up to 96 rows, bf16 or scaled fp8");
  m.def("fill_rows", &fill_rows, "lists of numbers to rows of a host tensor");
  m.def("greedy_sample", &greedy_sample, "argmax sampling", py::arg("out"),
        py::arg("logits"), py::arg("logprob") = py::none());
  m.def("gumbel_sample", &gumbel_sample, "temperature sampling (hash RNG)",
        py::arg("out"), py::arg("logits"), py::arg("temperature"),
        py::arg("seeds"), py::arg("step"),
        py::arg("logprob") = py::none());
  m.def("rmsnorm_fp8", &rmsnorm_fp8, "rmsnorm with fused fp8 row quant");
  m.def("fused_add_rmsnorm_fp8", &fused_add_rmsnorm_fp8,
        "residual add + rmsnorm with fused fp8 row quant");
  m.def("silu_and_mul_fp8", &silu_and_mul_fp8, "SwiGLU with fused fp8 quant");
  m.def("quant_fp8", &quant_fp8, "bf16 -> fp8 row quant");
  m.def("nucleus_stats", &nucleus_stats, "per-row softmax max + Z");
  m.def("nucleus_accept", &nucleus_accept,
        "nucleus membership of sampled tokens (mass above < p, rank < k)");
  m.def("xgmi_alloc", &xgmi_alloc, "allocate + export the IPC comm buffer");
  m.def("xgmi_connect", &xgmi_connect, "open peer IPC buffers");
  m.def("xgmi_fused_allreduce_add_rmsnorm", &xgmi_fused_allreduce_add_rmsnorm,
        "one-shot xGMI all-reduce fused with residual add + RMSNorm");
  m.def("xgmi_error_count", &xgmi_error_count, "spin-wait timeout count");
  m.def("xgmi_max_elems", &xgmi_max_elems, "one-shot capacity (bf16 elems)");
  m.def("xgmi_shutdown", &xgmi_shutdown, "free/close comm buffers");
  m.def("sgmv", &sgmv, "segmented gather LoRA apply (one adapter segment)");
  m.def("lora_apply", &lora_apply,
        "LoRA apply over a batch of tokens with mixed adapters",
        py::arg("y"), py::arg("x"), py::arg("table"), py::arg("ids"),
        py::arg("max_rank"), py::arg("z") = py::none());
  register_chwbl(m);
}
