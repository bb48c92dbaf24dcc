// Paged-attention decode: the plan of a step's splits, and the launches of
// attention_decode.h.
#include <torch/extension.h>

#include <type_traits>

#include "attention_decode.h"

using namespace decode;

namespace {

// How the rows of a step are split, and in which order the splits are worked through.
// One workgroup; threads 8 c + r weigh candidate c over every eighth row.
//
// A CU reads at most about 56 GB/s (3000 keys of one head in one workgroup of 4, 6 or
// 12 waves: 33 us all of them), so a step takes as long as the CU with the most keys.
// M = CUs / kv heads splits fill the chip once. A candidate is a largest number of
// tiles to a split; it costs, in tiles, its largest split or that many rounds of the
// mean one, and kSplitCost a round for what a split costs beside its tiles. Splits go to
// the CUs in turn, so they are ordered largest first, and every second round backwards:
// each CU's share is about the same, and CUs with a split less than the others get the
// largest.
constexpr int kCandidates = 32, kPlanThreads = 8 * kCandidates, kPlanRows = 1024;
constexpr float kSplitCost = 6.f;  // tiles
constexpr int kLeastTiles = 8;     // that a split is cut to

DEV_INLINE int all_sum(int v) {
#pragma unroll
  for (int d = 1; d < 64; d *= 2) v += __shfl_xor(v, d);
  return v;
}

__global__ void __launch_bounds__(kPlanThreads) decode_plan_kernel(
    Item* __restrict__ items, Splits* __restrict__ rows, const int32_t* __restrict__ seq_lens,
    const int B, const int n_items, const int M, const int window, const int tile_keys) {
  // a row's tiles, then its splits and their size (from the front, padded with none)
  __shared__ __attribute__((aligned(16))) int tiles[kPlanRows], sizes[kPlanRows];
  __shared__ int lens[kPlanRows];
  __shared__ int total[kPlanThreads / 64];
  __shared__ float best_cost[kPlanThreads / 64];
  __shared__ int best_limit[kPlanThreads / 64];
  const int t = threadIdx.x, padded = (B + 7) / 8 * 8;
  int mine = 0;
  for (int i = t; i < padded; i += kPlanThreads) {
    int n = 0;
    if (i < B) {
      lens[i] = seq_lens[i];
      const int L = max(1, lens[i]);
      const int first = window > 0 ? max(0, L - window) / kBS * kBS : 0;
      n = (L - first + tile_keys - 1) / tile_keys;
    }
    tiles[i] = n;
    mine += n;
  }
  mine = all_sum(mine);
  if (t % 64 == 0) total[t / 64] = mine;
  __syncthreads();
  float all = 0.f;
#pragma unroll
  for (int w = 0; w < kPlanThreads / 64; ++w) all += (float)total[w];
  // candidate c: splits of at most all / (3 M 0.9^c) tiles
  const int c = t / 8;
  const int limit =
      max(kLeastTiles, (int)ceilf(all / (3.f * M * __builtin_amdgcn_exp2f(-0.152003f * c))));
  float n = 0.f, large = 0.f;
  const float inv = 1.f / limit;
  for (int i = t % 8; i < padded; i += 8) {
    const float x = (float)tiles[i], k = fminf(ceilf(x * inv), (float)kMaxSplits);
    n += k;
    large = fmaxf(large, k > 0.f ? x * __builtin_amdgcn_rcpf(k) : 0.f);
  }
#pragma unroll
  for (int d = 1; d < 8; d *= 2) {
    n += __shfl_xor(n, d);
    large = fmaxf(large, __shfl_xor(large, d));
  }
  float cost = fmaxf(large, ceilf(n / M) * all / n) + kSplitCost * n / M;
  int of = limit;
#pragma unroll
  for (int d = 8; d < 64; d *= 2) {
    const float other = __shfl_xor(cost, d);
    const int l = __shfl_xor(of, d);
    if (other < cost || (other == cost && l > of)) {
      cost = other;
      of = l;
    }
  }
  if (t % 64 == 0) {
    best_cost[t / 64] = cost;
    best_limit[t / 64] = of;
  }
  __syncthreads();
#pragma unroll
  for (int w = 0; w < kPlanThreads / 64; ++w) {
    if (best_cost[w] < cost || (best_cost[w] == cost && best_limit[w] > of)) {
      cost = best_cost[w];
      of = best_limit[w];
    }
  }
  for (int i = t; i < padded; i += kPlanThreads) {
    const int x = tiles[i], k = min(kMaxSplits, (x + of - 1) / of);
    // size in front: rows by it, their splits (up to 16) below
    sizes[i] = k ? ((x + k - 1) / k) << 5 | k : 0;
  }
  __syncthreads();
  for (int i = t; i < B; i += kPlanThreads) {
    const int own = sizes[i] >> 5, k_own = sizes[i] & 31;
    int first = 0, N = 0;
#pragma unroll 4
    for (int j = 0; j < padded; j += 4) {
      const int4 four = *reinterpret_cast<const int4*>(sizes + j);
      const int e[4] = {four.x, four.y, four.z, four.w};
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        const int size = e[q] >> 5, k = e[q] & 31;
        N += k;
        if (size > own || (size == own && j + q < i)) first += k;
      }
    }
    rows[i] = {first, k_own};
    const int rounds = (N + M - 1) / M, rest = N - (rounds - 1) * M;  // CUs of the last one
    const int L = lens[i];
    int round = first / M, x = first - round * M;
    for (int k = 0; k < k_own; ++k) {
      int cu;
      if (round == rounds - 1) cu = round % 2 ? rest - 1 - x : x;
      else if (round % 2) cu = x < rest ? rest - 1 - x : M - 1 - (x - rest);
      else cu = x < M - rest ? rest + x : x - (M - rest);
      items[round * M + cu] = {i, L, (uint16_t)k, (uint16_t)k_own, first + k};
      if (++x == M) {
        x = 0;
        ++round;
      }
    }
    if (i == 0) total[0] = N;
  }
  __syncthreads();
  for (int i = total[0] + t; i < n_items; i += kPlanThreads) items[i] = {-1, 0, 0, 0, 0};
}
}  // namespace

// How often a row's keys are split without a plan: until there are 512 workgroups (two a CU).
// The lengths are not known here; more splits cost in the merge, and a row that
// is much longer than the others is worked through by its own splits alone. At
// head size 256, whose workgroups read a row at half the rate of those at 128,
// many rows are split once more for that (576). Head size 128: 40 rows of
// 100-700 keys, 8 kv heads 22.4 us at 512, 21.1 at 256, 22.5 at 1536; of 1500-4000 96, 111
// at 256, 94; one row of 3000 among 7 idle ones 11.3, 14.5 at 256, 10.1; 96 rows of 100-300,
// 4 kv heads 15.8, 13.2 at 256, 18.9. Head size 256: 128 rows of 300 but one of 8000, 4
// kv heads 181 at 512, 113 at 576, 90 at 1536; 8 rows of 3500, e5m2 cache, 8 kv heads 31.5
// at 512, 39 at 576, 36 at 1536; 40 rows of 100-700, e5m2 cache, 4 kv heads 23.8, 24.0 and
// 27.2. A split has at least 32 keys of the widest row, 16 at head size 256.
// KUBEAI_DECODE_SPLIT_TARGET overrides it (steps with a plan do not ask).
int paged_decode_splits(int rows, int n_kv, int hd, int max_blocks) {
  static const int forced = []() {
    const char* e = getenv("KUBEAI_DECODE_SPLIT_TARGET");
    return e ? atoi(e) : 0;
  }();
  const int64_t wgs = (int64_t)rows * n_kv;
  const int target = forced > 0 ? forced : hd == 256 && wgs > 64 ? 576 : 512;
  const int tiles = hd == 256 ? max_blocks : (max_blocks + 1) / 2;
  return (int)std::max<int64_t>(
      1, std::min({(int64_t)kMaxSplits, (int64_t)tiles, (target + wgs - 1) / wgs}));
}

// The splits of a step's rows, for paged_attention_decode over any caches of this many
// kv heads, head size, element and window while the lengths are these.
torch::Tensor paged_decode_plan(torch::Tensor seq_lens, int64_t n_kv, int64_t hd,
                                int64_t element_size, int64_t window) {
  TORCH_CHECK(seq_lens.scalar_type() == torch::kInt32 && seq_lens.is_contiguous() &&
              seq_lens.is_cuda() && seq_lens.dim() == 1);
  const int B = (int)seq_lens.size(0);
  TORCH_CHECK(B >= 1 && B <= kPlanRows, "1 to ", kPlanRows, " rows");
  TORCH_CHECK(n_kv >= 1 && (hd == 128 || hd == 256) && (element_size == 1 || element_size == 2));
  const int M = std::max<int64_t>(1, kCUs / n_kv);
  const int64_t n_items = plan_items(B, n_kv);
  auto plan = torch::empty({4 * n_items + 2 * B}, seq_lens.options());
  auto* items = reinterpret_cast<Item*>(plan.data_ptr());
  hipLaunchKernelGGL(decode_plan_kernel, dim3(1), dim3(kPlanThreads), 0,
                     c10::hip::getCurrentHIPStream().stream(), items,
                     reinterpret_cast<Splits*>(items + n_items), seq_lens.data_ptr<int32_t>(),
                     B, (int)n_items, M, (int)window,
                     kBS * blocks_per_tile((int)hd, (int)element_size));
  HIP_CHECK_KERNEL();
  return plan;
}

// out [B, n_q, hd] bf16, or with out_scale [B] fp8 rows with a scale each
static void attend(torch::Tensor out, const ushort* q, int64_t q_stride, const NewRows* fresh,
                   int B, int n_q, torch::Tensor k_cache, torch::Tensor v_cache,
                   torch::Tensor block_tables, torch::Tensor seq_lens, double scale,
                   int64_t window, double softcap, c10::optional<torch::Tensor> out_scale,
                   c10::optional<torch::Tensor> plan) {
  const int hd = k_cache.size(3);
  TORCH_CHECK(out.is_contiguous() && out.numel() >= (int64_t)B * n_q * hd);
  TORCH_CHECK(k_cache.is_contiguous() && v_cache.is_contiguous());
  TORCH_CHECK(k_cache.scalar_type() == torch::kBFloat16 ||
              k_cache.scalar_type() == torch::kFloat8_e5m2);
  TORCH_CHECK(block_tables.scalar_type() == torch::kInt32);
  TORCH_CHECK(seq_lens.scalar_type() == torch::kInt32);
  block_tables = with_a_column(block_tables);
  const int n_kv = k_cache.size(1);
  const int max_blocks = block_tables.size(1);
  TORCH_CHECK(hd == 128 || hd == 256,
              "decode kernel supports head_dim 128 or 256");
  TORCH_CHECK(k_cache.size(2) == kBS, "decode kernel supports block_size=16");
  const int G = n_q / n_kv;
  TORCH_CHECK(n_q % n_kv == 0);
  if (B == 0) return;
  TORCH_CHECK(G == 1 || G == 2 || G == 4 || G == 5 || G == 6 || G == 8,
              "unsupported GQA group size ", G);
  const int n_splits = paged_decode_splits(B, n_kv, hd, max_blocks);
  const Item* items = nullptr;
  const Splits* row_splits = nullptr;
  int64_t parts = (int64_t)B * n_splits;
  if (plan.has_value()) {
    check_plan(*plan, B, n_kv);
    parts = plan_items(B, n_kv);
    items = reinterpret_cast<const Item*>(plan->data_ptr());
    row_splits = reinterpret_cast<const Splits*>(items + parts);
  }
  const bool fp8 = out_scale.has_value();
  TORCH_CHECK(out.scalar_type() == (fp8 ? torch::kFloat8_e4m3fn : torch::kBFloat16));
  if (fp8)
    TORCH_CHECK((items || n_splits > 1) && n_q <= 32 && out_scale->is_contiguous() &&
                    out_scale->scalar_type() == torch::kFloat32 && out_scale->numel() == B,
                "fp8 rows come from the merge of up to 32 heads");
  torch::Tensor part_o, part_ml;
  float *part_o_ptr = nullptr, *part_ml_ptr = nullptr;
  const bool merged = items || n_splits > 1;
  if (merged) {
    auto opts =
        torch::TensorOptions().device(k_cache.device()).dtype(torch::kFloat32);
    part_o = torch::empty({parts, n_q, (int64_t)hd}, opts);
    part_ml = torch::empty({parts, n_q, 2}, opts);
    part_o_ptr = part_o.data_ptr<float>();
    part_ml_ptr = part_ml.data_ptr<float>();
  }
  TORCH_CHECK(parts * n_kv < (int64_t)1 << 31);
  const dim3 grid((uint32_t)(parts * n_kv)), block(kBlockThreads);
  auto stream = c10::hip::getCurrentHIPStream().stream();
  auto with_new = [&](auto hdv, auto ct, auto cap, auto one, auto fresh_v, auto nb) {
    using CT = decltype(ct);
    hipLaunchKernelGGL(
        (paged_decode_kernel<decltype(hdv)::value, CT, decltype(cap)::value,
                             decltype(one)::value, decltype(fresh_v)::value,
                             decltype(nb)::value>),
        grid, block, 0, stream, fp8 ? nullptr : (ushort*)out.data_ptr(), q,
        (CT*)k_cache.data_ptr(), (CT*)v_cache.data_ptr(), block_tables.data_ptr<int32_t>(),
        seq_lens.data_ptr<int32_t>(), (float)scale, (float)softcap,
        (int)window, n_kv, G, max_blocks, q_stride, n_splits, items,
        fresh ? *fresh : NewRows{}, part_o_ptr, part_ml_ptr);
  };
  // No wave has more than one tile (12 rows of 500: 14.9 us with the loop's loads of no
  // bytes, 13.9 without): of a cache block, or up to twice as many keys of two, which are
  // faster than a loop of two (111 rows of 29-76 10.4 / 11.4).
  const int nb = blocks_per_tile(hd, k_cache.element_size());
  auto fit = [&](int blocks) {
    return !items && (max_blocks + blocks - 1) / blocks <= n_splits * kWaves;
  };
  const bool one = fit(nb), one_of_two = !one && !fresh && hd == 128 && nb == 1 && fit(2);
  auto launch = [&](auto hdv, auto ct, auto cap, auto one) {
    constexpr int HD = decltype(hdv)::value;
    const std::integral_constant<int, blocks_per_tile(HD, sizeof(ct))> own{};
    if constexpr (sizeof(ct) == 2) {
      if (fresh && fresh->sums.parts <= 4)
        return with_new(hdv, ct, cap, one, std::integral_constant<int, 4>{}, own);
      if (fresh) return with_new(hdv, ct, cap, one, std::integral_constant<int, 8>{}, own);
    }
    const std::integral_constant<int, 0> none{};
    if constexpr (sizeof(ct) == 2 && HD == 128 && decltype(one)::value) {
      if (one_of_two)
        return with_new(hdv, ct, cap, one, none, std::integral_constant<int, 2>{});
    }
    with_new(hdv, ct, cap, one, none, own);
  };
  auto with_cap = [&](auto hdv, auto ct) {
    auto with_one = [&](auto capped) {
      if (one || one_of_two) launch(hdv, ct, capped, std::true_type{});
      else launch(hdv, ct, capped, std::false_type{});
    };
    if (softcap > 0.0) with_one(std::true_type{});
    else with_one(std::false_type{});
  };
  auto with_hd = [&](auto ct) {
    if (hd == 256) with_cap(std::integral_constant<int, 256>{}, ct);
    else with_cap(std::integral_constant<int, 128>{}, ct);
  };
  if (k_cache.scalar_type() == torch::kFloat8_e5m2) with_hd((unsigned char)0);
  else with_hd((ushort)0);
  HIP_CHECK_KERNEL();
  if (fp8) {
    auto merge = [&](auto hdv, auto hpw) {
      hipLaunchKernelGGL(
          (decode_merge_fp8_kernel<decltype(hdv)::value, decltype(hpw)::value>), dim3(B),
          dim3(16 * WAVE_SIZE), 0, stream, (unsigned char*)out.data_ptr(),
          out_scale->data_ptr<float>(), nullptr, B, part_o_ptr, part_ml_ptr, row_splits, n_splits, n_q);
    };
    auto heads = [&](auto hdv) {
      if (n_q <= 16) merge(hdv, std::integral_constant<int, 1>{});
      else merge(hdv, std::integral_constant<int, 2>{});
    };
    if (hd == 256) heads(std::integral_constant<int, 256>{});
    else heads(std::integral_constant<int, 128>{});
    HIP_CHECK_KERNEL();
  } else if (merged) {
    const int64_t n_bh = (int64_t)B * n_q;
    const int wpb = 4;
    const dim3 mgrid((uint32_t)((n_bh + wpb - 1) / wpb)), mblock(wpb * WAVE_SIZE);
    if (hd == 256)
      hipLaunchKernelGGL((decode_merge_kernel<256>), mgrid, mblock, 0, stream,
                         (ushort*)out.data_ptr(), part_o_ptr, part_ml_ptr,
                         row_splits, n_splits, n_q, n_bh);
    else
      hipLaunchKernelGGL((decode_merge_kernel<128>), mgrid, mblock, 0, stream,
                         (ushort*)out.data_ptr(), part_o_ptr, part_ml_ptr,
                         row_splits, n_splits, n_q, n_bh);
    HIP_CHECK_KERNEL();
  }
}

void paged_attention_decode(torch::Tensor out, torch::Tensor q,
                            torch::Tensor k_cache, torch::Tensor v_cache,
                            torch::Tensor block_tables, torch::Tensor seq_lens,
                            double scale, int64_t window, double softcap,
                            c10::optional<torch::Tensor> out_scale,
                            c10::optional<torch::Tensor> plan) {
  TORCH_CHECK(q.stride(2) == 1 && q.stride(1) == q.size(2) && k_cache.dim() == 4 &&
              k_cache.size(3) == q.size(2));
  TORCH_CHECK(q.scalar_type() == torch::kBFloat16);
  attend(out, (const ushort*)q.data_ptr(), q.stride(0), nullptr, q.size(0), q.size(1), k_cache,
         v_cache, block_tables, seq_lens, scale, window, softcap, out_scale, plan);
}

// The same for rows whose queries, keys and values are a product's sums `part` (with
// the scales of fp8 operands), [parts, B, (n_q + 2 n_kv) hd]: rotated by positions, keys
// and values written to slots, which name the places of the rows' last keys (or < 0).
void paged_attention_decode_sums(torch::Tensor out, torch::Tensor part,
                                 c10::optional<torch::Tensor> sx,
                                 c10::optional<torch::Tensor> sw, int64_t n_q,
                                 torch::Tensor positions, torch::Tensor cos_sin,
                                 torch::Tensor slots, torch::Tensor k_cache,
                                 torch::Tensor v_cache, torch::Tensor block_tables,
                                 torch::Tensor seq_lens, double scale, int64_t window,
                                 double softcap, c10::optional<torch::Tensor> out_scale,
                                 c10::optional<torch::Tensor> plan) {
  TORCH_CHECK(k_cache.dim() == 4 && v_cache.sizes() == k_cache.sizes() &&
              v_cache.scalar_type() == torch::kBFloat16 &&
              k_cache.scalar_type() == torch::kBFloat16);
  const int64_t n_kv = k_cache.size(1), hd = k_cache.size(3), width = (n_q + 2 * n_kv) * hd;
  TORCH_CHECK(part.scalar_type() == torch::kFloat32 && part.is_contiguous() &&
              part.is_cuda() && part.dim() == 3 && part.size(0) >= 1 && part.size(0) <= 8 &&
              part.size(2) == width && ((uintptr_t)part.data_ptr() & 15) == 0);
  TORCH_CHECK((n_q / n_kv + 2) * hd / 8 <= kBlockThreads, "a thread has 8 columns");
  const int64_t B = part.size(1);
  TORCH_CHECK(seq_lens.numel() == B && block_tables.size(0) == B);
  TORCH_CHECK(positions.scalar_type() == torch::kInt32 && positions.numel() >= B &&
              positions.is_contiguous() && slots.scalar_type() == torch::kInt64 &&
              slots.numel() >= B && slots.is_contiguous());
  TORCH_CHECK(cos_sin.scalar_type() == torch::kFloat32 && cos_sin.is_contiguous() &&
              cos_sin.size(1) == hd && ((uintptr_t)cos_sin.data_ptr() & 15) == 0);
  TORCH_CHECK(sx.has_value() == sw.has_value());
  NewRows fresh{{part.data_ptr<float>(), nullptr, nullptr, (int)part.size(0), B * width,
                 (int)width},
                positions.data_ptr<int32_t>(), cos_sin.data_ptr<float>(),
                slots.data_ptr<int64_t>()};
  if (sx.has_value()) {
    TORCH_CHECK(sx->scalar_type() == torch::kFloat32 && sx->is_contiguous() &&
                sx->numel() == B && sw->scalar_type() == torch::kFloat32 &&
                sw->is_contiguous() && sw->numel() == width);
    fresh.sums.sx = sx->data_ptr<float>();
    fresh.sums.sw = sw->data_ptr<float>();
  }
  attend(out, nullptr, 0, &fresh, (int)B, (int)n_q, k_cache, v_cache, block_tables, seq_lens,
         scale, window, softcap, out_scale, plan);
}
