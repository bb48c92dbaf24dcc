// Paged flash-attention prefill (causal, GQA, prefix-cache aware) for gfx950.
//
// Semantics: kubeai_amd/ops/ref.py::paged_attention_prefill — new (chunk)
// query tokens attend to the full paged KV cache (which already contains
// this chunk's K/V via reshape_and_cache).
//
// Structure:
//  - workgroup = 4 waves over one kv head: GB = min(G, 4) of the group's
//    query heads x 4/GB subtiles of 32 query rows. The waves share each
//    staged tile of KVB keys, so a K/V byte fetched from L2 feeds 128 query
//    rows; two workgroups (head size 128) share a CU and overlap one's
//    softmax with the other's matrix instructions.
//  - S^T = K.Q^T and O^T += V^T.P^T on v_mfma_f32_32x32x16_bf16. Both keep
//    the query in the accumulator's column (lane & 31): running maximum, sum
//    and rescale are per-lane scalars. The sum over keys does not care about
//    their order, so P's accumulator registers are the second product's
//    operand as they stand (two rows converted per instruction, no exchange
//    between lanes) once V is read with the same key order: register j of
//    step ks in half `hi` is key 16 ks + 4 hi + (j & 3) + 8 (j >> 2), and
//    ds_read_b64_tr_b16 fetches four consecutive keys of a column.
//  - K and V tiles lie row-major in LDS, 16-byte units XOR-swizzled: K by
//    row & 7 (32 rows of one unit per read), V so that the four rows of one
//    16-lane transposing read fall in disjoint banks.
//  - LDS is double-buffered, the next tile's global loads issue before this
//    tile's compute; its cache blocks are looked up one tile earlier with
//    scalar loads.
//  - the grid numbers the query tiles of the whole packed step (find_tile),
//    kv head fastest: a step of one long prompt and many padding runs
//    launches no empty rows of blocks, and with 8 kv heads each XCD works on
//    one head, whose keys and values stay in its 4 MB L2. (A grid with the
//    sequence fastest put a lone prompt's tiles on two of the eight XCDs
//    when three padding runs came with it.) Late tiles, which see the most
//    keys, start first.
//
// Bound by the softmax's vector instructions against the matrix
// instructions: per 64 keys a wave issues 32 MFMAs (1024 cycles) and about
// as many cycles of max / exp2 / convert.
// Measured (us; before: 8-wave kernel for plain causal head size 128, 16-row
// kernel for the rest):
//   heads 32/8 x 128, one prompt of 2048                205 ->  69 (501 TF/s)
//     the same with 3 padding runs                      510 ->  68
//   8192                                               1840 -> 666 (826 TF/s)
//   8192, window 4096                                  2797 -> 488
//   512 new tokens behind 3584                          414 -> 100
//   six turns of 62-100 behind 365-587, 4 padding runs   72 ->  23
//   heads 64/8 x 128, 4096                              927 -> 360
//   heads 8/4 x 256, 3029 + 2145, cap, window 4096     1574 -> 268 (211 TF/s)
// Head size 256 holds 128 accumulator registers of O, so one wave a SIMD
// and 32-key tiles (a 64-key tile's two buffers would need 128 KB).
//
// Fragment layouts:
//   A[M=32][K=16]: lane l holds A[l&31][(l>>5)*8 + j], j=0..7
//   B[K=16][N=32]: lane l holds B[(l>>5)*8 + j][l&31]
//   C[M=32][N=32]: lane l holds C[(r&3) + 8*(r>>2) + 4*(l>>5)][l&31]
//   ds_read_b64_tr_b16: in each group of 16 lanes, lane l's element j comes
//   from the 8 bytes addressed by lane 4j + (l>>2), element l&3
#include <torch/extension.h>

#include "common.h"

namespace {

constexpr int kBS = 16;  // cache block size (tokens)
constexpr int kQB = 32;  // query rows per wave
constexpr int kNW = 4;   // waves per workgroup

typedef __attribute__((ext_vector_type(8))) short bf16x8;
typedef __attribute__((ext_vector_type(4))) short bf16x4;
typedef __attribute__((ext_vector_type(16))) float f32x16;
typedef __attribute__((ext_vector_type(2))) float f32x2;
typedef __attribute__((ext_vector_type(2))) __bf16 bf16x2;
typedef __attribute__((ext_vector_type(4))) uint32_t u32x4;
typedef __attribute__((address_space(3))) bf16x4 lds_bf16x4;

// run s of the packed stream owns the tile numbers from (start[s] - start[0])
// / size + s on (never fewer than it needs): T / size + n_seq numbers cover
// every batch. The runs may be a part of a longer stream (start[0] > 0).
DEV_INLINE int find_tile(const int32_t* start, int n_seq, int size, int n,
                         int* tile) {
  const int base = start[0];
  int lo = 0, hi = n_seq - 1;
  while (lo < hi) {
    const int mid = (lo + hi + 1) >> 1;
    if ((start[mid] - base) / size + mid <= n) lo = mid;
    else hi = mid - 1;
  }
  *tile = n - ((start[lo] - base) / size + lo);
  return lo;
}

// CT = cache element type: ushort (bf16) or unsigned char (fp8 e5m2,
// converted to bf16 while staging). CAP: capped scores. WIN: keys in
// (pos - window, pos] only.
template <int HD, int GB, typename CT, bool WIN, bool CAP>
__launch_bounds__(kNW * WAVE_SIZE, HD == 128 ? 2 : 1) __global__
void paged_prefill_kernel(
    ushort* __restrict__ out,          // [Tq, n_q, HD]
    const ushort* __restrict__ q,      // [Tq, n_q, HD], rows strided
    const CT* __restrict__ k_cache,    // [nb, n_kv, 16, HD]
    const CT* __restrict__ v_cache,
    const int32_t* __restrict__ block_tables,     // [B, max_blocks]
    const int32_t* __restrict__ query_start_loc,  // [B+1]
    const int32_t* __restrict__ seq_lens,         // [B]
    const float scale, const float softcap, const int window,
    const int n_kv, const int G, const int n_seq, const int max_blocks,
    const int64_t q_stride, const int n_tiles_q) {
  constexpr int KVB = HD == 128 ? 64 : 32;  // keys per staged tile
  constexpr int NSUB = KVB / 32;
  constexpr int NBK = KVB / kBS;            // cache blocks per tile
  constexpr int RS = kNW / GB;              // row subtiles per workgroup
  constexpr int QR = RS * kQB;              // query rows per workgroup
  constexpr int UPR = HD / 8;               // 16-byte units per row
  constexpr int NSTG = KVB * UPR / (kNW * WAVE_SIZE);  // units per thread
  constexpr int NC = HD / 16;               // contraction steps of S
  constexpr int ND = HD / 32;               // column blocks of O

  const int hg_n = G / GB;
  const int kh = blockIdx.x % n_kv;
  const int rest = blockIdx.x / n_kv;
  const int hg = rest % hg_n;
  int tile;
  const int b = __builtin_amdgcn_readfirstlane(
      find_tile(query_start_loc, n_seq, QR, n_tiles_q - 1 - rest / hg_n, &tile));
  const int s0 = query_start_loc[b];
  const int q_len = query_start_loc[b + 1] - s0;
  const int row_lo = __builtin_amdgcn_readfirstlane(tile) * QR;
  if (row_lo >= q_len) return;  // whole workgroup

  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / WAVE_SIZE);
  const int lane = threadIdx.x % WAVE_SIZE;
  const int hi = lane >> 5;
  const int ln31 = lane & 31;
  const int n_q = n_kv * G;
  const int head = kh * G + hg * GB + wave / RS;
  const int wrow0 = row_lo + (wave % RS) * kQB;  // wave's first row in the run

  const int L = seq_lens[b];
  const int ctx = L - q_len;
  const int n_rows = min(QR, q_len - row_lo);
  const int kv_limit = ctx + row_lo + n_rows;  // exclusive, whole workgroup
  const int n_tiles = (kv_limit + KVB - 1) / KVB;
  const int kt0 = WIN ? max(0, ctx + row_lo - window + 1) / KVB : 0;
  const int last_blk = (kv_limit - 1) / kBS;

  __shared__ __attribute__((aligned(16))) char lds[2][2][KVB * HD * 2];

  // ---- queries in registers, B operand per 16-wide step ------------------
  // (a negative scale turns the signs here, so that the largest product is
  // the largest score)
  bf16x8 q_frag[NC];
  {
    const int row = min(wrow0 + ln31, q_len - 1);
    const ushort* qp =
        q + (int64_t)(s0 + row) * q_stride + (int64_t)head * HD + hi * 8;
#pragma unroll
    for (int c = 0; c < NC; ++c) {
      q_frag[c] = *reinterpret_cast<const bf16x8*>(qp + c * 16);
      if (scale < 0.f) {
#pragma unroll
        for (int j = 0; j < 8; ++j) q_frag[c][j] ^= (short)0x8000;
      }
    }
  }
  // (never 0: a masked score is -inf times this)
  const float c2 = fmaxf(fabsf(scale) * (CAP ? 1.0f : kLog2e), 1e-30f);
  const SoftCap cap(CAP ? softcap : 1.0f);
  const int qpos = ctx + wrow0 + ln31;
  const int row_pos_lo = ctx + wrow0;                        // wave's rows
  const int row_pos_hi = ctx + min(wrow0 + kQB, q_len) - 1;  // (may be empty)

  f32x16 o_acc[ND];
#pragma unroll
  for (int d = 0; d < ND; ++d)
#pragma unroll
    for (int r = 0; r < 16; ++r) o_acc[d][r] = 0.f;
  float m_run = -INFINITY, l_run = 0.f;  // l_run: this lane's half of the keys

  // ---- staging: thread's unit i is row (tid / UPR) + i * rows_per_pass ----
  constexpr int RPP = kNW * WAVE_SIZE / UPR;  // rows per pass: 16 or 8
  const int st_row = threadIdx.x / UPR;
  const int st_unit = threadIdx.x % UPR;
  const int32_t* bt = block_tables + (int64_t)b * max_blocks;
  // offset inside a cache block of this thread's unit, even and odd passes
  const int st_src = (st_row % kBS) * HD + st_unit * 8;
  int k_dst[NSTG], v_dst[NSTG];
#pragma unroll
  for (int i = 0; i < NSTG; ++i) {
    const int r = st_row + i * RPP;
    const int vs = ((r & 3) << 1) | ((r >> 2) & 1);
    k_dst[i] = r * HD * 2 + ((st_unit ^ (r & 7)) << 4);
    v_dst[i] = r * HD * 2 + ((st_unit ^ vs) << 4);
  }
  bf16x8 st_k[NSTG], st_v[NSTG];
  int blk_next[NBK];
  auto look_up = [&](int kt) {
#pragma unroll
    for (int j = 0; j < NBK; ++j)
      blk_next[j] = bt[min(kt * NBK + j, last_blk)];
  };
  auto load_tile = [&](int kt) {
    const int valid = kv_limit - kt * KVB;
#pragma unroll
    for (int i = 0; i < NSTG; ++i) {
      const int64_t blk = blk_next[i * RPP / kBS];
      const int64_t base = (blk * n_kv + kh) * (kBS * HD) + (i * RPP % kBS) * HD;
      if constexpr (sizeof(CT) == 2) {
        st_k[i] = *reinterpret_cast<const bf16x8*>(k_cache + base + st_src);
        st_v[i] = *reinterpret_cast<const bf16x8*>(v_cache + base + st_src);
      } else {
        const ushort8 kc = e5m2x8_to_bf16x8(
            *reinterpret_cast<const uint64_t*>(k_cache + base + st_src));
        const ushort8 vc = e5m2x8_to_bf16x8(
            *reinterpret_cast<const uint64_t*>(v_cache + base + st_src));
        st_k[i] = __builtin_bit_cast(bf16x8, kc);
        st_v[i] = __builtin_bit_cast(bf16x8, vc);
      }
      // rows past the last key: their P is 0, but 0 * stale NaN is not
      if (valid < KVB && st_row + i * RPP >= valid) st_v[i] = bf16x8{};
    }
  };
  auto write_tile = [&](int buf) {
#pragma unroll
    for (int i = 0; i < NSTG; ++i) {
      *reinterpret_cast<bf16x8*>(&lds[buf][0][k_dst[i]]) = st_k[i];
      *reinterpret_cast<bf16x8*>(&lds[buf][1][v_dst[i]]) = st_v[i];
    }
  };

  // lane's LDS offsets: K unit (2c + hi) ^ (row & 7) for c & 3; V unit
  // (4d + u) ^ swizzle for d & 1, the rest are immediates
  int k_off[4], v_off[2];
#pragma unroll
  for (int c = 0; c < 4; ++c)
    k_off[c] = ln31 * HD * 2 + (((2 * c + hi) ^ (ln31 & 7)) << 4);
  {
    const int r = 4 * hi + ((lane >> 2) & 3);
    const int vs = ((r & 3) << 1) | (r >> 2);
    const int u = ((lane >> 4) & 1) * 2 + ((lane & 3) >> 1);
#pragma unroll
    for (int d = 0; d < 2; ++d)
      v_off[d] = r * HD * 2 + (((4 * d + u) ^ vs) << 4) + (lane & 1) * 8;
  }

  look_up(kt0);
  load_tile(kt0);
  look_up(kt0 + 1);
  write_tile(0);
  __syncthreads();

  for (int kt = kt0; kt < n_tiles; ++kt) {
    const int cur = (kt - kt0) & 1;
    const int kv_start = kt * KVB;
    const bool have_next = kt + 1 < n_tiles;
    if (have_next) {
      load_tile(kt + 1);
      look_up(kt + 2);
    }

    // tiles all of whose keys lie after (or, windowed, before) the wave's rows
    const bool live = kv_start <= row_pos_hi &&
                      (!WIN || kv_start + KVB - 1 > row_pos_lo - window);
    if (live) {
      // ---- S^T = K . Q^T -------------------------------------------------
      f32x16 s[NSUB];
      const char* kb = lds[cur][0];
#pragma unroll
      for (int sub = 0; sub < NSUB; ++sub)
#pragma unroll
        for (int r = 0; r < 16; ++r) s[sub][r] = 0.f;
#pragma unroll
      for (int c = 0; c < NC; ++c)
#pragma unroll
        for (int sub = 0; sub < NSUB; ++sub) {
          const bf16x8 k_frag = *reinterpret_cast<const bf16x8*>(
              kb + k_off[c & 3] + (c >> 2) * 128 + sub * 32 * HD * 2);
          s[sub] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(k_frag, q_frag[c],
                                                           s[sub], 0, 0, 0);
        }

      // one wave a SIMD has nobody to cover a read of K: four are kept ahead
      // (heads 8/4 x 256, 3029 + 2145: 255 -> 235 us, each read waited for
      // before; two waves a SIMD, at head size 128, cover it themselves)
      if constexpr (HD == 256) {
        constexpr int kMfma = 0x008, kLdsRead = 0x100, kAhead = 4;
        __builtin_amdgcn_sched_group_barrier(kLdsRead, kAhead, 0);
#pragma unroll
        for (int c = 0; c < NC - kAhead; ++c) {
          __builtin_amdgcn_sched_group_barrier(kMfma, 1, 0);
          __builtin_amdgcn_sched_group_barrier(kLdsRead, 1, 0);
        }
        __builtin_amdgcn_sched_group_barrier(kMfma, kAhead, 0);
      }

      // ---- mask, running maximum -----------------------------------------
      if constexpr (CAP) cap.apply(s, c2);
      const bool inside = kv_start + KVB - 1 <= row_pos_lo &&
                          (!WIN || kv_start > row_pos_hi - window);
      if (!inside) {
        const int hi_kv = qpos - kv_start;  // last visible key of the tile
        const int lo_kv = WIN ? hi_kv - window + 1 : 0;
#pragma unroll
        for (int sub = 0; sub < NSUB; ++sub)
#pragma unroll
          for (int r = 0; r < 16; ++r) {
            const int kv = sub * 32 + (r & 3) + 8 * (r >> 2) + 4 * hi;
            const bool see = kv <= hi_kv && (!WIN || kv >= lo_kv);
            s[sub][r] = see ? s[sub][r] : -INFINITY;
          }
      }
      float pmax = s[0][0];
#pragma unroll
      for (int sub = 0; sub < NSUB; ++sub)
#pragma unroll
        for (int r = 0; r < 16; ++r) pmax = fmaxf(pmax, s[sub][r]);
      {  // the other half of the keys
        const auto sw = __builtin_amdgcn_permlane32_swap(
            __float_as_uint(pmax), __float_as_uint(pmax), false, false);
        pmax = fmaxf(__uint_as_float(sw[0]), __uint_as_float(sw[1]));
      }
      const float to_log2 = CAP ? kLog2e : c2;
      pmax = (pmax == -INFINITY) ? pmax : pmax * to_log2;
      // the maximum may lag by 2^11 before everything is rescaled
      if (!__all(pmax <= m_run + 11.0f)) {
        const float m_new = fmaxf(m_run, pmax);
        const float corr = __builtin_amdgcn_exp2f(
            m_run - (m_new == -INFINITY ? 0.f : m_new));
        l_run *= corr;
#pragma unroll
        for (int d = 0; d < ND; ++d)
#pragma unroll
          for (int r = 0; r < 16; ++r) o_acc[d][r] *= corr;
        m_run = m_new;
      }
      const float m_use = (m_run == -INFINITY) ? 0.f : m_run;

      // ---- P, its sum, and the bf16 operand ------------------------------
      bf16x8 p_frag[2 * NSUB];
#pragma unroll
      for (int sub = 0; sub < NSUB; ++sub)
#pragma unroll
        for (int ks = 0; ks < 2; ++ks) {
          u32x4 pk;
#pragma unroll
          for (int j = 0; j < 4; ++j) {
            f32x2 p;
            p[0] = __builtin_amdgcn_exp2f(
                fmaf(s[sub][ks * 8 + 2 * j], to_log2, -m_use));
            p[1] = __builtin_amdgcn_exp2f(
                fmaf(s[sub][ks * 8 + 2 * j + 1], to_log2, -m_use));
            l_run += p[0];
            l_run += p[1];
            pk[j] = __builtin_bit_cast(uint32_t,
                                       __builtin_convertvector(p, bf16x2));
          }
          p_frag[sub * 2 + ks] = __builtin_bit_cast(bf16x8, pk);
        }

      // ---- O^T += V^T . P^T ----------------------------------------------
      const char* vb = lds[cur][1];
#pragma unroll
      for (int ks = 0; ks < 2 * NSUB; ++ks)
#pragma unroll
        for (int d = 0; d < ND; ++d) {
          const char* va = vb + v_off[d & 1] + (d >> 1) * 128 + ks * 16 * HD * 2;
          const bf16x4 v0 = __builtin_amdgcn_ds_read_tr16_b64_v4i16(
              (lds_bf16x4*)(va));
          const bf16x4 v1 = __builtin_amdgcn_ds_read_tr16_b64_v4i16(
              (lds_bf16x4*)(va + 8 * HD * 2));
          const bf16x8 v_frag =
              __builtin_shufflevector(v0, v1, 0, 1, 2, 3, 4, 5, 6, 7);
          o_acc[d] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(
              v_frag, p_frag[ks], o_acc[d], 0, 0, 0);
        }
    }

    // one barrier per tile: the other buffer's last reads ended before the
    // previous barrier
    if (have_next) write_tile(cur ^ 1);
    __syncthreads();
  }

  // ---- normalize and write ------------------------------------------------
  l_run += __shfl_xor(l_run, 32, 64);
  const float inv_l = (l_run > 0.f) ? 1.0f / l_run : 0.f;
  if (wrow0 + ln31 < q_len) {
    ushort* op = out + ((int64_t)(s0 + wrow0 + ln31) * n_q + head) * HD + 4 * hi;
#pragma unroll
    for (int d = 0; d < ND; ++d)
#pragma unroll
      for (int rq = 0; rq < 4; ++rq) {
        ushort4_t o;
#pragma unroll
        for (int j = 0; j < 4; ++j)
          o[j] = f32_to_bf16(o_acc[d][rq * 4 + j] * inv_l);
        *reinterpret_cast<ushort4_t*>(op + d * 32 + rq * 8) = o;
      }
  }
}

}  // namespace

void paged_attention_prefill(torch::Tensor out, torch::Tensor q,
                             torch::Tensor k_cache, torch::Tensor v_cache,
                             torch::Tensor block_tables,
                             torch::Tensor query_start_loc,
                             torch::Tensor seq_lens, double scale,
                             int64_t window, double softcap) {
  TORCH_CHECK(q.stride(2) == 1 && q.stride(1) == q.size(2));
  TORCH_CHECK(out.is_contiguous());
  TORCH_CHECK(k_cache.is_contiguous() && v_cache.is_contiguous());
  TORCH_CHECK(q.scalar_type() == torch::kBFloat16);
  TORCH_CHECK(k_cache.scalar_type() == torch::kBFloat16 ||
              k_cache.scalar_type() == torch::kFloat8_e5m2);
  TORCH_CHECK(block_tables.scalar_type() == torch::kInt32);
  TORCH_CHECK(query_start_loc.scalar_type() == torch::kInt32);
  TORCH_CHECK(seq_lens.scalar_type() == torch::kInt32);
  const int n_q = q.size(1), hd = q.size(2);
  const int n_kv = k_cache.size(1);
  const int B = seq_lens.size(0);
  const int max_blocks = block_tables.size(1);
  TORCH_CHECK(hd == 128 || hd == 256,
              "prefill kernel supports head_dim 128 or 256");
  TORCH_CHECK(k_cache.size(2) == kBS);
  const int G = n_q / n_kv;
  TORCH_CHECK(n_q % n_kv == 0);
  TORCH_CHECK(G == 1 || G == 2 || G == 4 || G == 8,
              "unsupported GQA group size ", G);
  const int Tq = q.size(0);
  if (Tq == 0 || B == 0) return;
  const int GB = std::min(G, 4);
  const int qr = kNW / GB * kQB;
  const int n_tiles_q = Tq / qr + B;  // see find_tile
  const int64_t blocks = (int64_t)n_tiles_q * (G / GB) * n_kv;
  auto stream = c10::hip::getCurrentHIPStream().stream();
  const bool fp8_cache = k_cache.scalar_type() == torch::kFloat8_e5m2;
#define LAUNCH(HDV, GBV, CT, WINV, CAPV)                                     \
  hipLaunchKernelGGL((paged_prefill_kernel<HDV, GBV, CT, WINV, CAPV>),       \
                     dim3((uint32_t)blocks), dim3(kNW * WAVE_SIZE), 0,       \
                     stream, (ushort*)out.data_ptr(),                        \
                     (const ushort*)q.data_ptr(),                            \
                     (const CT*)k_cache.data_ptr(),                          \
                     (const CT*)v_cache.data_ptr(),                          \
                     block_tables.data_ptr<int32_t>(),                       \
                     query_start_loc.data_ptr<int32_t>(),                    \
                     seq_lens.data_ptr<int32_t>(), (float)scale,             \
                     (float)softcap, (int)window, n_kv, G, B, max_blocks,    \
                     q.stride(0), n_tiles_q)
#define LAUNCH_MASK(HDV, GBV, CT)                                            \
  do {                                                                       \
    if (softcap > 0.0) {                                                     \
      if (window > 0) LAUNCH(HDV, GBV, CT, true, true);                      \
      else LAUNCH(HDV, GBV, CT, false, true);                                \
    } else {                                                                 \
      if (window > 0) LAUNCH(HDV, GBV, CT, true, false);                     \
      else LAUNCH(HDV, GBV, CT, false, false);                               \
    }                                                                        \
  } while (0)
#define LAUNCH_CT(HDV, GBV)                                                  \
  do {                                                                       \
    if (fp8_cache) LAUNCH_MASK(HDV, GBV, unsigned char);                     \
    else LAUNCH_MASK(HDV, GBV, ushort);                                      \
  } while (0)
#define LAUNCH_HD(GBV)                                                       \
  do {                                                                       \
    if (hd == 256) LAUNCH_CT(256, GBV);                                      \
    else LAUNCH_CT(128, GBV);                                                \
  } while (0)
  switch (GB) {
    case 1: LAUNCH_HD(1); break;
    case 2: LAUNCH_HD(2); break;
    default: LAUNCH_HD(4); break;
  }
#undef LAUNCH_HD
#undef LAUNCH_CT
#undef LAUNCH_MASK
#undef LAUNCH
  HIP_CHECK_KERNEL();
}
