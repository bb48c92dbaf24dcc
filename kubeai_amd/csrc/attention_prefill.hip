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
//    rows; at head size 128 two workgroups share a CU and overlap one's
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
//  - head size 128: LDS is double-buffered, the next tile's global loads issue
//    before this tile's compute; its cache blocks are looked up one tile earlier
//    with scalar loads. Head size 256 of more than a few keys: paged_prefill_wide_kernel.
//  - the grid numbers the query tiles of the whole packed step (find_tile),
//    kv head fastest: a step of one long prompt and many padding runs
//    launches no empty rows of blocks, and with 8 kv heads each XCD works on
//    one head, whose keys and values stay in its 4 MB L2. (A grid with the
//    sequence fastest put a lone prompt's tiles on two of the eight XCDs
//    when three padding runs came with it.) Late tiles, which see the most
//    keys, start first.
//
// Bound, at head size 128, by the softmax's vector instructions beside the matrix
// instructions (per 64 keys a wave issues 32 MFMAs, 1024 cycles, and about as many
// cycles of max / exp2 / convert; of 8192's cycles the matrix cores have 42 %, those
// 43, LDS 53) and the card's power: forms with 5 % fewer cycles run at 5 % less clock.
// Measured (us; before: 8-wave kernel for plain causal head size 128, 16-row
// kernel for the rest):
//   heads 32/8 x 128, one prompt of 2048                205 ->  69 (501 TF/s)
//     the same with 3 padding runs                      510 ->  68
//   8192                                               1840 -> 666 (826 TF/s)
//   8192, window 4096                                  2797 -> 488
//   512 new tokens behind 3584                          414 -> 100
//   six turns of 62-100 behind 365-587, 4 padding runs   72 ->  23
//   heads 64/8 x 128, 4096                              927 -> 360
//   heads 8/4 x 256, 3029 + 2145, cap, window 4096     1574 -> 146 (385 TF/s)
//
// Fragment layouts:
//   A[M=32][K=16]: lane l holds A[l&31][(l>>5)*8 + j], j=0..7
//   B[K=16][N=32]: lane l holds B[(l>>5)*8 + j][l&31]
//   C[M=32][N=32]: lane l holds C[(r&3) + 8*(r>>2) + 4*(l>>5)][l&31]
//   ds_read_b64_tr_b16: in each group of 16 lanes, lane l's element j comes
//   from the 8 bytes addressed by lane 4j + (l>>2), element l&3
#include <torch/extension.h>

#include <algorithm>
#include <type_traits>

#include "attention_decode.h"
#include "common.h"

namespace {

constexpr int kBS = 16;  // cache block size (tokens)
constexpr int kQB = 32;  // query rows per wave
constexpr int kNW = 4;   // waves per workgroup
// Head size 256, at most so many keys a workgroup: one tile after the other instead of
// three under way at a time, whose beginning and end take longer (us, that / one after the
// other: 4 tokens 10.4 / 6.2, 20 10.8 / 7.1, 52 + 64 15.5 / 13.6). Over 399 steps of 1 to 40
// runs one after the other takes 0.64 of the time up to 32 keys, 0.85 up to 96, 0.96 up
// to 160, 0.99 up to 192, 1.04 up to 288 and 1.28 above 600.
constexpr int kFewKeys = 192;

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

// Head size 128, and 256 where no row has many keys (kFewKeys). CT = cache element
// type: ushort (bf16) or unsigned char (fp8 e5m2, converted to bf16 while staging). CAP:
// capped scores. WIN: keys in (pos - window, pos] only.
constexpr int tile_keys(int hd) { return hd == 128 ? 64 : 32; }
template <int HD>
using Tiles = char[2][2][tile_keys(HD) * HD * 2];  // places, K and V

template <int HD, int GB, typename CT, bool WIN, bool CAP>
DEV_INLINE void attend_rows(
    Tiles<HD>& lds, const int block,
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
  constexpr int KVB = tile_keys(HD);  // keys per staged tile
  constexpr int NSUB = KVB / 32;
  constexpr int NBK = KVB / kBS;            // cache blocks per tile
  constexpr int RS = kNW / GB;              // row subtiles per workgroup
  constexpr int QR = RS * kQB;              // query rows per workgroup
  constexpr int UPR = HD / 8;               // 16-byte units per row
  constexpr int NSTG = KVB * UPR / (kNW * WAVE_SIZE);  // units per thread
  constexpr int NC = HD / 16;               // contraction steps of S
  constexpr int ND = HD / 32;               // column blocks of O

  const int hg_n = G / GB;
  const int kh = block % n_kv;
  const int rest = block / n_kv;
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

template <int HD, int GB, typename CT, bool WIN, bool CAP>
__launch_bounds__(kNW * WAVE_SIZE, HD == 128 ? 2 : 1) __global__
void paged_prefill_kernel(
    ushort* __restrict__ out, const ushort* __restrict__ q, const CT* __restrict__ k_cache,
    const CT* __restrict__ v_cache, const int32_t* __restrict__ block_tables,
    const int32_t* __restrict__ query_start_loc, const int32_t* __restrict__ seq_lens,
    const float scale, const float softcap, const int window, const int n_kv, const int G,
    const int n_seq, const int max_blocks, const int64_t q_stride, const int n_tiles_q) {
  __shared__ __attribute__((aligned(16))) Tiles<HD> lds;
  attend_rows<HD, GB, CT, WIN, CAP>(lds, blockIdx.x, out, q, k_cache, v_cache, block_tables,
                                    query_start_loc, seq_lens, scale, softcap, window, n_kv, G,
                                    n_seq, max_blocks, q_stride, n_tiles_q);
}

// A step's prompt portions and its decode rows (head size 128, planned splits) in one
// launch: neither fills the chip by itself, and each is a chain of latencies. The first
// workgroups are the prompts', the longest of them first; the decode splits go where
// there is room beside and behind them, two workgroups a CU by the prompts' registers.
// us, two launches / this, each with the merge (heads 32/8): 32 rows of 100-700 and six
// turns of 48-112 behind 300-600 43.0 / 36.7, to fp8 46.0 / 38.8; 28 rows and four prompts
// of 20-120 25.4 / 18.7; 40 rows of 50-1000 and 17 tokens 30.1 / 22.1, 300 tokens 37.1 /
// 27.0, 2000 tokens 91.9 / 82.7, 6000 tokens 372 / 366; 96 of 1500-4000 and 100 tokens
// 208 / 199; one row and 20 tokens 13.4 / 9.1. The results are the same bits.
template <int GB, typename CT, bool WIN, bool CAP>
__launch_bounds__(kNW * WAVE_SIZE, 2) __global__ void step_attention_kernel(
    ushort* __restrict__ out,  // [T, n_q, 128], the decode rows first
    ushort* __restrict__ decode_out,  // the same, or null: parts of all decode rows
    const ushort* __restrict__ q, CT* k_cache, CT* v_cache,
    const int32_t* __restrict__ prompt_tables, const int32_t* __restrict__ query_start_loc,
    const int32_t* __restrict__ prompt_lens, const int32_t* __restrict__ decode_tables,
    const int32_t* __restrict__ decode_lens, const float scale, const float softcap,
    const int window, const int n_kv, const int G, const int n_seq, const int prompt_blocks,
    const int decode_blocks, const int64_t q_stride, const int n_tiles_q, const int n_decode,
    const int prompt_wgs, const decode::Item* __restrict__ plan, float* __restrict__ part_o,
    float* __restrict__ part_ml) {
  static_assert(kNW == decode::kWaves);
  using Own = decode::Lds<128, CT, 0>;
  __shared__ __attribute__((aligned(16))) char mem[std::max(sizeof(Tiles<128>), sizeof(Own))];
  if ((int)blockIdx.x < prompt_wgs) {
    attend_rows<128, GB, CT, WIN, CAP>(
        *reinterpret_cast<Tiles<128>*>(mem), blockIdx.x, out + (int64_t)n_decode * n_kv * G * 128,
        q + n_decode * q_stride, k_cache, v_cache, prompt_tables, query_start_loc, prompt_lens,
        scale, softcap, window, n_kv, G, n_seq, prompt_blocks, q_stride, n_tiles_q);
  } else {
    decode::attend_split<128, CT, CAP, false, 0>(
        *reinterpret_cast<Own*>(mem), blockIdx.x - prompt_wgs, decode_out, q, k_cache, v_cache,
        decode_tables, decode_lens, scale, softcap, window, n_kv, G, decode_blocks, q_stride, 1,
        plan, decode::NewRows{}, part_o, part_ml);
  }
}

// one place of the ring after another
DEV_INLINE int ring3(int i) { return i >= 3 ? i - 3 : i; }

// v is worked out here: the compiler would take it to where it is read, behind the
// matrix instructions that are to cover it
DEV_INLINE void here(float& v) { asm volatile("" : "+v"(v)); }
DEV_INLINE void here(uint32_t& v) { asm volatile("" : "+v"(v)); }

// f(B), ... f(E - 1) with the numbers as types
template <int B, int E, typename F>
DEV_INLINE void each(const F& f) {
  if constexpr (B < E) {
    f(std::integral_constant<int, B>{});
    each<B + 1, E>(f);
  }
}

// Head size 256: O and Q take 192 registers of a lane, so there is one wave a SIMD, and
// what it waits for nobody else covers. So three tiles of 32 keys are under way at a
// time: S of tile t + 1, the softmax of tile t and P V of tile t - 1, none of which
// waits for another. Behind each of the 32 matrix instructions of an iteration stands a
// part of the rest, in this order (32 cycles for it; at one wave an instruction takes 5
// to issue, whatever it is, and that is what bounds the loop now: about 400 of them):
// reads of V, then of the next K, into registers; the softmax, no step of which waits for
// another of its slot; registers to LDS (three places for K and V each), the next
// tiles' loads and the blocks after them.
//   heads 8/4 x 256, 3029 + 2145: 231 us -> 115, capped, no window 262 -> 141; 500 capped
// 41 -> 32
// The same at head size 128, 64 rows a wave: 8192 as long as with two waves a SIMD and
// half the rows (611 us, 606: more clocks at a higher rate; the card's power), shorter
// prompts 1.3 times.
// 2^rs_bits waves are on the rows of a head.
template <typename CT, bool WIN, bool CAP>
__launch_bounds__(kNW * WAVE_SIZE, 1) __global__ void paged_prefill_wide_kernel(
    ushort* __restrict__ out,          // [Tq, n_q, HD]
    const ushort* __restrict__ q,      // [Tq, n_q, HD], rows strided
    const CT* __restrict__ k_cache,    // [nb, n_kv, 16, HD]
    const CT* __restrict__ v_cache,
    const int32_t* __restrict__ block_tables,     // [B, max_blocks]
    const int32_t* __restrict__ query_start_loc,  // [B+1]
    const int32_t* __restrict__ seq_lens,         // [B]
    const float scale, const float softcap, const int window,
    const int n_kv, const int G, const int n_seq, const int max_blocks,
    const int64_t q_stride, const int n_tiles_q, const int rs_bits) {
  constexpr int HD = 256;
  constexpr int KVB = 32;                   // keys per tile
  constexpr int NBK = KVB / kBS;            // cache blocks per tile
  constexpr int UPR = HD / 8;               // 16-byte units per row
  constexpr int NSTG = KVB * UPR / (kNW * WAVE_SIZE);  // units per thread
  constexpr int NC = HD / 16;               // contraction steps of S
  constexpr int ND = HD / 32;               // column blocks of O
  constexpr int TB = KVB * HD * 2;          // bytes of a tile in LDS

  const int GB = kNW >> rs_bits;            // heads per workgroup
  const int QR = kQB << rs_bits;            // its rows
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
  const int head = kh * G + hg * GB + (wave >> rs_bits);
  const int wrow0 = row_lo + (wave & ((1 << rs_bits) - 1)) * kQB;  // wave's first row in the run

  const int L = seq_lens[b];
  const int ctx = L - q_len;
  const int n_rows = min(QR, q_len - row_lo);
  const int kv_limit = ctx + row_lo + n_rows;  // exclusive, whole workgroup
  const int n_tiles = (kv_limit + KVB - 1) / KVB;
  const int kt0 = WIN ? max(0, ctx + row_lo - window + 1) / KVB : 0;
  const int last_blk = (kv_limit - 1) / kBS;
  // tiles with keys that the wave's rows see: [t_lo, t_hi) (none: never)
  const int row_pos_lo = ctx + wrow0;
  const int row_pos_hi = ctx + min(wrow0 + kQB, q_len) - 1;
  const bool any = wrow0 < q_len;
  const int t_lo = !any ? 1 << 30 : WIN ? max(0, row_pos_lo - window + 1) / KVB : 0;
  const int t_hi = any ? row_pos_hi / KVB + 1 : 1 << 30;

  // K: three places; V: three and zeros, what the first tile has in front of it
  __shared__ __attribute__((aligned(16))) char lds_k[3 * TB], lds_v[4 * TB];

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
      asm volatile("" : "+a"(q_frag[c]));  // leaves the others to the softmax
    }
  }
  // (never 0: a masked score is -inf times this)
  const float c2 = fmaxf(fabsf(scale) * (CAP ? 1.0f : kLog2e), 1e-30f);
  const float to_log2 = CAP ? kLog2e : c2;
  const SoftCap cap(CAP ? softcap : 1.0f);

  f32x16 o_acc[ND];
  float m_run = -INFINITY, l_run = 0.f;  // l_run: this lane's half of the keys
#pragma unroll
  for (int d = 0; d < ND; ++d) {
#pragma unroll
    for (int r = 0; r < 16; ++r) o_acc[d][r] = 0.f;
    // (of a constant at the loop's entry the compiler makes 16 loop variables)
    asm volatile("" : "+a"(o_acc[d]));
  }

  // ---- staging: thread's unit i is row (tid / UPR) + i * rows_per_pass ----
  constexpr int RPP = kNW * WAVE_SIZE / UPR;  // rows per pass: 8
  constexpr int PB = NSTG / NBK;              // passes per cache block
  const int st_row = threadIdx.x / UPR;
  const int st_unit = threadIdx.x % UPR;
  const int32_t* bt = block_tables + (int64_t)b * max_blocks;
  const uint32_t st_src = ((st_row % kBS) * HD + st_unit * 8) * sizeof(CT);
  const char* k_head = (const char*)(k_cache + (int64_t)kh * (kBS * HD));
  const char* v_head = (const char*)(v_cache + (int64_t)kh * (kBS * HD));
  const uint64_t blk_bytes = (uint64_t)n_kv * (kBS * HD) * sizeof(CT);
  int k_dst[NSTG], v_dst[NSTG];
#pragma unroll
  for (int i = 0; i < NSTG; ++i) {
    const int r = st_row + i * RPP;
    const int vs = ((r & 3) << 1) | ((r >> 2) & 1);
    k_dst[i] = r * HD * 2 + ((st_unit ^ (r & 7)) << 4);
    v_dst[i] = r * HD * 2 + ((st_unit ^ vs) << 4);
  }
  typedef typename std::conditional<sizeof(CT) == 2, bf16x8, uint64_t>::type Raw;
  // block j of tile kt (past the last key: the last one again)
  auto block = [&](int kt, int j) { return (uint32_t)bt[min(kt * NBK + j, last_blk)]; };
  auto load = [&](const char* head, uint32_t blk, int i) {
    return *reinterpret_cast<const Raw*>(head + blk * blk_bytes +
                                         i % PB * RPP * HD * sizeof(CT) + st_src);
  };
  auto widen = [](const Raw& r) {
    if constexpr (sizeof(CT) == 2) return r;
    else return __builtin_bit_cast(bf16x8, e5m2x8_to_bf16x8(r));
  };
  auto put_k = [&](int base, int i, const Raw& st) {
    *reinterpret_cast<bf16x8*>(&lds_k[base + k_dst[i]]) = widen(st);
  };
  // rows past the last key: their P is 0, but 0 * stale NaN is not
  auto put_v = [&](int base, int i, const Raw& st, int valid) {
    bf16x8 v = widen(st);
    if (valid < KVB) {
      if (st_row + i * RPP >= valid) v = bf16x8{};
      asm volatile("" ::: "memory");  // (a branch, not a selection for every tile)
    }
    *reinterpret_cast<bf16x8*>(&lds_v[base + v_dst[i]]) = v;
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
  bf16x8 kf[NC], vf[2 * ND];
  auto read_k = [&](int c, int base) {  // base: of the tile's place
    kf[c] = *reinterpret_cast<const bf16x8*>(&lds_k[base + k_off[c & 3] + (c >> 2) * 128]);
  };
  auto read_v = [&](int i, int base) {  // i: 16 keys (i / ND), 32 columns (i % ND)
    const int ks = i / ND, d = i % ND;
    const char* va = &lds_v[base + v_off[d & 1] + (d >> 1) * 128 + ks * 16 * HD * 2];
    const bf16x4 v0 = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_bf16x4*)(va));
    const bf16x4 v1 =
        __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_bf16x4*)(va + 8 * HD * 2));
    vf[i] = __builtin_shufflevector(v0, v1, 0, 1, 2, 3, 4, 5, 6, 7);
  };

  // scores and weights of the current tile and of the next / the last one
  f32x16 s[2];
  bf16x8 p[2][2] = {};

  constexpr int NQ = NC, NP = 2 * ND, SLOTS = NQ + NP;  // matrix instructions
  constexpr int NW = 16;                                // scores of a lane
  constexpr int kCapItems = CAP ? NW : 0;               // one score each
  constexpr int kFirstMax = kCapItems + (CAP ? 1 : 0);  // 4 scores each
  constexpr int kFirstUpdate = kFirstMax + NW / 4;      // in two steps
  constexpr int kFirstWeight = kFirstUpdate + 2;        // in three, one behind another
  constexpr int kItems = kFirstWeight + NW + 2;
  // weight of the items in front of item i (10 cycles), the first item behind matrix
  // instruction t
  constexpr auto before = [](int i) constexpr {
    int w = 0;
    for (int k = 0; k < i; ++k)
      w += k < kCapItems ? 6 : k < kFirstMax ? 2 : k < kFirstUpdate ? 1 : 3;
    return w;
  };
  constexpr int kWeight = before(kItems);
  constexpr auto item_of = [before](int t) constexpr {
    int i = 0;
    while (i < kItems && before(i) * SLOTS / kWeight < t) ++i;
    return i;
  };

  Raw st_k[NSTG], st_v[NSTG];
  uint32_t blk_k[NBK], blk_v[NBK];
  auto iteration = [&](auto parity, int kt, int place, int v_base, int k_base) {
    constexpr int J = decltype(parity)::value;
    // what the registers hold goes to LDS, then the next tiles' loads, then the blocks of
    // those behind them
    const int to_k = place * TB, to_v = ring3(place + 1) * TB;
    const int valid = kv_limit - (kt + 1) * KVB;
    auto staging = [&](auto slot) {
      constexpr int t = decltype(slot)::value;
      constexpr int n = SLOTS / 2 / (2 * NSTG);  // slots a write or a load
      if constexpr (t % n == n - 1) {
        constexpr int i = t / n % (2 * NSTG), j = i % NSTG;
        if constexpr (t < SLOTS / 2) {
          if constexpr (i < NSTG) put_k(to_k, j, st_k[j]);
          else put_v(to_v, j, st_v[j], valid);
        } else if constexpr (i < NSTG) {
          st_k[j] = load(k_head, blk_k[j / PB], j);
          if constexpr (j % PB == PB - 1) blk_k[j / PB] = block(kt + 5, j / PB);
        } else {
          st_v[j] = load(v_head, blk_v[j / PB], j);
          if constexpr (j % PB == PB - 1) blk_v[j / PB] = block(kt + 3, j / PB);
        }
      }
    };
    f32x16& sc = s[J];
    const int kv_start = kt * KVB;
    float pmax, m_use, corr;
    bool grow = false;
    float amax = 0.f;
    f32x16 raw;
    const bool inside =
        kv_start + KVB - 1 <= row_pos_lo && (!WIN || kv_start > row_pos_hi - window);
    auto mask = [&] {
      if (inside) return;
      const int hi_kv = row_pos_lo + ln31 - kv_start;  // last visible key of the tile
      const int lo_kv = WIN ? hi_kv - window + 1 : 0;
#pragma unroll
      for (int r = 0; r < 16; ++r) {
        const int kv = (r & 3) + 8 * (r >> 2) + 4 * hi;
        const bool see = kv <= hi_kv && (!WIN || kv >= lo_kv);
        sc[r] = see ? sc[r] : -INFINITY;
      }
    };
    float top, t[NW], e[NW];
    auto item = [&](auto number) {
      constexpr int i = decltype(number)::value;
      if constexpr (i < kCapItems) {
        const float x = sc[i] * c2;
        raw[i] = x;
        amax = fmaxf(amax, fabsf(x));
        float y = cap.small(x);
        here(y);
        sc[i] = y;
      } else if constexpr (i < kFirstMax) {
        if (__builtin_expect(__any(amax >= cap.edge), 0)) {
#pragma unroll
          for (int r = 0; r < 16; ++r) {
            float l = cap.large(raw[r]);
            here(l);  // a selection, not a branch per value
            sc[r] = fabsf(raw[r]) >= cap.edge ? l : sc[r];
          }
        }
        mask();
      } else if constexpr (i < kFirstUpdate) {
        constexpr int r = (i - kFirstMax) * 4;
        const float m = fmaxf(fmaxf(sc[r], sc[r + 1]), r ? pmax : sc[r]);
        pmax = fmaxf(fmaxf(sc[r + 2], sc[r + 3]), m);
        here(pmax);
      } else if constexpr (i == kFirstUpdate) {
        // the other half of the keys
        const auto sw = __builtin_amdgcn_permlane32_swap(
            __float_as_uint(pmax), __float_as_uint(pmax), false, false);
        top = fmaxf(__uint_as_float(sw[0]), __uint_as_float(sw[1])) * to_log2;
        here(top);
      } else if constexpr (i < kFirstWeight) {
        // the maximum may lag by 2^11 before everything is rescaled
        grow = top > m_run + 11.0f;
        corr = grow ? __builtin_amdgcn_exp2f(m_run - top) : 1.0f;
        m_run = grow ? top : m_run;
        l_run *= corr;
        m_use = m_run == -INFINITY ? 0.f : m_run;
        here(m_use);
        here(l_run);
      } else {
        constexpr int w = i - kFirstWeight;  // no step waits for one of its own slot
        if constexpr (w >= 2) {
          constexpr int k = w - 2;
          l_run += e[k];
          here(l_run);
          if constexpr (k % 2) {
            f32x2 both = {e[k - 1], e[k]};
            uint32_t h = __builtin_bit_cast(uint32_t, __builtin_convertvector(both, bf16x2));
            here(h);
            u32x4 all = __builtin_bit_cast(u32x4, p[J][k / 8]);
            all[k % 8 / 2] = h;
            p[J][k / 8] = __builtin_bit_cast(bf16x8, all);
          }
        }
        if constexpr (w >= 1 && w <= NW) {
          e[w - 1] = __builtin_amdgcn_exp2f(t[w - 1]);
          here(e[w - 1]);
        }
        if constexpr (w < NW) {
          t[w] = fmaf(sc[w], to_log2, -m_use);
          here(t[w]);
        }
      }
    };
    if constexpr (!CAP) mask();
    each<0, SLOTS>([&](auto slot) {
      constexpr int t = decltype(slot)::value;
      if constexpr (t < NQ) {
        f32x16 z = {};
        if constexpr (t > 0) z = s[J ^ 1];
        s[J ^ 1] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(kf[t], q_frag[t], z, 0, 0, 0);
        each<2 * ND * t / NQ, 2 * ND * (t + 1) / NQ>(
            [&](auto i) { read_v(decltype(i)::value, v_base); });
      } else {
        constexpr int x = t - NQ;
        o_acc[x % ND] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(
            vf[x], p[J ^ 1][x / ND], o_acc[x % ND], 0, 0, 0);
        each<NC * (t - NQ) / NP, NC * (t - NQ + 1) / NP>(
            [&](auto c) { read_k(decltype(c)::value, k_base); });
      }
      staging(slot);
      each<item_of(t), t + 1 < SLOTS ? item_of(t + 1) : kItems>(item);
      __builtin_amdgcn_sched_barrier(0);
    });
    // (read in the registers that the softmax reaches; no read of LDS goes beyond)
    asm volatile("" : "+v"(s[J ^ 1])::"memory");
    if (__any(grow)) {
      // in the registers that only matrix instructions (and moves) reach: taken through
      // the others the compiler would move all of O there and back for each unit.
      // (s_nop: a matrix instruction's result is there after up to 18 cycles' worth)
      asm volatile("s_nop 15\n\ts_nop 15");
#pragma unroll
      for (int d = 0; d < ND; ++d) {
#pragma unroll
        for (int r = 0; r < 16; ++r) {
          float o = o_acc[d][r], x;
          asm volatile("v_accvgpr_read_b32 %1, %0\n\tv_mul_f32 %1, %1, %2\n\t"
                       "v_accvgpr_write_b32 %0, %1"
                       : "+a"(o), "=&v"(x)
                       : "v"(corr));
          o_acc[d][r] = o;
        }
        asm volatile("" : "+a"(o_acc[d]));
      }
      asm volatile("s_nop 7");
    }
  };
  for (int i = threadIdx.x * 16; i < TB; i += kNW * WAVE_SIZE * 16)
    *reinterpret_cast<bf16x8*>(&lds_v[3 * TB + i]) = bf16x8{};

  // ---- at the start of tile t LDS has K of t .. t + 2, V of t - 1 and t, the registers
  // K of t + 3 and V of t + 1. Tile kt0 + i lies in place i % 3 ----------------------
  {
    Raw first[4][NSTG];
#pragma unroll
    for (int i = 0; i < NSTG; ++i) {
#pragma unroll
      for (int k = 0; k < 3; ++k) first[k][i] = load(k_head, block(kt0 + k, i / PB), i);
      first[3][i] = load(v_head, block(kt0, i / PB), i);
    }
#pragma unroll
    for (int i = 0; i < NSTG; ++i) {
#pragma unroll
      for (int k = 0; k < 3; ++k) put_k(k * TB, i, first[k][i]);
      put_v(0, i, first[3][i], kv_limit - kt0 * KVB);
    }
  }
#pragma unroll
  for (int i = 0; i < NSTG; ++i) {
    st_k[i] = load(k_head, block(kt0 + 3, i / PB), i);
    st_v[i] = load(v_head, block(kt0 + 1, i / PB), i);
  }
#pragma unroll
  for (int j = 0; j < NBK; ++j) {
    blk_k[j] = block(kt0 + 4, j);
    blk_v[j] = block(kt0 + 2, j);
  }
  __syncthreads();

  each<0, NC>([&](auto c) { read_k(decltype(c)::value, 0); });
#pragma unroll
  for (int r = 0; r < 16; ++r) s[0][r] = 0.f;
#pragma unroll
  for (int c = 0; c < NC; ++c)
    s[0] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(kf[c], q_frag[c], s[0], 0, 0, 0);
  each<0, NC>([&](auto c) { read_k(decltype(c)::value, TB); });
  int place = 0;  // of the current tile
  // V of tile t, zeros for one that the wave's rows do not see (its P is 0)
  auto v_of = [&](int t) {
    return (t >= t_lo && t < t_hi ? ring3(place + 2) : 3) * TB;
  };
  // (an odd number of tiles: one more, of no key that a row sees)
  int kt = kt0;
  for (; kt < n_tiles; kt += 2) {
    iteration(std::integral_constant<int, 0>{}, kt, place, v_of(kt - 1),
              ring3(place + 2) * TB);
    __syncthreads();
    place = ring3(place + 1);
    iteration(std::integral_constant<int, 1>{}, kt + 1, place, v_of(kt),
              ring3(place + 2) * TB);
    __syncthreads();
    place = ring3(place + 1);
  }
  const int v_last = v_of(kt - 1);
  each<0, 2 * ND>([&](auto number) {
    constexpr int x = decltype(number)::value;
    read_v(x, v_last);
    o_acc[x % ND] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(vf[x], p[1][x / ND],
                                                            o_acc[x % ND], 0, 0, 0);
  });

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
  // at most, of a workgroup's rows
  const int64_t keys =
      std::min((int64_t)max_blocks * kBS, window > 0 ? window + qr : INT64_MAX);
  auto stream = c10::hip::getCurrentHIPStream().stream();
  const bool fp8_cache = k_cache.scalar_type() == torch::kFloat8_e5m2;
  auto launch = [&](auto kernel, auto ct, auto... more) {
    using CT = decltype(ct);
    hipLaunchKernelGGL(kernel, dim3((uint32_t)blocks), dim3(kNW * WAVE_SIZE), 0, stream,
                       (ushort*)out.data_ptr(), (const ushort*)q.data_ptr(),
                       (const CT*)k_cache.data_ptr(), (const CT*)v_cache.data_ptr(),
                       block_tables.data_ptr<int32_t>(),
                       query_start_loc.data_ptr<int32_t>(), seq_lens.data_ptr<int32_t>(),
                       (float)scale, (float)softcap, (int)window, n_kv, G, B, max_blocks,
                       q.stride(0), n_tiles_q, more...);
  };
  auto masks = [&](auto f) {
    if (softcap > 0.0) {
      if (window > 0) f(std::true_type{}, std::true_type{});
      else f(std::false_type{}, std::true_type{});
    } else {
      if (window > 0) f(std::true_type{}, std::false_type{});
      else f(std::false_type{}, std::false_type{});
    }
  };
  auto sizes = [&](auto ct) {
    using CT = decltype(ct);
    masks([&](auto win, auto cap) {
      constexpr bool W = decltype(win)::value, C = decltype(cap)::value;
      auto heads = [&](auto hdv) {
        constexpr int HD = decltype(hdv)::value;
        if (GB == 1) launch(paged_prefill_kernel<HD, 1, CT, W, C>, ct);
        else if (GB == 2) launch(paged_prefill_kernel<HD, 2, CT, W, C>, ct);
        else launch(paged_prefill_kernel<HD, 4, CT, W, C>, ct);
      };
      if (hd == 128) {
        heads(std::integral_constant<int, 128>{});
      } else if (keys <= kFewKeys) {
        heads(std::integral_constant<int, 256>{});
      } else {
        const int rs_bits = GB == 4 ? 0 : GB == 2 ? 1 : 2;
        launch(paged_prefill_wide_kernel<CT, W, C>, ct, rs_bits);
      }
    });
  };
  if (fp8_cache) sizes((unsigned char)0);
  else sizes((ushort)0);
  HIP_CHECK_KERNEL();
}

// paged_attention_prefill of rows n_decode.. of q [T, n_q, 128] and paged_attention_decode
// of those before, by a plan, in one launch and the merge of the decode rows' splits. out
// [T, n_q, 128] bf16, or (out_scale fp32 [T]) [T, n_q * 128] fp8 rows with a scale each,
// which the merge makes of up to 32 heads.
void paged_attention_step(torch::Tensor out, c10::optional<torch::Tensor> out_scale,
                          torch::Tensor q, int64_t n_decode, torch::Tensor k_cache,
                          torch::Tensor v_cache, torch::Tensor decode_tables,
                          torch::Tensor decode_lens, torch::Tensor plan,
                          torch::Tensor prompt_tables, torch::Tensor query_start_loc,
                          torch::Tensor prompt_lens, double scale, int64_t window,
                          double softcap) {
  TORCH_CHECK(q.dim() == 3 && q.stride(2) == 1 && q.stride(1) == 128 && q.size(2) == 128 &&
              q.scalar_type() == torch::kBFloat16 && q.is_cuda());
  TORCH_CHECK(k_cache.is_contiguous() && v_cache.is_contiguous() && k_cache.dim() == 4 &&
              v_cache.sizes() == k_cache.sizes() && k_cache.size(2) == kBS &&
              k_cache.size(3) == 128 && v_cache.scalar_type() == k_cache.scalar_type());
  TORCH_CHECK(k_cache.scalar_type() == torch::kBFloat16 ||
              k_cache.scalar_type() == torch::kFloat8_e5m2);
  for (const auto& t : {decode_tables, decode_lens, prompt_tables, query_start_loc, prompt_lens})
    TORCH_CHECK(t.scalar_type() == torch::kInt32 && t.is_contiguous() && t.is_cuda());
  const int64_t T = q.size(0), n_q = q.size(1);
  const int n_kv = k_cache.size(1), G = n_q / n_kv, B = prompt_lens.numel();
  const int64_t D = n_decode, Tq = T - D;
  TORCH_CHECK(n_q % n_kv == 0 && (G == 1 || G == 2 || G == 4 || G == 8),
              "unsupported GQA group size ", G);
  TORCH_CHECK(D >= 1 && Tq >= 1 && B >= 1 && decode_lens.numel() == D &&
              decode_tables.dim() == 2 && decode_tables.size(0) == D &&
              prompt_tables.dim() == 2 && prompt_tables.size(0) == B &&
              query_start_loc.numel() == B + 1);
  decode_tables = decode::with_a_column(decode_tables);
  decode::check_plan(plan, D, n_kv);
  const bool fp8 = out_scale.has_value();
  TORCH_CHECK(out.is_contiguous() && out.is_cuda() && out.numel() == T * n_q * 128 &&
              out.scalar_type() == (fp8 ? torch::kFloat8_e4m3fn : torch::kBFloat16));
  if (fp8)
    TORCH_CHECK(n_q <= 32 && out_scale->is_contiguous() && out_scale->is_cuda() &&
                out_scale->scalar_type() == torch::kFloat32 && out_scale->numel() == T);
  const int64_t items = decode::plan_items(D, n_kv);
  const auto* item = reinterpret_cast<const decode::Item*>(plan.data_ptr());
  const auto* splits = reinterpret_cast<const decode::Splits*>(item + items);
  const auto opts = q.options().dtype(torch::kFloat32);
  auto part_o = torch::empty({items, n_q, 128}, opts), part_ml = torch::empty({items, n_q, 2}, opts);
  auto rows = fp8 ? torch::empty({T, n_q, 128}, q.options()) : out;
  const int GB = std::min(G, 4), qr = kNW / GB * kQB;
  const int n_tiles_q = Tq / qr + B;  // see find_tile
  const int64_t prompt_wgs = (int64_t)n_tiles_q * (G / GB) * n_kv;
  TORCH_CHECK(prompt_wgs + items * n_kv < (int64_t)1 << 31);
  auto stream = c10::hip::getCurrentHIPStream().stream();
  auto launch = [&](auto gb, auto ct, auto win, auto cap) {
    using CT = decltype(ct);
    hipLaunchKernelGGL(
        (step_attention_kernel<decltype(gb)::value, CT, decltype(win)::value,
                               decltype(cap)::value>),
        dim3((uint32_t)(prompt_wgs + items * n_kv)), dim3(kNW * WAVE_SIZE), 0, stream,
        (ushort*)rows.data_ptr(), fp8 ? nullptr : (ushort*)rows.data_ptr(),
        (const ushort*)q.data_ptr(), (CT*)k_cache.data_ptr(), (CT*)v_cache.data_ptr(),
        prompt_tables.data_ptr<int32_t>(), query_start_loc.data_ptr<int32_t>(),
        prompt_lens.data_ptr<int32_t>(), decode_tables.data_ptr<int32_t>(),
        decode_lens.data_ptr<int32_t>(), (float)scale, (float)softcap, (int)window, n_kv, G, B,
        (int)prompt_tables.size(1), (int)decode_tables.size(1), q.stride(0), n_tiles_q, (int)D,
        (int)prompt_wgs, item, part_o.data_ptr<float>(), part_ml.data_ptr<float>());
  };
  auto masks = [&](auto gb, auto ct) {
    if (window > 0) {
      if (softcap > 0.0) launch(gb, ct, std::true_type{}, std::true_type{});
      else launch(gb, ct, std::true_type{}, std::false_type{});
    } else {
      if (softcap > 0.0) launch(gb, ct, std::false_type{}, std::true_type{});
      else launch(gb, ct, std::false_type{}, std::false_type{});
    }
  };
  auto heads = [&](auto ct) {
    if (GB == 1) masks(std::integral_constant<int, 1>{}, ct);
    else if (GB == 2) masks(std::integral_constant<int, 2>{}, ct);
    else masks(std::integral_constant<int, 4>{}, ct);
  };
  if (k_cache.scalar_type() == torch::kFloat8_e5m2) heads((unsigned char)0);
  else heads((ushort)0);
  HIP_CHECK_KERNEL();
  if (fp8) {
    auto merge = [&](auto hpw) {
      hipLaunchKernelGGL((decode::decode_merge_fp8_kernel<128, decltype(hpw)::value>),
                         dim3((uint32_t)T), dim3(16 * WAVE_SIZE), 0, stream,
                         (unsigned char*)out.data_ptr(), out_scale->data_ptr<float>(),
                         (const ushort*)rows.data_ptr(), (int)D, part_o.data_ptr<float>(),
                         part_ml.data_ptr<float>(), splits, 1, (int)n_q);
    };
    if (n_q <= 16) merge(std::integral_constant<int, 1>{});
    else merge(std::integral_constant<int, 2>{});
  } else {
    const int64_t n_bh = D * n_q;
    hipLaunchKernelGGL((decode::decode_merge_kernel<128>), dim3((uint32_t)((n_bh + 3) / 4)),
                       dim3(4 * WAVE_SIZE), 0, stream, (ushort*)out.data_ptr(),
                       part_o.data_ptr<float>(), part_ml.data_ptr<float>(), splits, 1, (int)n_q,
                       n_bh);
  }
  HIP_CHECK_KERNEL();
}
