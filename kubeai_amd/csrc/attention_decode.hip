// Paged-attention decode (one new token per sequence) for gfx950.
//
// Semantics: kubeai_amd/ops/ref.py::paged_attention_decode.
//
// Structure:
//  - workgroup = (sequence, kv head, split of the keys); the waves of a row's splits
//    take tiles in turn, each with its own softmax state; the G query heads of the
//    group share every key. A tile is one cache block (32 keys over an e5m2 cache at
//    head size 128): 145 registers and three waves a SIMD, where tiles of 32 keys take
//    209 and leave room for two (28 rows of 100-700 in 3 splits 17.9 us, 15.9). The first
//    look-up in the block table does not wait for the row's length.
//  - which splits there are, and in which order, is worked out on the device once a
//    step (decode_plan_kernel below), by the rows' lengths.
//  - S^T = K.Q^T on v_mfma_f32_16x16x32_bf16: a lane reads 16 bytes of one
//    key straight into the operand (16 keys x 64 contiguous bytes per load,
//    no LDS), the query heads are columns (lane & 15; those past G repeat the
//    last head). Scores of 4 keys per block lie in the lane, a maximum is two
//    lane swaps, the sum stays per lane until the end.
//  - O^T += V^T.P^T: the score registers are the second product's operand as
//    they stand. V needs its keys along a lane: it goes through a
//    wave-private LDS tile (row-major, 16-byte units XOR-swizzled, no
//    barriers) and comes back through ds_read_b64_tr_b16.
//  - the weights keep their 24 bits: they are cut into three bf16 parts of 8
//    bits that are multiplied one after the other into the same fp32 sum. A
//    part that would be 0 is 2^-100 (or the weight, if that is less): times an
//    infinite value 0 would be NaN.
//  - the next tile's K and V are in flight while this one is computed (two
//    register sets), and the blocks of the one after it are being looked up. Past the
//    last tile the loads are of no bytes: in a branch they had the compiler wait, in
//    front of each tile, for the next one's loads as well (96 rows of 1500-4000 228 us).
// Bound by reading the cache. The form before this (scores and weighted sum
// on the vector ALUs) issued about 150 LDS operations per 16 keys, most of
// them the lane permutes that passed a weight to every lane; here it is 12.
// Measured, kernel + merge of the splits, us (the same number of splits for every row
// and tiles of 32 keys -> planned):
//   heads 32/8 x 128, 40 rows of 100-700 keys         23.2 -> 18.8, to fp8 25.3 -> 20.1
//   96 rows of 1500-4000                             209 -> 195 (5.8 TB/s)
//   64 rows of 100-2000                              60.9 -> 53.4
//   40 rows of 200, one of 4000                      34.9 -> 15.8, to fp8 37.1 -> 19.6
//   8 rows of 3584                                    28.8 -> 25.6
//   1 row of 3000 and 7 idle ones                     12.6 -> 8.7
//   12 rows of 500                                    13.2 -> 10.5
//   96 rows of 100-300, one split each                20.5 -> 19.8 (unplanned 18.8)
//   heads 8/4 x 256, 40 rows of 100-700               21.9 -> 18.4
//     64 rows of 100-2000                             65.1 -> 60.3
//     96 rows of 2000                                 139 -> 139.5
// At head size 256, over
// a bf16 cache the query lies in LDS: with it in registers 25 were spilled, and
// the reloads waited for the loads in flight (the last two 236 us).
#include <torch/extension.h>

#include <type_traits>

#include "common.h"

namespace {

constexpr int kWaves = 4;
constexpr int kBlockThreads = kWaves * WAVE_SIZE;
constexpr int kBS = 16;      // cache block size (tokens)
constexpr int kMaxSplits = 16;
constexpr int kMaxG = 8;
constexpr int kCUs = 256;

typedef __attribute__((ext_vector_type(8))) short bf16x8;
typedef __attribute__((ext_vector_type(4))) short bf16x4;
typedef __attribute__((ext_vector_type(4))) float f32x4;
typedef __attribute__((address_space(3))) bf16x4 lds_bf16x4;

// One split of a row; a row's splits, which lie behind one another.
struct alignas(16) Item {
  int row, len;  // row < 0: none
  uint16_t split, splits;
  int part;      // where its results go
};
struct alignas(8) Splits {
  int first, n;
};

// Rows that are still sums (common.h: ProductSums, [parts, B, (n_q + 2 n_kv) hd]).
struct NewRows {
  ProductSums sums;
  const int32_t* positions;  // [B]
  const float* cos_sin;      // [max_pos, hd]
  const int64_t* slots;      // [B]; < 0: the row's key is in the cache or nowhere
};

// Cache blocks of a tile.
constexpr int blocks_per_tile(int hd, int element) { return hd == 128 && element == 1 ? 2 : 1; }

// Waves a SIMD holds: 145 registers at head size 128, 256 at 256.
constexpr int waves_per_simd(int hd) { return hd == 128 ? 3 : 2; }

// 16 (or 8) bytes a lane from base + at, zeros if size is 0
template <typename T>
DEV_INLINE T buffer_load(const void* base, int size, int at) {
  T v{};
#ifdef __HIP_DEVICE_COMPILE__
  const auto r = __builtin_amdgcn_make_buffer_rsrc((void*)base, 0, size, 0x00020000);
  if constexpr (sizeof(T) == 16)
    v = __builtin_bit_cast(T, __builtin_amdgcn_raw_buffer_load_b128(r, at, 0, 0));
  else
    v = __builtin_bit_cast(T, __builtin_amdgcn_raw_buffer_load_b64(r, at, 0, 0));
#endif
  return v;
}

// no load moves over it: the caches are not __restrict__, so the compiler takes the
// asm to write them
DEV_INLINE void in_order() {
  __builtin_amdgcn_sched_barrier(0);
  asm volatile("" ::: "memory");
  __builtin_amdgcn_sched_barrier(0);
}

// combine a value over the four 16-lane groups that hold the same column
template <typename F>
DEV_INLINE float over_groups(float v, F&& f) {
  const auto a = __builtin_amdgcn_permlane32_swap(
      __float_as_uint(v), __float_as_uint(v), false, false);
  v = f(__uint_as_float(a[0]), __uint_as_float(a[1]));
  const auto b = __builtin_amdgcn_permlane16_swap(
      __float_as_uint(v), __float_as_uint(v), false, false);
  return f(__uint_as_float(b[0]), __uint_as_float(b[1]));
}

// CT = cache element type: ushort (bf16) or unsigned char (fp8 e5m2,
// converted to bf16 on the way in, exactly). CAP: s = cap * tanh(s / cap)
// after scaling and before masking. ONE: no wave has more than one tile.
// NEW: the rows' queries, keys and values are a product's sums still, of up to so many
// parts. Every workgroup adds and rotates its own query heads and the key, a unit of 8
// columns a thread, with the first tile's loads on their way behind the sums'; the one
// that has the row's last tile writes key and value to the cache, and takes them from
// LDS for that tile. us with the merge, rotation as a
// launch before / here: 40 rows of 100-700, sums in 4 parts, to fp8 25.0 / 22.2, bf16 23.5 /
// 21.0; 8 rows, sums in 8 parts 18.2 / 14.8, 14.9 / 11.6.
template <int HD, typename CT, bool CAP, bool ONE, int NEW>
__launch_bounds__(kBlockThreads, waves_per_simd(HD)) __global__ void paged_decode_kernel(
    ushort* __restrict__ out,            // [B, n_q, hd] bf16, or null: parts of all rows
    const ushort* __restrict__ q,        // [B, n_q, hd] bf16
    CT* k_cache,                         // [nb, n_kv, bs, hd]
    CT* v_cache,
    const int32_t* __restrict__ block_tables,  // [B, max_blocks]
    const int32_t* __restrict__ seq_lens,      // [B]
    const float scale, const float softcap, const int window,
    const int n_kv, const int G, const int max_blocks,
    const int64_t q_stride, const int row_splits,
    const Item* __restrict__ plan,  // or null: row_splits splits of every row
    const NewRows fresh,
    float* __restrict__ part_o,    // [splits of all rows, n_q, hd]
    float* __restrict__ part_ml) { // [splits of all rows, n_q, 2]
  constexpr int NB = blocks_per_tile(HD, sizeof(CT));
  constexpr int NC = HD / 32;            // contraction steps of S
  constexpr int ND = HD / 16;            // row blocks of O^T
  constexpr int NV = HD / 32;            // 16-byte V units per lane and block
  const int item = blockIdx.x / n_kv, kh = blockIdx.x % n_kv;
  int b, split, n_splits, L, part_row = item;
  if (plan) {
    const Item it = plan[item];
    if (it.row < 0) return;
    b = it.row;
    split = it.split;
    n_splits = it.splits;
    L = it.len;
    part_row = it.part;
  } else {
    b = item / row_splits;
    split = item % row_splits;
    n_splits = row_splits;
    L = seq_lens[b];
  }
  const int n_q = n_kv * G;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / WAVE_SIZE);
  const int lane = threadIdx.x % WAVE_SIZE;
  const int col = lane & 15, grp = lane >> 4;
  const int n_blocks = (L + kBS - 1) / kBS;
  // sliding window: the query (position L-1) attends keys in
  // (L-1-window, L-1]; splits divide the visible blocks only
  int w0 = 0, blk_base = 0;
  if (window > 0) {
    w0 = max(0, L - window);
    blk_base = w0 / kBS;
  }
  const int n_units = (n_blocks - blk_base + NB - 1) / NB;  // tiles
  // the waves of all splits take tiles in turn
  const int turn = kWaves * n_splits;

  constexpr int kVTile = NB * kBS * HD;  // elements of a wave's V tile
  constexpr size_t kSmem = sizeof(ushort) * kWaves * kVTile >
                                   sizeof(float) * kWaves * kMaxG * HD
                               ? sizeof(ushort) * kWaves * kVTile
                               : sizeof(float) * kWaves * kMaxG * HD;
  __shared__ __attribute__((aligned(16))) char smem[kSmem];
  __shared__ float merge_ml[kWaves][kMaxG][2];
  char* vt = smem + wave * kVTile * 2;

  // Head size 256 over a bf16 cache: two tiles of K and V and the sums leave no
  // registers for the query; it lies in LDS, 16-byte units XORed with the head.
  constexpr bool kQLds = HD == 256 && sizeof(CT) == 2;
  __shared__ __attribute__((aligned(16))) ushort q_lds[kQLds || NEW > 0 ? kMaxG * HD : 8];
  static_assert(NEW == 0 || sizeof(CT) == 2);  // (over an e5m2 cache 116 registers were spilled)
  __shared__ __attribute__((aligned(16))) CT new_kv[2][NEW > 0 ? HD : 16];
  bf16x8 q_frag[kQLds ? 1 : NC];
  const ushort* qp = q + (int64_t)b * q_stride + (int64_t)kh * G * HD;
  const int q_head = min(col, G - 1);
  if constexpr (NEW > 0) {
    // (below, behind the first tile's loads)
  } else if constexpr (kQLds) {
    for (int i = threadIdx.x; i < G * (HD / 8); i += kBlockThreads) {
      const int g = i / (HD / 8), u = i % (HD / 8);
      *reinterpret_cast<bf16x8*>(&q_lds[g * HD + ((u ^ g) << 3)]) =
          *reinterpret_cast<const bf16x8*>(qp + i * 8);
    }
    __syncthreads();
  } else {
#pragma unroll
    for (int c = 0; c < NC; ++c)
      q_frag[c] = *reinterpret_cast<const bf16x8*>(qp + q_head * HD + grp * 8 + c * 32);
  }
  auto query = [&](int c) -> bf16x8 {
    if constexpr (kQLds)
      return *reinterpret_cast<const bf16x8*>(
          &q_lds[q_head * HD + (((c * 4 + grp) ^ q_head) << 3)]);
    else
      return q_frag[c];
  };
  const float c2 = CAP ? scale : scale * kLog2e;
  const SoftCap cap(CAP ? softcap : 1.0f);

  f32x4 o_acc[ND];
#pragma unroll
  for (int d = 0; d < ND; ++d) o_acc[d] = f32x4{0.f, 0.f, 0.f, 0.f};
  float m_run = -INFINITY, l_run = 0.f;  // l_run: this lane's keys

  const int32_t* bt = block_tables + (int64_t)b * max_blocks;
  using Unit = std::conditional_t<sizeof(CT) == 2, bf16x8, uint64_t>;
  Unit kf[2][NB][NC], vf[2][NB][NV];
  auto to_bf16 = [](const Unit& u) -> bf16x8 {
    if constexpr (sizeof(CT) == 2) return u;
    else return __builtin_bit_cast(bf16x8, e5m2x8_to_bf16x8(u));
  };
  // the cache blocks of tile t (past the last one: any entry of the table, not used).
  // Without a window the first look-up does not wait for the row's length.
  struct Blocks {
    int at[NB];
  };
  auto look_up = [&](int t) {
    Blocks o;
#pragma unroll
    for (int j = 0; j < NB; ++j)
      o.at[j] = bt[min(blk_base + t * NB + j, max_blocks - 1)];
    return o;
  };
  constexpr int kBlockBytes = kBS * HD * sizeof(CT);
  const int k_at = (col * HD + grp * 8) * sizeof(CT), v_at = lane * 8 * sizeof(CT);
  // blocks behind the last one: loads of no bytes
  auto load_tile = [&](int set, int t, const Blocks& blocks) {
#pragma unroll
    for (int j = 0; j < NB; ++j) {
      const int size = blk_base + t * NB + j < n_blocks ? kBlockBytes : 0;
      const int64_t base = ((int64_t)blocks.at[j] * n_kv + kh) * (kBS * HD);
#pragma unroll
      for (int c = 0; c < NC; ++c)
        kf[set][j][c] =
            buffer_load<Unit>(k_cache + base, size, k_at + c * 32 * (int)sizeof(CT));
#pragma unroll
      for (int i = 0; i < NV; ++i)
        vf[set][j][i] = buffer_load<Unit>(v_cache + base, size,
                                          v_at + i * WAVE_SIZE * 8 * (int)sizeof(CT));
    }
  };

  // LDS offsets of the transposing reads: keys 4 grp + (lane >> 2 & 3) of a
  // block, columns 16 d + 4 (lane & 3); units of rows r are XORed with
  // 2 (r & 3), which spreads the four rows of a 16-lane read over the banks
  const int tr_row = 4 * grp + ((lane >> 2) & 3);
  const int tr_x = ((lane >> 2) & 3) << 1;
  const int tr_u = (lane & 3) >> 1;  // unit within the 32 bytes
  const char* tr_base = vt + tr_row * HD * 2 + (lane & 1) * 8;

  int new_tile = -1;  // the tile whose last key is still in LDS
  auto compute = [&](int set, int t) {
    const int tok0 = (blk_base + t * NB) * kBS;
    const bool whole = tok0 >= w0 && tok0 + NB * kBS <= L;
    if constexpr (NEW > 0) {
      if (t == new_tile) {
#pragma unroll
        for (int j = 0; j < NB; ++j) {
          const int row = L - 1 - tok0 - j * kBS;  // (in this block or not)
#pragma unroll
          for (int c = 0; c < NC; ++c)
            if (col == row)
              kf[set][j][c] = *reinterpret_cast<const Unit*>(&new_kv[0][c * 32 + grp * 8]);
#pragma unroll
          for (int i = 0; i < NV; ++i) {
            const int e = lane + i * WAVE_SIZE;
            if (e / (HD / 8) == row)
              vf[set][j][i] = *reinterpret_cast<const Unit*>(&new_kv[1][e % (HD / 8) * 8]);
          }
        }
      }
    }
    // ---- V to LDS ------------------------------------------------------
#pragma unroll
    for (int j = 0; j < NB; ++j)
#pragma unroll
      for (int i = 0; i < NV; ++i) {
        const int e = lane + i * WAVE_SIZE;  // 16-byte unit of the block
        const int row = e / (HD / 8), un = e % (HD / 8);
        bf16x8 v = to_bf16(vf[set][j][i]);
        // rows past the end: their weight is 0, but 0 * stale NaN is not
        if (!whole && tok0 + j * kBS + row >= L) v = bf16x8{};
        *reinterpret_cast<bf16x8*>(
            vt + (j * kBS + row) * HD * 2 + ((un ^ ((row & 3) << 1)) << 4)) = v;
      }
    // ---- scores ----------------------------------------------------------
    f32x4 s[NB];
#pragma unroll
    for (int j = 0; j < NB; ++j) {
      s[j] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int c = 0; c < NC; ++c)
        s[j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(
            to_bf16(kf[set][j][c]), query(c), s[j], 0, 0, 0);
    }
    if constexpr (CAP) cap.apply(s, c2);
    float tmax = -INFINITY;
#pragma unroll
    for (int j = 0; j < NB; ++j)
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        float x = s[j][i] * (CAP ? kLog2e : c2);
        const int tok = tok0 + j * kBS + grp * 4 + i;
        if (!whole && (tok >= L || tok < w0)) x = -INFINITY;
        s[j][i] = x;
        tmax = fmaxf(tmax, x);
      }
    tmax = over_groups(tmax, [](float a, float c) { return fmaxf(a, c); });
    // the maximum may lag by 2^11 before everything is rescaled
    if (!__all(tmax <= m_run + 11.0f)) {
      const float m_new = fmaxf(m_run, tmax);
      const float corr =
          __builtin_amdgcn_exp2f(m_run - (m_new == -INFINITY ? 0.f : m_new));
      l_run *= corr;
#pragma unroll
      for (int d = 0; d < ND; ++d) o_acc[d] *= corr;
      m_run = m_new;
    }
    const float m_use = (m_run == -INFINITY) ? 0.f : m_run;
    // ---- weights, in three bf16 parts --------------------------------------
    short p_part[3][NB * 4];
#pragma unroll
    for (int j = 0; j < NB; ++j)
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        float p = __builtin_amdgcn_exp2f(s[j][i] - m_use);
        l_run += p;
        const float least = fminf(p, 0x1p-100f);
#pragma unroll
        for (int k = 0; k < 3; ++k) {
          const uint32_t top = __float_as_uint(p) & 0xffff0000u;
          p_part[k][j * 4 + i] = (short)(top >> 16);
          p = fmaxf(p - __uint_as_float(top), least);
        }
      }
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    __builtin_amdgcn_wave_barrier();
    // ---- O^T += V^T . P^T ------------------------------------------------
#pragma unroll
    for (int d = 0; d < ND; ++d) {
      const char* a = tr_base + (((2 * d + tr_u) ^ tr_x) << 4);
      const bf16x4 v0 =
          __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_bf16x4*)(a));
      if constexpr (NB == 2) {
        const bf16x4 v1 = __builtin_amdgcn_ds_read_tr16_b64_v4i16(
            (lds_bf16x4*)(a + kBS * HD * 2));
        const bf16x8 v =
            __builtin_shufflevector(v0, v1, 0, 1, 2, 3, 4, 5, 6, 7);
#pragma unroll
        for (int k = 0; k < 3; ++k) {
          bf16x8 p;
#pragma unroll
          for (int i = 0; i < 8; ++i) p[i] = p_part[k][i];
          o_acc[d] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(v, p, o_acc[d],
                                                             0, 0, 0);
        }
      } else {
#pragma unroll
        for (int k = 0; k < 3; ++k) {
          bf16x4 p;
#pragma unroll
          for (int i = 0; i < 4; ++i) p[i] = p_part[k][i];
          o_acc[d] = __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(v0, p, o_acc[d],
                                                               0, 0, 0);
        }
      }
    }
    // the next tile's V is stored after these reads (LDS operations of a
    // wave run in order)
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    __builtin_amdgcn_wave_barrier();
  };

  // (no load in a branch: where paths of more and of fewer loads meet, the compiler
  // waits for all of them)
  const int first = split * kWaves + wave;
  const Blocks start = look_up(first);
  if constexpr (NEW > 0) {
    constexpr int HALF = HD / 2, UPH = HD / 8;  // units a head
    // the lanes 2 i and 2 i + 1 have units half a head apart; all threads load (past
    // the last unit: that again), none in a branch
    const int at_unit = min((int)threadIdx.x, (G + 2) * UPH - 2 + (int)(threadIdx.x & 1));
    const int head = at_unit / UPH, half = at_unit & 1;  // G: the key, G + 1: the value
    const int u = at_unit % UPH / 2 * 8;                 // the pair's column in a half
    const int col0 = (head < G ? kh * G + head : head == G ? n_q + kh : n_q + n_kv + kh) * HD +
                     u + half * HALF;
    const ProductSums& sums = fresh.sums;
    const int at = max(0, L - 1);  // the new key's place in the row
    const int64_t slot = fresh.slots[b];
    const float* cs = fresh.cos_sin + (int64_t)fresh.positions[b] * HD + u;
    const int last = bt[min(at / kBS, max_blocks - 1)];
    f32x4 part[NEW][2];
    const float* row = sums.part + (int64_t)b * sums.N + col0;
#pragma unroll
    for (int k = 0; k < NEW; ++k) {
      const auto* from =
          reinterpret_cast<const f32x4*>(row + min(k, sums.parts - 1) * sums.stride);
      part[k][0] = from[0];
      part[k][1] = from[1];
    }
    const int cols[1] = {col0};
    const SumScales<1> by(sums, b, cols);
    f32x4 cv[2], sv[2];
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      cv[i] = reinterpret_cast<const f32x4*>(cs)[i];
      sv[i] = reinterpret_cast<const f32x4*>(cs + HALF)[i];
    }
    in_order();
    load_tile(0, first, start);
    in_order();
    f32x4 x[2] = {f32x4{0.f, 0.f, 0.f, 0.f}, f32x4{0.f, 0.f, 0.f, 0.f}};
#pragma unroll
    for (int i = 0; i < 2; ++i)
#pragma unroll
      for (int k = 0; k < NEW; ++k)
        if (k < sums.parts) x[i] += part[k][i];
    ushort8 o;
#pragma unroll
    for (int j = 0; j < 8; ++j) {
      float f = x[j / 4][j % 4];
      if (sums.sx) f = f * by.sx * by.sw[0][j];
      o[j] = f32_to_bf16(f);
      const float own = bf16_to_f32(o[j]), other = __shfl_xor(own, 1);
      const float c = cv[j / 4][j % 4], s = sv[j / 4][j % 4];
      if (head <= G) o[j] = f32_to_bf16(half ? own * c + other * s : own * c - other * s);
    }
    // the waves' turns go on over the splits
    const bool owner = (max(n_units, 1) - 1) / kWaves % n_splits == split;
    if (threadIdx.x < (G + 2) * UPH) {
      const int unit = u / 8 + half * (UPH / 2);
      if (head < G) {
        *reinterpret_cast<ushort8*>(&q_lds[head * HD + ((unit ^ head) << 3)]) = o;
      } else {
        *reinterpret_cast<ushort8*>(&new_kv[head - G][unit * 8]) = o;
        if (owner && slot >= 0) {
          CT* cache = head == G ? k_cache : v_cache;
          *reinterpret_cast<ushort8*>(
              cache + ((slot / kBS * n_kv + kh) * kBS + slot % kBS) * HD + unit * 8) = o;
        }
      }
    }
    new_tile = slot >= 0 && slot == (int64_t)last * kBS + at % kBS ? n_units - 1 : -1;
    __syncthreads();
    if constexpr (!kQLds) {
#pragma unroll
      for (int c = 0; c < NC; ++c)
        q_frag[c] = *reinterpret_cast<const bf16x8*>(
            &q_lds[q_head * HD + (((c * 4 + grp) ^ q_head) << 3)]);
    }
  }
  if (first < n_units) {
    if constexpr (NEW == 0) load_tile(0, first, start);
    if constexpr (ONE) {
      compute(0, first);
    } else {
      Blocks even, odd = look_up(first + turn);
      for (int t = first; t < n_units; t += 2 * turn) {
        load_tile(1, t + turn, odd);
        even = look_up(t + 2 * turn);
        in_order();
        compute(0, t);
        in_order();
        load_tile(0, t + 2 * turn, even);
        odd = look_up(t + 3 * turn);
        in_order();
        if (t + turn < n_units) compute(1, t + turn);
      }
    }
  }

  // ---- merge the waves -----------------------------------------------------
  l_run = over_groups(l_run, [](float a, float c) { return a + c; });
  __syncthreads();  // the V tiles are free
  float* merge_o = reinterpret_cast<float*>(smem);  // [wave][G][HD]
  if (col < G) {
    float* mo = merge_o + (wave * G + col) * HD + grp * 4;
#pragma unroll
    for (int d = 0; d < ND; ++d)
      *reinterpret_cast<f32x4*>(mo + d * 16) = o_acc[d];
    if (grp == 0) {
      merge_ml[wave][col][0] = m_run;
      merge_ml[wave][col][1] = l_run;
    }
  }
  __syncthreads();
  for (int i = threadIdx.x; i < G * (HD / 4); i += kBlockThreads) {
    const int g = i / (HD / 4), e = i % (HD / 4) * 4;
    float m_star = -INFINITY;
#pragma unroll
    for (int w = 0; w < kWaves; ++w) m_star = fmaxf(m_star, merge_ml[w][g][0]);
    const float m_use = (m_star == -INFINITY) ? 0.f : m_star;
    float l_star = 0.f;
    f32x4 o = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int w = 0; w < kWaves; ++w) {
      const float c = __builtin_amdgcn_exp2f(merge_ml[w][g][0] - m_use);
      l_star += merge_ml[w][g][1] * c;
      o += *reinterpret_cast<const f32x4*>(merge_o + (w * G + g) * HD + e) * c;
    }
    const int64_t head = (int64_t)b * n_q + kh * G + g;
    const int64_t part = (int64_t)part_row * n_q + kh * G + g;
    if (n_splits == 1 && out) {
      const float inv_l = 1.0f / l_star;
      ushort4_t r;
#pragma unroll
      for (int k = 0; k < 4; ++k) r[k] = f32_to_bf16(o[k] * inv_l);
      *reinterpret_cast<ushort4_t*>(out + head * HD + e) = r;
    } else {
      // partial results (an empty split writes m = -inf, l = 0, o = 0)
      *reinterpret_cast<f32x4*>(part_o + part * HD + e) = o;
      if (e == 0) {
        part_ml[part * 2] = m_star;
        part_ml[part * 2 + 1] = l_star;
      }
    }
  }
}

// Merged values of one query head, 2 or 4 a lane, rounded to bf16. The lanes read
// all splits' (m, l) at once; the rows of O are on their way before those are used, up
// to 16 at a time (as many as a row has splits), 4 where there are no more.
template <int HD>
struct Merged {
  static constexpr int EPL = HD / 64;
  typedef __attribute__((ext_vector_type(EPL))) float vec;
  ushort v[EPL];
  float ms, ls;
  const vec* po;
  int64_t step;
  int n;
  vec o[kMaxSplits];

  // the head's parts lie n_q apart, at first + head and on
  template <int MOST>
  DEV_INLINE void load(const float* part_o, const float* part_ml, Splits of, int n_q,
                       int head) {
    const int lane = threadIdx.x % WAVE_SIZE;
    const int64_t first = (int64_t)of.first * n_q + head;
    n = of.n;
    step = (int64_t)n_q * 64;
    const float* pml = part_ml + (first + (int64_t)min(lane, n - 1) * n_q) * 2;
    po = reinterpret_cast<const vec*>(part_o + first * HD) + lane;
    ms = pml[0];
    ls = pml[1];
#pragma unroll
    for (int k = 0; k < MOST; ++k) o[k] = po[min(k, n - 1) * step];
  }
  template <int MOST>
  DEV_INLINE void finish() {
    const int lane = threadIdx.x % WAVE_SIZE;
    const float m_star = wave_reduce_max(ms);
    const float c = __builtin_amdgcn_exp2f(ms - (m_star == -INFINITY ? 0.f : m_star));
    const float l_star = wave_reduce_sum(lane < n ? ls * c : 0.f);
    vec sum;
#pragma unroll
    for (int e = 0; e < EPL; ++e) sum[e] = 0.f;
#pragma unroll
    for (int k = 0; k < MOST; ++k)
      if (k < n) sum += o[k] * __uint_as_float(__builtin_amdgcn_readlane(__float_as_uint(c), k));
    const float inv_l = 1.0f / l_star;
#pragma unroll
    for (int e = 0; e < EPL; ++e) v[e] = f32_to_bf16(sum[e] * inv_l);
  }
};

// a row's splits, from the plan or the same number for all
DEV_INLINE Splits splits_of(const Splits* plan, int n, int row) {
  return plan ? plan[row] : Splits{row * n, n};
}

// Merge the splits' results: one wave per (sequence, query head). A planned row that
// was not split has its result.
template <int HD>
__global__ void decode_merge_kernel(
    ushort* __restrict__ out,             // [B, n_q, hd]
    const float* __restrict__ part_o, const float* __restrict__ part_ml,
    const Splits* __restrict__ plan, const int n_splits, const int n_q,
    const int64_t n_bh) {
  constexpr int EPL = HD / 64;
  const int64_t bh = (int64_t)blockIdx.x * (blockDim.x / WAVE_SIZE) +
                     threadIdx.x / WAVE_SIZE;
  if (bh >= n_bh) return;
  const Splits of = splits_of(plan, n_splits, (int)(bh / n_q));
  if (of.n == 1) return;
  Merged<HD> m;
  auto merge = [&](auto most) {
    m.template load<decltype(most)::value>(part_o, part_ml, of, n_q, (int)(bh % n_q));
    m.template finish<decltype(most)::value>();
  };
  if (of.n <= 4) merge(std::integral_constant<int, 4>{});
  else merge(std::integral_constant<int, kMaxSplits>{});
  ushort* oh = out + bh * HD + EPL * (threadIdx.x % WAVE_SIZE);
#pragma unroll
  for (int e = 0; e < EPL; e += 2)
    *reinterpret_cast<uint32_t*>(oh + e) = ((uint32_t)m.v[e + 1] << 16) | m.v[e];
}

// The same, and the row (all heads of a sequence) to fp8 with one scale, as the
// conversion of the merged bf16 row has it: one workgroup of 16 waves per row,
// HPW heads a wave, one after the other: a chain of loads each, so only for few of
// them (ops.decode_fp8_merges). Bound by its launch: 40 rows of 32 x 128 in 2 splits,
// merge and conversion 9.6 us, this 5.1 (in a profile; beside the attention 1 less).
template <int HD, int HPW>
__launch_bounds__(16 * WAVE_SIZE) __global__ void decode_merge_fp8_kernel(
    unsigned char* __restrict__ out,      // [B, n_q * hd]
    float* __restrict__ out_scale,        // [B]
    const float* __restrict__ part_o, const float* __restrict__ part_ml,
    const Splits* __restrict__ plan, const int n_splits, const int n_q) {
  constexpr int EPL = HD / 64;
  const int wave = threadIdx.x / WAVE_SIZE, lane = threadIdx.x % WAVE_SIZE;
  const int64_t row = blockIdx.x;
  const Splits of = splits_of(plan, n_splits, (int)row);
  __shared__ float red[16];
  float vals[HPW][EPL];
  float amax = 0.f;
  Merged<HD> m[HPW];
  auto merge = [&](auto most) {
    constexpr int MOST = decltype(most)::value;
#pragma unroll
    for (int h = 0; h < HPW; ++h)  // (past the last head: that again)
      m[h].template load<MOST>(part_o, part_ml, of, n_q, min(h * 16 + wave, n_q - 1));
#pragma unroll
    for (int h = 0; h < HPW; ++h) {
      m[h].template finish<MOST>();
#pragma unroll
      for (int e = 0; e < EPL; ++e) {
        vals[h][e] = bf16_to_f32(m[h].v[e]);
        amax = fmaxf(amax, fabsf(vals[h][e]));
      }
    }
  };
  if (of.n <= 4) merge(std::integral_constant<int, 4>{});
  else merge(std::integral_constant<int, kMaxSplits>{});
  amax = wave_reduce_max(amax);
  if (lane == 0) red[wave] = amax;
  __syncthreads();
  float gmax = 1e-6f;
#pragma unroll
  for (int w = 0; w < 16; ++w) gmax = fmaxf(gmax, red[w]);
  if (threadIdx.x == 0) out_scale[row] = gmax / 448.0f;
  const float inv_scale = 448.0f / gmax;
#pragma unroll
  for (int h = 0; h < HPW; ++h) {
    const int head = h * 16 + wave;
    if (head < n_q) {
      unsigned char* to = out + (row * n_q + head) * HD + EPL * lane;
      int w = __builtin_amdgcn_cvt_pk_fp8_f32(vals[h][0] * inv_scale,
                                              vals[h][1] * inv_scale, 0, false);
      if constexpr (EPL == 4) {
        w = __builtin_amdgcn_cvt_pk_fp8_f32(vals[h][2] * inv_scale,
                                            vals[h][3] * inv_scale, w, true);
        *reinterpret_cast<uint32_t*>(to) = (uint32_t)w;
      } else {
        *reinterpret_cast<ushort*>(to) = (ushort)w;
      }
    }
  }
}


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
constexpr int kPlanThreads = 256, kCandidates = 32, kPlanRows = 1024;
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
// 100-700 keys, 8 kv heads 23.0 us at 512, 25.6 at 1536; one row of 3000 among 7
// idle ones 13.6 at 512, 17.0 at 1536. Head size 256: 128 rows of 300 but one
// of 8000, 4 kv heads 224 us at 512, 122 at 576, 87 at 1536; 8 rows of 3500, e5m2
// cache, 8 kv heads 33 at 512, 42 at 576; 40 rows of 100-700, e5m2 cache, 4 kv
// heads 19.3 at 512 and 576, 22 at 768, 25 at 1536. (Measured with tiles of 32 keys.) A
// split has at least 32 keys of the widest row, 16 at head size 256. KUBEAI_DECODE_SPLIT_TARGET overrides for tuning sweeps.
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
// kv heads, head size, element and window while the lengths are these: int32 [4 items +
// 2 rows], the items in front.
torch::Tensor paged_decode_plan(torch::Tensor seq_lens, int64_t n_kv, int64_t hd,
                                int64_t element_size, int64_t window) {
  TORCH_CHECK(seq_lens.scalar_type() == torch::kInt32 && seq_lens.is_contiguous() &&
              seq_lens.is_cuda() && seq_lens.dim() == 1);
  const int B = (int)seq_lens.size(0);
  TORCH_CHECK(B >= 1 && B <= kPlanRows, "1 to ", kPlanRows, " rows");
  TORCH_CHECK(n_kv >= 1 && (hd == 128 || hd == 256) && (element_size == 1 || element_size == 2));
  const int M = std::max<int64_t>(1, kCUs / n_kv);
  const int64_t n_items = 3 * M + B;  // (what the first candidate may need)
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
    TORCH_CHECK(plan->scalar_type() == torch::kInt32 && plan->is_contiguous() &&
                plan->is_cuda() && plan->dim() == 1 && plan->numel() >= 6 * B &&
                (plan->numel() - 2 * B) % 4 == 0 && ((uintptr_t)plan->data_ptr() & 15) == 0);
    parts = (plan->numel() - 2 * B) / 4;
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
  auto with_new = [&](auto hdv, auto ct, auto cap, auto one, auto fresh_v) {
    using CT = decltype(ct);
    hipLaunchKernelGGL(
        (paged_decode_kernel<decltype(hdv)::value, CT, decltype(cap)::value,
                             decltype(one)::value, decltype(fresh_v)::value>),
        grid, block, 0, stream, fp8 ? nullptr : (ushort*)out.data_ptr(), q,
        (CT*)k_cache.data_ptr(), (CT*)v_cache.data_ptr(), block_tables.data_ptr<int32_t>(),
        seq_lens.data_ptr<int32_t>(), (float)scale, (float)softcap,
        (int)window, n_kv, G, max_blocks, q_stride, n_splits, items,
        fresh ? *fresh : NewRows{}, part_o_ptr, part_ml_ptr);
  };
  auto launch = [&](auto hdv, auto ct, auto cap, auto one) {
    if constexpr (sizeof(ct) == 2) {
      if (fresh && fresh->sums.parts <= 4)
        return with_new(hdv, ct, cap, one, std::integral_constant<int, 4>{});
      if (fresh) return with_new(hdv, ct, cap, one, std::integral_constant<int, 8>{});
    }
    with_new(hdv, ct, cap, one, std::integral_constant<int, 0>{});
  };
  // (12 rows of 500: 14.9 us with the loop's loads of no bytes, 13.9 without)
  const int nb = blocks_per_tile(hd, k_cache.element_size());
  const bool one = !items && (max_blocks + nb - 1) / nb <= n_splits * kWaves;
  auto with_cap = [&](auto hdv, auto ct) {
    auto with_one = [&](auto capped) {
      if (one) launch(hdv, ct, capped, std::true_type{});
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
          out_scale->data_ptr<float>(), part_o_ptr, part_ml_ptr, row_splits, n_splits, n_q);
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
