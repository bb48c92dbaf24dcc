// Products of many rows: y[i] = x[i] w^T, or for the rows of every expert e of a
// mixture y[i] = x[src[i]] w[e]^T in one launch; bf16 or fp8 e4m3 (W8A8 with row
// and column scales), fp32 accumulation. What the epilogue makes of them: bf16
// rows, fp32 sums of a part of K, or in bf16 silu or tanh-gelu(gate) * up of stacked
// gate and up columns (in fp32, rounded once) or relu(.)^2 times a weight per row.
//
// Bound by the matrix cores (and the power they draw: dense bf16 runs at 1.65
// GHz here), as long as nothing keeps them waiting. What it takes:
//  - 4 waves, one per SIMD, in 2 x 2, each up to 4 x 4 matrix instructions of
//    32 x 32. At 128 x 128 per wave LDS feeds 64 bytes a cycle; 8 waves of 128 x
//    64 need 96, and with the 32 that are written that is all it has.
//  - operands go straight to LDS, 16 bytes a lane. A CU takes 64 bytes a cycle of
//    those loads, and a wave that issues its 16 loads of a step at once stands
//    still for 1000 cycles; so one is put behind each matrix instruction (each
//    second of bf16). 28672 x 4096, 2048 rows, us, all at once / spread: fp8 261
//    / 205, bf16 439 / 376.
//  - the operands of the next chunk of K are read from LDS while the current
//    one's are multiplied. The barrier of a step lies in front of its last
//    chunk: everyone has the step's last operands in registers, so its place
//    in LDS can be written, and the next step's have landed.
//  - memory answers after 1 to 2 us, a step takes 1. At 256 x 256 two steps are 128
//    KB; the last 32 KB hold a third step of w, which comes from memory, where
//    x comes from L2: 2 places for A, 3 for B.
//  - the loads write 64 lanes in a row: the swizzle that keeps the reads free of
//    bank conflicts (16-byte unit u of row r lies at u ^ (r & 7)) is made by
//    the lane's choice of source. They are buffer loads: rows past the end and
//    the steps past the last read nothing, so the loop has no tail.
//  - results go through LDS, 32 rows of a wave at a time, so that whole lines are
//    stored (fp8, the same product: 27000 cycles a tile when stored from the
//    accumulators, 13000 now; the loop takes 83000).
//  - an XCD's tiles are consecutive, up to 8 row tiles down one column, then the
//    next column: they read the same rows of w from its L2.
// us, weights out of cache, library / this: fp8 28672 x 4096 384 rows 60 / 45, 2048
// rows 228 / 211, 8192 rows 764 / 743; 4096 x 4096 384 rows 14.9 / 12.0; 4096 x 14336
// 4480 rows 264 / 233; bf16 28672 x 4096 384 rows 83 / 84, 2048 rows 333 / 391 (1.65
// GHz; the library stays); 128256 x 4096 96 rows 225 / 207. 28672 x 4096 with silu
// and up, as two launches / here: bf16 384 rows 92 / 89.
#pragma once

#include <algorithm>
#include <type_traits>

#include "common.h"

namespace tiled {

enum Epilogue { kRows, kSums, kSilu, kGelu, kSquare };

struct Args {
  ushort* y;        // [R, columns]
  float* part;      // kSums: [parts, R, N]
  const char *x, *w;
  const float *sx, *sw;     // fp8: per row of x, [E, N]
  const float* row_weight;  // kSquare: [R]
  const int *bounds, *src;  // experts: E row counts or E + 1 offsets; rows of x
  bool offsets;
  int E, R, N, KB, k_part;      // N: columns of w; KB, k_part: bytes of K
  int64_t ldx, ldw, ew, xbytes;  // bytes
  bool wide;                     // rows of y begin on 16 bytes
};

// tile shapes: WM x WN matrix instructions a wave, places in LDS for A and B (96 KB
// and more: one workgroup a CU)
struct Shape {
  int wm, wn, na, nb;
  constexpr int rows() const { return 64 * wm; }
  constexpr int cols() const { return 64 * wn; }
};
constexpr Shape kShapes[] = {{4, 4, 2, 3}, {3, 4, 2, 3}, {4, 3, 2, 3}, {3, 3, 3, 3},
                             {2, 4, 3, 3}, {3, 2, 3, 3}, {2, 2, 4, 4}, {1, 2, 4, 4},
                             {1, 1, 6, 6}};
constexpr int kNumShapes = sizeof(kShapes) / sizeof(kShapes[0]);
// the last shape is for the sums of few rows alone (tiled_gemm.hip: narrow_sums)
constexpr int kNarrow = kNumShapes - 1;

void launch_fp8(int shape, Epilogue epi, const Args& a, int grid);
void launch_bf16(int shape, Epilogue epi, const Args& a, int grid);

constexpr int kStep = 128;  // bytes of K per step

typedef __attribute__((ext_vector_type(8))) short bf16x8;
typedef __attribute__((ext_vector_type(4))) short bf16x4;
typedef __attribute__((ext_vector_type(16))) float f32x16;
typedef __attribute__((ext_vector_type(4))) int i32x4;
typedef __attribute__((ext_vector_type(8))) int i32x8;
typedef __attribute__((ext_vector_type(4))) __bf16 bf4;
typedef __attribute__((ext_vector_type(4))) float f32x4;

// 16 bytes a lane from base + voff + soff to l + 16 * lane; lanes past `size`
// bytes read nothing
DEV_INLINE void load_lds16(const char* base, int size, char* l, int voff, int soff) {
#ifdef __HIP_DEVICE_COMPILE__
  const auto r = __builtin_amdgcn_make_buffer_rsrc((void*)base, 0, size, 0x00020000);
  __builtin_amdgcn_raw_ptr_buffer_load_lds(
      r, (__attribute__((address_space(3))) uint32_t*)l, 16, voff, soff, 0, 0);
#endif
}

DEV_INLINE void barrier() {
  __builtin_amdgcn_sched_barrier(0);
  asm volatile("" ::: "memory");
  __builtin_amdgcn_s_barrier();
  asm volatile("" ::: "memory");
  __builtin_amdgcn_sched_barrier(0);
}

// own LDS reads are done, all but the last N loads have landed
template <int N>
DEV_INLINE void wait_loads() {
  static_assert(N < 64);
  __builtin_amdgcn_s_waitcnt((N & 15) | ((N >> 4) << 14) | 0x70);
}

struct Work {
  int expert, row, rows, col, part;  // rows == 0: nothing to do
};

// Sums over the lanes up to this one.
DEV_INLINE int lane_sums(int v) {
#pragma unroll
  for (int d = 1; d < 64; d *= 2) {
    const int a = __shfl_up(v, d);
    if ((int)(threadIdx.x & 63) >= d) v += a;
  }
  return v;
}

// workgroups go to the XCDs in turn: each XCD gets consecutive ones of `all`
DEV_INLINE int tile_of(int all) {
  const int per = all / 8, rem = all % 8, xcd = blockIdx.x % 8, seq = blockIdx.x / 8;
  return seq >= per + (xcd < rem) ? -1 : xcd * per + min(xcd, rem) + seq;
}

// place of tile `at` among row_tiles x nt: bands of up to 8 row tiles, down
// each column
DEV_INLINE void place(int at, int row_tiles, int nt, int* row, int* col) {
  const int band = at / (8 * nt);
  at -= band * 8 * nt;
  const int high = min(8, row_tiles - band * 8);
  *row = band * 8 + at % high;
  *col = at / high;
}

// What this workgroup does, from the experts' row counts (or offsets).
template <int BM>
DEV_INLINE Work find_tile(const Args& a, int nt) {
  const int R = a.R, E = a.E;
  if (!a.bounds) {  // one matrix, K perhaps in parts
    const int row_tiles = (R + BM - 1) / BM, tiles = row_tiles * nt;
    const int id = tile_of(gridDim.x), part = id / tiles;
    Work k{0, 0, 0, 0, part};
    place(id - part * tiles, row_tiles, nt, &k.row, &k.col);
    k.row *= BM;
    k.rows = min(BM, R - k.row);
    return k;
  }
  const int lane = threadIdx.x & 63;
  const int* bounds = a.bounds;
  auto count = [&](int e) {
    return e >= E ? 0 : a.offsets ? bounds[e + 1] - bounds[e] : bounds[e];
  };
  int total = 0;  // row tiles
  for (int base = 0; base < E; base += 64) {
    total += __shfl(lane_sums((count(base + lane) + BM - 1) / BM), 63);
  }
  const int id = tile_of(total * nt);
  if (id < 0) return {0, 0, 0, 0, 0};
  int tiles0 = 0, rows0 = 0;
  for (int base = 0; base < E; base += 64) {
    const int c = count(base + lane), t = (c + BM - 1) / BM;
    const int tiles = lane_sums(t), rows = lane_sums(c);
    const uint64_t past = __ballot(id < (tiles0 + tiles) * nt);
    if (past) {
      const int f = __ffsll((unsigned long long)past) - 1;
      const int mine = __shfl(t, f), first = rows0 + __shfl(rows - c, f);
      const int end = min(rows0 + __shfl(rows, f), R);
      int row, col;
      place(id - (tiles0 + __shfl(tiles - t, f)) * nt, mine, nt, &row, &col);
      row = first + row * BM;
      return {base + f, row, max(0, min(BM, end - row)), col, 0};
    }
    tiles0 += __shfl(tiles, 63);
    rows0 += __shfl(rows, 63);
  }
  return {0, 0, 0, 0, 0};
}

template <bool FP8, int SHAPE, Epilogue EPI>
__global__ __launch_bounds__(256, 1) void tiled_kernel(const Args a) {
  constexpr Shape S = kShapes[SHAPE];
  constexpr int WM = S.wm, WN = S.wn, NA = S.na, NB = S.nb;
  static_assert(NA >= 2 && (NB == NA || (NA == 2 && NB == 3)));
  constexpr int BM = S.rows(), BN = S.cols();
  constexpr bool kHalves = EPI == kSilu || EPI == kGelu;  // gate | up columns
  static_assert(!kHalves || (WN % 2 == 0 && !FP8));
  constexpr int OUT = kHalves ? BN / 2 : BN;  // columns of the result
  constexpr int AC = BM / 32, BC = BN / 32, L = AC + BC;  // loads per wave and step
  constexpr int SA = BM * kStep, SB = BN * kStep;
  constexpr int CW = WN * 32, PITCH = CW * 4 + 16;  // a wave's result rows in LDS
  constexpr int kBytes = std::max(NA * SA + NB * SB, 4 * 32 * PITCH + BM * 4);
  __shared__ __attribute__((aligned(16))) char lds[kBytes];

  const int N = a.N, cols = kHalves ? N / 2 : N;  // of the result
  Work work = find_tile<BM>(a, (cols + OUT - 1) / OUT);
  // the same in every lane: buffers are described in scalar registers
  work.expert = __builtin_amdgcn_readfirstlane(work.expert);
  work.row = __builtin_amdgcn_readfirstlane(work.row);
  work.rows = __builtin_amdgcn_readfirstlane(work.rows);
  work.col = __builtin_amdgcn_readfirstlane(work.col);
  work.part = __builtin_amdgcn_readfirstlane(work.part);
  if (work.rows <= 0) return;
  const int m0 = work.row, rows = work.rows, n0 = work.col * OUT;
  const int k0 = work.part * a.k_part;
  const int steps = (min(a.KB, k0 + a.k_part) - k0) / kStep;

  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int lane = threadIdx.x & 63, l31 = lane & 31, hi = lane >> 5;
  const int wm = wave & 1, wn = wave >> 1;
  // a load covers 8 rows; offsets of the wave's rows from the tile's first
  const int unit = ((lane & 7) ^ (lane >> 3)) * 16;
  int ao[AC], bo[BC];
#pragma unroll
  for (int i = 0; i < AC; i++) {
    const int m = (wave * AC + i) * 8 + (lane >> 3);
    ao[i] = (a.src ? a.src[m0 + min(m, rows - 1)] : m) * (int)a.ldx + unit;
  }
#pragma unroll
  for (int i = 0; i < BC; i++) {
    int n = (wave * BC + i) * 8 + (lane >> 3);
    if constexpr (kHalves) {  // a wave's columns: half gate, half up
      n = n / CW * (CW / 2) + n % (CW / 2) + (n % CW >= CW / 2 ? cols : 0);
    }
    bo[i] = n * (int)a.ldw + unit;
  }
  const char* xb = a.src ? a.x : a.x + m0 * a.ldx;
  const char* wb = a.w + work.expert * a.ew + n0 * a.ldw;
  const int xn = a.src ? (int)a.xbytes : (rows - 1) * (int)a.ldx + a.KB;
  const int wn_ = ((kHalves ? N - n0 : min(N - n0, BN)) - 1) * (int)a.ldw + a.KB;
  // One row tile: the workgroups begin at columns of K apart. At the same ones of
  // rows of 2^n bytes they wait for the same few of the memory's channels (us, weights
  // out of cache, all at the first / apart: fp8 28672 x 4096 40 rows 32.0 / 25.9, 65536
  // x 8192 121 / 101, 128256 x 4096 117 / 108; bf16 28672 x 4096 40 rows 53.6 / 45.5;
  // 36864 x 4608 47.3 / 47.3). With more row tiles they would lose what they share.
  // (Only in tiles of few rows: in the others it costs 1 % of a large product. Not of
  // sums, whose parts lie apart and have few steps: 1080 x 2944 x 1408 bf16 16.9 us with it,
  // 15.7.)
  constexpr bool kApart = WM <= 2 && EPI != kSums;
  int first = 0;
  if constexpr (kApart) {
    if (!a.bounds && a.R <= BM && a.k_part == a.KB)
      first = (int)((blockIdx.x >> 3) * 2u % (uint32_t)steps);
  }
  auto column = [&](int s) {
    if constexpr (!kApart) return k0 + s * kStep;
    return k0 + (s + first < steps ? s + first : s + first - steps) * kStep;
  };
  // load l of a batch: the AC of step sa of x, then the BC of step sb of w
  auto load = [&](int l, int pa, int sa, int pb, int sb) {
    if (l < AC) {
      load_lds16(xb, sa < steps ? xn : 0, lds + pa * SA + (wave * AC + l) * 1024, ao[l],
                 column(sa));
    } else {
      load_lds16(wb, sb < steps ? wn_ : 0, lds + NA * SA + pb * SB + (wave * BC + l - AC) * 1024,
                 bo[l - AC], column(sb));
    }
  };

  constexpr int C = FP8 ? 2 : 4;              // chunks of K a step
  // A sum for each chunk of a step where there are few parts: the error grows with the
  // terms that are added one behind the other (bf16 4096 x 14336 in 4 parts 3.7e-7 of the
  // result, 2.5e-7 in the 8 that other tiles have, 1.7e-7 with these sums).
  constexpr int SUMS = SHAPE == kNarrow ? C : 1;
  f32x16 sums[SUMS][WN][WM];
#pragma unroll
  for (int u = 0; u < SUMS; u++) {
#pragma unroll
    for (int i = 0; i < WN; i++) {
#pragma unroll
      for (int j = 0; j < WM; j++) {
#pragma unroll
        for (int r = 0; r < 16; r++) sums[u][i][j][r] = 0.f;
      }
    }
  }
  auto& acc = sums[0];
  constexpr int MF = WM * WN, RO = WM + WN;   // products, operands a chunk
  typename std::conditional<FP8, i32x8, bf16x8>::type va[2][WM], vb[2][WN];
  // operand o of chunk c: b[0], a[0], the other b, the other a
  auto read = [&](int o, int buf, int pa, int pb, int c) {
    const bool isb = o == 0 || (o > 1 && o <= WN);
    const int i = isb ? (o ? o - 1 : 0) : (o == 1 ? 0 : o - WN);
    const char* p = isb ? lds + NA * SA + pb * SB + (wn * CW + i * 32 + l31) * kStep
                        : lds + pa * SA + ((wm * WM + i) * 32 + l31) * kStep;
    if constexpr (FP8) {
      const i32x4 lo = *(const i32x4*)(p + (((4 * c + 2 * hi) ^ (l31 & 7)) << 4));
      const i32x4 up = *(const i32x4*)(p + (((4 * c + 2 * hi + 1) ^ (l31 & 7)) << 4));
      const i32x8 v = __builtin_shufflevector(lo, up, 0, 1, 2, 3, 4, 5, 6, 7);
      if (isb) vb[buf][i] = v;
      else va[buf][i] = v;
    } else {
      const bf16x8 v = *(const bf16x8*)(p + (((2 * c + hi) ^ (l31 & 7)) << 4));
      if (isb) vb[buf][i] = v;
      else va[buf][i] = v;
    }
  };
  auto multiply = [&](int t, int c) {
    const int j = t / WN, i = t % WN, buf = c & 1;
    auto& acc = sums[c % SUMS];
    if constexpr (FP8) {  // block scales of 1
      acc[i][j] = __builtin_amdgcn_mfma_scale_f32_32x32x64_f8f6f4(
          vb[buf][i], va[buf][j], acc[i][j], 0, 0, 0, 0x7f7f7f7f, 0, 0x7f7f7f7f);
    } else {
      acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(vb[buf][i], va[buf][j], acc[i][j],
                                                          0, 0, 0);
    }
  };

  // What the epilogue scales by. A lane has row l31 of each 32 when it puts its
  // sums into LDS and, where rows are 2^n units, the same 8 columns of each row
  // that it takes out.
  constexpr int UR = (kHalves ? CW / 2 : CW) / 8;  // units of 8 results a row
  constexpr bool kFixed = 64 % UR == 0;
  float rs[WM], rw = 0.f;
  if constexpr (FP8 && EPI != kSums) {
#pragma unroll
    for (int j = 0; j < WM; j++) {
      const int m = m0 + min((wm * WM + j) * 32 + l31, rows - 1);
      rs[j] = a.sx[a.src ? a.src[m] : m];
    }
  }
  if constexpr (EPI == kSquare) rw = a.row_weight[m0 + min((int)threadIdx.x, rows - 1)];
  f32x4 cs[2];
  auto columns = [&](int n) {
    const float* s = a.sw + (int64_t)work.expert * N;
    cs[0] = *(const f32x4*)(s + min(n, cols - 4));
    cs[1] = *(const f32x4*)(s + min(n + 4, cols - 4));
  };
  if constexpr (FP8 && EPI != kSums && kFixed) columns(n0 + wn * UR * 8 + lane % UR * 8);

  // Batch s loads step s + NA of x and s + NB of w into the places that step s
  // leaves, spread over the C * MF products from its barrier to the next:
  // begun(g) loads lie in front of product g.
  auto begun = [](int g) {
    const int n = FP8 ? g : g / 2;
    return n < L ? n : L;
  };
#pragma unroll
  for (int s = -NB; s < 0; s++) {
    const int end = s < -1 ? L : begun(MF);
#pragma unroll
    for (int l = 0; l < L; l++) {
      if (l < end && (l >= AC || s + NA >= 0)) load(l, s + NA, s + NA, s + NB, s + NB);
    }
  }
  __builtin_amdgcn_sched_barrier(0);
  constexpr int kLater = (NA - 2) * L + (NB - NA) * BC;  // loads behind the next step's
  wait_loads<kLater + std::min(L, FP8 ? MF : MF / 2)>();
  barrier();
#pragma unroll
  for (int o = 0; o < RO; o++) read(o, 0, 0, 0, 0);
  int pa = 0, pb = 0, la = NA - 1, lb = NB - 1;  // places of this and of the last step
  for (int s = 0; s < steps; s++) {
    const int na = pa + 1 == NA ? 0 : pa + 1, nb = pb + 1 == NB ? 0 : pb + 1;
#pragma unroll
    for (int c = 0; c < C; c++) {
      const bool last = c == C - 1;
      if (last) {
        __builtin_amdgcn_sched_barrier(0);
        wait_loads<kLater>();
        barrier();
      }
#pragma unroll
      for (int t = 0; t < MF; t++) {
#pragma unroll
        for (int o = 0; o < RO; o++) {  // (bounds that unroll)
          if (o < RO * t / MF || o >= RO * (t + 1) / MF) continue;
          if (last) read(o, (c + 1) & 1, na, nb, 0);
          else read(o, (c + 1) & 1, pa, pb, c + 1);
        }
        multiply(t, c);
        const int g = last ? t : (c + 1) * MF + t;
        const int end = g == C * MF - 1 ? L : begun(g + 1);
#pragma unroll
        for (int l = 0; l < L; l++) {
          if (l < begun(g) || l >= end) continue;
          if (last) load(l, pa, s + NA, pb, s + NB);
          else load(l, la, s - 1 + NA, lb, s - 1 + NB);
        }
        __builtin_amdgcn_sched_barrier(0);
      }
    }
    la = pa;
    lb = pb;
    pa = na;
    pb = nb;
  }
  wait_loads<0>();
  barrier();
#pragma unroll
  for (int u = SUMS / 2; u > 0; u /= 2) {
#pragma unroll
    for (int c = 0; c < u; c++) {
#pragma unroll
      for (int i = 0; i < WN; i++) {
#pragma unroll
        for (int j = 0; j < WM; j++) sums[c][i][j] += sums[c + u][i][j];
      }
    }
  }

  // A lane's sums are row l31 and, four at a time, columns 8 q + 4 hi: all the
  // first halves of 8 columns lie in front of all the second ones.
  char* own = lds + wave * 32 * PITCH;
  float* weights = (float*)(lds + 4 * 32 * PITCH);
  if constexpr (EPI == kSquare) {
    if (threadIdx.x < BM) weights[threadIdx.x] = rw;
    __syncthreads();
  }
  ushort* y = a.y;
#pragma unroll
  for (int j = 0; j < WM; j++) {
#pragma unroll
    for (int i = 0; i < WN; i++) {
#pragma unroll
      for (int q = 0; q < 4; q++) {
        f32x4 v;
#pragma unroll
        for (int t = 0; t < 4; t++) {
          v[t] = acc[i][j][q * 4 + t];
          if constexpr (FP8 && EPI != kSums) v[t] *= rs[j];
        }
        *(f32x4*)(own + l31 * PITCH + hi * (CW * 2) + (i * 4 + q) * 16) = v;
      }
    }
    __builtin_amdgcn_wave_barrier();
#pragma unroll
    for (int k = 0; k < (32 * UR + 63) / 64; k++) {
      const int at = k * 64 + lane, r = at / UR, u = at % UR;
      if (32 * UR % 64 && r >= 32) continue;
      const char* p = own + r * PITCH + u * 16;
      const int row = (wm * WM + j) * 32 + r, n = n0 + (wn * UR + u) * 8;
      f32x4 v[2] = {*(const f32x4*)p, *(const f32x4*)(p + CW * 2)}, up[2];
      if constexpr (kHalves) {
        up[0] = *(const f32x4*)(p + UR * 16);
        up[1] = *(const f32x4*)(p + UR * 16 + CW * 2);
      }
      if (row >= rows || n >= cols) continue;
      const int m = m0 + row;
      if constexpr (EPI == kSums) {
        float* o = a.part + ((int64_t)work.part * a.R + m) * N + n;
        *(f32x4*)o = v[0];
        if (n + 4 < N) *(f32x4*)(o + 4) = v[1];
        continue;
      }
      if constexpr (FP8 && EPI != kSums) {
        if constexpr (!kFixed) columns(n);
#pragma unroll
        for (int h = 0; h < 2; h++) {
#pragma unroll
          for (int t = 0; t < 4; t++) v[h][t] *= cs[h][t];
        }
      }
      bf16x4 o[2];
#pragma unroll
      for (int h = 0; h < 2; h++) {
        if constexpr (kHalves) {
#pragma unroll
          for (int t = 0; t < 4; t++) {
            const float g = v[h][t];
            float z = g;  // gelu: 0.5 (1 + tanh y) = 1 / (1 + e^-2y)
            if constexpr (EPI == kGelu) z = 1.5957691216057308f * (g + 0.044715f * g * g * g);
            v[h][t] = g / (1.0f + __expf(-z)) * up[h][t];
          }
        }
        bf4 b = __builtin_convertvector(v[h], bf4);
        if constexpr (EPI == kSquare) {
#pragma unroll
          for (int t = 0; t < 4; t++) {
            const float f = fmaxf((float)b[t], 0.f);
            v[h][t] = f * f * weights[row];
          }
          b = __builtin_convertvector(v[h], bf4);
        }
        o[h] = __builtin_bit_cast(bf16x4, b);
      }
      ushort* to = y + (int64_t)m * cols + n;
      if (a.wide) {
        *(bf16x8*)to = __builtin_shufflevector(o[0], o[1], 0, 1, 2, 3, 4, 5, 6, 7);
      } else {
        *(bf16x4*)to = o[0];
        if (n + 4 < cols) *(bf16x4*)(to + 4) = o[1];
      }
    }
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_sched_barrier(0);
  }
}

template <bool FP8, Epilogue EPI>
void launch(int shape, const Args& a, int grid) {
  auto stream = c10::hip::getCurrentHIPStream().stream();
  auto go = [&](auto s) {
    constexpr int i = decltype(s)::value;
    if constexpr (EPI == kSums ||
                  (i != kNarrow && ((EPI != kSilu && EPI != kGelu) || kShapes[i].wn % 2 == 0))) {
      hipLaunchKernelGGL((tiled_kernel<FP8, i, EPI>), dim3(grid), dim3(256), 0, stream, a);
    } else {
      TORCH_CHECK(false, "no such tile");
    }
  };
  switch (shape) {
    case 0: go(std::integral_constant<int, 0>{}); break;
    case 1: go(std::integral_constant<int, 1>{}); break;
    case 2: go(std::integral_constant<int, 2>{}); break;
    case 3: go(std::integral_constant<int, 3>{}); break;
    case 4: go(std::integral_constant<int, 4>{}); break;
    case 5: go(std::integral_constant<int, 5>{}); break;
    case 6: go(std::integral_constant<int, 6>{}); break;
    case 7: go(std::integral_constant<int, 7>{}); break;
    case 8: go(std::integral_constant<int, 8>{}); break;
    default: TORCH_CHECK(false, "no such tile");
  }
  HIP_CHECK_KERNEL();
}

}  // namespace tiled
