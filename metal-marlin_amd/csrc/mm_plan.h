// Which kernel a product of more than 32 rows takes, and how it splits K: host code
// only, no HIP, so that the choice can be checked anywhere.
#pragma once
#include <algorithm>
#include <cstddef>

namespace mmplan {
constexpr int PLAN_PF_BK = 64;     // k per chunk of the prefill tiles
constexpr int PLAN_MID_BK = 128;   // of the mid-sized tiles

#ifndef MM_PF_KS_BLOCKS
#define MM_PF_KS_BLOCKS 200   // split K while the grid has fewer blocks than this
#endif

inline int cdiv(int a, int b) { return (a + b - 1) / b; }

// Above 32 rows the dispatch takes whichever kernel a time model says is fastest:
// the mid-sized tiles (mm_mid.h) or the prefill tiles of 256, 128 or 64 rows.
// A grid runs in rounds of 256 blocks (one per CU) of K / ks k each, and a last one
// that is little cheaper when it is not full; a K split adds its hand-off or
// reduction.  The constants are fitted, FP4 and INT4 apart, to 1900 shapes timed on
// every kernel under sustained load (the clock is power limited): M = 33 .. 8192,
// N = 512 .. 28672, K = 640 .. 14336, groups of 32 .. 128, Marlin, row-packed and
// pair forms; the model is within 2-6% (rms) of them, and the kernel it picks is on
// average 0.1% and at most 11% slower than the best of them.  The rules before it lost
// more: no mid-sized tiles, 256-row ones from 240 blocks on, 30-39% on average; and
// one model fitted to FP4 at K = 4096 for all, up to 41% (us of the kernel it took, of
// the best: 4096 -> 4096, M = 1600 71 mid, 62 on 128 rows; INT4 3968 -> 856, M = 2048
// 46 mid, 35 on 128 rows; INT4 4096 -> 28672, M = 384 153 mid, 132 on 256 rows).
struct TileCost {
  double base, round;        // us per launch, per round
  double full, part, grow;   // us per round at K = 4096: full; not full, plus its growth
  double a, bc;              // us per MB of activations; of weights and results
  double split, partial;     // us of a K split, and per MB of its partial sums
  double g64, g32;           // factor of groups that are a multiple of 64 only, of 32
};
enum { T_MID, T_256, T_128, T_128_FEW, T_64 };   // T_128_FEW: one row tile
constexpr TileCost COST[5][2] = {
    // FP4, INT4
    {{1.7, 2.0, 16.6, 8.7, 8.5, 0.18, 0.04, 0, 0, 1.08, 1.07},
     {2.8, 2.0, 23.9, 18.8, 5.3, 0.15, 0.03, 0, 0, 1.20, 1.15}},
    {{1.2, 6.1, 108, 80, 22.5, 0, 0.09, 0, 0, 1, 1.12},
     {4.9, 1.9, 129, 108, 10.4, 0.04, 0.07, 0, 0, 1, 1.24}},
    {{3.1, 3.0, 66.4, 40.8, 25, 0, 0.02, 5.1, 0.17, 1, 1.23},
     {5.4, 1.1, 86.5, 68.6, 15.1, 0, 0.01, 4.8, 0.21, 1, 1.32}},
    {{3.8, 1.8, 46, 49.5, 0, 0.02, 0.02, 2.5, 0.40, 0.92, 1.37},
     {5.6, 1.9, 61.8, 66, 0, 0.02, 0, 2.9, 0.33, 0.95, 1.42}},
    {{2.7, 2.7, 35.3, 32.5, 0, 0.02, 0, 2.4, 0.44, 0.95, 1.39},
     {2.6, 2.6, 48.2, 46.8, 0, 0.02, 0, 3.2, 0.44, 0.98, 1.31}}};
// Mid-sized tiles, at most one block per CU: up to 128 blocks (64 columns each)
// and above, where the time per k grows as the last CUs fill.
struct MidCost {
  double base64, slope64;    // us, us at K = 4096
  double base, slope, grow;
  double a, bc, split, partial, g64, g32;
};
constexpr MidCost COST_MID_ONE[2] = {{3.9, 10.9, 4.2, 13, 5.6, 0.10, 0.03, 2.2, 0.22, 1.16, 1.15},
                                     {4.8, 12.7, 3.5, 30, 1, 0.05, 0.02, 2.6, 0.20, 1.33, 1.33}};

template <class C>
inline double group_factor(const C& c, int g) {
  return g % 128 == 0 ? 1 : (g % 64 == 0 ? c.g64 : c.g32);
}
// Blocks of k k each, ks of them per tile; an M x N x K product.
inline double tiles_us(int kernel, bool int4, long blocks, double k, int ks, double part_mb, int M,
                       int N, int K, int g) {
  const double a_mb = 2e-6 * M * K, bc_mb = 0.5e-6 * N * K + 2e-6 * M * N;
  if (kernel == T_MID && blocks <= 256) {
    const MidCost& c = COST_MID_ONE[int4];
    const double kg = group_factor(c, g) * k / 4096, x = blocks / 256.0;
    return (blocks <= 128 ? c.base64 + c.slope64 * kg
                          : c.base + (c.slope + c.grow * x * x * x) * kg) +
           c.a * a_mb + c.bc * bc_mb + (ks > 1 ? c.split + c.partial * part_mb : 0);
  }
  const TileCost& c = COST[kernel][int4];
  const long n = blocks / 256;
  const double x = (blocks % 256) / 256.0;
  const double last = x > 0 ? c.part + c.grow * (kernel == T_MID ? x : x * x) : 0;
  return c.base + c.round * (n + (x > 0)) + group_factor(c, g) * k / 4096 * (c.full * n + last) +
         c.a * a_mb + c.bc * bc_mb + (ks > 1 ? c.split + c.partial * part_mb : 0);
}

// Prefill plan: tile config (0: 256x256, 1: 128x256, 2: 64x256) and K split.
struct PrefillPlan {
  int cfg;
  int ksplit;
  double us;
};

inline PrefillPlan plan_prefill_cfg(int cfg, int M, int N, int K, int g, bool int4) {
  PrefillPlan p{cfg, 1, 0};
  const long blocks = (long)cdiv(M, 256 >> cfg) * cdiv(N, 256);
  // Split K when the grid cannot fill the 256 CUs; every split keeps >= 8
  // chunks of 64 k so the pipeline stays full.  (256 x 256 tiles are taken only
  // where one round of them beats two of 128 x 256.)
  const int nch = K / PLAN_PF_BK;
  if (cfg != 0)
    while (blocks * p.ksplit < MM_PF_KS_BLOCKS && nch / (p.ksplit * 2) >= 8) p.ksplit *= 2;
  p.us = tiles_us(cfg == 0 ? T_256 : (cfg == 2 ? T_64 : (M <= 128 ? T_128_FEW : T_128)), int4,
                  blocks * p.ksplit, (double)K / p.ksplit, p.ksplit, p.ksplit * (4e-6 * M * N), M,
                  N, K, g);
  return p;
}

inline PrefillPlan plan_prefill(int M, int N, int K, int g, bool int4) {
  const PrefillPlan p = plan_prefill_cfg(M > 64 ? 1 : 2, M, N, K, g, int4);
  if (M <= 128) return p;
  const PrefillPlan big = plan_prefill_cfg(0, M, N, K, g, int4);
  return big.us < p.us ? big : p;
}

// Enough for either format and any group size: 256-row tiles do not split K.
inline size_t prefill_ws_bytes(int M, int N, int K) {
  const int ks = plan_prefill_cfg(M > 64 ? 1 : 2, M, N, K, PLAN_PF_BK, false).ksplit;
  return ks > 1 ? (size_t)ks * M * N * sizeof(float) : 0;
}

// Mid plan.  Tiles of 64 rows x 128 columns (8 waves, two blocks per CU), K split
// while that fits one block per CU and leaves each split 8 chunks; 64 columns
// where the split grid still leaves half the CUs idle; 128 rows where 65..128
// rows have more 64-row tiles than CUs.  Measured on MI355X, FP4 g = 128, us
// before (prefill tiles) -> mid:
//   M = 64:  4096 -> 2 x 14336 (SwiGLU) 31.5 -> 24.3, 4096 -> 6144 18.8 -> 12.1,
//            4096 -> 4096 17.0 -> 10.7, 4096 -> 1024 13.9 -> 9.4
//   M = 100: 4096 -> 2 x 14336 43.1 -> 35.6, 4096 -> 4096 20.9 -> 13.1,
//            14336 -> 4096 28.0 -> 24.1
//   M = 512: 4096 -> 4096 31.8 -> 22.1; INT4 4096 -> 6144 59.6 -> 50.5
//   row-packed M = 100: 4096 -> 2 x 14336 44.2 -> 35.2, 14336 -> 4096 28.0 -> 22.3;
//            M = 300 122.8 -> 93.6 and 67.4 -> 52.8
// What bounds it is LDS traffic and the matrix cores together.
struct MidPlan {
  int rb, wn;   // 32-row blocks and 64-column groups per tile; wn == 0: not a mid-sized product
  int ks, cps;  // K splits, chunks per split
};

// The mid-sized tiles that the product would take.  ct: 128-column tiles of the
// product (the pair and multi forms count their own).
inline MidPlan plan_mid_tiles(int M, long ct, int K) {
  MidPlan p{2, 0, 1, 0};
  const int nch = K / PLAN_MID_BK;
  const long tiles = ct * cdiv(M, 64);
  if (M <= 32 || K % PLAN_MID_BK != 0 || nch < 4) return p;
  p.wn = 2;
  if (M > 64 && M <= 128 && tiles > 256) p.rb = 4;
  while (tiles * (p.ks + 1) <= 256 && nch / (p.ks + 1) >= 8) ++p.ks;
  p.cps = cdiv(nch, p.ks);
  p.ks = cdiv(nch, p.cps);
  if (tiles * p.ks <= 128) p.wn = 1;
  return p;
}

inline double mid_us(const MidPlan& p, int M, long ct, int N, int K, int g, bool int4) {
  const long blocks = ct * cdiv(M, 64) * p.ks;
  return tiles_us(T_MID, int4, blocks, (double)p.cps * PLAN_MID_BK, p.ks,
                  blocks * (64 * 128 * 4e-6), M, N, K, g);
}

// The mid-sized plan of a product over N columns in ct tiles, wn == 0 where the
// prefill tiles (other_us) are faster.  FP4 up to 128 rows, and INT4 above 64 with
// more tiles than CUs, always take it: the prefill tiles were slower everywhere.
inline MidPlan choose_mid(int M, long ct, int N, int K, int g, bool int4, double other_us) {
  MidPlan p = plan_mid_tiles(M, ct, K);
  if (p.wn == 0 || (M <= 128 && (!int4 || ct * cdiv(M, 64) > 256))) return p;
  if (mid_us(p, M, ct, N, K, g, int4) > other_us) p.wn = 0;
  return p;
}
inline MidPlan plan_mid(int M, int N, int K, int g, bool int4) {
  return choose_mid(M, cdiv(N, 128), N, K, g, int4, plan_prefill(M, N, K, g, int4).us);
}
}  // namespace mmplan
