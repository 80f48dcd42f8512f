// The plan of a pipelined GEMM call and the numbering of its tiles: host code, and the part of the
// kernels that maps blocks to tiles.  Compiles for the host alone too, where the tests read it.
#pragma once
#include <cstdint>

#ifdef __HIPCC__
#include <hip/hip_runtime.h>
#define GP_HD __host__ __device__ __forceinline__
#else
#define GP_HD inline
#endif

namespace qmm {

constexpr int GP_MAX_SPLIT = 8;

// A call's blocks: [0, whole_tiles) run whole tiles, the others the S K-ranges of the tiles
// that are left (whole_tiles on).  Tiles are numbered in groups of 4 x tiles walked down x
// tiles first, and each XCD (the hardware hands it the blocks b with b % 8 = its number)
// takes a contiguous run of them, so the ~32 blocks resident on one XCD cover a 4 x 8 patch of
// (x rows, W rows) and share those operands in that XCD's L2.  Of a call that is all split, at
// few x tiles, the x tiles of one W range of one K range run next to each other, so that they
// share its W.
// PAIR (the MLP, whose tile holds half a tile's columns of gate and the same of up): tiles 2 t and
// 2 t + 1 are the halves of tile t of one matrix alone.
struct GpBlock {
  int t, tm, tn, kr;
  bool split;
};
template <bool PAIR>
GP_HD void gp_tile_at(int t, int tiles_m, int tiles_n, int *tm, int *tn) {
  constexpr int G = 4;
  const int half = t & 1;
  if (PAIR) t >>= 1;
  const int first = t / (G * tiles_n) * G, gm = tiles_m - first < G ? tiles_m - first : G, i = t - first * tiles_n;
  *tm = first + i % gm;
  *tn = PAIR ? 2 * (i / gm) + half : i / gm;
}
GP_HD int gp_xcd_run(int b, int n) {
  const int base = n / 8, rem = n % 8, x = b % 8;
  return x * base + (x < rem ? x : rem) + b / 8;
}
template <bool PAIR = false>
GP_HD GpBlock gp_block(int b, int tiles_m, int tiles_n, int whole_tiles, int S) {
  GpBlock r;
  r.split = b >= whole_tiles;
  r.kr = 0;
  if (!r.split) {
    r.t = gp_xcd_run(b, whole_tiles);
  } else {
    const int left = tiles_m * tiles_n * (PAIR ? 2 : 1) - whole_tiles, u = gp_xcd_run(b - whole_tiles, left * S);
    const int gm = whole_tiles == 0 && tiles_m <= 4 ? (PAIR ? 2 * tiles_m : tiles_m) : 1;
    r.kr = u / gm % S;
    r.t = whole_tiles + u / (gm * S) * gm + u % gm;
  }
  gp_tile_at<PAIR>(r.t, tiles_m, tiles_n, &r.tm, &r.tn);
  return r;
}

// ---------------------------------------------------------------- the plan of a call

// A tile size: TM x TN, per_cu blocks of it on a CU, and its measured cost: us per K step with
// 1, 2, .. blocks on every CU, and us per round beside that.
struct GpCost {
  int TM, TN, per_cu;
  float round, step[3];
};
struct GpPlan {
  int cfg, whole, left, S;  // whole tiles, then `left` tiles split S ways along K
  float us;                 // estimated
};
// The least estimated time over every tile size and every split of the tiles left after the
// whole rounds (at most max_split ways, one round of blocks, at least 4 K steps each, in
// units of `unit` steps).  Where several blocks share a CU, the last round may instead give
// every CU `more` whole tiles and the split ones run beside them.  A split adds the reduce: its
// launch and its partial sums' traffic.
inline GpPlan gp_plan(const GpCost *costs, int n, int M, int64_t N, int steps, int unit, int cus,
                      int max_split = GP_MAX_SPLIT) {
  if (cus <= 0) cus = 256;  // (no device answers: the launch reports it)
  GpPlan best{0, 0, 0, 1, 0.f};
  float best_us = 1e30f;
  const int units = (steps + unit - 1) / unit;
  for (int c = 0; c < n; ++c) {
    const GpCost &d = costs[c];
    const int64_t T = (int64_t)((M + d.TM - 1) / d.TM) * ((N + d.TN - 1) / d.TN);
    const int64_t slots = (int64_t)cus * d.per_cu, rounds = T / slots;
    for (int more = 0; more < d.per_cu; ++more) {
      const int64_t whole = rounds * slots + (int64_t)more * cus, left = T - whole;
      if (left < 0) break;
      for (int S = 1; S <= max_split; ++S) {
        if (S > 1 && (left == 0 || left * S > slots - (int64_t)more * cus || units < S || steps < 4 * S)) break;
        if (more && left && S == 1) continue;  // (the same blocks as more = 0)
        const int mine = (units + S - 1) / S * unit, split_steps = mine < steps ? mine : steps;
        int per = more + (int)((left * S + cus - 1) / cus);  // blocks on a CU in the last round
        if (per > d.per_cu) per = d.per_cu;
        float us = (float)rounds * ((float)steps * d.step[d.per_cu - 1] + d.round);
        if (more) us += (float)(steps - split_steps) * d.step[more - 1];
        if (per) us += (float)split_steps * d.step[per - 1] + d.round;
        if (S > 1) us += 1.5f + (float)left * S * (M < d.TM ? M : d.TM) * d.TN * 8.f / 6.6e6f;
        if (us < best_us) best_us = us, best = GpPlan{c, (int)whole, (int)left, S, us};
      }
    }
  }
  if (best.S == 1) best.whole += best.left, best.left = 0;
  return best;
}

// The plan of an MLP's gate and up in one launch (tiles numbered in pairs, see gp_block) whose
// sums run in the order of the two calls it replaces, so that its result is theirs bit for bit.
// The order of a column's sums depends only on the split S of its tile along K: where `one`, a
// call's own plan, splits no tile, or all, any of the n_pair tile sizes that have the form does,
// with that split (the least estimated time); where it splits the last tiles, its own tile size
// and twice its tiles.  cfg -1: that size has no MLP form, or the two calls and the activation (at
// 2.7 TB/s) are estimated faster, as where their tile has no MLP form and twice the next one's
// blocks need another round: nvfp4 20 x 17408 x 5120 50 us in one launch, 40 in three calls; mxfp8
// 200 x 17408 x 5120 130 and 121 (64 rows: 63 and 75; 2048 rows: 572 and 614).
inline GpPlan gp_plan_pair(const GpCost *costs, int n_pair, const GpPlan &one, int M, int64_t N, int steps, int unit,
                           int cus) {
  if (cus <= 0) cus = 256;
  if (one.whole && one.left) return GpPlan{one.cfg < n_pair ? one.cfg : -1, 2 * one.whole, 2 * one.left, one.S, 0.f};
  GpPlan best{-1, 0, 0, one.S, 0.f};
  float best_us = 2.f * one.us + 3.f + (float)M * (float)N * 6.f / 2.7e6f;
  const int units = (steps + unit - 1) / unit, mine = (units + one.S - 1) / one.S * unit;
  for (int c = 0; c < n_pair; ++c) {
    const GpCost &d = costs[c];
    const int64_t T = (int64_t)((M + d.TM - 1) / d.TM) * ((N + d.TN - 1) / d.TN) * 2, blocks = T * one.S;
    if (blocks > INT32_MAX) continue;
    const int64_t slots = (int64_t)cus * d.per_cu, rounds = blocks / slots;
    const int per = (int)((blocks - rounds * slots + cus - 1) / cus), n = mine < steps ? mine : steps;
    float us = (float)rounds * ((float)n * d.step[d.per_cu - 1] + d.round);
    if (per) us += (float)n * d.step[per - 1] + d.round;
    if (one.S > 1) us += 1.5f + (float)blocks * (M < d.TM ? M : d.TM) * d.TN * 8.f / 6.6e6f;
    if (us < best_us) best_us = us, best = GpPlan{c, one.S > 1 ? 0 : (int)T, one.S > 1 ? (int)T : 0, one.S, us};
  }
  return best;
}

// ---------------------------------------------------------------- the tile sizes and their costs

// Dense bf16 (DnGeom).  Measured on calls of whole rounds and of one block per CU, weights cold: on
// 18 shapes of 300 to 2048 rows the plan's choice takes 1.02 times the best tile's time on average, at
// most 1.07, on 39 of 9 rows up 1.05 and 1.35 (1000 x 10240 x 5120: 256 x 160 tiles fill one round of
// 256 CUs, 95 us; 256 x 256 ones, 160 of them, 99).
inline constexpr GpCost DN_COST[] = {{256, 256, 1, 3.f, {1.24f}},         {256, 160, 1, 3.f, {1.10f}},
                                     {192, 256, 1, 3.f, {1.20f}},         {256, 128, 1, 3.f, {0.91f}},
                                     {128, 128, 2, 3.f, {0.64f, 0.90f}},  {64, 128, 2, 3.f, {0.56f, 0.74f}},
                                     {64, 64, 3, 3.f, {0.42f, 0.57f, 0.72f}}};

// nvfp4 (NvGeom).  Fitted to 45 shapes of 5 to 1930 rows, two thirds under 400, with every tile and split:
// rms error 7%, the plan's choice 1.01 of the best of them on average, at most 1.26.  On 19 others
// of 300 to 2048 rows the choice is 1.01 of the best on average, at most 1.08; the estimate itself is
// low there, as the clock is under full load: measured 0.94 to 1.27 times it, 1.11 on average.
inline constexpr GpCost NV_COST[] = {{256, 256, 1, 9.7f, {1.10f}},         {192, 256, 1, 8.9f, {0.86f}},
                                     {128, 256, 1, 9.7f, {0.58f}},         {128, 128, 2, 7.8f, {0.42f, 0.69f}},
                                     {64, 128, 2, 8.6f, {0.26f, 0.43f}},   {32, 128, 3, 8.4f, {0.22f, 0.34f, 0.48f}}};

// mxfp8 (MxGeom).  Fitted to 50 shapes of 5 to 1930 rows likewise: rms error 8%, the choice 1.01 of the
// best on average, at most 1.18.  On 22 others of 300 to 2048 rows 1.02, at most 1.19 (W of 20000 rows
// and more at K of 1100: two blocks of 128 x 128 on a CU overlap their rounds, which the plan prices
// one after the other); measured 0.73 to 1.34 times the estimate.  The last two have no MLP form: a
// wave's column blocks are not pairs.
inline constexpr GpCost MX_COST[] = {{256, 256, 1, 13.9f, {1.05f}},        {192, 256, 1, 13.4f, {0.83f}},
                                     {128, 256, 1, 13.6f, {0.61f}},        {128, 128, 2, 12.2f, {0.49f, 0.76f}},
                                     {64, 128, 2, 12.5f, {0.28f, 0.46f}},  {256, 160, 1, 13.7f, {0.72f}},
                                     {32, 128, 2, 11.8f, {0.24f, 0.40f}}};

// The K elements of a step, and the steps of a W stage (what a split divides).
constexpr int GP_STEP = 64, NV_UNIT = 4, MX_UNIT = 2;
// The plans of a call; mlp: of gate and up [N, K] in one launch, cfg -1 if that is not done.
// Dense: split, whether there is scratch for the partial sums of tiles split along K.
inline GpPlan plan_dense(int M, int64_t N, int K, bool split, int cus) {
  return gp_plan(DN_COST, sizeof(DN_COST) / sizeof(DN_COST[0]), M, N, (K + GP_STEP - 1) / GP_STEP, 1, cus,
                 split ? GP_MAX_SPLIT : 1);
}
inline GpPlan plan_nvfp4(int M, int64_t N, int K, bool mlp, int cus) {
  constexpr int n = sizeof(NV_COST) / sizeof(NV_COST[0]);
  const int steps = (K + GP_STEP - 1) / GP_STEP;
  const GpPlan one = gp_plan(NV_COST, n, M, N, steps, NV_UNIT, cus);
  return mlp ? gp_plan_pair(NV_COST, n - 1, one, M, N, steps, NV_UNIT, cus) : one;
}
inline GpPlan plan_mxfp8(int M, int64_t N, int K, bool mlp, int cus) {
  constexpr int n = sizeof(MX_COST) / sizeof(MX_COST[0]);
  const int steps = (K + GP_STEP - 1) / GP_STEP;
  const GpPlan one = gp_plan(MX_COST, n, M, N, steps, MX_UNIT, cus);
  return mlp ? gp_plan_pair(MX_COST, n - 2, one, M, N, steps, MX_UNIT, cus) : one;
}

}  // namespace qmm
