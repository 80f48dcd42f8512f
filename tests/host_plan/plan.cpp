// The GEMMs' plan and tile numbering (mlx-runner_amd/csrc/gemm_plan.h) compiled for the host.
//   plan            lines "KIND M N K" (dense, nvfp4, mxfp8, nvfp4-mlp, mxfp8-mlp) on 256 CUs ->
//                   "TMxTN whole|split|both" or "none"
//   plan numbering  random calls: every tile of a call runs once whole or once per K range, and the
//                   MLP's halves of a tile run as that tile runs in a projection's own call
#include <cstdint>
#include <cstdio>
#include <cstring>
#include <random>
#include <vector>

#include "gemm_plan.h"
using namespace qmm;

static int plans() {
  char kind[16];
  int M, K;
  long N;
  while (std::scanf("%15s %d %ld %d", kind, &M, &N, &K) == 4) {
    const bool mlp = std::strstr(kind, "-mlp");
    const bool dense = !std::strcmp(kind, "dense"), nv = !std::strncmp(kind, "nvfp4", 5);
    const GpPlan p = dense ? plan_dense(M, N, K, true, 256) : nv ? plan_nvfp4(M, N, K, mlp, 256) : plan_mxfp8(M, N, K, mlp, 256);
    if (p.cfg < 0) {
      std::puts("none");
      continue;
    }
    const GpCost &c = (dense ? DN_COST : nv ? NV_COST : MX_COST)[p.cfg];
    std::printf("%dx%d %s\n", c.TM, c.TN, !p.left ? "whole" : !p.whole ? "split" : "both");
  }
  return 0;
}

#define CHECK(x) \
  if (!(x)) return std::printf("call %d: %s\n", it, #x), 1
static int numbering() {
  std::mt19937 rng(7);
  for (int it = 0; it < 5000; ++it) {
    const int tm = 1 + rng() % 12, tn = 1 + rng() % 80, T = tm * tn;
    const int whole = rng() % 4 == 0 ? 0 : rng() % 3 == 0 ? T : rng() % (T + 1), S = whole == T ? 1 : 2 + rng() % 7;
    std::vector<int> ranges(T);            // of each tile: 1 whole, S split
    std::vector<unsigned> seen(T), half(2 * T);  // bit k: K range k ran
    for (int b = 0; b < whole + (T - whole) * S; ++b) {
      const GpBlock g = gp_block<false>(b, tm, tn, whole, S);
      CHECK(g.tm >= 0 && g.tm < tm && g.tn >= 0 && g.tn < tn && g.kr >= 0 && g.kr < S);
      const int id = g.tm * tn + g.tn;
      ranges[id] = g.split ? S : 1;
      CHECK(!(seen[id] >> g.kr & 1));
      seen[id] |= 1u << g.kr;
    }
    for (int id = 0; id < T; ++id) CHECK(ranges[id] > 0 && seen[id] == (1u << ranges[id]) - 1);
    for (int b = 0; b < 2 * whole + 2 * (T - whole) * S; ++b) {
      const GpBlock g = gp_block<true>(b, tm, tn, 2 * whole, S);
      CHECK(g.tm >= 0 && g.tm < tm && g.tn >= 0 && g.tn < 2 * tn && g.kr >= 0 && g.kr < S);
      CHECK((g.split ? S : 1) == ranges[g.tm * tn + g.tn / 2]);
      int rm, rn;  // the reduce finds the tile by its number
      gp_tile_at<true>(g.t, tm, tn, &rm, &rn);
      CHECK(rm == g.tm && rn == g.tn && g.split == (g.t >= 2 * whole));
      const int id = g.tm * 2 * tn + g.tn;
      CHECK(!(half[id] >> g.kr & 1));
      half[id] |= 1u << g.kr;
    }
    for (int id = 0; id < 2 * T; ++id) CHECK(half[id] == (1u << ranges[id / (2 * tn) * tn + id % (2 * tn) / 2]) - 1);
  }
  // an MLP's plan splits as the projection's own, whatever the sizes
  for (int it = 0; it < 20000; ++it) {
    const int M = 9 + rng() % 2500, K = 64 * (1 + rng() % 280);
    const int64_t N = 1 + rng() % 40000;
    const bool nv = rng() & 1;
    const GpCost *cost = nv ? NV_COST : MX_COST;
    const GpPlan one = nv ? plan_nvfp4(M, N, K, false, 256) : plan_mxfp8(M, N, K, false, 256);
    const GpPlan p = nv ? plan_nvfp4(M, N, K, true, 256) : plan_mxfp8(M, N, K, true, 256);
    if (p.cfg < 0) continue;
    const int64_t T = (int64_t)((M + cost[p.cfg].TM - 1) / cost[p.cfg].TM) * ((N + cost[p.cfg].TN - 1) / cost[p.cfg].TN);
    CHECK(p.S == one.S && p.whole + p.left == 2 * T && (p.left > 0) == (one.left > 0) && (p.whole > 0) == (one.whole > 0));
    if (one.whole && one.left) CHECK(p.cfg == one.cfg && p.whole == 2 * one.whole && p.left == 2 * one.left);
  }
  std::puts("ok");
  return 0;
}

int main(int argc, char **argv) { return argc > 1 && !std::strcmp(argv[1], "numbering") ? numbering() : plans(); }
