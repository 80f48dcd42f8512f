// nvfp4 prefill GEMM on the bf16 MFMA (v_mfma_f32_32x32x16_bf16).
//
// y[M, N] = x[M, K] @ deq(W)[N, K].T, W in nvfp4 (E2M1 nibbles, one E4M3 scale
// per 16), x bf16, fp32 accumulation, bf16 out.
//
// Why bf16 MFMA: an E2M1 value times an E4M3 scale has up to 6 significant bits,
// which no 8-bit MFMA operand format holds, and the scaled MFMAs take only
// E8M0 scales per 32; in bf16 (8 bits) the dequantized weight is exact.
//
// What bounds it: at tall x the matrix cores at the clock the power limit leaves (a large
// bf16 library product reaches ~1.45 PFLOP/s here), at short x the latency of a step.  So:
//   * K steps of 64, x by DMA in whole 128-byte cache lines per row into a ring of SX
//     stages.  A row's W piece of a step is 32 bytes, so W moves in stages of four steps,
//     128 bytes per row as well, with their scales; two such stages are four steps of lead,
//     which covers the ~1.2 us that cold W takes.
//   * The waves lie side by side along W (1 x 4), so that one wave of the block dequantizes
//     a W element (VALU work), in pairs spread between the MFMAs of the sub-step before it
//     is used, beside the reads of that sub-step's x; one barrier per K step.
//   * The tile height is chosen per call (nv_plan), and the tiles left over after the whole
//     rounds are split along K over the idle CUs, fp32 partial sums reduced in K order
//     (deterministic) by a second kernel.
// Measured, us per call, weights cold (M x N x K; the former kernel, two groups of waves in
// turns with W moved 32 bytes per row and step, in brackets): 2048 x 16480 x 5120  271 (318,
// 1.28 PFLOP/s now), 2048 x 34816 x 5120  544 (567), 500 x 10240 x 5120  57 (63), 48 x 17408 x
// 5120  23-26 (26-30), 200 x 6144 x 5120  26-31 (32).  256 x 256 tiles in 8 waves of 128 x 64, which dequantize every element
// twice: 276 in the first.  K that is not a multiple of 64, which ran gemm.hip's kernel:
// 33 x 1000 x 1056 28 -> 9.4.
#include <type_traits>

#include "gemm_pipe.h"
#include "qmm_device.h"
#include "qmm_launch.h"

namespace qmm {

namespace {
constexpr int V_BK = GP_STEP;   // K elements of a step: 128 bytes of an x row, 32 of a W row
constexpr int V_SS = NV_UNIT;    // steps of a W stage: 128 bytes of a W row, 16 of its scales
// A block's tile: WM x WN waves of (32 FI) x (32 FJ); LDS rings of SX stages of x (a step
// each) and two stages of W and its scales (V_SS steps each).
template <int FI_, int FJ_, int WM_, int WN_, int SX_>
struct NvGeom {
  static constexpr int FI = FI_, FJ = FJ_, WM = WM_, WN = WN_, SX = SX_;
  static constexpr int TM = 32 * FI * WM, TN = 32 * FJ * WN, NW = WM * WN, THREADS = 64 * NW;
  static constexpr int XT = TM * 128, WT = TN * 128, ST = TN * 16;
  static constexpr int WOFF = SX * XT, SOFF = WOFF + 2 * WT;  // the rings' places
  static constexpr int LDS = SOFF + 2 * ST;
  static constexpr int NX = TM / 8 / NW;           // x DMAs per wave per step
  static constexpr int NWD = TN / 8 / NW;          // W DMAs per wave per stage, in two halves:
  static constexpr int NA = NWD / 2 + 1, NB = NWD - NWD / 2;  // NA with the scales' one
  static_assert(TM / 8 % NW == 0 && TN / 8 % NW == 0 && TN % 64 == 0 && NW % 2 == 0 && SX >= 2 && SX <= 4, "");
  static constexpr int REGION = 32 * (64 * FJ + 32);
  static_assert(NW * REGION <= LDS, "the epilogue regions fit the rings");
  // DMAs that may be in flight at the barrier of step j of a stage (see the kernel): those
  // issued after x of the next step, and at j = 3 none of the next W stage's
  static constexpr int in_flight(int j) {
    int n = (SX - 2) * NX;
    for (int i = j + 1 - SX; i < j; ++i) n += (i & 3) == 3 ? NA : (i & 3) == 0 ? NB : 0;
    return j == 3 && n > 2 * NX ? 2 * NX : j == 3 && SX < 4 ? (SX - 2) * NX : n;
  }
};
}  // namespace

// Zeros that stand for the pieces of the last step and stage past K.
__device__ const uint4 nv_zero = {0, 0, 0, 0};

// 16-byte piece p of a row's 128 bytes is stored at slot p ^ nv_swz(row).
__device__ __forceinline__ int nv_swz(int r) { return (r & 7) ^ ((r >> 3) & 1); }

// MLP: the tile's W rows are two matrices', 32-row blocks of gate and of up in turn (row
// blocks 2 b and 2 b + 1 of a tile are rows 32 b + [0, 32) of the tile's TN / 2), and the
// result is silu(gate) * up, TN / 2 columns of it per tile.
template <class G, bool MLP>
__global__ __launch_bounds__(G::THREADS, G::LDS <= 81920 ? 2 * G::NW / 4 : G::NW / 4) void gemm_nvfp4_kernel(
    const uint16_t *__restrict__ x, const uint8_t *__restrict__ w, const uint8_t *__restrict__ sp,
    const uint8_t *__restrict__ w_up, const uint8_t *__restrict__ sp_up, const YOut yo, int M, int N, int K,
    int whole_tiles, int S, float *__restrict__ part) {
  constexpr int FI = G::FI, FJ = G::FJ, NX = G::NX, NWD = G::NWD, SX = G::SX;
  constexpr int TC = MLP ? G::TN / 2 : G::TN;  // columns of y per tile
  static_assert(!MLP || FJ % 2 == 0, "a wave holds gate and up of a column");
  extern __shared__ __attribute__((aligned(16))) uint8_t lds[];
  const uint32_t lds0 = lds_addr(lds);
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int wm = wave % G::WM, wn = wave / G::WM;
  const int tiles_m = (M + G::TM - 1) / G::TM, tiles_n = (N + G::TN - 1) / G::TN;
  const int steps = (K + V_BK - 1) / V_BK, stages = (steps + V_SS - 1) / V_SS;
  const GpBlock blk = gp_block<MLP>(blockIdx.x, tiles_m, tiles_n, whole_tiles, S);
  const int m0 = blk.tm * G::TM, n0 = blk.tn * TC;
  if (MLP && n0 >= N) return;  // the second half of the last pair (its partial sums are not read either)
  // the block's W stages [g_begin, g_end) and steps [s_begin, s_end)
  const int g_begin = blk.split ? (int)((int64_t)blk.kr * stages / S) : 0;
  const int g_end = blk.split ? (int)((int64_t)(blk.kr + 1) * stages / S) : stages;
  const int s_begin = g_begin * V_SS, s_end = min(g_end * V_SS, steps);

  // A DMA fills 1 KiB: rows 8 g + [0, 8) of a stage of x (or W), g = wave + NW i; lane l the
  // 16-byte slot l % 8 of row l / 8, which holds piece (l % 8) ^ swz(row) of the row's 128 bytes.
  const int64_t wrow = K >> 1;
  const uint8_t *xb = (const uint8_t *)x + (int64_t)m0 * K * 2;
  const int dr = 8 * wave + (lane >> 3), dp = (lane & 7) ^ nv_swz(dr);  // rows 8 NW apart share a swizzle
  uint32_t xo[NX], wo[NWD];
  const uint8_t *wb[MLP ? NWD : 1];
#pragma unroll
  for (int i = 0; i < NX; ++i) xo[i] = (uint32_t)(min(m0 + dr + 8 * G::NW * i, M - 1) - m0) * (uint32_t)(2 * K) + dp * 16;
  if constexpr (!MLP) wb[0] = w + (int64_t)n0 * wrow;
#pragma unroll
  for (int i = 0; i < NWD; ++i) {
    const int q = wave + G::NW * i, r = dr + 8 * G::NW * i;  // 8 rows of one 32-row block
    int row = r;
    if constexpr (MLP) {
      wb[i] = ((q >> 2) & 1 ? w_up : w) + (int64_t)n0 * wrow;
      row = (r >> 6) * 32 + (r & 31);
    }
    wo[i] = (uint32_t)((min(n0 + row, N - 1) - n0) * wrow) + dp * 16;
  }
  // scales: the tile-major copy holds, per 256 rows and step, 256 dwords; a stage's V_SS x TN
  // dwords take TN / 64 DMAs of four rows per lane, one per wave (the waves past that repeat one)
  const int sq = (wave % (G::TN / 64)) * 64 + lane, sd = sq / (G::TN / 4), st = sq % (G::TN / 4) * 4;
  const int sr = min(n0 + (MLP ? (st >> 6) * 32 + (st & 31) : st), ((N + 255) & ~255) - 4);
  const uint8_t *sb = (MLP && (st >> 5) & 1 ? sp_up : sp) + ((int64_t)(sr >> 8) * steps * 256 + (sr & 255)) * 4;
  const uint32_t sl = (uint32_t)(G::SOFF + (wave % (G::TN / 64)) * 1024);

  auto issue_x = [&](int i, int s) __attribute__((always_inline)) {
    gp_dma16s(xb + (int64_t)s * 128, xo[i], lds0 + (uint32_t)((s % SX) * G::XT + (wave + G::NW * i) * 1024));
  };
  auto issue_w = [&](int i, int g) __attribute__((always_inline)) {
    gp_dma16s(wb[MLP ? i : 0] + (int64_t)g * 128, wo[i], lds0 + (uint32_t)(G::WOFF + (g & 1) * G::WT + (wave + G::NW * i) * 1024));
  };
  // (a stage's steps past the last one repeat it)
  auto issue_s = [&](int g) __attribute__((always_inline)) {
    gp_dma16(sb + (int64_t)min(g * V_SS + sd, steps - 1) * 1024, lds0 + sl + (uint32_t)((g & 1) * G::ST));
  };
  // the x DMAs of step s, a whole one or the rows' last, whose pieces past K are zeros
  auto issue_x_any = [&](int s) __attribute__((always_inline)) {
#pragma unroll
    for (int i = 0; i < NX; ++i) {
      if ((s + 1) * V_BK <= K) {
        issue_x(i, s);
      } else {
        const uint8_t *p = xb + xo[i] + (int64_t)s * 128;
        if (s * V_BK + 8 * dp >= K) p = (const uint8_t *)&nv_zero;
        gp_dma16(p, lds0 + (uint32_t)((s % SX) * G::XT + (wave + G::NW * i) * 1024));
      }
    }
  };
  // W DMAs [i0, i1) of stage g, likewise
  auto issue_w_any = [&](int i0, int i1, int g) __attribute__((always_inline)) {
#pragma unroll
    for (int i = 0; i < NWD; ++i) {
      if (i < i0 || i >= i1) continue;
      if ((g + 1) * V_SS * V_BK <= K) {
        issue_w(i, g);
      } else {
        const uint8_t *p = wb[MLP ? i : 0] + wo[i] + (int64_t)g * 128;
        if (g * V_SS * V_BK + 32 * dp >= K) p = (const uint8_t *)&nv_zero;
        gp_dma16(p, lds0 + (uint32_t)(G::WOFF + (g & 1) * G::WT + (wave + G::NW * i) * 1024));
      }
    }
  };

  // Fragments (32x32x16 bf16 operands: lane l holds row l % 32 and half fh = l / 32 of the 16
  // K): sub-step ks takes the step's elements 32 fh + 8 ks + [0, 8), piece 4 fh + ks of the x
  // row; a lane's four W pieces are then the 16 bytes 2 j + fh of the W row (step j of its
  // stage), and their scales bytes 2 fh and 2 fh + 1 of the row's dword.
  const int fr = lane & 31, fh = lane >> 5;
  const int ra = wm * 32 * FI + fr, rb = wn * 32 * FJ + fr;
  const int oa = ra * 128 + 16 * ((4 * fh) ^ nv_swz(ra));
  const int ob = G::WOFF + rb * 128 + 16 * (fh ^ nv_swz(rb));
  const int os = G::SOFF + rb * 4 + 2 * fh;

  f32x16_t acc[FI][FJ];
#pragma unroll
  for (int i = 0; i < FI; ++i)
#pragma unroll
    for (int j = 0; j < FJ; ++j)
#pragma unroll
      for (int v = 0; v < 16; ++v) acc[i][j][v] = 0.f;

  bf16x8_t af[2][FI], bf[2][FJ];  // sub-step ks's fragments, in set ks % 2
  uint4 wq[FJ];                   // the step's W fragments as stored
  uint32_t wsc[FJ];
  auto read_x = [&](int s, int ks, int i) __attribute__((always_inline)) {
    af[ks & 1][i] = *(const bf16x8_t *)(lds + (s % SX) * G::XT + (oa ^ (16 * ks)) + 4096 * i);
  };
  auto read_w = [&](int s, int j) __attribute__((always_inline)) {
    const int g = s >> 2, t = s & 3;
    wq[j] = *(const uint4 *)(lds + (g & 1) * G::WT + (ob ^ (32 * t)) + 4096 * j);
    wsc[j] = *(const uint16_t *)(lds + (g & 1) * G::ST + os + t * (G::TN * 4) + 128 * j);
  };
  // pair p (of 4) of W fragment j for sub-step ks: E2M1 -> f32, times the scale, -> bf16, exact
  auto deq = [&](int ks, int j, int p) __attribute__((always_inline)) {
    const uint32_t word = ks == 0 ? wq[j].x : ks == 1 ? wq[j].y : ks == 2 ? wq[j].z : wq[j].w;
    const float sc = ks < 2 ? __builtin_amdgcn_cvt_f32_fp8((int)wsc[j], 0) : __builtin_amdgcn_cvt_f32_fp8((int)wsc[j], 1);
    f32x2_t v;
    if (p == 0) v = fp4x2_to_f32x2<0>(word);
    else if (p == 1) v = fp4x2_to_f32x2<1>(word);
    else if (p == 2) v = fp4x2_to_f32x2<2>(word);
    else v = fp4x2_to_f32x2<3>(word);
    bf[ks & 1][j][2 * p] = (__bf16)(v.x * sc);
    bf[ks & 1][j][2 * p + 1] = (__bf16)(v.y * sc);
  };
  constexpr int NM = FI * FJ, ND = 4 * FJ;  // MFMAs and dequantized pairs of a sub-step

  // Order of the DMAs: W and scales of the first stage, x of the first SX steps, the first
  // half of the second stage; then at each step s, x of step s + SX followed by the second
  // half of the next W stage (at a stage's first step) or the first half of the one after
  // (at its last step).
  issue_w_any(0, NWD, g_begin);
  issue_s(g_begin);
#pragma unroll 1
  for (int t = 0; t < SX && s_begin + t < s_end; ++t) issue_x_any(s_begin + t);
  if (g_begin + 1 < g_end) {
    issue_w_any(0, NWD / 2, g_begin + 1);
    issue_s(g_begin + 1);
  }
  if (g_begin + 1 < g_end && s_end - s_begin >= SX) gp_wait_barrier<(SX - 1) * NX + G::NA>();
  else gp_wait_barrier<0>();
#pragma unroll
  for (int j = 0; j < FJ; ++j) read_w(s_begin, j);
#pragma unroll
  for (int i = 0; i < FI; ++i) read_x(s_begin, 0, i);
#pragma unroll
  for (int d = 0; d < ND; ++d) deq(0, d % FJ, d / FJ);

  // Step s = V_SS g + T.  Sub-step ks's MFMAs run beside the reads and the dequantization of
  // the next sub-step's fragments.  Before sub-step 3 every read of the step's stages is done
  // and, after the barrier, every wave's: its x stage, and after a W stage's last step that
  // stage, are refilled.
  // MODE 2: all of it whole; 3: as 2, but no W stage g + 2; 1: whatever is in the range, each
  // barrier waiting for every DMA.
  auto step = [&](auto mode_c, auto t_c, int g) __attribute__((always_inline)) {
    constexpr int MODE = decltype(mode_c)::value, T = decltype(t_c)::value;
    const int s = V_SS * g + T;
#pragma unroll
    for (int ks = 0; ks < 4; ++ks) {
      if (ks == 3) {
        if constexpr (MODE >= 2) gp_wait_barrier<G::in_flight(T)>();
        else gp_wait_barrier<0>();
        __builtin_amdgcn_sched_barrier(0);
        if constexpr (MODE == 1) {
          if (s + SX < s_end) issue_x_any(s + SX);
          if (T == 0 && g + 1 < g_end) issue_w_any(NWD / 2, NWD, g + 1);
          if (T == 3 && g + 2 < g_end) {
            issue_w_any(0, NWD / 2, g + 2);
            issue_s(g + 2);
          }
        }
      }
      // the DMAs of this sub-step: x, then W, the scales last
      constexpr int NWH = T == 0 ? G::NB : T == 3 && MODE == 2 ? G::NA : 0;
      constexpr int W0 = T == 0 ? NWD / 2 : 0;
      constexpr int NI = NX + NWH;
#pragma unroll
      for (int m = 0; m < NM; ++m) {
        if (ks == 3) {
          if constexpr (MODE >= 2) {
#pragma unroll
            for (int i = m * NI / NM; i < (m + 1) * NI / NM; ++i) {
              if (i < NX) issue_x(i, s + SX);
              else if (T == 0) issue_w(W0 + i - NX, g + 1);
              else if (i - NX < NWD / 2) issue_w(i - NX, g + 2);
              else issue_s(g + 2);
            }
          }
          if (m == 0) {
#pragma unroll
            for (int j = 0; j < FJ; ++j) read_w(s + 1, j);
          }
#pragma unroll
          for (int i = m * FI / NM; i < (m + 1) * FI / NM; ++i) read_x(s + 1, 0, i);
          // the W fragments have arrived by the second half
          if (2 * m >= NM || NM == 1) {
            constexpr int H = NM - NM / 2;
            const int mm = m - NM / 2;
#pragma unroll
            for (int d = mm * ND / H; d < (mm + 1) * ND / H; ++d) deq(0, d % FJ, d / FJ);
          }
        } else {
#pragma unroll
          for (int i = m * FI / NM; i < (m + 1) * FI / NM; ++i) read_x(s, ks + 1, i);
#pragma unroll
          for (int d = m * ND / NM; d < (m + 1) * ND / NM; ++d) deq(ks + 1, d % FJ, d / FJ);
        }
        const int j = m / FI, i = m % FI;
        acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(af[ks & 1][i], bf[ks & 1][j], acc[i][j], 0, 0, 0);
        __builtin_amdgcn_sched_barrier(0);
      }
    }
  };
  using I0 = std::integral_constant<int, 0>;
  using I1 = std::integral_constant<int, 1>;
  using I2 = std::integral_constant<int, 2>;
  using I3 = std::integral_constant<int, 3>;
  int g = g_begin;
  // the stages whose SX steps ahead and W stage ahead are whole (MODE 3: and W stage g + 2 is not)
  const int whole = min(g_end, K / (V_SS * V_BK));
#pragma unroll 1
  for (; g + 2 < whole; ++g) {
    step(I2{}, I0{}, g);
    step(I2{}, I1{}, g);
    step(I2{}, I2{}, g);
    step(I2{}, I3{}, g);
  }
  if (g + 2 == whole && whole == g_end) {
    step(I3{}, I0{}, g);
    step(I3{}, I1{}, g);
    step(I3{}, I2{}, g);
    step(I3{}, I3{}, g);
    ++g;
  }
#pragma unroll 1
  for (; g < g_end; ++g) {
    const int n = s_end - V_SS * g;
    step(I1{}, I0{}, g);
    if (n > 1) step(I1{}, I1{}, g);
    if (n > 2) step(I1{}, I2{}, g);
    if (n > 3) step(I1{}, I3{}, g);
  }
  gp_lds_barrier();

  const int row0 = m0 + wm * 32 * FI;
  if (blk.split) {
    gp_store_partial<FI, FJ, G::NW>(acc, part + (size_t)((blk.t - whole_tiles) * S + blk.kr) * G::TM * G::TN, wave, lane,
                                    M - row0);
    return;
  }
  const bool vec = yout_vec(yo);
  uint8_t *region = lds + wave * G::REGION;
  if constexpr (MLP) {
    f32x16_t h[FI][FJ / 2];
    gp_silu_mul<FI, FJ>(acc, h);
    gp_store_rows<FI, FJ / 2, 0>(h, region, lane, yo, M, row0, n0 + wn * 16 * FJ, N, vec);
  } else {
    gp_store_rows<FI, FJ, 0>(acc, region, lane, yo, M, row0, n0 + wn * 32 * FJ, N, vec);
  }
}

template <class G, bool MLP>
__global__ __launch_bounds__(256) void gemm_nvfp4_reduce_kernel(const float *__restrict__ part, const YOut yo, int M,
                                                                int N, int whole_tiles, int S) {
  gp_reduce_tile<G, MLP>(part, yo, M, N, whole_tiles, S, blockIdx.x * 256 + threadIdx.x);
}

// ---------------------------------------------------------------- the plan

namespace {
using Nv256 = NvGeom<8, 2, 1, 4, 2>;  // 256 x 256
using Nv192 = NvGeom<6, 2, 1, 4, 2>;  // 192 x 256
using NvW = NvGeom<4, 2, 1, 4, 2>;    // 128 x 256
using Nv128 = NvGeom<4, 1, 1, 4, 2>;  // 128 x 128, two blocks per CU
using Nv64 = NvGeom<2, 1, 1, 4, 4>;   // 64 x 128, two blocks per CU
using Nv32 = NvGeom<1, 1, 1, 4, 4>;   // 32 x 128, three blocks per CU
}  // namespace

// The MLP form needs a wave's column blocks in pairs: at 128 columns, 2 x 2 waves.
using Nv128M = NvGeom<2, 2, 2, 2, 2>;  // 128 x 128, two blocks per CU
using Nv64M = NvGeom<1, 2, 2, 2, 4>;   // 64 x 128, two blocks per CU

static GpPlan nv_plan(const QmmArgs &a) { return plan_nvfp4(a.M, a.N, a.K, a.w_up != nullptr, device_cu_count()); }

template <class G, bool MLP>
static hipError_t launch_nv(const QmmArgs &a, const GpPlan &p, const uint8_t *sp, const uint8_t *sp_up, float *part,
                            hipStream_t st) {
  static std::atomic<uint64_t> lds_set{0};
  hipError_t e = ensure_dynamic_lds(lds_set, (const void *)gemm_nvfp4_kernel<G, MLP>, G::LDS);
  if (e != hipSuccess) return e;
  const YOut yo = yout_of(a);  // y, or a grouped call's parts
  hipLaunchKernelGGL((gemm_nvfp4_kernel<G, MLP>), dim3(p.whole + p.left * p.S), dim3(G::THREADS), G::LDS, st,
                     (const uint16_t *)a.x, a.w, sp, a.w_up, sp_up, yo, a.M, a.N, a.K, p.whole, p.S, part);
  e = hipGetLastError();
  if (e != hipSuccess || p.left == 0) return e;
  constexpr int RB = G::NW * G::FI * (MLP ? G::FJ / 2 : G::FJ);
  hipLaunchKernelGGL((gemm_nvfp4_reduce_kernel<G, MLP>), dim3(p.left * RB), dim3(256), 0, st, (const float *)part, yo,
                     a.M, a.N, p.whole, p.S);
  return hipGetLastError();
}

// K % 32: 16-byte W pieces; x and W rows 16-byte aligned for the DMA.
bool gemm_nvfp4_ok(const QmmArgs &a) {
  return a.mode == NVFP4 && !a.x_f32 && a.K % 32 == 0 && a.K > 0 && a.M > 0 && a.N > 0 && (uintptr_t)a.x % 16 == 0 &&
         (uintptr_t)a.w % 16 == 0 && (uintptr_t)a.w_up % 16 == 0 && (!a.w_up || nv_plan(a).cfg >= 0);
}

// Workspace: the scales repacked tile-major, unless they come so, then the split tiles' fp32
// partial sums.
size_t gemm_nvfp4_workspace(const QmmArgs &a) {
  const GpPlan p = nv_plan(a);
  const size_t sw = tiled_scales_bytes(a.N, a.K / 16);
  return (a.s_tiled ? 0 : sw) + (a.w_up && !a.s_up_tiled ? sw : 0) +
         (size_t)p.left * p.S * NV_COST[p.cfg].TM * NV_COST[p.cfg].TN * sizeof(float);
}

hipError_t launch_gemm_nvfp4(const QmmArgs &a, void *ws, hipStream_t st) {
  if (!gemm_nvfp4_ok(a)) return hipErrorInvalidValue;
  const uint8_t *sp = (const uint8_t *)a.s_tiled, *sp_up = (const uint8_t *)a.s_up_tiled;
  uint8_t *next = (uint8_t *)ws;
  const size_t sw = tiled_scales_bytes(a.N, a.K / 16);  // (a multiple of 1 KiB)
  hipError_t e = hipSuccess;
  if (!sp) {
    e = launch_repack_scales(a.s, a.N, a.K / 16, (uint32_t *)next, st);
    sp = next, next += sw;
  }
  if (e == hipSuccess && a.w_up && !sp_up) {
    e = launch_repack_scales(a.s_up, a.N, a.K / 16, (uint32_t *)next, st);
    sp_up = next, next += sw;
  }
  if (e != hipSuccess) return e;
  float *part = (float *)next;
  const GpPlan p = nv_plan(a);
  if (a.w_up) {
    switch (p.cfg) {
      case 0: return launch_nv<Nv256, true>(a, p, sp, sp_up, part, st);
      case 1: return launch_nv<Nv192, true>(a, p, sp, sp_up, part, st);
      case 2: return launch_nv<NvW, true>(a, p, sp, sp_up, part, st);
      case 3: return launch_nv<Nv128M, true>(a, p, sp, sp_up, part, st);
      default: return launch_nv<Nv64M, true>(a, p, sp, sp_up, part, st);
    }
  }
  switch (p.cfg) {
    case 0: return launch_nv<Nv256, false>(a, p, sp, sp_up, part, st);
    case 1: return launch_nv<Nv192, false>(a, p, sp, sp_up, part, st);
    case 2: return launch_nv<NvW, false>(a, p, sp, sp_up, part, st);
    case 3: return launch_nv<Nv128, false>(a, p, sp, sp_up, part, st);
    case 4: return launch_nv<Nv64, false>(a, p, sp, sp_up, part, st);
    default: return launch_nv<Nv32, false>(a, p, sp, sp_up, part, st);
  }
}

}  // namespace qmm
