// Dense bf16 linear y[M, N] = x[M, K] @ w[N, K].T (linear, src/model.zig:200-211): bf16
// operands, fp32 accumulation, bf16 out (RNE).  x of up to 8 rows runs a GEMV
// (gemv_bf16_kernel), taller x a pipelined GEMM on v_mfma_f32_32x32x16_bf16.
//
// The GEMM.  What bounds it: at tall x the matrix cores at the clock the power limit leaves
// (a large library product reaches ~1.45 PFLOP/s here, not 2.5), and before that the time a
// K step's operands take from L2 or HBM, ~1.2 us cold; at short x the weight stream.  So:
//   * K steps of 64: a row's piece of a step is 128 bytes, a whole cache line.  With steps
//     of 32 each line was fetched twice, by two steps (M = 1000, N = 10240, K = 5120 in
//     256 x 256 tiles: 126 us whatever the ring's depth, 99 us with 64).
//   * Operands go to LDS by DMA, x into a ring of SX stages and W into a deeper one of SW:
//     x is re-read by every W tile and comes from L2, W comes from HBM and needs the longer
//     lead.  256 x 256 tiles: rings of 2 + 2 stages (128 KiB) 120 us, 2 + 3 (160 KiB, all
//     of the LDS) 99 us.
//   * Each wave reads the next sub-step's fragments (of 16 K) beside the current sub-step's
//     MFMAs and meets the others at one barrier per K step; DMAs are issued one at a time
//     between MFMAs.
//   * The tile is chosen per call (dense_plan below): the sizes differ in operand bytes per
//     MFMA, in how they divide M x N, and in rounds of the chip.  Tiles left over after the
//     whole rounds are split along K over the idle CUs in the same launch, fp32 partial
//     sums reduced in K order (deterministic) by a second kernel.  Without scratch for
//     them (a call that is being captured: a replay may run beside other calls of the
//     stream) every tile is whole.
// Measured, us per call, inputs changing from call to call (M x N x K; the former
// kernel, 128 x 128 tiles through registers without a pipeline, in brackets):
//   1000 x 10240 x 5120  92 (172), 2048 x 34816 x 5120  570 = 1.28 PFLOP/s,
//   512 x 6144 x 5120  45, 64 x 10240 x 5120  27 (110; without scratch 40),
//   16 x 17408 x 5120  39 (131; 53).
#include <type_traits>

#include "gemm_pipe.h"
#include "qmm_device.h"
#include "qmm_launch.h"

namespace qmm {

// ---------------------------------------------------------------- x of a few rows

// A workgroup of W waves per 4 W rows, its lanes over 16-byte (8-element) chunks of them, U chunks
// in flight per lane; the waves' sums are added in wave order.  Bound by the weight stream, so by
// the bytes in flight: with one wave per 4 rows and one chunk each, a CU had 20 KiB of 5120 rows
// in flight, and short matrices left most CUs without a wave (us,
// before and now: 5120 x 17408 at 2 rows 30.6 -> 28.9, 1024 x 5120 at 1 row 7.1 -> 3.9, 703 x
// 6912 at 4 rows 11.4 -> 6.3).
template <int M, int W, int U>
__global__ __launch_bounds__(64 * W) void gemv_bf16_kernel(const uint16_t *__restrict__ x, const uint16_t *__restrict__ w,
                                                           uint16_t *__restrict__ y, int N, int K) {
  constexpr int R = 4;
  __shared__ float part[W][R * M];
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int n0 = blockIdx.x * R;
  const int C = K >> 3;
  float acc[R][M];
#pragma unroll
  for (int r = 0; r < R; ++r)
#pragma unroll
    for (int m = 0; m < M; ++m) acc[r][m] = 0.f;
  auto dot8 = [](float t, uint4 q, uint4 xv) __attribute__((always_inline)) {
    t = dot2_bf16(__builtin_bit_cast(bf16x2_t, q.x), xv.x, t);
    t = dot2_bf16(__builtin_bit_cast(bf16x2_t, q.y), xv.y, t);
    t = dot2_bf16(__builtin_bit_cast(bf16x2_t, q.z), xv.z, t);
    return dot2_bf16(__builtin_bit_cast(bf16x2_t, q.w), xv.w, t);
  };
  int c = tid;
  // chunks c + 64 W u of the rows, u < U
  if constexpr (U > 1)
    for (; c + 64 * W * (U - 1) < C; c += 64 * W * U) {
      uint4 q[U][R];
#pragma unroll
      for (int u = 0; u < U; ++u)
#pragma unroll
        for (int r = 0; r < R; ++r) {
          const int n = n0 + r < N ? n0 + r : N - 1;
          q[u][r] = load_stream16((const uint4 *)(w + (int64_t)n * K) + c + 64 * W * u);
        }
#pragma unroll
      for (int u = 0; u < U; ++u)
#pragma unroll
        for (int m = 0; m < M; ++m) {
          const uint4 xv = ((const uint4 *)(x + (int64_t)m * K))[c + 64 * W * u];
#pragma unroll
          for (int r = 0; r < R; ++r) acc[r][m] = dot8(acc[r][m], q[u][r], xv);
        }
    }
  for (; c < C; c += 64 * W) {
    uint4 q[R];
#pragma unroll
    for (int r = 0; r < R; ++r) {
      const int n = n0 + r < N ? n0 + r : N - 1;
      q[r] = load_stream16((const uint4 *)(w + (int64_t)n * K) + c);
    }
#pragma unroll
    for (int m = 0; m < M; ++m) {
      const uint4 xv = ((const uint4 *)(x + (int64_t)m * K))[c];
#pragma unroll
      for (int r = 0; r < R; ++r) acc[r][m] = dot8(acc[r][m], q[r], xv);
    }
  }
  float out = 0.f;
#pragma unroll
  for (int r = 0; r < R; ++r)
#pragma unroll
    for (int m = 0; m < M; ++m) {
      const float t = wave_sum(acc[r][m]);
      out = (lane == r * M + m) ? t : out;
    }
  if constexpr (W > 1) {
    if (lane < R * M) part[wave][lane] = out;
    __syncthreads();
    if (wave) return;
    out = 0.f;
    if (lane < R * M) {
#pragma unroll
      for (int v = 0; v < W; ++v) out += part[v][lane];
    }
  }
  if (lane < R * M) {
    const int r = lane / M, m = lane % M;
    if (n0 + r < N) y[(int64_t)m * N + n0 + r] = f32_to_bf16_rne(out);
  }
}

template <int M>
static void launch_gemv(const uint16_t *x, const uint16_t *w, uint16_t *y, int N, int K, hipStream_t st) {
  // Several waves per row group where the groups alone give a CU under 6 waves and every lane
  // still has a chunk; from there on one wave and one chunk each (at 12288 x 5120 four waves and
  // two chunks measured 22.4 -> 23.9 us at 4 rows, 300 x 1024 eight waves 4.0 -> 5.2).
  const int groups = (N + 3) / 4, cus = device_cu_count(), chunks = K >> 3;
  const dim3 grid(groups);
  if (groups < 2 * cus && chunks >= 512) hipLaunchKernelGGL((gemv_bf16_kernel<M, 8, 2>), grid, dim3(512), 0, st, x, w, y, N, K);
  else if (groups < 6 * cus && chunks >= (M <= 4 ? 256 : 512)) hipLaunchKernelGGL((gemv_bf16_kernel<M, 4, 2>), grid, dim3(256), 0, st, x, w, y, N, K);
  else if (groups < 4 * cus && chunks >= 128) hipLaunchKernelGGL((gemv_bf16_kernel<M, 2, 1>), grid, dim3(128), 0, st, x, w, y, N, K);
  else hipLaunchKernelGGL((gemv_bf16_kernel<M, 1, 1>), grid, dim3(64), 0, st, x, w, y, N, K);
}

// x of up to 8 rows, the sizes of decode calls, runs the GEMV, which needs no scratch: a program
// may capture those calls, forbid allocation around them and issue them from several threads.
// (At 6-8 rows the GEMM's split tiles are faster, GEMV / GEMM in us: 10240 x 5120 at 6 rows 29 / 25,
// 5120 x 17408 at 8 rows 47 / 38; but their partial sums are scratch of the stream.)
static bool linear_gemv(int M) { return M <= QMV_MAX_M; }

// ---------------------------------------------------------------- taller x

namespace {
constexpr int D_BK = GP_STEP;  // K elements of a step: 128 bytes of a row
// A block's tile: WM x WN waves of (32 FI) x (32 FJ); LDS rings of SX stages of x rows and
// SW >= SX stages of W rows.
template <int FI_, int FJ_, int WM_, int WN_, int SX_, int SW_>
struct DnGeom {
  static constexpr int FI = FI_, FJ = FJ_, WM = WM_, WN = WN_, SX = SX_, SW = SW_;
  static constexpr int TM = 32 * FI * WM, TN = 32 * FJ * WN, NW = WM * WN, THREADS = 64 * NW;
  static constexpr int XT = TM * 128, WT = TN * 128;         // a stage of x, of W
  static constexpr int LDS = SX * XT + SW * WT;
  static constexpr int NX = TM / 8 / NW, NWD = TN / 8 / NW;  // x and W DMAs per wave per step
  static_assert(TM / 8 % NW == 0 && TN / 8 % NW == 0 && SX >= 2 && SW > SX, "whole DMAs per wave");
  static constexpr int REGION = 32 * (64 * FJ + 32);
  static_assert(NW * REGION <= LDS, "the epilogue regions fit the rings");
};
}  // namespace

// Zeros that stand for the pieces of the last K step past K.
__device__ const uint4 dn_zero = {0, 0, 0, 0};

// 16-byte piece p of a row's 128 bytes is stored at slot p ^ dn_swz(row).
__device__ __forceinline__ int dn_swz(int r) { return (r & 7) ^ ((r >> 3) & 1); }

template <class G>
__global__ __launch_bounds__(G::THREADS, G::LDS <= 81920 ? 2 * G::NW / 4 : G::NW / 4) void gemm_dense_kernel(
    const uint16_t *__restrict__ x, const uint16_t *__restrict__ w, uint16_t *__restrict__ y, int M, int N, int K,
    int whole_tiles, int S, float *__restrict__ part) {
  constexpr int FI = G::FI, FJ = G::FJ, NX = G::NX, NWD = G::NWD, SX = G::SX, SW = G::SW;
  extern __shared__ __attribute__((aligned(16))) uint8_t lds[];
  const uint32_t lds0 = lds_addr(lds);
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int wm = wave % G::WM, wn = wave / G::WM;
  const int tiles_m = (M + G::TM - 1) / G::TM, tiles_n = (N + G::TN - 1) / G::TN;
  const int steps = (K + D_BK - 1) / D_BK;
  const GpBlock blk = gp_block(blockIdx.x, tiles_m, tiles_n, whole_tiles, S);
  const int m0 = blk.tm * G::TM, n0 = blk.tn * G::TN;
  const int s_begin = blk.split ? (int)((int64_t)blk.kr * steps / S) : 0;
  const int s_end = blk.split ? (int)((int64_t)(blk.kr + 1) * steps / S) : steps;

  // A DMA fills 1 KiB: rows 8 g + [0, 8) of a stage of x (or W), g = wave + NW i; lane l the
  // 16-byte slot l % 8 of row l / 8, which holds piece (l % 8) ^ swz(row) of the row's step.
  const uint8_t *xb = (const uint8_t *)x + (int64_t)m0 * K * 2, *wb = (const uint8_t *)w + (int64_t)n0 * K * 2;
  const int dr = 8 * wave + (lane >> 3), dp = (lane & 7) ^ dn_swz(dr);  // rows 8 NW apart share a swizzle
  static_assert(G::NW % 2 == 0, "");
  uint32_t xo[NX], wo[NWD];
#pragma unroll
  for (int i = 0; i < NX; ++i) xo[i] = (uint32_t)(min(m0 + dr + 8 * G::NW * i, M - 1) - m0) * (uint32_t)(2 * K) + dp * 16;
#pragma unroll
  for (int i = 0; i < NWD; ++i) wo[i] = (uint32_t)(min(n0 + dr + 8 * G::NW * i, N - 1) - n0) * (uint32_t)(2 * K) + dp * 16;
  auto issue_x = [&](int i, int s) __attribute__((always_inline)) {
    gp_dma16s(xb + (int64_t)s * 128, xo[i], lds0 + (uint32_t)((s % SX) * G::XT + (wave + G::NW * i) * 1024));
  };
  auto issue_w = [&](int i, int s) __attribute__((always_inline)) {
    gp_dma16s(wb + (int64_t)s * 128, wo[i], lds0 + (uint32_t)(SX * G::XT + (s % SW) * G::WT + (wave + G::NW * i) * 1024));
  };
  // all x (W) DMAs of step s, a whole one or the rows' last, whose pieces past K are zeros
  auto issue_any = [&](bool isx, int s) __attribute__((always_inline)) {
    const bool past = s * D_BK + 8 * dp >= K;
#pragma unroll
    for (int i = 0; i < (NX > NWD ? NX : NWD); ++i) {
      if (isx ? i >= NX : i >= NWD) continue;
      if ((s + 1) * D_BK <= K) {
        if (isx) issue_x(i, s);
        else issue_w(i, s);
      } else {
        const uint8_t *p = (isx ? xb + xo[i < NX ? i : 0] : wb + wo[i < NWD ? i : 0]) + (int64_t)s * 128;
        if (past) p = (const uint8_t *)&dn_zero;
        gp_dma16(p, lds0 + (uint32_t)((isx ? (s % SX) * G::XT : SX * G::XT + (s % SW) * G::WT) + (wave + G::NW * i) * 1024));
      }
    }
  };

  const int fr = lane & 31, fh = lane >> 5;
  const int ra = wm * 32 * FI + fr, rb = wn * 32 * FJ + fr;
  const int oa = ra * 128 + 16 * (fh ^ dn_swz(ra));
  const int ob = SX * G::XT + rb * 128 + 16 * (fh ^ dn_swz(rb));

  f32x16_t acc[FI][FJ];
#pragma unroll
  for (int i = 0; i < FI; ++i)
#pragma unroll
    for (int j = 0; j < FJ; ++j)
#pragma unroll
      for (int v = 0; v < 16; ++v) acc[i][j][v] = 0.f;

  // sub-step ks's fragments, in register set ks % 2
  bf16x8_t af[2][FI], bf[2][FJ];
  auto read = [&](int s, int ks, int q) __attribute__((always_inline)) {
    if (q < FJ) bf[ks & 1][q] = *(const bf16x8_t *)(lds + (s % SW) * G::WT + (ob ^ (32 * ks)) + 4096 * q);
    else af[ks & 1][q - FJ] = *(const bf16x8_t *)(lds + (s % SX) * G::XT + (oa ^ (32 * ks)) + 4096 * (q - FJ));
  };
  constexpr int NR = FI + FJ, NM = FI * FJ;

  // Order of the DMAs: W(0 .. SW - SX - 1), then x(t), W(t + SW - SX) for t = 0, 1, ..
#pragma unroll 1
  for (int t = SX - SW; t < SX; ++t) {
    if (t >= 0 && s_begin + t < s_end) issue_any(true, s_begin + t);
    if (t < SX - 1 && s_begin + t + SW - SX < s_end) issue_any(false, s_begin + t + SW - SX);
  }
  if (s_end - s_begin >= SW) gp_wait_barrier<(SX - 1) * (NX + NWD)>();
  else gp_wait_barrier<0>();
#pragma unroll
  for (int q = 0; q < NR; ++q) read(s_begin, 0, q);

  // Step s.  Sub-step ks's MFMAs run beside the reads of the next sub-step's fragments.
  // Before sub-step 3 every read of stage s is done and, after the barrier, every wave's:
  // its x stage is refilled with step s + SX beside sub-step 3, its W stage with step
  // s + SW beside the next step's first sub-steps.
  // MODE 2: those DMAs are whole; 1: any, if in the range; 0: as 1, and the next stage
  // needs every DMA.
  auto step = [&](auto mode_c, int s) __attribute__((always_inline)) {
    constexpr int MODE = decltype(mode_c)::value;
#pragma unroll
    for (int ks = 0; ks < 4; ++ks) {
      if (ks == 3) {
        if constexpr (MODE > 0) gp_wait_barrier<NWD + (SX - 2) * (NX + NWD)>();
        else gp_wait_barrier<0>();
        __builtin_amdgcn_sched_barrier(0);
      }
      if constexpr (MODE < 2) {
        if (ks == 0 && s + SW - 1 < s_end) issue_any(false, s + SW - 1);
        if (ks == 3 && s + SX < s_end) issue_any(true, s + SX);
      }
#pragma unroll
      for (int m = 0; m < NM; ++m) {
        if constexpr (MODE == 2) {
          if (ks == 3) {
#pragma unroll
            for (int i = m * NX / NM; i < (m + 1) * NX / NM; ++i) issue_x(i, s + SX);
          } else if (ks < 2) {
            constexpr int H = (NWD + 1) / 2;
#pragma unroll
            for (int i = m * H / NM; i < (m + 1) * H / NM; ++i)
              if (ks * H + i < NWD) issue_w(ks * H + i, s + SW - 1);
          }
        }
#pragma unroll
        for (int q = m * NR / NM; q < (m + 1) * NR / NM; ++q) read(ks == 3 ? s + 1 : s, (ks + 1) & 3, q);
        const int j = m / FI, i = m % FI;
        acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(af[ks & 1][i], bf[ks & 1][j], acc[i][j], 0, 0, 0);
        __builtin_amdgcn_sched_barrier(0);
      }
    }
  };
  int s = s_begin;
  constexpr int LEAD = SW - 1 > SX ? SW - 1 : SX;
  const int whole = K % D_BK == 0 ? s_end : (s_end < steps ? s_end : steps - 1);  // steps [s_begin, whole) are whole
#pragma unroll 1
  for (; s + LEAD < whole; ++s) step(std::integral_constant<int, 2>{}, s);
#pragma unroll 1
  for (; s + SW - 1 < s_end; ++s) step(std::integral_constant<int, 1>{}, s);
#pragma unroll 1
  for (; s < s_end; ++s) step(std::integral_constant<int, 0>{}, s);
  gp_lds_barrier();

  const int row0 = m0 + wm * 32 * FI, col0 = n0 + wn * 32 * FJ;
  if (blk.split) {
    gp_store_partial<FI, FJ, G::NW>(acc, part + (size_t)((blk.t - whole_tiles) * S + blk.kr) * G::TM * G::TN, wave, lane,
                                    M - row0);
    return;
  }
  const YOut yo = yout_one(y, N);
  gp_store_rows<FI, FJ, 0>(acc, lds + wave * G::REGION, lane, yo, M, row0, col0, N, yout_vec(yo));
}

template <class G>
__global__ __launch_bounds__(256) void gemm_dense_reduce_kernel(const float *__restrict__ part, uint16_t *__restrict__ y,
                                                               int M, int N, int whole_tiles, int S) {
  gp_reduce_tile<G>(part, yout_one(y, N), M, N, whole_tiles, S, blockIdx.x * 256 + threadIdx.x);
}

// ---------------------------------------------------------------- the plan

namespace {
using Dn256 = DnGeom<4, 2, 2, 4, 2, 3>;   // 256 x 256
using Dn160 = DnGeom<2, 5, 4, 1, 2, 4>;   // 256 x 160
using Dn192 = DnGeom<3, 4, 2, 2, 2, 3>;   // 192 x 256
using DnH = DnGeom<4, 2, 2, 2, 2, 4>;     // 256 x 128
using Dn128 = DnGeom<2, 2, 2, 2, 2, 3>;   // 128 x 128, two blocks per CU
using Dn64 = DnGeom<2, 1, 1, 4, 2, 4>;    // 64 x 128, two blocks per CU
using DnS = DnGeom<1, 1, 2, 2, 2, 4>;     // 64 x 64, three blocks per CU
}  // namespace

// (split: with scratch for the partial sums of tiles split along K)
static GpPlan dense_plan(int M, int N, int K, bool split) {
  return plan_dense(M, N, K, split, device_cu_count());
}

template <class G>
static hipError_t launch_dense_cfg(const uint16_t *x, const uint16_t *w, uint16_t *y, int M, int N, int K,
                                   const GpPlan &p, float *part, hipStream_t st) {
  static std::atomic<uint64_t> lds_set{0};
  hipError_t e = ensure_dynamic_lds(lds_set, (const void *)gemm_dense_kernel<G>, G::LDS);
  if (e != hipSuccess) return e;
  hipLaunchKernelGGL((gemm_dense_kernel<G>), dim3(p.whole + p.left * p.S), dim3(G::THREADS), G::LDS, st, x, w, y, M, N,
                     K, p.whole, p.S, part);
  e = hipGetLastError();
  if (e != hipSuccess || p.left == 0) return e;
  constexpr int RB = G::NW * G::FI * G::FJ * 4 * 64 / 256;
  hipLaunchKernelGGL((gemm_dense_reduce_kernel<G>), dim3(p.left * RB), dim3(256), 0, st, (const float *)part, y, M, N,
                     p.whole, p.S);
  return hipGetLastError();
}

static hipError_t launch_dense_plan(const uint16_t *x, const uint16_t *w, uint16_t *y, int M, int N, int K,
                                    const GpPlan &p, float *part, hipStream_t st) {
  switch (p.cfg) {
    case 0: return launch_dense_cfg<Dn256>(x, w, y, M, N, K, p, part, st);
    case 1: return launch_dense_cfg<Dn160>(x, w, y, M, N, K, p, part, st);
    case 2: return launch_dense_cfg<Dn192>(x, w, y, M, N, K, p, part, st);
    case 3: return launch_dense_cfg<DnH>(x, w, y, M, N, K, p, part, st);
    case 4: return launch_dense_cfg<Dn128>(x, w, y, M, N, K, p, part, st);
    case 5: return launch_dense_cfg<Dn64>(x, w, y, M, N, K, p, part, st);
    default: return launch_dense_cfg<DnS>(x, w, y, M, N, K, p, part, st);
  }
}

size_t linear_bf16_workspace(int M, int N, int K) {
  if (linear_gemv(M)) return 0;
  const GpPlan p = dense_plan(M, N, K, true);
  return (size_t)p.left * p.S * DN_COST[p.cfg].TM * DN_COST[p.cfg].TN * sizeof(float);
}

hipError_t launch_linear_bf16(const uint16_t *x, const uint16_t *w, uint16_t *y, int M, int N, int K, void *ws,
                              hipStream_t st) {
  if (K % 16 != 0 || M <= 0 || N <= 0) return hipErrorInvalidValue;
  if (!linear_gemv(M)) return launch_dense_plan(x, w, y, M, N, K, dense_plan(M, N, K, ws != nullptr), (float *)ws, st);
  switch (M) {
#define QMM_GEMV_CASE(MM) \
  case MM: launch_gemv<MM>(x, w, y, N, K, st); break;
    QMM_GEMV_CASE(1) QMM_GEMV_CASE(2) QMM_GEMV_CASE(3) QMM_GEMV_CASE(4)
    QMM_GEMV_CASE(5) QMM_GEMV_CASE(6) QMM_GEMV_CASE(7) QMM_GEMV_CASE(8)
#undef QMM_GEMV_CASE
  }
  return hipGetLastError();
}

}  // namespace qmm
