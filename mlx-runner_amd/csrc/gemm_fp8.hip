// mxfp8 prefill GEMM on the gfx950 scaled fp8 MFMA (v_mfma_scale_f32_32x32x64_f8f6f4).
//
// y[M, N] = x[M, K] @ deq(W)[N, K].T, W in mxfp8 (E4M3 bytes, one E8M0 scale per 32).
//
// The MFMA takes both operands in an 8-bit format with one E8M0 scale per row
// and 32-wide K block -- exactly the mxfp8 weight layout, consumed raw.  x is
// bf16 (8 significant bits); one E4M3 pass would keep 4 and miss the output
// tolerance, so a pre-pass splits x per 32-block into
//     x = hi * 2^(sh-127) + lo * 2^(sl-127)      (hi, lo E4M3; sh, sl E8M0)
// with the scale chosen as 2^ceil(log2(amax/448)) (no element is clamped).
// bf16's 8 bits fit in two 4-bit E4M3 significands, so the split is exact
// except for elements below ~2^-9 of their block's max.  The GEMM then issues
// two scaled MFMAs (hi, lo) per weight fragment into the same accumulator:
// the weight tile is loaded once, the MFMA work doubles.
//
// What bounds it: at tall x the matrix cores at the clock the power limit leaves (a large
// fp8 library product reaches ~3.07 PFLOP/s here; 2048 x 34816 x 5120 runs at 2.8-2.9, hi and
// lo both counted), at short x the latency of a step.  So:
//   * K steps of 64: a row's hi and lo bytes of a step lie together, 128 bytes, a cache line;
//     W moves in stages of two steps, 128 bytes per row too (64 wasted half of each line).
//   * x and W go to LDS rings by DMA; the lo fragments are read beside the products of the
//     hi parts, the next step's beside those of the lo parts; one barrier per step.
//   * The tile is chosen per call (mx_plan), and the tiles left over after the whole rounds are
//     split along K over the idle CUs, fp32 partial sums reduced in K order (deterministic) by
//     a second kernel.
// Measured, us per call with the split, weights cold (M x N x K; the former kernel, two groups
// of waves in turns, two barriers per step, in brackets): 2048 x 5120 x 17408  272-287 (320),
// 2048 x 17408 x 5120  269 (282), 200 x 5120 x 17408  54 (61), 48 x 17408 x 5120  28-35 (37-46),
// 385 x 4129 x 1280  20 (32); K % 128 = 64, which ran an unpipelined kernel: 68 x 27408 x 3392
// 41 (199).
// gate, up and silu(gate) * up of an MLP in one launch (MLP below), 2048 x (2 x 17408) x 5120 with
// the split of x: 572 us, against 614 for the three calls, whose result it gives bit for bit
// (gp_plan_pair; on another box 620, and 600 with the last tiles split as suits one launch best).
#include <type_traits>

#include "gemm_pipe.h"
#include "qmm_device.h"
#include "qmm_launch.h"

namespace qmm {

// ---------------------------------------------------------------- x split pre-pass

constexpr int X_BK = GP_STEP;  // K elements of a step: 64 bytes of hi and 64 of lo of an x row

// The split of 16 consecutive elements (lane pair l, l ^ 1 shares a 32-block): E4M3
// hi / lo words and the block's exponents th, tl.
__device__ __forceinline__ void split16(const uint4 q0, const uint4 q1, uint32_t (&hw)[4], uint32_t (&lw)[4], int &th,
                                        int &tl) {
  const uint32_t w8[8] = {q0.x, q0.y, q0.z, q0.w, q1.x, q1.y, q1.z, q1.w};
  float v[16];
  float amax = 0.f;
#pragma unroll
  for (int t = 0; t < 8; ++t) {
    v[2 * t] = __uint_as_float(w8[t] << 16);
    v[2 * t + 1] = __uint_as_float(w8[t] & 0xFFFF0000u);
  }
#pragma unroll
  for (int t = 0; t < 16; ++t) amax = fmaxf(amax, fabsf(v[t]));
  amax = fmaxf(amax, __shfl_xor(amax, 1));
  th = amax > 0.f ? ceil_scale_exp(amax) : -127;
  // hi straight from the bf16 pairs (the conversion divides by 2^th and rounds to nearest
  // even), then back to f32 times 2^th for the residual, which is exact in f32
  const float sh = e8m0_scale_operand(th);
  float rmax = 0.f;
#pragma unroll
  for (int t = 0; t < 4; ++t) {
    i16x2_t c = {0, 0};
    c = __builtin_amdgcn_cvt_scalef32_pk_fp8_bf16(c, __builtin_bit_cast(bf16x2_t, w8[2 * t]), sh, false);
    c = __builtin_amdgcn_cvt_scalef32_pk_fp8_bf16(c, __builtin_bit_cast(bf16x2_t, w8[2 * t + 1]), sh, true);
    hw[t] = __builtin_bit_cast(uint32_t, c);
    const f32x2_t b0 = __builtin_amdgcn_cvt_scalef32_pk_f32_fp8(hw[t], sh, false);
    const f32x2_t b1 = __builtin_amdgcn_cvt_scalef32_pk_f32_fp8(hw[t], sh, true);
    v[4 * t] -= b0.x;
    v[4 * t + 1] -= b0.y;
    v[4 * t + 2] -= b1.x;
    v[4 * t + 3] -= b1.y;
#pragma unroll
    for (int u = 0; u < 4; ++u) rmax = fmaxf(rmax, fabsf(v[4 * t + u]));
  }
  rmax = fmaxf(rmax, __shfl_xor(rmax, 1));
  tl = rmax > 0.f ? ceil_scale_exp(rmax) : -127;
  const float sl = e8m0_scale_operand(tl);
#pragma unroll
  for (int t = 0; t < 4; ++t) {
    i16x2_t c = {0, 0};
    c = __builtin_amdgcn_cvt_scalef32_pk_fp8_f32(c, v[4 * t], v[4 * t + 1], sl, false);
    c = __builtin_amdgcn_cvt_scalef32_pk_fp8_f32(c, v[4 * t + 2], v[4 * t + 3], sl, true);
    lw[t] = __builtin_bit_cast(uint32_t, c);
  }
}

// x [rows, K] -> xs: per row and step 128 bytes, the step's 64 hi then its 64 lo bytes (zeros
// past K), rows of steps x 128 bytes; and the block scales, a dword per row and step (hi and
// lo of the step's first 32-block, then of its second), tile-major: for each 256 rows and pair
// of steps, 2 x 256 consecutive dwords.  A wave takes 16 rows x U steps; in each step lane l
// takes row l / 4, 16 elements l % 4 of the step.  All reads are issued before the first is
// split.  Rows past `rows` (up to the 16-row group) read the last row and store nothing.
template <int U>
__global__ __launch_bounds__(256) void split_x_kernel(const uint16_t *__restrict__ x, int rows, int K, int steps,
                                                      uint8_t *__restrict__ xs, uint32_t *__restrict__ sx) {
  const int lane = threadIdx.x & 63;
  const int su = (steps + U - 1) / U, w = blockIdx.x * 4 + (threadIdx.x >> 6);
  const int rg = w / su, st0 = U * (w - rg * su);
  if (16 * rg >= rows) return;  // (the grid is whole blocks; a wave leaves as one)
  const int r = 16 * rg + (lane >> 2), c = lane & 3;
  const uint16_t *src = x + (int64_t)min(r, rows - 1) * K + 16 * c;
  uint4 q[U][2];
#pragma unroll
  for (int u = 0; u < U; ++u) {
    q[u][0] = q[u][1] = make_uint4(0, 0, 0, 0);
    if (X_BK * (st0 + u) + 16 * c < K) {
      q[u][0] = *(const uint4 *)(src + X_BK * (st0 + u));
      q[u][1] = *(const uint4 *)(src + X_BK * (st0 + u) + 8);
    }
  }
  const int pairs = (steps + 1) / 2;
#pragma unroll
  for (int u = 0; u < U; ++u) {
    const int st = st0 + u;
    if (st >= steps) break;
    uint32_t hw[4], lw[4];
    int th, tl;
    split16(q[u][0], q[u][1], hw, lw, th, tl);
    uint32_t sc = (uint32_t)(th + 127) | (uint32_t)(tl + 127) << 8;
    sc |= (uint32_t)__shfl_xor((int)sc, 2) << 16;  // lanes 0 of 4: the step's two blocks
    if (r < rows) {
      uint8_t *o = xs + ((int64_t)r * steps + st) * 128 + 16 * c;
      *(uint4 *)o = make_uint4(hw[0], hw[1], hw[2], hw[3]);
      *(uint4 *)(o + 64) = make_uint4(lw[0], lw[1], lw[2], lw[3]);
      if (c == 0) sx[(((int64_t)(r >> 8) * pairs + (st >> 1)) * 2 + (st & 1)) * 256 + (r & 255)] = sc;
    }
  }
}

// ---------------------------------------------------------------- GEMM

namespace {
// A block's tile: WM x WN waves of (32 FI) x (32 FJ); LDS rings of SX stages of x (a step
// each) and SW stages of W and of the scales (two steps each: 128 bytes of a W row, the dword
// of its four block scales and an x row's two).
template <int FI_, int FJ_, int WM_, int WN_, int SX_, int SW_>
struct MxGeom {
  static constexpr int FI = FI_, FJ = FJ_, WM = WM_, WN = WN_, SX = SX_, SW = SW_;
  static constexpr int TM = 32 * FI * WM, TN = 32 * FJ * WN, NW = WM * WN, THREADS = 64 * NW;
  static constexpr int XT = TM * 128, WT = TN * 128;
  static constexpr int SD = (TN + 2 * TM + 255) / 256;  // scale DMAs of a stage
  static constexpr int WOFF = SX * XT, SOFF = WOFF + SW * WT, ST = SD * 1024;
  static constexpr int LDS = SOFF + SW * ST;
  static constexpr int NX = TM / 8 / NW;       // x DMAs per wave per step
  static constexpr int NWD = TN / 8 / NW + 1;  // W DMAs and one of the scales' per wave per stage
  static_assert(TM / 8 % NW == 0 && TN / 8 % NW == 0 && TN % 4 == 0 && NW % 2 == 0 && SD <= NW, "");
  // (step 2 g + 1 of the kernel's MODE 3, g + SW the range's end, brings x of step 2 g + 1 + SX, which
  // has to be one of the range's 2 (g + SW))
  static_assert(SX >= 2 && SW >= 2 && SX <= 2 * SW - 2, "");
  static constexpr int REGION = 32 * (64 * FJ + 32);
  static_assert(NW * REGION <= LDS, "the epilogue regions fit the rings");
  // DMAs that may be in flight at the barrier of an even (odd) step s: x of step i + SX is
  // issued in step i, and W stage (i - 1) / 2 + SW after it when i is odd; x of step s + 1
  // has to be there and, at an odd step, the next W stage.
  static constexpr int issued(int from, int to) {  // in steps from .. to - 1
    int n = 0;
    for (int i = from; i < to; ++i) n += NX + (i & 1 ? NWD : 0);
    return n;
  }
  static constexpr int in_flight(int s) {
    const int i0 = s + 1 - SX, nx = (i0 & 1 ? NWD : 0) + issued(i0 + 1, s);
    const int nw = issued(s + 2 - 2 * SW + 1, s);
    return (s & 1) && nw < nx ? nw : nx;
  }
};
}  // namespace

// Zeros that stand for the pieces of the last stage past K.
__device__ const uint4 mx_zero = {0, 0, 0, 0};

// 16-byte piece p of a row's 128 bytes is stored at slot p ^ mx_swz(row).
__device__ __forceinline__ int mx_swz(int r) { return (r & 7) ^ ((r >> 3) & 1); }

// MLP: the tile's W rows are two matrices', 32-row blocks of gate and of up in turn (row
// block 2 b and 2 b + 1 of a tile are rows 32 b + [0, 32) of the tile's TN / 2), and the
// result is silu(gate) * up, TN / 2 columns of it per tile.
template <class G, bool MLP>
__global__ __launch_bounds__(G::THREADS, G::LDS <= 81920 ? 2 * G::NW / 4 : G::NW / 4) void gemm_mxfp8_kernel(
    const uint8_t *__restrict__ xs, const uint32_t *__restrict__ sx, const uint8_t *__restrict__ w,
    const uint8_t *__restrict__ sp, const uint8_t *__restrict__ w_up, const uint8_t *__restrict__ sp_up, const YOut yo,
    int M, int N, int K, int whole_tiles, int S, float *__restrict__ part) {
  constexpr int FI = G::FI, FJ = G::FJ, NX = G::NX, NWD = G::NWD, SX = G::SX, SW = G::SW;
  constexpr int TC = MLP ? G::TN / 2 : G::TN;  // columns of y per tile
  static_assert(!MLP || FJ % 2 == 0, "a wave holds gate and up of a column");
  extern __shared__ __attribute__((aligned(16))) uint8_t lds[];
  const uint32_t lds0 = lds_addr(lds);
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int wm = wave % G::WM, wn = wave / G::WM;
  const int tiles_m = (M + G::TM - 1) / G::TM, tiles_n = (N + G::TN - 1) / G::TN;
  const int steps = (K + X_BK - 1) / X_BK, stages = (steps + 1) / 2;
  const GpBlock blk = gp_block<MLP>(blockIdx.x, tiles_m, tiles_n, whole_tiles, S);
  const int m0 = blk.tm * G::TM, n0 = blk.tn * TC;
  if (MLP && n0 >= N) return;  // the second half of the last pair (its partial sums are not read either)
  const int g_begin = blk.split ? (int)((int64_t)blk.kr * stages / S) : 0;
  const int g_end = blk.split ? (int)((int64_t)(blk.kr + 1) * stages / S) : stages;
  const int s_begin = g_begin * 2, s_end = min(g_end * 2, steps);

  // A DMA fills 1 KiB: rows 8 q + [0, 8) of a stage of x (or W), q = wave + NW i; lane l the
  // 16-byte slot l % 8 of row l / 8, which holds piece (l % 8) ^ swz(row) of the row's 128 bytes.
  const int64_t xrow = (int64_t)steps * 128;
  const uint8_t *xb = xs + (int64_t)m0 * xrow;
  const int dr = 8 * wave + (lane >> 3), dp = (lane & 7) ^ mx_swz(dr);  // rows 8 NW apart share a swizzle
  uint32_t xo[NX], wo[NWD - 1];
  const uint8_t *wb[MLP ? NWD - 1 : 1];
#pragma unroll
  for (int i = 0; i < NX; ++i) xo[i] = (uint32_t)((min(m0 + dr + 8 * G::NW * i, M - 1) - m0) * xrow) + dp * 16;
  if constexpr (!MLP) wb[0] = w + (int64_t)n0 * K;
#pragma unroll
  for (int i = 0; i < NWD - 1; ++i) {
    const int q = wave + G::NW * i, r = dr + 8 * G::NW * i;  // 8 rows of one 32-row block
    int row = r;
    if constexpr (MLP) {
      wb[i] = ((q >> 2) & 1 ? w_up : w) + (int64_t)n0 * K;
      row = (r >> 6) * 32 + (r & 31);
    }
    wo[i] = (uint32_t)(min(n0 + row, N - 1) - n0) * (uint32_t)K + dp * 16;
  }
  // scales: dword d of a stage's ring slot is W row d's (d < TN), then x row r's of step t at
  // TN + t TM + r; a DMA moves four dwords per lane, 256 in all, wave v the v % SD-th (lanes past
  // the last dword repeat it)
  const int n256 = (N + 255) & ~255, m256 = (M + 255) & ~255;
  const int sq = min((wave % G::SD) * 256 + 4 * lane, G::TN + 2 * G::TM - 4);
  const uint8_t *sb;
  uint32_t sstep;  // bytes from a stage's to the next's
  if (sq < G::TN) {
    const int mat = MLP ? (sq >> 5) & 1 : 0, row = min(n0 + (MLP ? (sq >> 6) * 32 + (sq & 31) : sq), n256 - 4);
    sb = (mat ? sp_up : sp) + ((int64_t)(row >> 8) * stages * 256 + (row & 255)) * 4;
    sstep = 1024;
  } else {
    const int t = (sq - G::TN) / G::TM, row = min(m0 + (sq - G::TN) % G::TM, m256 - 4);
    sb = (const uint8_t *)sx + (((int64_t)(row >> 8) * stages * 2 + t) * 256 + (row & 255)) * 4;
    sstep = 2048;
  }

  auto issue_x = [&](int i, int s) __attribute__((always_inline)) {
    gp_dma16s(xb + (int64_t)s * 128, xo[i], lds0 + (uint32_t)((s % SX) * G::XT + (wave + G::NW * i) * 1024));
  };
  auto w_slot = [&](int i, int g) __attribute__((always_inline)) {
    return lds0 + (uint32_t)(G::WOFF + (g % SW) * G::WT + (wave + G::NW * i) * 1024);
  };
  auto issue_w = [&](int i, int g) __attribute__((always_inline)) {  // the last one: the scales
    if (i < NWD - 1) gp_dma16s(wb[MLP ? i : 0] + (int64_t)g * 128, wo[i], w_slot(i, g));
    else gp_dma16(sb + (int64_t)g * sstep, lds0 + (uint32_t)(G::SOFF + (g % SW) * G::ST + (wave % G::SD) * 1024));
  };
  // stage g's W, whole or the rows' last, whose pieces past K are zeros
  auto issue_w_any = [&](int g) __attribute__((always_inline)) {
#pragma unroll
    for (int i = 0; i < NWD; ++i) {
      if ((g + 1) * 2 * X_BK <= K || i == NWD - 1) {
        issue_w(i, g);
      } else {
        const uint8_t *p = wb[MLP ? i : 0] + wo[i] + (int64_t)g * 128;
        if (g * 2 * X_BK + 16 * dp >= K) p = (const uint8_t *)&mx_zero;
        gp_dma16(p, w_slot(i, g));
      }
    }
  };

  // Fragments (32x32x64 operands: lane l holds row l % 32, K bytes 16 fh + [0, 16) and 32 + 16 fh
  // + [0, 16), fh = l / 32, and the scale of block fh): x hi pieces fh and fh + 2 of the row's 128
  // bytes, lo fh + 4 and fh + 6; W, step t of its stage, 4 t + fh and 4 t + fh + 2.
  const int fr = lane & 31, fh = lane >> 5;
  const int ra = wm * 32 * FI + fr, rb = wn * 32 * FJ + fr;
  const int oa = ra * 128 + 16 * (fh ^ mx_swz(ra));
  const int ob = G::WOFF + rb * 128 + 16 * (fh ^ mx_swz(rb));
  const int osw = G::SOFF + rb * 4 + fh, osx = G::SOFF + (G::TN + ra) * 4 + 2 * fh;

  f32x16_t acc[FI][FJ];
#pragma unroll
  for (int i = 0; i < FI; ++i)
#pragma unroll
    for (int j = 0; j < FJ; ++j)
#pragma unroll
      for (int v = 0; v < 16; ++v) acc[i][j][v] = 0.f;

  i32x8_t ah[FI], al[FI], bf[2][FJ];  // W in set s % 2
  // block scales (x: hi in byte 0, lo in byte 1), also in set s % 2: the MFMA reads its scale
  // registers after issue, so none is written by the instructions that follow it
  int sa[2][FI], sbw[2][FJ];
  auto frag = [&](const uint8_t *p, int o) __attribute__((always_inline)) {
    const uint4 u0 = *(const uint4 *)(p + o), u1 = *(const uint4 *)(p + (o ^ 32));
    return i32x8_t{(int)u0.x, (int)u0.y, (int)u0.z, (int)u0.w, (int)u1.x, (int)u1.y, (int)u1.z, (int)u1.w};
  };
  auto read_hi = [&](auto t_c, int s, int i) __attribute__((always_inline)) {
    constexpr int T = decltype(t_c)::value;  // s % 2
    ah[i] = frag(lds + (s % SX) * G::XT + 4096 * i, oa);
    sa[T][i] = *(const uint16_t *)(lds + ((s >> 1) % SW) * G::ST + osx + T * (4 * G::TM) + 128 * i);
  };
  auto read_lo = [&](int s, int i) __attribute__((always_inline)) {
    al[i] = frag(lds + (s % SX) * G::XT + 4096 * i, oa ^ 64);
  };
  auto read_w = [&](auto t_c, int s, int j) __attribute__((always_inline)) {
    constexpr int T = decltype(t_c)::value;
    bf[T][j] = frag(lds + ((s >> 1) % SW) * G::WT + 4096 * j, ob ^ (64 * T));
    sbw[T][j] = *(lds + ((s >> 1) % SW) * G::ST + osw + 2 * T + 128 * j);
  };
  constexpr int NM = FI * FJ;
  using I0 = std::integral_constant<int, 0>;
  using I1 = std::integral_constant<int, 1>;
  using I2 = std::integral_constant<int, 2>;
  using I3 = std::integral_constant<int, 3>;

  // The DMAs' order: step i brings x of step i + SX and, when odd, then W stage (i - 1) / 2 + SW
  // (relative to the range's first step); here the steps before the first.
#pragma unroll 1
  for (int i = 1 - 2 * SW; i < 0; ++i) {
    if (i + SX >= 0 && s_begin + i + SX < s_end) {
#pragma unroll
      for (int q = 0; q < NX; ++q) issue_x(q, s_begin + i + SX);
    }
    if ((i & 1) && g_begin + (i - 1) / 2 + SW < g_end) issue_w_any(g_begin + (i - 1) / 2 + SW);
  }
  if (g_end - g_begin >= SW && s_end - s_begin >= SX) gp_wait_barrier<G::in_flight(1)>();
  else gp_wait_barrier<0>();
#pragma unroll
  for (int j = 0; j < FJ; ++j) read_w(I0{}, s_begin, j);
#pragma unroll
  for (int i = 0; i < FI; ++i) read_hi(I0{}, s_begin, i);

  // Step s = 2 g + T: the products of the hi parts beside the reads of the lo parts; then every
  // read of the step's stages is done and, after the barrier, every wave's: the products of the
  // lo parts beside the next step's reads and the DMAs that refill the x stage and, after its
  // second step, the W stage.
  // MODE 2: those are whole and in the range; 3: no W stage g + SW; 1: whatever is in the range,
  // each barrier waiting for every DMA.
  auto step = [&](auto mode_c, auto t_c, int g) __attribute__((always_inline)) {
    constexpr int MODE = decltype(mode_c)::value, T = decltype(t_c)::value;
    const int s = 2 * g + T;
#pragma unroll
    for (int m = 0; m < NM; ++m) {
#pragma unroll
      for (int i = m * FI / NM; i < (m + 1) * FI / NM; ++i) read_lo(s, i);
      const int j = m / FI, i = m % FI;
      acc[i][j] = __builtin_amdgcn_mfma_scale_f32_32x32x64_f8f6f4(ah[i], bf[T][j], acc[i][j], 0, 0, 0, sa[T][i], 0,
                                                                  sbw[T][j]);
      __builtin_amdgcn_sched_barrier(0);
    }
    if constexpr (MODE >= 2) gp_wait_barrier<G::in_flight(T)>();
    else gp_wait_barrier<0>();
    __builtin_amdgcn_sched_barrier(0);
    if constexpr (MODE == 1) {
      if (s + SX < s_end) {
#pragma unroll
        for (int q = 0; q < NX; ++q) issue_x(q, s + SX);
      }
      if (T == 1 && g + SW < g_end) issue_w_any(g + SW);
    }
    constexpr int NI = MODE == 1 ? 0 : NX + (T == 1 && MODE == 2 ? NWD : 0), NR = FJ + FI;
#pragma unroll
    for (int m = 0; m < NM; ++m) {
#pragma unroll
      for (int i = m * NI / NM; i < (m + 1) * NI / NM; ++i) {
        if (i < NX) issue_x(i, s + SX);
        else issue_w(i - NX, g + SW);
      }
#pragma unroll
      for (int q = m * NR / NM; q < (m + 1) * NR / NM; ++q) {
        if (q < FJ) read_w(std::integral_constant<int, 1 - T>{}, s + 1, q);
        else read_hi(std::integral_constant<int, 1 - T>{}, s + 1, q - FJ);
      }
      const int j = m / FI, i = m % FI;
      acc[i][j] = __builtin_amdgcn_mfma_scale_f32_32x32x64_f8f6f4(al[i], bf[T][j], acc[i][j], 0, 0, 1, sa[T][i], 0,
                                                                  sbw[T][j]);
      __builtin_amdgcn_sched_barrier(0);
    }
  };
  int g = g_begin;
  const int whole = min(g_end, K / (2 * X_BK));  // the stages that are whole
#pragma unroll 1
  for (; g + SW < whole; ++g) {
    step(I2{}, I0{}, g);
    step(I2{}, I1{}, g);
  }
  if (g + SW == whole && whole == g_end) {
    step(I3{}, I0{}, g);
    step(I3{}, I1{}, g);
    ++g;
  }
#pragma unroll 1
  for (; g < g_end; ++g) {
    step(I1{}, I0{}, g);
    if (2 * g + 1 < s_end) step(I1{}, I1{}, g);
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
__global__ __launch_bounds__(256) void gemm_mxfp8_reduce_kernel(const float *__restrict__ part, const YOut yo, int M,
                                                                int N, int whole_tiles, int S) {
  gp_reduce_tile<G, MLP>(part, yo, M, N, whole_tiles, S, blockIdx.x * 256 + threadIdx.x);
}

// ---------------------------------------------------------------- the plan

namespace {
using Mx256 = MxGeom<4, 4, 2, 2, 2, 2>;  // 256 x 256
using Mx192 = MxGeom<3, 4, 2, 2, 2, 2>;  // 192 x 256
using MxW = MxGeom<2, 4, 2, 2, 3, 3>;    // 128 x 256
using Mx128 = MxGeom<2, 2, 2, 2, 2, 2>;  // 128 x 128, two blocks per CU
using Mx64 = MxGeom<1, 2, 2, 2, 3, 3>;   // 64 x 128, two blocks per CU
using Mx160 = MxGeom<2, 5, 4, 1, 2, 2>;  // 256 x 160
using Mx32 = MxGeom<1, 1, 1, 4, 3, 3>;   // 32 x 128, two blocks per CU
}  // namespace

static GpPlan mx_plan(const QmmArgs &a) { return plan_mxfp8(a.M, a.N, a.K, a.w_up != nullptr, device_cu_count()); }

// The workspace: the split x, its scales, the repacked W scales that do not come tile-major,
// and the split tiles' fp32 partial sums; each part a multiple of 256 bytes.
struct MxWs {
  size_t xs, sx, sw, part;
};
static MxWs mx_ws(const QmmArgs &a, const GpPlan &p) {
  const size_t steps = (a.K + X_BK - 1) / X_BK, rows = ((size_t)a.M + 255) & ~(size_t)255;
  MxWs ws;
  ws.xs = ((size_t)a.M * steps * 128 + 255) & ~(size_t)255;
  ws.sx = rows * ((steps + 1) / 2 * 2) * 4;
  ws.sw = tiled_scales_bytes(a.N, a.K / 32);
  ws.part = (size_t)p.left * p.S * MX_COST[p.cfg].TM * MX_COST[p.cfg].TN * sizeof(float);
  return ws;
}

template <class G, bool MLP>
static hipError_t launch_mx_tiles(const QmmArgs &a, const GpPlan &p, const uint8_t *xs, const uint32_t *sx,
                                  const uint8_t *sp, const uint8_t *sp_up, float *part, hipStream_t st) {
  static std::atomic<uint64_t> lds_set{0};
  hipError_t e = ensure_dynamic_lds(lds_set, (const void *)gemm_mxfp8_kernel<G, MLP>, G::LDS);
  if (e != hipSuccess) return e;
  const YOut yo = yout_of(a);  // y, or a grouped call's parts
  hipLaunchKernelGGL((gemm_mxfp8_kernel<G, MLP>), dim3(p.whole + p.left * p.S), dim3(G::THREADS), G::LDS, st, xs, sx, a.w,
                     sp, a.w_up, sp_up, yo, a.M, a.N, a.K, p.whole, p.S, part);
  e = hipGetLastError();
  if (e != hipSuccess || p.left == 0) return e;
  constexpr int RB = G::NW * G::FI * (MLP ? G::FJ / 2 : G::FJ);
  hipLaunchKernelGGL((gemm_mxfp8_reduce_kernel<G, MLP>), dim3(p.left * RB), dim3(256), 0, st, (const float *)part, yo, a.M,
                     a.N, p.whole, p.S);
  return hipGetLastError();
}

hipError_t launch_repack_scales(const uint8_t *s, int64_t N, int nb, uint32_t *out, hipStream_t st) {
  const int dpr = (nb + 3) / 4;
  const bool dwords = nb % 4 == 0 && (uintptr_t)s % 4 == 0, wide = dwords && dpr % 4 == 0 && (uintptr_t)s % 16 == 0;
  const int64_t threads = ((N + 255) & ~(int64_t)255) * dpr / (wide ? 4 : 1);
  const int64_t blocks = (threads + 255) / 256 < 65536 ? (threads + 255) / 256 : 65536;
  if (wide)
    hipLaunchKernelGGL(repack_scales_kernel<4>, dim3(blocks), dim3(256), 0, st, s, N, nb, out);
  else if (dwords)
    hipLaunchKernelGGL(repack_scales_kernel<1>, dim3(blocks), dim3(256), 0, st, s, N, nb, out);
  else
    hipLaunchKernelGGL(repack_scales_kernel<0>, dim3(blocks), dim3(256), 0, st, s, N, nb, out);
  return hipGetLastError();
}

size_t tiled_scales_bytes(int64_t N, int nb) { return (((size_t)N + 255) & ~(size_t)255) * (size_t)((nb + 3) / 4 * 4); }

int gemm_tiled_scale_bytes_per_row(const QmmArgs &a) {
  if (qmm_on_decode(a)) return 0;
  return gemm_mxfp8_ok(a) ? a.K / 32 : gemm_nvfp4_ok(a) ? a.K / 16 : 0;
}

// K % 64: the row lengths whose results the split of x has always served; an odd number of 32-blocks
// runs gemm.hip's kernel, whose products are exact (a padded half step here would be ten times
// faster, but of its outputs 1.2% round the other way than the exact sums, of that kernel's 0.01%).
// x and W rows 16-byte aligned.
bool gemm_mxfp8_ok(const QmmArgs &a) {
  return a.mode == MXFP8 && !a.x_f32 && a.K % X_BK == 0 && a.K > 0 && a.M > 0 && a.N > 0 && (uintptr_t)a.x % 16 == 0 &&
         (uintptr_t)a.w % 16 == 0 && (uintptr_t)a.w_up % 16 == 0 && (!a.w_up || mx_plan(a).cfg >= 0);
}

size_t gemm_mxfp8_workspace(const QmmArgs &a) {
  const MxWs ws = mx_ws(a, mx_plan(a));
  return ws.xs + ws.sx + (a.s_tiled ? 0 : ws.sw) + (a.w_up && !a.s_up_tiled ? ws.sw : 0) + ws.part;
}

hipError_t launch_gemm_mxfp8(const QmmArgs &a, void *workspace, hipStream_t st) {
  if (!gemm_mxfp8_ok(a)) return hipErrorInvalidValue;
  const int steps = (a.K + X_BK - 1) / X_BK;
  const GpPlan p = mx_plan(a);
  const MxWs ws = mx_ws(a, p);
  uint8_t *xs = (uint8_t *)workspace, *next = xs + ws.xs + ws.sx;
  uint32_t *sx = (uint32_t *)(xs + ws.xs);
  // U steps per wave: enough waves to fill the chip first, then 4 for the loads in flight
  const int64_t rg = ((int64_t)a.M + 15) / 16;
  const int U = rg * steps >= 4 * 4096 ? 4 : 1;
  const int64_t waves = rg * ((steps + U - 1) / U);
  if (waves >= ((int64_t)1 << 31)) return hipErrorInvalidValue;
  if (U == 4)
    hipLaunchKernelGGL(split_x_kernel<4>, dim3((waves + 3) / 4), dim3(256), 0, st, (const uint16_t *)a.x, a.M, a.K, steps, xs, sx);
  else
    hipLaunchKernelGGL(split_x_kernel<1>, dim3((waves + 3) / 4), dim3(256), 0, st, (const uint16_t *)a.x, a.M, a.K, steps, xs, sx);
  hipError_t e = hipGetLastError();
  const uint8_t *sp = (const uint8_t *)a.s_tiled, *sp_up = (const uint8_t *)a.s_up_tiled;
  if (e == hipSuccess && !sp) {
    e = launch_repack_scales(a.s, a.N, a.K / 32, (uint32_t *)next, st);
    sp = next, next += ws.sw;
  }
  if (e == hipSuccess && a.w_up && !sp_up) {
    e = launch_repack_scales(a.s_up, a.N, a.K / 32, (uint32_t *)next, st);
    sp_up = next, next += ws.sw;
  }
  if (e != hipSuccess) return e;
  float *part = (float *)next;
  if (a.w_up) {
    switch (p.cfg) {
      case 0: return launch_mx_tiles<Mx256, true>(a, p, xs, sx, sp, sp_up, part, st);
      case 1: return launch_mx_tiles<Mx192, true>(a, p, xs, sx, sp, sp_up, part, st);
      case 2: return launch_mx_tiles<MxW, true>(a, p, xs, sx, sp, sp_up, part, st);
      case 3: return launch_mx_tiles<Mx128, true>(a, p, xs, sx, sp, sp_up, part, st);
      default: return launch_mx_tiles<Mx64, true>(a, p, xs, sx, sp, sp_up, part, st);
    }
  }
  switch (p.cfg) {
    case 0: return launch_mx_tiles<Mx256, false>(a, p, xs, sx, sp, sp_up, part, st);
    case 1: return launch_mx_tiles<Mx192, false>(a, p, xs, sx, sp, sp_up, part, st);
    case 2: return launch_mx_tiles<MxW, false>(a, p, xs, sx, sp, sp_up, part, st);
    case 3: return launch_mx_tiles<Mx128, false>(a, p, xs, sx, sp, sp_up, part, st);
    case 4: return launch_mx_tiles<Mx64, false>(a, p, xs, sx, sp, sp_up, part, st);
    case 5: return launch_mx_tiles<Mx160, false>(a, p, xs, sx, sp, sp_up, part, st);
    default: return launch_mx_tiles<Mx32, false>(a, p, xs, sx, sp, sp_up, part, st);
  }
}

}  // namespace qmm
