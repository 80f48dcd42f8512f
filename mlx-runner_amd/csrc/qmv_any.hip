// nvfp4 decode matmul for x of 3-8 rows at row lengths the scaled-MFMA kernels (qmv_mfma.hip)
// have no instance for: any K that is a multiple of 128.
//
// y[M, N] = x[M, K] @ deq(W)[N, K].T, x and y bf16, fp32 accumulation; with MLP
// silu(x @ gate.T) * (x @ up.T).
//
// What bounds it: the dequantization (~2 VALU ops per weight), whatever the rows; the unpacking
// GEMV's work grows with every row of x, and the prefill GEMM pays a step's latency and a
// reduce.  us per call, N x K, weights cold:
//                        3 rows        4 rows        6 rows (GEMV at 3-4 rows and GEMM at 6 before)
//   14336 x 4096      16.8 -> 11.1  19.3 -> 11.6  15.4 -> 12.4
//   30000 x 2560      28.0 -> 16.8  33.5 -> 16.6  17.5 -> 17.4
//   5120 x 8192       18.9 -> 13.8  23.5 -> 13.9  (two passes: GEMM 13.5, here 15.5)
//   6144 x 2048        8.5 -> 7.1    9.8 -> 6.9    9.8 -> 7.0
//   MLP 14336 x 4096 with its down projection 4096 x 14336: 50.5 -> 36.0, 59.5 -> 37.1, 58.9 -> 41.2
#include "qmm_device.h"
#include "qmm_launch.h"

namespace qmm {

namespace {
constexpr int QA_SLICE = 256, QA_MAXQ = 16, QA_FLUSH_MAX = 8, QA_WAVES = 20;
// A wave's LDS: 16 rows of a slice's W bytes (pitch + 16: rows fall in distinct banks) and of its scales.
constexpr int QA_PITCH = 128 + 16, QA_TILE = 16 * QA_PITCH + 16 * 16;
__device__ __forceinline__ void qa_barrier() { asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory"); }
}  // namespace

// Work split: a workgroup owns a contiguous row range (rbase rows, one more in the first rrem
// workgroups), its Q waves the K slices p Q + q of 256 elements in P passes.  A unit is 16
// rows (MLP: 8 gate rows and the same 8 up rows) x one slice: loaded 1 KiB contiguous per
// instruction, changed in layout through the wave's LDS tile, dequantized to bf16 (exact) and
// multiplied with all 16 x rows at once (v_mfma_f32_16x16x32_bf16; x stays in registers for a
// pass, rows from M on are zero).
//   MFMA c of a unit (of 8) takes elements 64 h + 8 c + [0, 8) for lane group h, so a lane
// reads 32 contiguous bytes; E2M1 times its E4M3 scale is exact in bf16.  Slices of 256, not 512:
// half the registers of x, so that 20 waves fit a CU (14336 x 4096 at 3 rows: 11.2 against 12.0
// us, 30000 x 2560 16.4 against 19.7).
// Output lane (n, h), element v: x row 4 h + v, W row n.  Partial sums go to LDS per (row
// block, x row, wave) and are summed over the waves in a fixed order; later passes continue
// them.  The half of the last slice that is past K has zero x and re-reads its row.
template <bool MLP>
__global__ __launch_bounds__(64 * QA_MAXQ) void qmv_any_kernel(int N, int K, int M, int F, int P, int rbase, int rrem,
                                                               const uint16_t *__restrict__ x,
                                                               const uint8_t *__restrict__ w,
                                                               const uint8_t *__restrict__ s,
                                                               const uint8_t *__restrict__ w2,
                                                               const uint8_t *__restrict__ s2, const YOut yo) {
  constexpr int RB = MLP ? 8 : 16;                       // output rows per unit
  extern __shared__ __attribute__((aligned(16))) uint8_t lds[];
  const int tid = threadIdx.x, lane = tid & 63, Q = blockDim.x >> 6;
  const int q = __builtin_amdgcn_readfirstlane(tid >> 6);
  uint8_t *wt = lds + q * QA_TILE, *st = wt + 16 * QA_PITCH;
  float *part = (float *)(lds + Q * QA_TILE);  // [F][M][Q][16]
  const int b = blockIdx.x;
  const int r_begin = b * rbase + min(b, rrem), r_end = r_begin + rbase + (b < rrem ? 1 : 0);
  const int nrb = (r_end - r_begin + RB - 1) / RB;
  const int n = lane & 15, h = lane >> 4;
  const uint32_t wrow = (uint32_t)(K >> 1), srow = (uint32_t)(K >> 4);

  // sums of row blocks [rb0, rb0 + cnt) over the waves
  auto flush = [&](int rb0, int cnt) __attribute__((always_inline)) {
    qa_barrier();
    const int items = cnt * M * RB;
    for (int t = tid; t < items; t += blockDim.x) {
      const int nn = t % RB, m = t / RB % M, rbi = t / (RB * M);
      const int row = r_begin + RB * (rb0 + rbi) + nn;
      const float *pp = part + ((rbi * M + m) * Q) * 16 + nn;
      float a = 0.f, u = 0.f;
      for (int qq = 0; qq < Q; ++qq) {
        a += pp[16 * qq];
        if constexpr (MLP) u += pp[16 * qq + 8];
      }
      if (row < r_end) *yo.at(m, row) = f32_to_bf16_rne(MLP ? silu_mul_bf16(a, u) : a);
    }
    qa_barrier();
  };

  for (int p = 0; p < P; ++p) {
    const int k0 = QA_SLICE * (p * Q + q);
    if (k0 < K) {  // (one pass: always)
      const int kv = min(QA_SLICE, K - k0);  // elements of the slice, a multiple of 128
      bf16x8_t af[8];
      {
        const bool live = n < M;
        const uint16_t *xp = x + (int64_t)(live ? n : 0) * K + k0;
#pragma unroll
        for (int c = 0; c < 8; ++c) {
          const int k = 64 * h + 8 * c;
          uint4 v = *(const uint4 *)(xp + (k < kv ? k : 0));
          if (!live || k >= kv) v = make_uint4(0, 0, 0, 0);
          af[c] = __builtin_bit_cast(bf16x8_t, v);
        }
      }
      // Load i, lane l: row 8 i + l / 8, 16-byte piece l % 8 of the slice; scales: row l / 4, dword
      // l % 4.  Rows past the range re-read its last row.
      const int wq = 16 * (lane & 7), sq = 4 * (lane & 3);
      const uint32_t woff = (uint32_t)(k0 >> 1) + (wq < kv >> 1 ? wq : 0), soff = (uint32_t)(k0 >> 4) + (sq < kv >> 4 ? sq : 0);
      uint4 wv[2];
      uint32_t sv;
      auto load_unit = [&](int rb) __attribute__((always_inline)) {
        auto row_of = [&](int rr) __attribute__((always_inline)) {
          return (uint32_t)min(r_begin + RB * rb + (MLP ? rr & 7 : rr), r_end - 1);
        };
#pragma unroll
        for (int i = 0; i < 2; ++i) {
          const int rr = 8 * i + (lane >> 3);
          wv[i] = load_stream16((MLP && rr >= 8 ? w2 : w) + row_of(rr) * wrow + woff);
        }
        sv = *(const uint32_t *)((MLP && lane >= 32 ? s2 : s) + row_of(lane >> 2) * srow + soff);
      };
      load_unit(0);
      int rbf = 0;  // rb % F
      for (int rb = 0; rb < nrb; ++rb) {
        // registers -> tile, then the next unit's loads; a wave's LDS accesses run in order
#pragma unroll
        for (int i = 0; i < 2; ++i)
          *(uint4 *)(wt + (8 * i + (lane >> 3)) * QA_PITCH + 16 * (lane & 7)) = wv[i];
        *(uint32_t *)(st + 4 * lane) = sv;
        if (rb + 1 < nrb) load_unit(rb + 1);
        float *slot = part + (size_t)(rbf * M) * Q * 16 + q * 16 + n;
        f32x4_t acc = {0.f, 0.f, 0.f, 0.f};
        if (p > 0) {
#pragma unroll
          for (int v = 0; v < 4; ++v)
            if (4 * h + v < M) acc[v] = slot[(4 * h + v) * Q * 16];
        }
        const uint32_t sc = *(const uint32_t *)(st + n * 16 + 4 * h);
        uint4 wd[2];
#pragma unroll
        for (int i = 0; i < 2; ++i) wd[i] = *(const uint4 *)(wt + n * QA_PITCH + 32 * h + 16 * i);
#pragma unroll
        for (int c = 0; c < 8; ++c) {
          const uint4 &u = wd[c >> 2];
          const uint32_t word = (c & 3) == 0 ? u.x : (c & 3) == 1 ? u.y : (c & 3) == 2 ? u.z : u.w;
          acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(af[c], deq8_nvfp4(word, (sc >> (8 * (c >> 1))) & 0xFF), acc, 0, 0, 0);
        }
#pragma unroll
        for (int v = 0; v < 4; ++v)
          if (4 * h + v < M) slot[(4 * h + v) * Q * 16] = acc[v];
        if (P == 1 && (rbf + 1 == F || rb + 1 == nrb)) flush(rb - rbf, rbf + 1);
        rbf = rbf + 1 == F ? 0 : rbf + 1;
      }
    }
  }
  if (P > 1) flush(0, nrb);
}

namespace {
struct QaShape {
  int Q, P, grid, F, lds;  // F = 0: does not fit
};
}  // namespace
static QaShape qa_shape(const QmmArgs &a) {
  const int slices = (a.K + QA_SLICE - 1) / QA_SLICE, RB = a.w_up ? 8 : 16;
  QaShape g;
  g.P = (slices + QA_MAXQ - 1) / QA_MAXQ;
  g.Q = (slices + g.P - 1) / g.P;
  const int per_cu = QA_WAVES / g.Q, cus = device_cu_count();
  const int rbs = (a.N + RB - 1) / RB;
  g.grid = rbs < cus * per_cu ? rbs : cus * per_cu;
  g.F = 0;
  if (g.grid <= 0) return g;
  const int nrb = ((a.N + g.grid - 1) / g.grid + RB - 1) / RB;
  int F = nrb < QA_FLUSH_MAX ? nrb : QA_FLUSH_MAX;
  if (g.P > 1) F = nrb;
  const int room = (160 * 1024) / per_cu;
  while (F > 0 && g.Q * QA_TILE + F * a.M * g.Q * 64 > room) F = g.P > 1 ? 0 : F - 1;
  g.F = F;
  g.lds = g.Q * QA_TILE + F * a.M * g.Q * 64;
  return g;
}

// Where it is faster: than the unpacking GEMV at 3-4 rows except on short matrices (4096 x
// 4096 at 3 rows 8.1 against 5.9 us, 5120 x 4096 8.2 against 8.7, 4096 x 12288 15.7 against
// 17.8); than the prefill GEMM at 5-8 rows in one pass (5120 x 8192 15.5 against 13.5), at 7-8 up
// to 16384 rows of W (the partial sums' traffic grows with both: 30000 x 2560 at 8 rows 19.2
// against 15.3, 14336 x 4096 13.6 against 15.1).
bool qmv_any_ok(const QmmArgs &a) {
  if (a.mode != NVFP4 || a.x_f32 || a.M < 3 || a.M > 8 || a.N < 4096 || a.K <= 0 || a.K % 128 != 0) return false;
  const bool one_pass = a.K <= QA_SLICE * QA_MAXQ;
  if (a.M <= 4 ? a.N < 5120 && one_pass : !one_pass || (a.M > 6 && a.N > 16384)) return false;
  if (((uintptr_t)a.x | (uintptr_t)a.w | (uintptr_t)a.w_up) & 15) return false;
  if (((uintptr_t)a.s | (uintptr_t)a.s_up) & 3) return false;
  if ((int64_t)a.N * (a.K / 2) >= ((int64_t)1 << 32)) return false;  // 32-bit offsets within a matrix
  return qa_shape(a).F > 0;
}

template <bool MLP>
static hipError_t launch_qa(const QmmArgs &a, hipStream_t st) {
  const QaShape g = qa_shape(a);
  static std::atomic<uint64_t> lds_set{0};
  const hipError_t e = ensure_dynamic_lds(lds_set, (const void *)qmv_any_kernel<MLP>, 160 * 1024);
  if (e != hipSuccess) return e;
  hipLaunchKernelGGL((qmv_any_kernel<MLP>), dim3(g.grid), dim3(64 * g.Q), g.lds, st, a.N, a.K, a.M, g.F, g.P,
                     a.N / g.grid, a.N % g.grid, (const uint16_t *)a.x, a.w, a.s, a.w_up, a.s_up, yout_of(a));
  return hipGetLastError();
}

hipError_t launch_qmv_any(const QmmArgs &a, hipStream_t st) {
  if (!qmv_any_ok(a)) return hipErrorInvalidValue;
  return a.w_up ? launch_qa<true>(a, st) : launch_qa<false>(a, st);
}

}  // namespace qmm
