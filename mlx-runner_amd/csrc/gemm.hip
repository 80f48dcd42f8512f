// Quantized matmul for more than 8 rows at row lengths the pipelined GEMMs do not take: nvfp4 with K
// a multiple of 16 but not of 32 (rows their 16-byte DMA pieces do not divide), mxfp8 with K a
// multiple of 32 but not of 64.  The mxfp8 GEMM of gemm_fp8.hip could pad the latter, but its
// fp8 MFMA on a split x is the coarser arithmetic: at 200 x 1000 x 1056 it rounds 1.17% of the
// outputs the other way than the exact sums, this kernel 0.008%.  What that precision costs: 147 x
// 2181 x 8672 takes 325 us here and 25 there.
//
// y[M, N] = x[M, K] @ deq(W)[N, K].T through the same call sites (src/engine.zig:364-382).
//
// Tiling (gfx950, wave64, 256 threads):
//   block tile 128 (x rows) x 128 (W rows), K step 32;
//   each thread stages 16 elements of one x row and 16 of one W row into LDS;
//   W elements are unpacked with the gfx950 converters, so LDS holds bf16:
//     nvfp4: E2M1 times its E4M3 scale in f32, exact in bf16 (at most 6
//            significant bits, magnitudes 2^-10 .. 2688);
//     mxfp8: the E4M3 codes unscaled (exact in bf16).  A K step is one 32-element
//            scale block, so each step's MFMA sums go to a temporary and are added
//            to the accumulator times the W row's E8M0 scale in f32: a weight whose
//            f32 (or bf16) dequant would overflow or underflow still multiplies x
//            as its true value, as in the other kernels;
//   4 waves in 2x2, each owning 64x64 of the tile as 2x2 v_mfma_f32_32x32x16_bf16
//   accumulators (fp32); epilogue rounds to bf16 (RNE).
#include "qmm_device.h"
#include "qmm_launch.h"

namespace qmm {

namespace {
constexpr int BM = 128, BN = 128, BK = 32, LDK = BK + 8;  // LDS row pitch (bf16), 80 bytes
}

__device__ __forceinline__ uint32_t pack_bf16x2(float a, float b) {
  return (uint32_t)f32_to_bf16_rne(a) | ((uint32_t)f32_to_bf16_rne(b) << 16);
}

// 16 consecutive W elements of row n starting at k (k a multiple of 16) as 8 bf16 pairs
// (mxfp8: unscaled codes, the block's scale in *sc_out; nvfp4: dequantized).
template <int MODE>
__device__ __forceinline__ void load_w16(const uint8_t *__restrict__ w, const uint8_t *__restrict__ s, int64_t n,
                                         int k, int K, uint32_t out[8], float *sc_out) {
  if constexpr (MODE == MXFP8) {
    const uint4 q = *(const uint4 *)(w + n * (int64_t)K + k);
    *sc_out = e8m0_to_f32(s[n * (int64_t)(K >> 5) + (k >> 5)]);
    const uint32_t d[4] = {q.x, q.y, q.z, q.w};
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      out[2 * j] = __builtin_bit_cast(uint32_t, fp8x2_to_bf16x2<false>(d[j]));
      out[2 * j + 1] = __builtin_bit_cast(uint32_t, fp8x2_to_bf16x2<true>(d[j]));
    }
  } else {
    const uint2 q = *(const uint2 *)(w + n * (int64_t)(K >> 1) + (k >> 1));
    const float sc = __builtin_amdgcn_cvt_f32_fp8((int)s[n * (int64_t)(K >> 4) + (k >> 4)], 0);
    const uint32_t d[2] = {q.x, q.y};
#pragma unroll
    for (int j = 0; j < 2; ++j) {
      f32x2_t a = fp4x2_to_f32x2<0>(d[j]), b = fp4x2_to_f32x2<1>(d[j]);
      f32x2_t c = fp4x2_to_f32x2<2>(d[j]), e = fp4x2_to_f32x2<3>(d[j]);
      out[4 * j + 0] = pack_bf16x2(a.x * sc, a.y * sc);
      out[4 * j + 1] = pack_bf16x2(b.x * sc, b.y * sc);
      out[4 * j + 2] = pack_bf16x2(c.x * sc, c.y * sc);
      out[4 * j + 3] = pack_bf16x2(e.x * sc, e.y * sc);
    }
  }
}

template <int MODE>
__global__ __launch_bounds__(256) void gemm_bf16_kernel(const uint16_t *__restrict__ x, const uint8_t *__restrict__ w,
                                                        const uint8_t *__restrict__ s, uint16_t *__restrict__ y, int M,
                                                        int N, int K) {
  __shared__ __attribute__((aligned(16))) uint16_t As[BM * LDK];
  __shared__ __attribute__((aligned(16))) uint16_t Bs[BN * LDK];
  __shared__ float Ss[MODE == MXFP8 ? BN : 1];  // mxfp8: the step's scale of each W row
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int wm = wave >> 1, wn = wave & 1;
  const int m0 = blockIdx.y * BM, n0 = blockIdx.x * BN;
  const int lrow = tid >> 1, lh = tid & 1;

  f32x16_t acc[2][2];
#pragma unroll
  for (int i = 0; i < 2; ++i)
#pragma unroll
    for (int j = 0; j < 2; ++j)
#pragma unroll
      for (int v = 0; v < 16; ++v) acc[i][j][v] = 0.f;

  for (int k0 = 0; k0 < K; k0 += BK) {
    const int kk = k0 + 16 * lh;
    uint4 a0 = {0, 0, 0, 0}, a1 = {0, 0, 0, 0};
    const int m = m0 + lrow;
    if (m < M && kk < K) {
      const uint4 *p = (const uint4 *)(x + (int64_t)m * K + kk);
      a0 = p[0];
      a1 = p[1];
    }
    uint32_t b[8] = {0, 0, 0, 0, 0, 0, 0, 0};
    float sc = 0.f;
    const int n = n0 + lrow;
    if (n < N && kk < K) load_w16<MODE>(w, s, n, kk, K, b, &sc);
    uint4 *ad = (uint4 *)(As + lrow * LDK + 16 * lh);
    ad[0] = a0;
    ad[1] = a1;
    uint4 *bd = (uint4 *)(Bs + lrow * LDK + 16 * lh);
    bd[0] = make_uint4(b[0], b[1], b[2], b[3]);
    bd[1] = make_uint4(b[4], b[5], b[6], b[7]);
    if constexpr (MODE == MXFP8)
      if (lh == 0) Ss[lrow] = sc;  // both halves of a row's step are one 32-block
    __syncthreads();
    f32x16_t part[2][2];
    if constexpr (MODE == MXFP8) {
#pragma unroll
      for (int i = 0; i < 2; ++i)
#pragma unroll
        for (int j = 0; j < 2; ++j)
#pragma unroll
          for (int v = 0; v < 16; ++v) part[i][j][v] = 0.f;
    }
#pragma unroll
    for (int kh = 0; kh < 2; ++kh) {
      bf16x8_t af[2], bf[2];
#pragma unroll
      for (int i = 0; i < 2; ++i)
        af[i] = *(const bf16x8_t *)(As + (wm * 64 + i * 32 + (lane & 31)) * LDK + kh * 16 + (lane >> 5) * 8);
#pragma unroll
      for (int j = 0; j < 2; ++j)
        bf[j] = *(const bf16x8_t *)(Bs + (wn * 64 + j * 32 + (lane & 31)) * LDK + kh * 16 + (lane >> 5) * 8);
#pragma unroll
      for (int i = 0; i < 2; ++i)
#pragma unroll
        for (int j = 0; j < 2; ++j) {
          if constexpr (MODE == MXFP8)
            part[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(af[i], bf[j], part[i][j], 0, 0, 0);
          else
            acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(af[i], bf[j], acc[i][j], 0, 0, 0);
        }
    }
    if constexpr (MODE == MXFP8) {
      // accumulator column = W row wn * 64 + j * 32 + lane % 32 of the tile
#pragma unroll
      for (int j = 0; j < 2; ++j) {
        const float scj = Ss[wn * 64 + j * 32 + (lane & 31)];
#pragma unroll
        for (int i = 0; i < 2; ++i)
#pragma unroll
          for (int v = 0; v < 16; ++v) acc[i][j][v] = __builtin_fmaf(part[i][j][v], scj, acc[i][j][v]);
      }
    }
    __syncthreads();
  }

#pragma unroll
  for (int i = 0; i < 2; ++i)
#pragma unroll
    for (int j = 0; j < 2; ++j) {
      const int col = n0 + wn * 64 + j * 32 + (lane & 31);
#pragma unroll
      for (int v = 0; v < 16; ++v) {
        const int row = m0 + wm * 64 + i * 32 + (v >> 2) * 8 + (lane >> 5) * 4 + (v & 3);
        if (row < M && col < N) y[(int64_t)row * N + col] = f32_to_bf16_rne(acc[i][j][v]);
      }
    }
}

bool gemm_ok(const QmmArgs &a) {
  // bf16 x; K a multiple of 16 (one nvfp4 group / half an mxfp8 group per loader).
  return !a.x_f32 && a.K % 16 == 0 && a.M > 0 && a.N > 0 && (a.mode != MXFP8 || a.K % 32 == 0);
}

hipError_t launch_gemm(const QmmArgs &a, hipStream_t st) {
  if (!gemm_ok(a)) return hipErrorInvalidValue;
  dim3 grid((a.N + BN - 1) / BN, (a.M + BM - 1) / BM);
  if (a.mode == MXFP8)
    hipLaunchKernelGGL((gemm_bf16_kernel<MXFP8>), grid, dim3(256), 0, st, (const uint16_t *)a.x, a.w, a.s,
                       (uint16_t *)a.y, a.M, a.N, a.K);
  else
    hipLaunchKernelGGL((gemm_bf16_kernel<NVFP4>), grid, dim3(256), 0, st, (const uint16_t *)a.x, a.w, a.s,
                       (uint16_t *)a.y, a.M, a.N, a.K);
  return hipGetLastError();
}

}  // namespace qmm
