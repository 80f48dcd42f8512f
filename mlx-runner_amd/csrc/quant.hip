// Dequantize (mlx_dequantize, src/mlx.zig:274) and quantize (mlx_quantize,
// src/mlx.zig:278) for the mxfp8 / nvfp4 layouts.
//
// Both move each byte once and are bound by memory (a large copy reaches ~5 TB/s here, read
// plus write): a thread takes chunks of 8 elements, 16 bytes of bf16, so that a wave's loads
// and stores cover whole lines, and UNROLL chunks at a time to keep enough of them in flight.
// The tensors are contiguous and K is a multiple of the group, so a chunk's words and scale
// follow from its index alone.  10240 x 5120, nvfp4, bf16: quantize 126 -> 26 us (one thread
// per group, 2-byte loads and a double-precision scale search before), dequantize 28 -> 28 us,
// 134 MB each: 5 TB/s.
//
// dequant: elements go through the same gfx950 converters the matmul kernels use, so the
// exhaustive dequant test pins the in-kernel unpack as well; the product with the group
// scale is one f32 multiply (exact for every finite in-range value).
//
// quantize: every rounding decision is exact (see the rule in qmm.h), so the result is
// bit-identical to the CPU restatement.
#include "qmm_device.h"
#include "qmm_launch.h"

namespace qmm {

constexpr int UNROLL = 4;
constexpr int CHUNK = 8;  // elements

// 16 bytes at an address of 2-byte alignment or better (a caller's array may be a view).
__device__ __forceinline__ uint4 load16u(const void *p) {
  uint4 v;
  __builtin_memcpy(&v, __builtin_assume_aligned(p, 2), 16);
  return v;
}
__device__ __forceinline__ void store16u(void *p, uint4 v) { __builtin_memcpy(__builtin_assume_aligned(p, 2), &v, 16); }

template <int MODE, bool OUT_F32>
__global__ __launch_bounds__(256) void dequant_kernel(const uint32_t *__restrict__ w, const uint8_t *__restrict__ s,
                                                      void *__restrict__ out, int64_t chunks) {
  const int64_t c0 = blockIdx.x * (int64_t)(256 * UNROLL) + threadIdx.x;
  uint32_t q[UNROLL][2], sc[UNROLL];
#pragma unroll
  for (int u = 0; u < UNROLL; ++u) {
    const int64_t c = min(c0 + 256 * u, chunks - 1);
    if constexpr (MODE == MXFP8) q[u][0] = w[2 * c], q[u][1] = w[2 * c + 1], sc[u] = s[c >> 2];
    else q[u][0] = w[c], sc[u] = s[c >> 1];
  }
#pragma unroll
  for (int u = 0; u < UNROLL; ++u) {
    const int64_t c = c0 + 256 * u;
    if (c >= chunks) break;
    float v[8];
    f32x2_t p[4];
    float f;
    if constexpr (MODE == MXFP8) {
      f = e8m0_to_f32(sc[u]);
      p[0] = fp8x2_to_f32x2<false>(q[u][0]), p[1] = fp8x2_to_f32x2<true>(q[u][0]);
      p[2] = fp8x2_to_f32x2<false>(q[u][1]), p[3] = fp8x2_to_f32x2<true>(q[u][1]);
    } else {
      f = __builtin_amdgcn_cvt_f32_fp8((int)sc[u], 0);
      p[0] = fp4x2_to_f32x2<0>(q[u][0]), p[1] = fp4x2_to_f32x2<1>(q[u][0]);
      p[2] = fp4x2_to_f32x2<2>(q[u][0]), p[3] = fp4x2_to_f32x2<3>(q[u][0]);
    }
#pragma unroll
    for (int j = 0; j < 4; ++j) v[2 * j] = p[j].x * f, v[2 * j + 1] = p[j].y * f;
    if constexpr (OUT_F32) {
      float *o = (float *)out + c * CHUNK;
      store16u(o, make_uint4(__float_as_uint(v[0]), __float_as_uint(v[1]), __float_as_uint(v[2]), __float_as_uint(v[3])));
      store16u(o + 4,
               make_uint4(__float_as_uint(v[4]), __float_as_uint(v[5]), __float_as_uint(v[6]), __float_as_uint(v[7])));
    } else {
      uint32_t d[4];
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        if constexpr (MODE == MXFP8) {
          d[j] = (uint32_t)f32_to_bf16_rne(v[2 * j]) | (uint32_t)f32_to_bf16_rne(v[2 * j + 1]) << 16;
        } else {  // E2M1 x E4M3 is exact in bf16: the upper halves; a NaN scale is the only NaN
          d[j] = __builtin_amdgcn_perm(__float_as_uint(v[2 * j + 1]), __float_as_uint(v[2 * j]), 0x07060302u);
          d[j] = f != f ? 0x7FC07FC0u : d[j];
        }
      }
      store16u((uint16_t *)out + c * CHUNK, make_uint4(d[0], d[1], d[2], d[3]));
    }
  }
}

template <int MODE, bool OUT_F32>
static void dequant_launch(const uint8_t *w, const uint8_t *s, int64_t chunks, void *out, hipStream_t st) {
  hipLaunchKernelGGL((dequant_kernel<MODE, OUT_F32>), dim3((chunks + 256 * UNROLL - 1) / (256 * UNROLL)), dim3(256), 0, st,
                     (const uint32_t *)w, s, out, chunks);
}

hipError_t launch_dequant(int mode, const uint8_t *w, const uint8_t *s, int64_t N, int64_t K, void *out,
                          bool out_f32, hipStream_t st) {
  const int64_t chunks = N * (K / CHUNK);
  if (chunks == 0) return hipSuccess;
  if (mode == MXFP8) out_f32 ? dequant_launch<MXFP8, true>(w, s, chunks, out, st) : dequant_launch<MXFP8, false>(w, s, chunks, out, st);
  else out_f32 ? dequant_launch<NVFP4, true>(w, s, chunks, out, st) : dequant_launch<NVFP4, false>(w, s, chunks, out, st);
  return hipGetLastError();
}

// ---------------------------------------------------------------- quantize

// E4M3 code of v in [0, 448] and back (v_cvt_pk_fp8_f32 rounds to nearest even).
__device__ __forceinline__ uint32_t e4m3_code(float v) {
  return (uint32_t)__builtin_amdgcn_cvt_pk_fp8_f32(v, 0.f, 0, false) & 0xFFu;
}
__device__ __forceinline__ float e4m3_value(uint32_t c) { return __builtin_amdgcn_cvt_f32_fp8((int)c, 0); }

// nvfp4 group scale: the E4M3 code nearest to amax / 6, ties to even, at most 448.  The
// rounded quotient's code c is at most one off; amax is compared with 6 times the midpoints
// beside it, 3 (v(c) + v(c +- 1)), which have at most 8 significant bits: exact in f32.
__device__ __forceinline__ uint32_t nvfp4_scale_code(float amax) {
  const uint32_t c = e4m3_code(fminf(amax * (1.f / 6.f), 448.f));
  const float v = e4m3_value(c);
  const bool odd = c & 1;
  const float hi = 3.f * (v + e4m3_value(c < 0x7Eu ? c + 1 : c)), lo = 3.f * (v + e4m3_value(c > 0u ? c - 1 : c));
  if (c < 0x7Eu && (amax > hi || (amax == hi && odd))) return c + 1;
  if (c > 0u && (amax < lo || (amax == lo && odd))) return c - 1;
  return c;
}

// E2M1 code (sign in bit 3, none on zero) of v for the scale sc >= 0, by comparisons with the
// exact products of the midpoints and sc: a tie takes the even code, NaN code 0.
__device__ __forceinline__ uint32_t e2m1_code(float v, float sc) {
  const float mids[7] = {0.25f, 0.75f, 1.25f, 1.75f, 2.5f, 3.5f, 5.0f};
  const float ax = fabsf(v);
  uint32_t c = 0;
#pragma unroll
  for (int t = 0; t < 7; ++t) c += (t & 1 ? ax >= mids[t] * sc : ax > mids[t] * sc) ? 1u : 0u;
  if (sc == 0.f) c = 0;
  return c && signbit(v) ? c | 8u : c;
}

// The largest of v over the LPG lanes (2 or 4) that share a group.
template <int LPG>
__device__ __forceinline__ uint32_t group_max(uint32_t v) {
  v = max(v, (uint32_t)__builtin_amdgcn_mov_dpp((int)v, 0xB1, 0xF, 0xF, true));               // lane ^ 1
  if constexpr (LPG == 4) v = max(v, (uint32_t)__builtin_amdgcn_mov_dpp((int)v, 0x4E, 0xF, 0xF, true));  // lane ^ 2
  return v;
}

// A chunk of 8 per lane; LPG lanes, adjacent, share a group's maximum.  |v| is compared by its
// bits, which order as the values do; groups that hold an infinity or a NaN (a NaN does not
// count towards the maximum) take the comparisons for every element.
template <int MODE, bool IN_F32>
__global__ __launch_bounds__(256) void quantize_kernel(const void *__restrict__ in, int64_t chunks,
                                                       uint32_t *__restrict__ wq, uint8_t *__restrict__ s) {
  constexpr int LPG = (MODE == MXFP8 ? 32 : 16) / CHUNK, NV = IN_F32 ? 2 : 1;
  const int64_t c0 = blockIdx.x * (int64_t)(256 * UNROLL) + threadIdx.x;
  uint4 q[UNROLL][NV];
#pragma unroll
  for (int u = 0; u < UNROLL; ++u)
#pragma unroll
    for (int i = 0; i < NV; ++i)
      q[u][i] = load16u((const uint8_t *)in + min(c0 + 256 * u, chunks - 1) * (16 * NV) + 16 * i);
#pragma unroll
  for (int u = 0; u < UNROLL; ++u) {
    const int64_t c = c0 + 256 * u;
    if (c >= chunks) break;  // chunks is a multiple of LPG: the lanes of a group leave together
    float v[8];
    uint32_t m = 0;  // f32 bits of the chunk's largest magnitude
    if constexpr (IN_F32) {
      const uint32_t d[8] = {q[u][0].x, q[u][0].y, q[u][0].z, q[u][0].w, q[u][NV - 1].x, q[u][NV - 1].y, q[u][NV - 1].z, q[u][NV - 1].w};
#pragma unroll
      for (int j = 0; j < 8; ++j) v[j] = __uint_as_float(d[j]), m = max(m, d[j] & 0x7FFFFFFFu);
    } else {
      const uint32_t d[4] = {q[u][0].x, q[u][0].y, q[u][0].z, q[u][0].w};
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        v[2 * j] = __uint_as_float(d[j] << 16), v[2 * j + 1] = __uint_as_float(d[j] & 0xFFFF0000u);
        m = max(m, max(d[j] << 16 & 0x7FFFFFFFu, d[j] & 0x7FFF0000u));
      }
    }
    m = group_max<LPG>(m);
    const bool finite = m < 0x7F800000u;
    if (!finite) {  // the largest that is not a NaN
      float a = 0.f;
#pragma unroll
      for (int j = 0; j < 8; ++j) a = fmaxf(a, fabsf(v[j]));
      m = group_max<LPG>(__float_as_uint(a));
    }
    const float amax = __uint_as_float(m);
    if constexpr (MODE == MXFP8) {
      int X = 0;
      if (m != 0) {
        const int e = (int)(m >> 23);
        X = (e == 0 ? 31 - __builtin_clz(m) - 149 : e - 127) - 8 + 127;  // floor(log2 amax) - 8
        X = X < 0 ? 0 : (X > 254 ? 254 : X);
      }
      uint32_t w[2];
#pragma unroll
      for (int h = 0; h < 2; ++h) {
        float p[4];
#pragma unroll
        for (int j = 0; j < 4; ++j) {
          // v / 2^(X - 127), exact for every value that can round to a nonzero code
          const float t = __builtin_ldexpf(v[4 * h + j], 127 - X);
          p[j] = t != t ? 0.f : __builtin_amdgcn_fmed3f(t, -448.f, 448.f);
        }
        int r = __builtin_amdgcn_cvt_pk_fp8_f32(p[0], p[1], 0, false);
        r = __builtin_amdgcn_cvt_pk_fp8_f32(p[2], p[3], r, true);
        const uint32_t mag = (uint32_t)r & 0x7F7F7F7Fu;  // no sign on zero
        w[h] = mag | ((uint32_t)r & (mag + 0x7F7F7F7Fu) & 0x80808080u);
      }
      uint2 o = make_uint2(w[0], w[1]);
      *(uint2 *)(wq + 2 * c) = o;
      if (c % LPG == 0) s[c / LPG] = (uint8_t)X;
    } else {
      const uint32_t code = m ? nvfp4_scale_code(amax) : 0u;
      const float sc = e4m3_value(code);
      uint32_t w = 0;
      if (IN_F32 || !finite || code == 0u) {
#pragma unroll
        for (int j = 0; j < 8; ++j) w |= e2m1_code(v[j], sc) << (4 * j);
      } else {
        // v / sc, exact where it is a midpoint, then the converter's nearest even.  (An 8-bit
        // over a 4-bit significand is a midpoint or at least 2^-15 of it away: every bf16 up
        // to 16 sc, which is more than a group of this scale holds, over every scale, and
        // every bf16 over the largest scale, gives the code of the comparisons.)
        const float inv = 1.f / sc;
        float p[8];
#pragma unroll
        for (int j = 0; j < 8; ++j) {
          const float q0 = v[j] * inv;
          const float q1 = __builtin_fmaf(__builtin_fmaf(-q0, sc, v[j]), inv, q0);
          p[j] = __builtin_amdgcn_fmed3f(q1, -6.f, 6.f);
        }
        w = __builtin_amdgcn_cvt_scalef32_pk_fp4_f32(w, p[0], p[1], 1.0f, 0);
        w = __builtin_amdgcn_cvt_scalef32_pk_fp4_f32(w, p[2], p[3], 1.0f, 1);
        w = __builtin_amdgcn_cvt_scalef32_pk_fp4_f32(w, p[4], p[5], 1.0f, 2);
        w = __builtin_amdgcn_cvt_scalef32_pk_fp4_f32(w, p[6], p[7], 1.0f, 3);
        const uint32_t mag = w & 0x77777777u;  // no sign on zero
        w = mag | (w & (mag + 0x77777777u) & 0x88888888u);
      }
      wq[c] = w;
      if (c % LPG == 0) s[c / LPG] = (uint8_t)code;
    }
  }
}

template <int MODE, bool IN_F32>
static void quantize_launch(const void *in, int64_t chunks, uint32_t *wq, uint8_t *s, hipStream_t st) {
  hipLaunchKernelGGL((quantize_kernel<MODE, IN_F32>), dim3((chunks + 256 * UNROLL - 1) / (256 * UNROLL)), dim3(256), 0,
                     st, in, chunks, wq, s);
}

hipError_t launch_quantize(int mode, const void *in, bool in_f32, int64_t N, int64_t K, uint32_t *wq, uint8_t *s,
                           hipStream_t st) {
  const int64_t chunks = N * (K / CHUNK);
  if (chunks == 0) return hipSuccess;
  if (mode == MXFP8) in_f32 ? quantize_launch<MXFP8, true>(in, chunks, wq, s, st) : quantize_launch<MXFP8, false>(in, chunks, wq, s, st);
  else in_f32 ? quantize_launch<NVFP4, true>(in, chunks, wq, s, st) : quantize_launch<NVFP4, false>(in, chunks, wq, s, st);
  return hipGetLastError();
}

__global__ void fill_zero_bytes_kernel(uint8_t *__restrict__ p, int64_t n) {
  if ((int64_t)threadIdx.x < n) p[threadIdx.x] = 0;
}

// Zero-fill (a kernel rather than hipMemsetAsync, so the op stays safe to
// record into a HIP graph).
__global__ __launch_bounds__(256) void fill_zero_kernel(uint32_t *__restrict__ p, int64_t words) {
  for (int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; i < words; i += (int64_t)gridDim.x * blockDim.x)
    p[i] = 0u;
}

hipError_t launch_fill_zero(void *p, size_t bytes, hipStream_t st) {
  const int64_t words = (int64_t)(bytes / 4);
  if (words > 0) {
    int64_t blocks = (words + 255) / 256;
    if (blocks > 65536) blocks = 65536;
    hipLaunchKernelGGL(fill_zero_kernel, dim3(blocks), dim3(256), 0, st, (uint32_t *)p, words);
  }
  if (bytes % 4) {
    // trailing bytes (odd-sized bf16 outputs): one more word-aligned store is not
    // possible without overrunning, so clear them with a byte kernel
    hipLaunchKernelGGL(fill_zero_bytes_kernel, dim3(1), dim3(64), 0, st, (uint8_t *)p + words * 4,
                       (int64_t)(bytes % 4));
  }
  return hipGetLastError();
}

int device_cu_count() {
  static std::atomic<int> cached[64];
  int dev = 0;
  if (hipGetDevice(&dev) != hipSuccess) {
    (void)hipGetLastError();
    return 0;
  }
  const bool slot = dev >= 0 && dev < 64;
  if (slot) {
    const int c = cached[dev].load(std::memory_order_relaxed);
    if (c > 0) return c;
  }
  int n = 0;
  if (hipDeviceGetAttribute(&n, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess || n <= 0) {
    (void)hipGetLastError();
    return 0;
  }
  if (slot) cached[dev].store(n, std::memory_order_relaxed);
  return n;
}

hipError_t ensure_dynamic_lds(std::atomic<uint64_t> &done, const void *kernel, int bytes) {
  int dev = 0;
  hipError_t e = hipGetDevice(&dev);
  if (e != hipSuccess) return e;
  const uint64_t bit = dev >= 0 && dev < 64 ? (uint64_t)1 << dev : 0;
  if (bit && (done.load(std::memory_order_acquire) & bit)) return hipSuccess;
  e = hipFuncSetAttribute(kernel, hipFuncAttributeMaxDynamicSharedMemorySize, bytes);
  if (e == hipSuccess && bit) done.fetch_or(bit, std::memory_order_release);
  return e;
}

}  // namespace qmm
