// The int8 tier on gfx950: per-row symmetric int8 quantization of
// activations and of (dequantized) weights. The int8 x int8 -> int32 GEMM
// itself runs on the bf16 GEMMs' tiles (tall.hip's int8 mode; below it qgemm.hip,
// operand mode kI8Ops: v_mfma_i32_32x32x32_i8, 128 int8 of K per step in the same
// 128-byte LDS rows) with the dequant epilogue fused:
//   y = bf16(fma(float(acc), sx[m] * sw[n], bias[n] or +0)).
// Integer accumulation is exact, so the int32 results are bit-identical to
// any other order of the same sum; the epilogue is a fixed f32 sequence.
//
// Reference: the int8 tier under MetalOps::dense_mma_ (I8GemmContext::gemm,
// src/ltx25-metal-ops.cc:386-391; contract at src/ltx25-metal-ops.h:810-817).
#include "common.h"

#include <type_traits>

namespace ltx25 {
namespace {

constexpr int kThreads = 256;
constexpr int kRowsPerBlock = kThreads / 64;   // one wave per row

// Both quantizers are bound by memory (the row in, its int8 out) where their
// arithmetic, two passes over values that stay in registers, keeps up: a copy of
// the bytes of 8160 x 4096 and of a 4096 x 4096 w8 weight is 27 us, both in one
// launch take 32 (29 and 18 us, then 24 and 18, in a launch each).

// 16-byte chunks a lane keeps in registers between the absmax pass and the
// quantize pass: the instance for a row's K keeps no more than it needs, up to
// kMaxChunks (K up to 8192 bf16, 16384 w8 codes); chunks past them are read again
// for the second pass.
constexpr int kMaxChunks = 16;

typedef uint16_t u16x2 __attribute__((ext_vector_type(2)));
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));

__device__ __forceinline__ uint32_t pk_max_u16(uint32_t a, uint32_t b)
{
  return __builtin_bit_cast(uint32_t, __builtin_elementwise_max(__builtin_bit_cast(u16x2, a),
                                                                __builtin_bit_cast(u16x2, b)));
}

__device__ __forceinline__ uint32_t pk_min_u16(uint32_t a, uint32_t b)
{
  return __builtin_bit_cast(uint32_t, __builtin_elementwise_min(__builtin_bit_cast(u16x2, a),
                                                                __builtin_bit_cast(u16x2, b)));
}

// q = clamp(rint(v / s), -127, 127) with v / s correctly rounded, given
// rs = 1 / s rounded, for four values packed low byte first. `exact` 0: s and rs
// are normal and no value is a NaN, so |v * rs| <= 127 (1 + 2^-23) needs no clamp
// and is within 127 * 2^-24 < 2^-17 of the quotient, 2^-18 more with that rounded;
// rint of it is rint(v / s) unless it lies within 2^-16 of a half-integer. The fma with 1.5 * 2^23 rounds it to the integer
// and holds that in its low bits; a second one gives its distance. Values near a
// half-integer take the division itself, tested once for the four, and so does
// every value with `exact` 1. A NaN gives -127; s <= 0 gives 0.
// 7 instructions a value with the unpacking and the absmax; with the product, the
// clamp and the distance apart it was 10, and both operands of 8160 x 4096 -> 4096
// (w8) took 35 us where they take 32.
__device__ __forceinline__ uint32_t q8x4(const float* v, float s, float rs, float exact)
{
  constexpr float kMagic = 12582912.0f;
  if (!(s > 0.0f)) { return 0u; }
  uint32_t bits[4];
  float off = exact;
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    const float m = fmaf(v[j], rs, kMagic);
    bits[j] = __float_as_uint(m);
    off = fmaxf(off, fabsf(fmaf(v[j], rs, kMagic - m)));
  }
  if (off > 0.5f - 0x1p-16f) {
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      bits[j] = __float_as_uint(fminf(fmaxf(rintf(v[j] / s), -127.0f), 127.0f) + kMagic);
    }
  }
  // the four low bytes: v_perm picks bytes 0..3 of its second operand, 4..7 of its first
  const uint32_t lo = __builtin_amdgcn_perm(bits[1], bits[0], 0x0c0c0400u);
  const uint32_t hi = __builtin_amdgcn_perm(bits[3], bits[2], 0x04000c0cu);
  return lo | hi;
}

// q8x4's `exact` for a row of scale s, `nan`: one of the values is a NaN
__device__ __forceinline__ float needs_division(float s, bool nan)
{
  return s >= 0x1p-126f && s <= 0x1p126f && !nan ? 0.0f : 1.0f;
}

__device__ __forceinline__ float wave_absmax(float amax)
{
  for (int off = 32; off > 0; off >>= 1) {
    amax = fmaxf(amax, __shfl_xor(amax, off, 64));
  }
  return amax;
}

// One wave per row: absmax, then q = clamp(rint(x / s), -127, 127),
// s = absmax / 127. Works on bf16 activations (values exact in f32). Lane l
// takes 16-byte chunks l, l + 64, ...: every load instruction of the wave
// covers 1 KB of the row, NC of them in flight per lane, and the row's
// maximum is a shuffle reduction (no LDS, no barrier). The absmax runs on the
// bf16 bits, two a time, sign bits cleared: their order is the values' order;
// a row with a NaN (bits past infinity's) takes its maximum again in floats,
// which passes NaNs over.
template <int NC>
__device__ __forceinline__ void quantize_row(const uint16_t* x, int8_t* q, float* scale, int m,
                                             int K)
{
  const int lane = threadIdx.x & 63;
  const uint16_t* xr = x + (size_t)m * K;
  int8_t* qr = q + (size_t)m * K;
  const int chunks = K / 8;
  u32x4 cache[NC];
#pragma unroll
  for (int c = 0; c < NC; ++c) {
    const int i = lane + c * 64;
    cache[c] = u32x4{0u, 0u, 0u, 0u};
    if (i < chunks) { cache[c] = *(const u32x4*)(xr + (size_t)i * 8); }
  }
  uint32_t mx = 0u;
  auto absmax8 = [&](const u32x4& v) {
#pragma unroll
    for (int j = 0; j < 4; ++j) { mx = pk_max_u16(mx, v[j] & 0x7fff7fffu); }
  };
#pragma unroll
  for (int c = 0; c < NC; ++c) { absmax8(cache[c]); }
  for (int i = lane + NC * 64; i < chunks; i += 64) {
    absmax8(*(const u32x4*)(xr + (size_t)i * 8));
  }
  const uint32_t top = mx >> 16 > (mx & 0xffffu) ? mx >> 16 : mx & 0xffffu;
  // bits of non-negative floats order as the floats do
  float amax = __uint_as_float(top << 16);
  const bool nan = __any(top > 0x7f80u);
  if (nan) {
    amax = 0.0f;
    for (int i = lane; i < chunks; i += 64) {
      const u32x4 v = *(const u32x4*)(xr + (size_t)i * 8);
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        amax = fmaxf(amax, fabsf(bf16_to_f32((uint16_t)(v[j] & 0xffffu))));
        amax = fmaxf(amax, fabsf(bf16_to_f32((uint16_t)(v[j] >> 16))));
      }
    }
  }
  amax = wave_absmax(amax);
  const float s = amax / 127.0f;
  const float rs = 1.0f / s;
  const float exact = needs_division(s, nan);
  if (lane == 0) { scale[m] = s; }
  auto quant8 = [&](const u32x4& v, int i) {
    float f[8];
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      f[2 * j] = __uint_as_float(v[j] << 16);
      f[2 * j + 1] = __uint_as_float(v[j] & 0xffff0000u);
    }
    *(uint2*)(qr + (size_t)i * 8) = make_uint2(q8x4(f, s, rs, exact), q8x4(f + 4, s, rs, exact));
  };
#pragma unroll
  for (int c = 0; c < NC; ++c) {
    const int i = lane + c * 64;
    if (i < chunks) { quant8(cache[c], i); }
  }
  for (int i = lane + NC * 64; i < chunks; i += 64) {
    quant8(*(const u32x4*)(xr + (size_t)i * 8), i);
  }
}

// The same for the dequantized values of a group-affine weight row,
// w = bf16(fma(scale, q, qbias)): one wave per row, one 16-byte load of
// codes (16 w8 or 32 w4 codes, all in one group) per chunk, kept in
// registers between the absmax and the quantize pass; 16-byte int8 stores.
// Within a group w is monotone in its code (the fma and the rounding are), so
// a chunk's absmax is that of its least and greatest code, found on the codes.
template <int BITS, int NC>
__device__ __forceinline__ void quantize_qrow(const uint8_t* codes, const uint16_t* scales,
                                              const uint16_t* qbias, int gshift, int gcols,
                                              int8_t* q, float* scale, int n, int K)
{
  constexpr int CPC = 128 / BITS;                 // codes per 16-byte chunk
  const int lane = threadIdx.x & 63;
  const uint8_t* cr = codes + (size_t)n * ((size_t)K * BITS / 8);
  const uint16_t* srow = scales + (size_t)n * gcols;
  const uint16_t* brow = qbias + (size_t)n * gcols;
  int8_t* qr = q + (size_t)n * K;
  const int chunks = K / CPC;
  u32x4 cache[NC];
  float sc[NC], zp[NC];
#pragma unroll
  for (int c = 0; c < NC; ++c) {
    const int i = lane + c * 64;
    cache[c] = u32x4{0u, 0u, 0u, 0u};
    sc[c] = zp[c] = 0.0f;
    if (i < chunks) {
      cache[c] = *(const u32x4*)(cr + (size_t)i * 16);
      sc[c] = bf16_to_f32(srow[(i * CPC) >> gshift]);
      zp[c] = bf16_to_f32(brow[(i * CPC) >> gshift]);
    }
  }
  float amax = 0.0f;
  bool nan = false;   // in one of the lane's own chunks, or infinities of both signs
  auto absmax_chunk = [&](const u32x4& c, float s, float b) {
    uint32_t lo = 0xffffffffu, hi = 0u;   // two u16 lanes of codes each
    auto two = [&](uint32_t v) {
      lo = pk_min_u16(lo, v);
      hi = pk_max_u16(hi, v);
    };
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      if constexpr (BITS == 8) {
        two(c[j] & 0x00ff00ffu);
        two((c[j] >> 8) & 0x00ff00ffu);
      } else {
#pragma unroll
        for (int t = 0; t < 4; ++t) { two((c[j] >> (4 * t)) & 0x000f000fu); }
      }
    }
    const uint32_t l = min(lo >> 16, lo & 0xffffu);
    const uint32_t h = max(hi >> 16, hi & 0xffffu);
    const float vl = bf16_to_f32(f32_to_bf16(fmaf(s, (float)l, b)));
    const float vh = bf16_to_f32(f32_to_bf16(fmaf(s, (float)h, b)));
    amax = fmaxf(amax, fmaxf(fabsf(vl), fabsf(vh)));
    // a group's value is a NaN only where the least or the greatest code's is
    nan = nan || __builtin_isnan(vl + vh);
  };
#pragma unroll
  for (int c = 0; c < NC; ++c) { absmax_chunk(cache[c], sc[c], zp[c]); }   // past the row: 0
  for (int i = lane + NC * 64; i < chunks; i += 64) {
    absmax_chunk(*(const u32x4*)(cr + (size_t)i * 16), bf16_to_f32(srow[(i * CPC) >> gshift]),
                 bf16_to_f32(brow[(i * CPC) >> gshift]));
  }
  amax = wave_absmax(amax);
  const float s = amax / 127.0f;
  const float rs = 1.0f / s;
  const float exact = needs_division(s, nan);
  if (lane == 0) { scale[n] = s; }
  auto quant_chunk = [&](const u32x4& c, float gs, float gb, int i) {
    uint32_t packed[CPC / 4];
#pragma unroll
    for (int t = 0; t < CPC / 4; ++t) {
      float v[4];
#pragma unroll
      for (int j = 0; j < 4; j += 2) {
        const int k = 4 * t + j;   // codes k and k + 1
        uint32_t c0, c1;
        if constexpr (BITS == 8) {
          c0 = (c[k >> 2] >> (8 * (k & 3))) & 0xffu;
          c1 = (c[k >> 2] >> (8 * (k & 3) + 8)) & 0xffu;
        } else {
          c0 = (c[k >> 3] >> (4 * (k & 7))) & 0xfu;
          c1 = (c[k >> 3] >> (4 * (k & 7) + 4)) & 0xfu;
        }
        const uint32_t w = pack_bf16x2(fmaf(gs, (float)c0, gb), fmaf(gs, (float)c1, gb));
        v[j] = __uint_as_float(w << 16);
        v[j + 1] = __uint_as_float(w & 0xffff0000u);
      }
      packed[t] = q8x4(v, s, rs, exact);
    }
#pragma unroll
    for (int t = 0; t < CPC / 16; ++t) {
      *(uint4*)(qr + (size_t)i * CPC + 16 * t) =
          make_uint4(packed[4 * t], packed[4 * t + 1], packed[4 * t + 2], packed[4 * t + 3]);
    }
  };
#pragma unroll
  for (int c = 0; c < NC; ++c) {
    const int i = lane + c * 64;
    if (i < chunks) { quant_chunk(cache[c], sc[c], zp[c], i); }
  }
  for (int i = lane + NC * 64; i < chunks; i += 64) {
    quant_chunk(*(const u32x4*)(cr + (size_t)i * 16), bf16_to_f32(srow[(i * CPC) >> gshift]),
                bf16_to_f32(brow[(i * CPC) >> gshift]), i);
  }
}

// The wave's row of the launch
__device__ __forceinline__ int wave_row()
{
  return __builtin_amdgcn_readfirstlane(blockIdx.x * kRowsPerBlock + (threadIdx.x >> 6));
}

template <int NC>
__global__ void __launch_bounds__(kThreads)
i8_quantize_rows_kernel(const uint16_t* x, int8_t* q, float* scale, int M, int K)
{
  const int m = wave_row();
  if (m < M) { quantize_row<NC>(x, q, scale, m, K); }
}

template <int BITS, int NC>
__global__ void __launch_bounds__(kThreads)
i8_quantize_qweight_kernel(const uint8_t* codes, const uint16_t* scales,
                           const uint16_t* qbias, int gshift, int gcols,
                           int8_t* q, float* scale, int N, int K)
{
  const int n = wave_row();
  if (n < N) { quantize_qrow<BITS, NC>(codes, scales, qbias, gshift, gcols, q, scale, n, K); }
}

// A linear's weight (BITS 16: bf16 rows) and activation in one launch, the weight's
// rows first: its codes' arithmetic runs under the activation's traffic.
// NC counts the activation's chunks per lane; a row of codes has half (w4 a
// quarter) as many.
template <int BITS, int NC>
__global__ void __launch_bounds__(kThreads)
i8_quantize_both_kernel(const void* w, const uint16_t* scales, const uint16_t* qbias, int gshift,
                        int gcols, int8_t* wq, float* sw, int N, const uint16_t* x, int8_t* xq,
                        float* sx, int M, int K)
{
  const int n = wave_row();
  if (n < N) {
    if constexpr (BITS == 16) {
      quantize_row<NC>((const uint16_t*)w, wq, sw, n, K);
    } else {
      constexpr int kC = NC * BITS / 16 > 2 ? NC * BITS / 16 : 2;
      quantize_qrow<BITS, kC>((const uint8_t*)w, scales, qbias, gshift, gcols, wq, sw, n, K);
    }
  } else if (n - N < M) {
    quantize_row<NC>(x, xq, sx, n - N, K);
  }
}

// go(integral_constant): the smallest instance whose lanes hold a row of
// `chunks` 16-byte chunks, or the largest
template <typename F>
void with_chunks(int chunks, F&& go)
{
  const int per_lane = (chunks + 63) / 64;
  if (per_lane <= 2) {
    go(std::integral_constant<int, 2>{});
  } else if (per_lane <= 4) {
    go(std::integral_constant<int, 4>{});
  } else if (per_lane <= 8) {
    go(std::integral_constant<int, 8>{});
  } else {
    go(std::integral_constant<int, kMaxChunks>{});
  }
}

int ilog2(int v)
{
  int s = 0;
  while ((1 << s) < v) { ++s; }
  return s;
}

}  // namespace

hipError_t launch_i8_quantize_rows(const uint16_t* x, int8_t* q, float* s,
                                   int M, int K, hipStream_t stream)
{
  const dim3 grid((unsigned)((M + kRowsPerBlock - 1) / kRowsPerBlock));
  with_chunks(K / 8, [&](auto nc) {
    hipLaunchKernelGGL((i8_quantize_rows_kernel<decltype(nc)::value>), grid, dim3(kThreads), 0,
                       stream, x, q, s, M, K);
  });
  return hipGetLastError();
}

hipError_t launch_i8_quantize_qweight(const void* codes,
                                      const uint16_t* scales,
                                      const uint16_t* qbias, int bits,
                                      int group, int8_t* q, float* s, int N,
                                      int K, hipStream_t stream)
{
  const int gshift = ilog2(group);
  const int gcols = K / group;
  const dim3 grid((unsigned)((N + kRowsPerBlock - 1) / kRowsPerBlock));
  with_chunks(K / (128 / bits), [&](auto nc) {
    constexpr int NC = decltype(nc)::value;
    if (bits == 8) {
      hipLaunchKernelGGL((i8_quantize_qweight_kernel<8, NC>), grid, dim3(kThreads), 0, stream,
                         (const uint8_t*)codes, scales, qbias, gshift, gcols, q, s, N, K);
    } else {
      hipLaunchKernelGGL((i8_quantize_qweight_kernel<4, NC>), grid, dim3(kThreads), 0, stream,
                         (const uint8_t*)codes, scales, qbias, gshift, gcols, q, s, N, K);
    }
  });
  return hipGetLastError();
}

hipError_t launch_i8_quantize_both(const void* w, const uint16_t* scales, const uint16_t* qbias,
                                   int bits, int group, int8_t* wq, float* sw, int N,
                                   const uint16_t* x, int8_t* xq, float* sx, int M, int K,
                                   hipStream_t stream)
{
  const int gshift = bits == 16 ? 0 : ilog2(group);
  const int gcols = bits == 16 ? 0 : K / group;
  const dim3 grid((unsigned)(((size_t)M + N + kRowsPerBlock - 1) / kRowsPerBlock));
  with_chunks(K / 8, [&](auto nc) {
    constexpr int NC = decltype(nc)::value;
    auto go = [&](auto kernel) {
      hipLaunchKernelGGL(kernel, grid, dim3(kThreads), 0, stream, w, scales, qbias, gshift, gcols,
                         wq, sw, N, x, xq, sx, M, K);
    };
    if (bits == 16) {
      go(i8_quantize_both_kernel<16, NC>);
    } else if (bits == 8) {
      go(i8_quantize_both_kernel<8, NC>);
    } else {
      go(i8_quantize_both_kernel<4, NC>);
    }
  });
  return hipGetLastError();
}

}  // namespace ltx25
