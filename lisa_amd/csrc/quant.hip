// Dequantize and quantize kernels (gfx950).
#include "lisaq_common.h"
#include "kernels.h"

namespace lisaq {

// affine_dequantize (quantized.metal:2735-2794; host form array_ops.rs:55-83):
// out = scale*q + bias, one rounding to bf16.  scale*q is exact in f32 (8-bit
// by <=8-bit significands), so this equals the host's (q*s)+b then cast.
template <int BITS>
__global__ __launch_bounds__(256) void dequant_kernel(const uint32_t* __restrict__ w,
                                                      const uint16_t* __restrict__ s,
                                                      const uint16_t* __restrict__ b,
                                                      uint16_t* __restrict__ out, int64_t words,
                                                      int64_t kq, int G, int gs) {
  constexpr int PACK = 32 / BITS;
  const int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x;
  if (i >= words) return;
  const int64_t r = i / kq;
  const int64_t c0 = (i - r * kq) * PACK;  // first K index of this word
  const int64_t g = r * G + c0 / gs;       // a word never straddles a group (gs % pack == 0)
  const float sc = bf2f(s[g]), bs = bf2f(b[g]);
  const uint32_t v = w[i];
  uint32_t o[PACK / 2];
#pragma unroll
  for (int e = 0; e < PACK / 2; ++e) {
    const float q0 = (float)((v >> (BITS * (2 * e))) & ((1u << BITS) - 1u));
    const float q1 = (float)((v >> (BITS * (2 * e + 1))) & ((1u << BITS) - 1u));
    o[e] = pack_bf2(fmaf(q0, sc, bs), fmaf(q1, sc, bs));
  }
  uint32_t* dst = reinterpret_cast<uint32_t*>(out + r * (kq * PACK) + c0);
  if constexpr (PACK == 4) {
    *reinterpret_cast<u32x2*>(dst) = u32x2{o[0], o[1]};
  } else if constexpr (PACK == 8) {
    *reinterpret_cast<u32x4*>(dst) = u32x4{o[0], o[1], o[2], o[3]};
  } else {
#pragma unroll
    for (int e = 0; e < PACK / 2; e += 4)
      *reinterpret_cast<u32x4*>(dst + e) = u32x4{o[e], o[e + 1], o[e + 2], o[e + 3]};
  }
}

int launch_dequantize(hipStream_t st, const uint32_t* w, const uint16_t* s, const uint16_t* b,
                      uint16_t* out, int64_t rows, int64_t K, int gs, int bits) {
  const int64_t kq = K * bits / 32;
  const int64_t words = rows * kq;
  if (words == 0) return LISAQ_OK;
  const int64_t blocks = (words + 255) / 256;
  if (bits == 4)
    hipLaunchKernelGGL(dequant_kernel<4>, dim3((unsigned)blocks), dim3(256), 0, st, w, s, b, out, words,
                       kq, (int)(K / gs), gs);
  else if (bits == 2)
    hipLaunchKernelGGL(dequant_kernel<2>, dim3((unsigned)blocks), dim3(256), 0, st, w, s, b, out, words,
                       kq, (int)(K / gs), gs);
  else if (bits == 8)
    hipLaunchKernelGGL(dequant_kernel<8>, dim3((unsigned)blocks), dim3(256), 0, st, w, s, b, out, words,
                       kq, (int)(K / gs), gs);
  else
    return set_error(LISAQ_EUNSUPPORTED, "dequantize: bits=%d not supported", bits);
  return check_launch("dequantize");
}

// ops::quantize (array_ops.rs:218-290), one thread per group.  Same f32
// operation sequence as the host loop, so codes, scales and biases are
// bit-identical to it (IEEE division, roundf = half away from zero).
template <typename T>
__device__ __forceinline__ float load_as_f32(const T* p, int64_t i);
template <>
__device__ __forceinline__ float load_as_f32<uint16_t>(const uint16_t* p, int64_t i) { return bf2f(p[i]); }
template <>
__device__ __forceinline__ float load_as_f32<float>(const float* p, int64_t i) { return p[i]; }

template <typename T>
__device__ __forceinline__ void store_from_f32(T* p, int64_t i, float v);
template <>
__device__ __forceinline__ void store_from_f32<uint16_t>(uint16_t* p, int64_t i, float v) { p[i] = f2bf(v); }
template <>
__device__ __forceinline__ void store_from_f32<float>(float* p, int64_t i, float v) { p[i] = v; }

template <typename T>
__global__ __launch_bounds__(256) void quant_kernel(const T* __restrict__ w, uint32_t* __restrict__ wq,
                                                    T* __restrict__ scales, T* __restrict__ biases,
                                                    int64_t ngroups, int gs, int bits) {
  const int64_t gid = blockIdx.x * (int64_t)blockDim.x + threadIdx.x;
  if (gid >= ngroups) return;
  const int64_t base = gid * gs;
  const float maxq = (float)((1u << bits) - 1u);
  float w_min = 3.40282347e38f, w_max = 0.0f;
  for (int i = 0; i < gs; ++i) {
    const float v = load_as_f32(w, base + i);
    w_min = fminf(w_min, v);
    w_max = fmaxf(w_max, v);
  }
  float scale = fmaxf(__fdiv_rn(w_max - w_min, maxq), 1e-7f);
  const bool side = fabsf(w_min) > fabsf(w_max);
  if (!side) scale = -scale;
  const float edge = side ? w_min : w_max;
  const float q0 = roundf(__fdiv_rn(edge, scale));
  const bool at_zero = q0 == 0.0f;
  if (!at_zero) scale = __fdiv_rn(edge, q0);
  const float bias = at_zero ? 0.0f : edge;
  store_from_f32(scales, gid, scale);
  store_from_f32(biases, gid, bias);
  const int pack = 32 / bits;
  const uint32_t mask = (1u << bits) - 1u;
  uint32_t* dst = wq + base / pack;
  for (int i0 = 0; i0 < gs; i0 += pack) {
    uint32_t word = 0;
    for (int e = 0; e < pack; ++e) {
      const float qf = fminf(roundf(__fdiv_rn(__fsub_rn(load_as_f32(w, base + i0 + e), bias), scale)), maxq);
      const int32_t q = (int32_t)qf;
      word |= ((uint32_t)q & mask) << (e * bits);
    }
    dst[i0 / pack] = word;
  }
}

// The same rule with 16 consecutive values per thread: GS / 16 neighbouring lanes
// own a group, so a wave reads 2 KB (bf16) of consecutive values and stores
// consecutive code words, and the group's range is two DPP reductions (minimum
// and maximum are exact in any order).  One thread per group reads 2 bytes at
// a stride of a whole group: every load touched 64 cache lines, and 9728 x 2560
// bf16 -> 4 bits took 950 us for 64 MB; here 17 us (3.7 TB/s).
//
// Codes: roundf(d), d = fl(a / s) with a = fl(v - bias) and, signs taken out, s > 0:
// without the IEEE division (~10 operations per value, and bf16 values meet
// halves often).  k = floor(a * fl(1 / s)) is the integer below d or, within the
// product's error of an integer, its neighbour; either way roundf(d) is k + 1 if
// d >= h and k if not, h = k + 1/2.  d >= h exactly where a / s >= h - g / 2, g the
// gap below h in f32 (the midpoint rounds to h, whose mantissa is even), i.e.
// (a - h s) + (g / 2) s >= 0.  Near a half a - h s is a multiple of ulp(s) / 2
// below 2^10 of them (h < 2^9 is a multiple of 1/2), so its fma is exact, and the
// second fma's rounding keeps the sum's sign.  A NaN stays one up to the minimum,
// which gives the largest code as roundf's path does.  Infinities and scales far
// from 1 divide.
template <int CTRL>
__device__ __forceinline__ float dpp_f32(float v) {
  return __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), CTRL, 0xF, 0xF, false));
}

constexpr int kQuantVals = 16;

template <typename T, int BITS, int GS>
__global__ __launch_bounds__(256) void quant16_kernel(const T* __restrict__ w, uint32_t* __restrict__ wq,
                                                      T* __restrict__ scales, T* __restrict__ biases,
                                                      int64_t nchunks) {
  constexpr int V = kQuantVals, L = GS / V;  // values per thread; lanes per group: 2, 4 or 8 of a 16-lane DPP row
  const int64_t c = blockIdx.x * (int64_t)blockDim.x + threadIdx.x;
  // (a group's chunks are all inside or all outside the matrix)
  if (c >= nchunks) return;
  float v[V];
  if constexpr (sizeof(T) == 2) {
#pragma unroll
    for (int i = 0; i < V / 8; ++i) {
      const u32x4 a = *reinterpret_cast<const u32x4*>(w + c * V + 8 * i);
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        v[8 * i + 2 * j] = bf2f_lo(a[j]);
        v[8 * i + 2 * j + 1] = bf2f_hi(a[j]);
      }
    }
  } else {
#pragma unroll
    for (int i = 0; i < V / 4; ++i) {
      const f32x4 a = *reinterpret_cast<const f32x4*>(w + c * V + 4 * i);
#pragma unroll
      for (int j = 0; j < 4; ++j) v[4 * i + j] = a[j];
    }
  }
  constexpr float maxq = (float)((1u << BITS) - 1u);
  float w_min = 3.40282347e38f, w_max = 0.0f;
#pragma unroll
  for (int j = 0; j < V; ++j) {
    w_min = fminf(w_min, v[j]);
    w_max = fmaxf(w_max, v[j]);
  }
  w_min = fminf(w_min, dpp_f32<0xB1>(w_min));  // lane ^ 1
  w_max = fmaxf(w_max, dpp_f32<0xB1>(w_max));
  if constexpr (L >= 4) {
    w_min = fminf(w_min, dpp_f32<0x4E>(w_min));  // lane ^ 2
    w_max = fmaxf(w_max, dpp_f32<0x4E>(w_max));
  }
  if constexpr (L >= 8) {
    w_min = fminf(w_min, dpp_f32<0x141>(w_min));  // mirrored half rows: the other four of eight
    w_max = fmaxf(w_max, dpp_f32<0x141>(w_max));
  }
  float scale = fmaxf(__fdiv_rn(w_max - w_min, maxq), 1e-7f);
  const bool side = fabsf(w_min) > fabsf(w_max);
  if (!side) scale = -scale;
  const float edge = side ? w_min : w_max;
  const float q0 = roundf(__fdiv_rn(edge, scale));
  const bool at_zero = q0 == 0.0f;
  if (!at_zero) scale = __fdiv_rn(edge, q0);
  const float bias = at_zero ? 0.0f : edge;
  const float sa = fabsf(scale), sg = scale < 0.0f ? -1.0f : 1.0f;
  const float r = __fdiv_rn(1.0f, sa), sb = -bias * sg, g2 = sa * 5.9604645e-8f;  // (2^-24 s)
  const bool sure = sa < 1e30f && sa > 1e-30f && fabsf(w_min) < 1e30f && w_max < 1e30f;
  float q[V];
#pragma unroll
  for (int j = 0; j < V; ++j) {
    const float a = fmaf(v[j], sg, sb);
    const float h = floorf(a * r) + 0.5f;
    // 2^p with p the exponent of the value below |h|: g / 2 = 2^p 2^-24
    const float e2p = __uint_as_float((__float_as_uint(h) - 1u) & 0x7F800000u);
    const float e = fmaf(e2p, g2, fmaf(-h, sa, a));
    q[j] = fminf(h + __builtin_copysignf(0.5f, e), maxq);
  }
  constexpr int NW = V * BITS / 32, CPH = 16 / BITS;  // words; codes per half word
  uint32_t o[NW];
  if (__all(sure)) {
    // half words as sums of powers (exact in f32), one conversion each
#pragma unroll
    for (int i = 0; i < NW; ++i) {
      uint32_t hw[2];
#pragma unroll
      for (int h = 0; h < 2; ++h) {
        const float* qq = q + (2 * i + h) * CPH;
        float t = qq[CPH - 1];
#pragma unroll
        for (int e = CPH - 2; e >= 0; --e) t = fmaf(t, (float)(1u << BITS), qq[e]);
        hw[h] = (uint32_t)t;
      }
      o[i] = hw[0] | (hw[1] << 16);
    }
  } else {
#pragma unroll
    for (int i = 0; i < NW; ++i) {
      o[i] = 0;
#pragma unroll
      for (int e = 0; e < 2 * CPH; ++e) {
        const float qf = fminf(roundf(__fdiv_rn(__fsub_rn(v[2 * CPH * i + e], bias), scale)), maxq);
        o[i] |= ((uint32_t)(int32_t)qf & ((1u << BITS) - 1u)) << (e * BITS);
      }
    }
  }
  if constexpr (NW == 4) *reinterpret_cast<u32x4*>(wq + c * 4) = u32x4{o[0], o[1], o[2], o[3]};
  else if constexpr (NW == 2) *reinterpret_cast<u32x2*>(wq + c * 2) = u32x2{o[0], o[1]};
  else wq[c] = o[0];
  if (c % L == 0) {
    store_from_f32(scales, c / L, scale);
    store_from_f32(biases, c / L, bias);
  }
}

template <typename T, int BITS>
static void launch_quant16(hipStream_t st, const T* w, uint32_t* wq, T* s, T* b, int64_t nchunks, int gs) {
  const dim3 grid((unsigned)((nchunks + 255) / 256));
  if (gs == 32) hipLaunchKernelGGL((quant16_kernel<T, BITS, 32>), grid, dim3(256), 0, st, w, wq, s, b, nchunks);
  else if (gs == 64) hipLaunchKernelGGL((quant16_kernel<T, BITS, 64>), grid, dim3(256), 0, st, w, wq, s, b, nchunks);
  else hipLaunchKernelGGL((quant16_kernel<T, BITS, 128>), grid, dim3(256), 0, st, w, wq, s, b, nchunks);
}

template <typename T>
static int launch_quantize_t(hipStream_t st, const T* w, uint32_t* wq, T* s, T* b, int64_t rows, int64_t K, int gs,
                             int bits) {
  const int64_t ngroups = rows * (K / gs);
  if (ngroups == 0) return LISAQ_OK;
  // sixteen values per thread where the group sizes and alignments of the packed
  // format's layers allow its loads and stores; anything else a thread per group
  const bool al = (uintptr_t)w % 16 == 0 && (uintptr_t)wq % 16 == 0;
  if (al && (gs == 32 || gs == 64 || gs == 128) && ngroups * gs / kQuantVals <= (int64_t)1 << 38) {
    const int64_t nchunks = ngroups * gs / kQuantVals;
    if (bits == 4) launch_quant16<T, 4>(st, w, wq, s, b, nchunks, gs);
    else if (bits == 2) launch_quant16<T, 2>(st, w, wq, s, b, nchunks, gs);
    else launch_quant16<T, 8>(st, w, wq, s, b, nchunks, gs);
    return check_launch("quantize");
  }
  hipLaunchKernelGGL(quant_kernel<T>, dim3((unsigned)((ngroups + 255) / 256)), dim3(256), 0, st, w, wq, s, b, ngroups,
                     gs, bits);
  return check_launch("quantize");
}

int launch_quantize(hipStream_t st, const void* w, int dtype, uint32_t* wq, void* s, void* b,
                    int64_t rows, int64_t K, int gs, int bits) {
  if (dtype == LISAQ_DTYPE_BF16)
    return launch_quantize_t(st, (const uint16_t*)w, wq, (uint16_t*)s, (uint16_t*)b, rows, K, gs, bits);
  return launch_quantize_t(st, (const float*)w, wq, (float*)s, (float*)b, rows, K, gs, bits);
}

}  // namespace lisaq
