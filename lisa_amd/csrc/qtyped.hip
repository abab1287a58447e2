// Quantized matmul for the compute dtypes and code widths outside the tuned
// bf16 2/4-bit kernels: x, scales, biases and y in bf16, f16 or f32 (the
// reference promotes all four to one dtype, ops/array_ops.rs:398-404) and
// 2-, 4- or 8-bit codes.
//
// Arithmetic contract, per the reference's templates on T:
//  * matvec (M < qmv_batch_limit; quantized.metal qmv_fast / qmv_wide,
//    :767-830, 996-1088): f32 throughout -- per 32-code chunk of one group,
//    y += scale * sum(x * q) + bias * sum(x), weights never rounded; y
//    rounded to T once;
//  * matmul (larger M; quantized.metal:1208-1326 with the block loader
//    :585-703): every weight dequantized to T, w = T(scale * q + bias) from an
//    f32 fma, then y = x . w^T with f32 accumulation, rounded to T once.
//
// Kernels: for the matvec x in LDS and several output rows per wave (a wave per
// output row for unaligned x or W).  For the matmul, of the problems that the
// bf16 2/4-bit matmul's kernel does not take in their type (f32, rows of an odd
// number of groups, addresses off its alignment): the matrix cores in bf16, f16
// or f32, and 64 x 64 register-tiled f32 FMA for an x off 16 bytes.
#include "lisaq_common.h"
#include "qmv.h"
#include "qmv_dev.h"
#include <utility>

namespace lisaq {

namespace {

// DT: 0 bf16, 1 f32, 2 f16 (the lisaq_dtype values)
template <int DT>
__device__ __forceinline__ float ld(const void* p, int64_t i) {
  if constexpr (DT == 0) return bf2f(static_cast<const uint16_t*>(p)[i]);
  else if constexpr (DT == 1) return static_cast<const float*>(p)[i];
  else return (float)static_cast<const _Float16*>(p)[i];
}
// float -> T (round to nearest even) -> float
template <int DT>
__device__ __forceinline__ float rnd(float v) {
  if constexpr (DT == 0) return bf2f(f2bf(v));
  else if constexpr (DT == 1) return v;
  else return (float)(_Float16)v;
}
template <int DT>
__device__ __forceinline__ void st(void* p, int64_t i, float v) {
  if constexpr (DT == 0) static_cast<uint16_t*>(p)[i] = f2bf(v);
  else if constexpr (DT == 1) static_cast<float*>(p)[i] = v;
  else static_cast<_Float16*>(p)[i] = (_Float16)v;
}

// code ci of a packed row (little-endian codes within each u32)
template <int BITS>
__device__ __forceinline__ uint32_t code(const uint32_t* row, int ci) {
  constexpr int PACK = 32 / BITS;
  return (row[ci / PACK] >> (BITS * (ci % PACK))) & ((1u << BITS) - 1u);
}

__device__ __forceinline__ float wsum64(float v) {
#pragma unroll
  for (int o = 32; o >= 1; o >>= 1) v += __shfl_xor(v, o);
  return v;
}

// Matvec: a wave per output row n; lane l takes the 32-code chunks l, l+64,
// ...; the rows of x in groups of MB.
template <int DT, int BITS, int GS>
__global__ __launch_bounds__(256) void qmv_typed_kernel(const void* x, const uint32_t* w, const void* s,
                                                        const void* b, void* y, int M, int N, int K) {
  constexpr int MB = 4;
  constexpr int WPC = BITS;  // u32 words per 32-code chunk
  const int lane = threadIdx.x & 63;
  const int n = blockIdx.x * 4 + (threadIdx.x >> 6);
  if (n >= N) return;
  const int C = K / 32, G = K / GS;
  const uint32_t* wrow = w + (int64_t)n * (K / (32 / BITS));
  for (int m0 = 0; m0 < M; m0 += MB) {
    float part[MB];
#pragma unroll
    for (int r = 0; r < MB; ++r) part[r] = 0.f;
    for (int c = lane; c < C; c += 64) {
      uint32_t wv[WPC];
#pragma unroll
      for (int i = 0; i < WPC; ++i) wv[i] = wrow[c * WPC + i];
      const int g = c * 32 / GS;
      const float sc = ld<DT>(s, (int64_t)n * G + g), bi = ld<DT>(b, (int64_t)n * G + g);
#pragma unroll
      for (int r = 0; r < MB; ++r) {
        const int m = m0 + r;
        if (m >= M) break;
        float dot = 0.f, xs = 0.f;
#pragma unroll
        for (int j = 0; j < 32; ++j) {
          const float xv = ld<DT>(x, (int64_t)m * K + c * 32 + j);
          const float q = (float)((wv[j / (32 / BITS)] >> (BITS * (j % (32 / BITS)))) & ((1u << BITS) - 1u));
          dot = fmaf(xv, q, dot);
          xs += xv;
        }
        part[r] = fmaf(sc, dot, fmaf(bi, xs, part[r]));
      }
    }
#pragma unroll
    for (int r = 0; r < MB; ++r) {
      const float t = wsum64(part[r]);
      if (lane == 0 && m0 + r < M) st<DT>(y, (int64_t)(m0 + r) * N + n, t);
    }
  }
}

// Matvec with x in LDS and several rows of W per wave: the kernel for x and W
// 16-byte aligned.  A lane takes pieces lane, lane + 64, ... of a row -- a piece
// is one load, 16 codes of 8 bits, 32 of 4 or 2 -- of RW rows at a time; each
// value of x read from LDS and each conversion of a code serve RW rows and MR
// rows of x.  Codes become f32 by v_cvt_f32_ubyte, and per piece (inside one group)
//   y += scale * sum(x * q) + bias * sum(x),
// all in f32, sum(x) of a piece once per workgroup.
// Two steps of loads are in flight over the wave's whole stream of rows, the
// first ones across the barriers of the staging of x (LDS only).  They are
// unconditional: behind a branch the compiler waits for every load in flight
// before each step (f16 8-bit 1000 x 8192 one row 5.4 -> 7.4 us; four or eight
// steps in flight, whose loads wait in line before the first: 5.5 / 6.5).
// What bounds it: one row of x, the stream of W; from two rows on VALU issue
// (per code ~(4.9 + 2.5 MR) cycles of a SIMD).  us: bf16 8-bit 9728 x 2560 1 row
// 5.9 (4.4 TB/s); 2560 x 9728 1 row 8.1, 2 rows 11.3; f16 8-bit 17408 x 5120 1
// row 19, 12 rows 70; 5120 x 17408 12 rows 90; f32 4-bit 17408 x 5120 1 row 17.
// x in LDS: planes of 16 bytes, plane q of every piece side by side (a wave's
// reads of a plane are contiguous), then the sums.
template <int DT, int BITS>
struct Piece {
  static constexpr int P = BITS == 8 ? 16 : 32;      // codes
  static constexpr int WORDS = P * BITS / 32;        // u32 words: 4, 4 or 2
  static constexpr int V = DT == 1 ? 4 : 8;          // values of x per 16-byte plane
  static constexpr int PL = P / V;                   // planes
  static constexpr int SZ = DT == 1 ? 4 : 2;         // bytes of a value
};

// codes V q .. V q + V - 1 of a piece as f32
template <int BITS, int V, int q>
__device__ __forceinline__ void piece_codes(const uint32_t* w, float* o) {
#pragma unroll
  for (int j = 0; j < V; ++j) {
    const int i = V * q + j;  // (compile-time after unrolling)
    if constexpr (BITS == 8) o[j] = (float)((w[i / 4] >> (8 * (i % 4))) & 0xFFu);
    else if constexpr (BITS == 4) o[j] = (float)((((w[i / 8] >> (4 * (i & 1))) & 0x0F0F0F0Fu) >> (8 * (i % 8 / 2))) & 0xFFu);
    else o[j] = (float)((((w[i / 16] >> (2 * (i & 3))) & 0x03030303u) >> (8 * (i % 16 / 4))) & 0xFFu);
  }
}

template <typename F, int... Q>
__device__ __forceinline__ void for_planes(F&& f, std::integer_sequence<int, Q...>) {
  (f(std::integral_constant<int, Q>{}), ...);
}

// Workgroup barrier over LDS only: loads from global memory stay in flight.
__device__ __forceinline__ void lds_barrier() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup", "local");
  __builtin_amdgcn_s_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");
}

template <int DT, int BITS, int GS, int MR, int RW>
__global__ __launch_bounds__(256) void qmv_typed_rows_kernel(const void* x, const uint32_t* w, const void* s,
                                                             const void* b, void* y, int M, int N, int K) {
  using Pc = Piece<DT, BITS>;
  typedef uint32_t wv_t __attribute__((ext_vector_type(Pc::WORDS)));
  constexpr int D = 2;
  extern __shared__ __attribute__((aligned(16))) unsigned char xsm[];
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int C = K / Pc::P, G = K / GS;
  const int64_t wstride = K / (32 / BITS);
  const int m0 = blockIdx.y * MR, mr = M - m0 < MR ? M - m0 : MR;
  float* const xsum = reinterpret_cast<float*>(xsm + (size_t)MR * K * Pc::SZ);  // [MR][C]
  // the wave's stream: steps 0 .. S - 1 of rows n0, of rows n0 + stride, ...; loads
  // are unconditional (clamped past a row's pieces and past the last row), so
  // that the waits count them
  struct Row {
    wv_t w[RW];
    float s[RW], b[RW];
  };
  const int S = (C + 63) / 64, stride = gridDim.x * 4 * RW;
  int ln = (blockIdx.x * 4 + wave) * RW, lt = 0;  // next step to load: rows, step
  // (wave-uniform bases: a load then has one 32-bit offset per lane)
  const uint32_t* wp[RW];
  const unsigned char *sp[RW], *bp[RW];
  auto set_rows = [&]() {
#pragma unroll
    for (int r = 0; r < RW; ++r) {
      const int64_t n = ln + r < N ? ln + r : N - 1;
      wp[r] = w + n * wstride;
      sp[r] = static_cast<const unsigned char*>(s) + n * G * Pc::SZ;
      bp[r] = static_cast<const unsigned char*>(b) + n * G * Pc::SZ;
    }
  };
  set_rows();
  auto load = [&](Row& o) {
    const int c = lt * 64 + lane, cc = c < C ? c : C - 1, g = cc * Pc::P / GS;
#pragma unroll
    for (int r = 0; r < RW; ++r) {
      o.w[r] = reinterpret_cast<const wv_t*>(wp[r])[cc];
      o.s[r] = ld<DT>(sp[r], g);
      o.b[r] = ld<DT>(bp[r], g);
    }
    if (++lt == S) {
      lt = 0;
      if (ln < N) ln += stride;
      set_rows();
    }
  };
  int n0 = ln, t = 0;
  Row ring[D];

  // x to LDS, U units per thread and turn with their loads together, then the
  // ring's first loads (rows past M: copies of the last, never stored)
  constexpr int U = MR >= 4 ? 1 : 4 / MR;
  const int units = C * Pc::PL;
  for (int e0 = tid; e0 < units; e0 += 256 * U) {
    u32x4 v[U][MR];
#pragma unroll
    for (int u = 0; u < U; ++u)
#pragma unroll
      for (int m = 0; m < MR; ++m)
        v[u][m] = reinterpret_cast<const u32x4*>(static_cast<const unsigned char*>(x) +
                                                 (int64_t)(m0 + (m < mr ? m : mr - 1)) * K * Pc::SZ)
            [e0 + 256 * u < units ? e0 + 256 * u : units - 1];
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const int e = e0 + 256 * u;
      if (e >= units) break;
#pragma unroll
      for (int m = 0; m < MR; ++m)
        reinterpret_cast<u32x4*>(xsm + (size_t)m * K * Pc::SZ)[(e % Pc::PL) * C + e / Pc::PL] = v[u][m];
    }
  }
#pragma unroll
  for (int i = 0; i < D; ++i) load(ring[i]);
  lds_barrier();
  // plane q of piece c of row m as f32
  auto plane = [&](int m, int q, int c, float* v) {
    const u32x4 a = reinterpret_cast<const u32x4*>(xsm + (size_t)m * K * Pc::SZ)[q * C + c];
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const uint32_t u = a[e];
      if constexpr (DT == 1) {
        v[e] = __uint_as_float(u);
      } else if constexpr (DT == 0) {
        v[2 * e] = __uint_as_float(u << 16);
        v[2 * e + 1] = __uint_as_float(u & 0xffff0000u);
      } else {
        v[2 * e] = (float)__builtin_bit_cast(_Float16, (uint16_t)(u & 0xffffu));
        v[2 * e + 1] = (float)__builtin_bit_cast(_Float16, (uint16_t)(u >> 16));
      }
    }
  };
  auto piece_sum = [&](int m, int c) {
    float sum = 0.f;
#pragma unroll
    for (int q = 0; q < Pc::PL; ++q) {
      float v[Pc::V];
      plane(m, q, c, v);
#pragma unroll
      for (int e = 0; e < Pc::V; ++e) sum += v[e];
    }
    return sum;
  };
  for (int i = tid; i < MR * C; i += 256) xsum[i] = piece_sum(i / C, i % C);
  lds_barrier();

  float part[RW][MR] = {};
  auto piece = [&](int c, const Row& o) {
    if (c >= C) return;
    float dot[RW][MR] = {};
    auto one = [&](auto qi) {
      constexpr int q = decltype(qi)::value;
      float xv[MR][Pc::V];
#pragma unroll
      for (int m = 0; m < MR; ++m) plane(m, q, c, xv[m]);
#pragma unroll
      for (int r = 0; r < RW; ++r) {
        uint32_t wd[Pc::WORDS];
#pragma unroll
        for (int e = 0; e < Pc::WORDS; ++e) wd[e] = o.w[r][e];
        float cv[Pc::V];
        piece_codes<BITS, Pc::V, q>(wd, cv);
#pragma unroll
        for (int e = 0; e < Pc::V; ++e)
#pragma unroll
          for (int m = 0; m < MR; ++m) dot[r][m] = fmaf(xv[m][e], cv[e], dot[r][m]);
      }
    };
    for_planes(one, std::make_integer_sequence<int, Pc::PL>{});
#pragma unroll
    for (int m = 0; m < MR; ++m) {
      const float xs = xsum[m * C + c];
#pragma unroll
      for (int r = 0; r < RW; ++r) part[r][m] = fmaf(o.s[r], dot[r][m], fmaf(o.b[r], xs, part[r][m]));
    }
  };
  // rows n0 .. done: their sums over the wave, stored, and the next rows
  auto finish = [&]() {
    float out = 0.f;
#pragma unroll
    for (int r = 0; r < RW; ++r)
#pragma unroll
      for (int m = 0; m < MR; ++m) {
        const float v = qmvdev::wave_sum(part[r][m]);
        out = lane == r * MR + m ? v : out;
        part[r][m] = 0.f;
      }
    const int r = lane / MR, m = lane % MR;
    if (lane < RW * MR && n0 + r < N && m < mr) st<DT>(y, (int64_t)(m0 + m) * N + n0 + r, out);
    t = 0;
    n0 += stride;
  };
  while (n0 < N) {
#pragma unroll
    for (int i = 0; i < D; ++i) {
      if (n0 < N) {  // (wave-uniform)
        piece(t * 64 + lane, ring[i]);
        if (++t == S) finish();
      }
      load(ring[i]);
    }
  }
}

// One row of f16 x and 4-bit codes of at most 4096 rows: a wave per output row on
// dot instructions, x from global memory (cached).  A code becomes the f16
// 1024 + q (bits 0x6400 | q), and q itself by a packed subtraction, both exact, so
// v_dot2_f32_f16 takes the pairs (q_j, q_j+4) of a word against (x_j, x_j+4);
// sum(x) of a piece by dots against (1, 1).  Short streams that the kernel
// above starts too late, staging x first (us, there / here): 2560 x 9728 8.4 /
// 7.1, 300 x 512 3.5 / 3.1, 1000 x 8192 4.9 / 4.8; 17408 x 5120 17.4 / 18.6.
typedef _Float16 f16x2 __attribute__((ext_vector_type(2)));

template <int GS>
__global__ __launch_bounds__(256) void qmv_f16_dot_kernel(const void* x, const uint32_t* w, const void* s,
                                                          const void* b, void* y, int M, int N, int K) {
  const int lane = threadIdx.x & 63;
  const int n = blockIdx.x * 4 + (threadIdx.x >> 6);
  if (n >= N) return;
  const int C = K / 32, G = K / GS;
  const uint32_t* wrow = w + (int64_t)n * (K / 8);
  const u32x4* xq = static_cast<const u32x4*>(x);
  const f16x2 k1024 = {(_Float16)1024.f, (_Float16)1024.f}, one = {(_Float16)1.f, (_Float16)1.f};
  float part = 0.f;
  for (int c = lane; c < C; c += 64) {
    const u32x4 wv = *reinterpret_cast<const u32x4*>(wrow + c * 4);
    const int g = c * 32 / GS;
    const float sc = ld<2>(s, (int64_t)n * G + g), bi = ld<2>(b, (int64_t)n * G + g);
    float dot = 0.f, xs = 0.f;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const u32x4 v = xq[c * 4 + i];  // values 32 c + 8 i .. + 7
      const uint32_t pr[4] = {__builtin_amdgcn_perm(v[2], v[0], 0x05040100u), __builtin_amdgcn_perm(v[2], v[0], 0x07060302u),
                              __builtin_amdgcn_perm(v[3], v[1], 0x05040100u), __builtin_amdgcn_perm(v[3], v[1], 0x07060302u)};
      const uint32_t wd = wv[i];
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const uint32_t q = ((wd >> (4 * j)) & 0x000F000Fu) | 0x64006400u;
        const f16x2 xp = __builtin_bit_cast(f16x2, pr[j]);
        dot = __builtin_amdgcn_fdot2(xp, __builtin_bit_cast(f16x2, q) - k1024, dot, false);
        xs = __builtin_amdgcn_fdot2(xp, one, xs, false);
      }
    }
    part = fmaf(sc, dot, fmaf(bi, xs, part));
  }
  const float t = wsum64(part);
  if (lane == 0) st<2>(y, n, t);
}

// Matmul: 64 x 64 output tile per workgroup, K in steps of 32 through LDS (x
// and the dequantized, T-rounded weights, both as f32), 4 x 4 outputs per
// thread.
template <int DT, int BITS, int GS>
__global__ __launch_bounds__(256) void qmm_typed_kernel(const void* x, const uint32_t* w, const void* s,
                                                        const void* b, void* y, int M, int N, int K) {
  constexpr int BM = 64, BN = 64, BK = 32, PAD = 4;
  __shared__ float xs[BK][BM + PAD];
  __shared__ float wt[BK][BN + PAD];
  const int tid = threadIdx.x, tx = tid % 16, ty = tid / 16;
  const int m0 = blockIdx.y * BM, n0 = blockIdx.x * BN;
  const int G = K / GS;
  const int64_t wrow = K / (32 / BITS);
  float acc[4][4] = {};
  for (int k0 = 0; k0 < K; k0 += BK) {
#pragma unroll
    for (int i = 0; i < BM * BK / 256; ++i) {
      const int e = tid + 256 * i, r = e / BK, kk = e % BK;
      xs[kk][r] = m0 + r < M ? ld<DT>(x, (int64_t)(m0 + r) * K + k0 + kk) : 0.f;
    }
    {
      const int r = tid / 4, kq = (tid % 4) * 8;  // 8 codes of row n0 + r
      const int n = n0 + r;
      if (n < N) {
        const uint32_t* row = w + (int64_t)n * wrow;
        const int g = (k0 + kq) / GS;  // (8 consecutive codes lie in one group: GS >= 32)
        const float sc = ld<DT>(s, (int64_t)n * G + g), bi = ld<DT>(b, (int64_t)n * G + g);
#pragma unroll
        for (int j = 0; j < 8; ++j) wt[kq + j][r] = rnd<DT>(fmaf(sc, (float)code<BITS>(row, k0 + kq + j), bi));
      } else {
#pragma unroll
        for (int j = 0; j < 8; ++j) wt[kq + j][r] = 0.f;
      }
    }
    __syncthreads();
#pragma unroll 8
    for (int kk = 0; kk < BK; ++kk) {
      float a[4], c[4];
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        a[i] = xs[kk][ty * 4 + i];
        c[i] = wt[kk][tx * 4 + i];
      }
#pragma unroll
      for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int j = 0; j < 4; ++j) acc[i][j] = fmaf(a[i], c[j], acc[i][j]);
    }
    __syncthreads();
  }
#pragma unroll
  for (int i = 0; i < 4; ++i)
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const int m = m0 + ty * 4 + i, n = n0 + tx * 4 + j;
      if (m < M && n < N) st<DT>(y, (int64_t)m * N + n, acc[i][j]);
    }
}

// Matmul on the matrix cores for the 16-bit compute dtypes (bf16, f16): the
// same contract -- every weight T(fma(scale, q, bias)), f32 accumulation, one
// rounding -- with v_mfma_f32_16x16x32_{bf16,f16}.  64 x 64 output tile per
// workgroup of four waves (each 32 x 32: 2 x 2 matrix tiles), K in steps of
// 32: each thread stages 8 values of x and dequantizes 8 weights of one row
// into two LDS buffers (rows padded to 80 bytes: a quarter-wave's 16-byte
// fragment reads hit distinct banks), so one barrier per step; the next
// step's x and code words are loaded while the current step's matrix
// instructions run.  x must be 16-byte aligned (the host checks).
typedef _Float16 f16x8 __attribute__((ext_vector_type(8)));

template <int DT>
__device__ __forceinline__ uint16_t bits16(float v) {
  if constexpr (DT == 0) return f2bf(v);
  else return __builtin_bit_cast(uint16_t, (_Float16)v);
}

template <int DT, int BITS, int GS, int TB>
__global__ __launch_bounds__(256) void qmm_typed_mfma_kernel(const void* x, const uint32_t* w, const void* s,
                                                             const void* b, void* y, int M, int N, int K) {
  static_assert(DT == 0 || DT == 2, "16-bit compute dtypes");
  static_assert(TB == 1 || TB == 2, "tile scale");
  // TB: 64 TB x 64 TB output tile, each wave 32 TB x 32 TB (2 TB x 2 TB matrix tiles)
  constexpr int BM = 64 * TB, BN = 64 * TB, BK = 32, RS = 40;  // LDS row stride: 40 16-bit values (80 bytes)
  constexpr int FT = 2 * TB;                                   // matrix tiles per wave and side
  __shared__ __attribute__((aligned(16))) uint16_t xa[2][BM * RS];
  __shared__ __attribute__((aligned(16))) uint16_t wb[2][BN * RS];
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int wm = (wave >> 1) * 32 * TB, wn = (wave & 1) * 32 * TB;  // the wave's quarter
  const int m0 = blockIdx.y * BM, n0 = blockIdx.x * BN;
  const int G = K / GS;
  // staging role: rows sr + 64 t of the tile (t < TB), values 8 c8 .. 8 c8 + 7 of the step
  const int sr = tid >> 2, c8 = (tid & 3) * 8;
  bool xok[TB];
  int nr[TB];
  const uint16_t* xrow[TB];
  const uint32_t* wrow[TB];
#pragma unroll
  for (int t = 0; t < TB; ++t) {
    const int r = sr + 64 * t;
    xok[t] = m0 + r < M;
    nr[t] = n0 + r < N ? n0 + r : N - 1;  // (rows past N: never stored)
    xrow[t] = static_cast<const uint16_t*>(x) + (int64_t)(xok[t] ? m0 + r : 0) * K;
    wrow[t] = w + (int64_t)nr[t] * (K / (32 / BITS));
  }
  u32x4 xv[TB];
  uint32_t cw[TB][BITS == 8 ? 2 : 1];
  float sc[TB], bi[TB];
  auto fetch = [&](int k0) {
    const int k = k0 + c8;
    const int g = k / GS;  // (8 consecutive codes lie in one group: GS >= 32)
#pragma unroll
    for (int t = 0; t < TB; ++t) {
      xv[t] = xok[t] ? *reinterpret_cast<const u32x4*>(xrow[t] + k) : u32x4{0u, 0u, 0u, 0u};
      if constexpr (BITS == 8) {
        cw[t][0] = wrow[t][k / 4];
        cw[t][1] = wrow[t][k / 4 + 1];
      } else if constexpr (BITS == 4) {
        cw[t][0] = wrow[t][k / 8];
      } else {
        cw[t][0] = wrow[t][k / 16] >> (2 * (k % 16));
      }
      sc[t] = ld<DT>(s, (int64_t)nr[t] * G + g);
      bi[t] = ld<DT>(b, (int64_t)nr[t] * G + g);
    }
  };
  auto stage = [&](int buf) {
#pragma unroll
    for (int t = 0; t < TB; ++t) {
      const int r = sr + 64 * t;
      *reinterpret_cast<u32x4*>(&xa[buf][r * RS + c8]) = xv[t];
      uint32_t h[4];
#pragma unroll
      for (int j = 0; j < 8; j += 2) {
        uint32_t q0, q1;
        if constexpr (BITS == 8) {
          q0 = (cw[t][j / 4] >> (8 * (j % 4))) & 0xFFu;
          q1 = (cw[t][j / 4] >> (8 * (j % 4 + 1))) & 0xFFu;
        } else {
          q0 = (cw[t][0] >> (BITS * j)) & ((1u << BITS) - 1u);
          q1 = (cw[t][0] >> (BITS * (j + 1))) & ((1u << BITS) - 1u);
        }
        h[j / 2] = (uint32_t)bits16<DT>(fmaf(sc[t], (float)q0, bi[t])) |
                   ((uint32_t)bits16<DT>(fmaf(sc[t], (float)q1, bi[t])) << 16);
      }
      *reinterpret_cast<u32x4*>(&wb[buf][r * RS + c8]) = u32x4{h[0], h[1], h[2], h[3]};
    }
  };
  f32x4 acc[FT][FT];
#pragma unroll
  for (int i = 0; i < FT; ++i)
#pragma unroll
    for (int j = 0; j < FT; ++j) acc[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};
  // fragment reads: row (lane & 15) of a 16-row tile, k values 8 (lane >> 4) ..
  const int fr = lane & 15, fk = (lane >> 4) * 8;
  fetch(0);
  stage(0);
  __syncthreads();
  for (int k0 = 0, buf = 0; k0 < K; k0 += BK, buf ^= 1) {
    const bool more = k0 + BK < K;
    if (more) fetch(k0 + BK);
    u32x4 af[FT], bf[FT];
#pragma unroll
    for (int i = 0; i < FT; ++i) {
      af[i] = *reinterpret_cast<const u32x4*>(&xa[buf][(wm + 16 * i + fr) * RS + fk]);
      bf[i] = *reinterpret_cast<const u32x4*>(&wb[buf][(wn + 16 * i + fr) * RS + fk]);
    }
#pragma unroll
    for (int i = 0; i < FT; ++i)
#pragma unroll
      for (int j = 0; j < FT; ++j) {
        if constexpr (DT == 0)
          acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(as_bf16x8(af[i]), as_bf16x8(bf[j]), acc[i][j], 0, 0, 0);
        else
          acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(f16x8, af[i]),
                                                             __builtin_bit_cast(f16x8, bf[j]), acc[i][j], 0, 0, 0);
      }
    if (more) stage(buf ^ 1);  // (buffer buf ^ 1 was last read before the previous barrier)
    __syncthreads();
  }
  // output element (row 4 (lane >> 4) + e, column lane & 15) of each 16 x 16 tile
#pragma unroll
  for (int i = 0; i < FT; ++i)
#pragma unroll
    for (int j = 0; j < FT; ++j)
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const int m = m0 + wm + 16 * i + 4 * (lane >> 4) + e, n = n0 + wn + 16 * j + (lane & 15);
        if (m < M && n < N) st<DT>(y, (int64_t)m * N + n, acc[i][j][e]);
      }
}

typedef void (*typed_fn)(const void*, const uint32_t*, const void*, const void*, void*, int, int, int);

// f32 matmul on the matrix cores: the same contract (weights are the f32
// fma(scale, q, bias), f32 accumulation) with v_mfma_f32_32x32x2_f32, each of
// four waves a 32 x 32 tile of f32 products.  Two forms:
//  * KS = false: a 64 x 64 tile, the waves its quarters, K in steps of 32;
//  * KS = true (fewer such tiles than compute units): a 32 x 32
//    tile, K in steps of 128 of which each wave takes 32, the four sums added
//    through LDS in wave order.
// Bounded by the matrix cores (157 TFLOP/s; a step is sixteen of their 64-cycle
// instructions per wave, its loads for the next step in flight).  The 64 x 64
// FMA tiles it replaced left most of the chip idle at small sizes and read
// every operand from LDS per product: 4-bit 64 x 4096 x 4096 458 -> 40 us, 256 x
// 4096 x 4096 561 -> 100 (86 TFLOP/s).
// LDS rows padded by 16 bytes: the 32 rows of a read fall on distinct banks.
template <int BITS, int GS, bool KS>
__global__ __launch_bounds__(256) void qmm_f32_mfma_kernel(const void* xv, const uint32_t* w, const void* sv,
                                                           const void* bv, void* yv, int M, int N, int K) {
  constexpr int T = KS ? 32 : 64, BK = KS ? 128 : 32, RS = BK + 4;  // tile, K step, LDS row in floats
  constexpr int TPR = 256 / T, VPT = BK / TPR;                     // staging threads per row, values per thread
  const float* const x = static_cast<const float*>(xv);
  const float* const s = static_cast<const float*>(sv);
  const float* const b = static_cast<const float*>(bv);
  float* const y = static_cast<float*>(yv);
  __shared__ __attribute__((aligned(16))) float xa[2][T * RS], wb[2][T * RS];
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, half = lane >> 5, col = lane & 31;
  const int m0 = blockIdx.y * T, n0 = blockIdx.x * T;
  const int wm = KS ? 0 : (wave >> 1) * 32, wn = KS ? 0 : (wave & 1) * 32, wk = KS ? wave * 32 : 0;
  const int G = K / GS;
  const int sr = tid / TPR, sc = (tid % TPR) * VPT;  // staging role: row, first value of the step
  const float* const xrow = x + (int64_t)(m0 + sr < M ? m0 + sr : M - 1) * K;  // (rows past the matrices: never stored)
  const int nr = n0 + sr < N ? n0 + sr : N - 1;
  const uint32_t* const wrow = w + (int64_t)nr * (K / (32 / BITS));
  constexpr int NW = VPT * BITS >= 32 ? VPT * BITS / 32 : 1;  // code words of a thread's values
  f32x4 xr[VPT / 4];
  uint32_t cw[NW];
  float scale, bias;
  auto fetch = [&](int k0) {
    const int k = k0 + sc;
    const bool in = k < K;  // (K is a multiple of 32, VPT of a thread lie inside or outside)
    const int kk = in ? k : 0;
#pragma unroll
    for (int i = 0; i < VPT / 4; ++i) {
      xr[i] = *reinterpret_cast<const f32x4*>(xrow + kk + 4 * i);
      if (!in) xr[i] = f32x4{0.f, 0.f, 0.f, 0.f};
    }
#pragma unroll
    for (int i = 0; i < NW; ++i) cw[i] = wrow[kk * BITS / 32 + i];
    if constexpr (VPT * BITS < 32) cw[0] >>= BITS * (kk % (32 / BITS));
    scale = in ? s[(int64_t)nr * G + kk / GS] : 0.f;
    bias = in ? b[(int64_t)nr * G + kk / GS] : 0.f;
  };
  auto stage = [&](int buf) {
#pragma unroll
    for (int i = 0; i < VPT / 4; ++i) {
      *reinterpret_cast<f32x4*>(&xa[buf][sr * RS + sc + 4 * i]) = xr[i];
      f32x4 v;
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const int j = 4 * i + e;
        v[e] = fmaf(scale, (float)((cw[j * BITS / 32] >> (BITS * (j % (32 / BITS)))) & ((1u << BITS) - 1u)), bias);
      }
      *reinterpret_cast<f32x4*>(&wb[buf][sr * RS + sc + 4 * i]) = v;
    }
  };
  f32x16 acc = {};
  fetch(0);
  stage(0);
  __syncthreads();
  for (int k0 = 0, buf = 0; k0 < K; k0 += BK, buf ^= 1) {
    const bool more = k0 + BK < K;
    if (more) fetch(k0 + BK);
    // half-wave h takes the values 16 h .. 16 h + 15 of the wave's 32
    const float* const ar = &xa[buf][(wm + col) * RS + wk + 16 * half];
    const float* const br = &wb[buf][(wn + col) * RS + wk + 16 * half];
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const f32x4 a = *reinterpret_cast<const f32x4*>(ar + 4 * i), c = *reinterpret_cast<const f32x4*>(br + 4 * i);
#pragma unroll
      for (int e = 0; e < 4; ++e) acc = __builtin_amdgcn_mfma_f32_32x32x2f32(a[e], c[e], acc, 0, 0, 0);
    }
    if (more) stage(buf ^ 1);  // (buffer buf ^ 1 was last read before the previous barrier)
    __syncthreads();
  }
  // the accumulator: column col, rows 8 (i / 4) + 4 half + i % 4
  if constexpr (KS) {
    float* const ex = xa[0];  // [4 waves][1024]
    static_assert(2 * T * RS >= 4 * 1024, "sums fit");
#pragma unroll
    for (int i = 0; i < 16; ++i) ex[wave * 1024 + i * 64 + lane] = acc[i];
    __syncthreads();
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const int i = wave * 4 + j, e = i * 64 + lane;
      const float t = ((ex[e] + ex[1024 + e]) + ex[2048 + e]) + ex[3072 + e];
      const int m = m0 + 8 * (i / 4) + 4 * half + i % 4, n = n0 + col;
      if (m < M && n < N) y[(int64_t)m * N + n] = t;
    }
  } else {
#pragma unroll
    for (int i = 0; i < 16; ++i) {
      const int m = m0 + wm + 8 * (i / 4) + 4 * half + i % 4, n = n0 + wn + col;
      if (m < M && n < N) y[(int64_t)m * N + n] = acc[i];
    }
  }
}

struct TypedRows {
  typed_fn fn;
  int rw;  // rows of W per wave
};

template <int DT, int BITS, int GS>
TypedRows pick_rows_mr(int MR, int RW) {
  if (MR == 1 && RW == 1) return {qmv_typed_rows_kernel<DT, BITS, GS, 1, 1>, 1};
  if (MR == 1 && RW == 2) return {qmv_typed_rows_kernel<DT, BITS, GS, 1, 2>, 2};
  if (MR == 1 && RW == 4) return {qmv_typed_rows_kernel<DT, BITS, GS, 1, 4>, 4};
  if (MR == 2 && RW == 1) return {qmv_typed_rows_kernel<DT, BITS, GS, 2, 1>, 1};
  if (MR == 2 && RW == 2) return {qmv_typed_rows_kernel<DT, BITS, GS, 2, 2>, 2};
  if (MR == 2 && RW == 4) return {qmv_typed_rows_kernel<DT, BITS, GS, 2, 4>, 4};
  if (MR == 4 && RW == 2) return {qmv_typed_rows_kernel<DT, BITS, GS, 4, 2>, 2};
  if (MR == 4 && RW == 4) return {qmv_typed_rows_kernel<DT, BITS, GS, 4, 4>, 4};
  return {nullptr, 0};
}

template <int DT>
TypedRows pick_rows_dt(int bits, int gs, int MR, int RW) {
  auto by_gs = [&](auto bt) -> TypedRows {
    constexpr int B = decltype(bt)::value;
    if (gs == 32) return pick_rows_mr<DT, B, 32>(MR, RW);
    if (gs == 64) return pick_rows_mr<DT, B, 64>(MR, RW);
    if (gs == 128) return pick_rows_mr<DT, B, 128>(MR, RW);
    return {nullptr, 0};
  };
  if constexpr (DT != LISAQ_DTYPE_BF16) {  // (bf16 with 2 and 4 bits: qmv*.hip, qmm*.h)
    if (bits == 2) return by_gs(std::integral_constant<int, 2>{});
    if (bits == 4) return by_gs(std::integral_constant<int, 4>{});
  }
  if (bits == 8) return by_gs(std::integral_constant<int, 8>{});
  return {nullptr, 0};
}

template <bool KS>
typed_fn pick_f32(int bits, int gs) {
  auto by_gs = [&](auto bt) -> typed_fn {
    constexpr int B = decltype(bt)::value;
    if (gs == 32) return qmm_f32_mfma_kernel<B, 32, KS>;
    if (gs == 64) return qmm_f32_mfma_kernel<B, 64, KS>;
    if (gs == 128) return qmm_f32_mfma_kernel<B, 128, KS>;
    return nullptr;
  };
  if (bits == 2) return by_gs(std::integral_constant<int, 2>{});
  if (bits == 4) return by_gs(std::integral_constant<int, 4>{});
  if (bits == 8) return by_gs(std::integral_constant<int, 8>{});
  return nullptr;
}

TypedRows pick_rows(int dtype, int bits, int gs, int MR, int RW) {
  if (dtype == LISAQ_DTYPE_BF16) return pick_rows_dt<0>(bits, gs, MR, RW);
  if (dtype == LISAQ_DTYPE_F32) return pick_rows_dt<1>(bits, gs, MR, RW);
  if (dtype == LISAQ_DTYPE_F16) return pick_rows_dt<2>(bits, gs, MR, RW);
  return {nullptr, 0};
}

template <int DT, int BITS, int TB>
typed_fn pick_mfma_gs(int gs) {
  if (gs == 32) return qmm_typed_mfma_kernel<DT, BITS, 32, TB>;
  if (gs == 64) return qmm_typed_mfma_kernel<DT, BITS, 64, TB>;
  if (gs == 128) return qmm_typed_mfma_kernel<DT, BITS, 128, TB>;
  return nullptr;
}

template <int DT, int TB>
typed_fn pick_mfma(int bits, int gs) {
  if constexpr (DT != LISAQ_DTYPE_BF16) {
    if (bits == 2) return pick_mfma_gs<DT, 2, TB>(gs);
    if (bits == 4) return pick_mfma_gs<DT, 4, TB>(gs);
  }
  if (bits == 8) return pick_mfma_gs<DT, 8, TB>(gs);
  return nullptr;
}

template <bool MV, int DT, int BITS>
typed_fn pick_gs(int gs) {
  if (gs == 32) return MV ? qmv_typed_kernel<DT, BITS, 32> : qmm_typed_kernel<DT, BITS, 32>;
  if (gs == 64) return MV ? qmv_typed_kernel<DT, BITS, 64> : qmm_typed_kernel<DT, BITS, 64>;
  if (gs == 128) return MV ? qmv_typed_kernel<DT, BITS, 128> : qmm_typed_kernel<DT, BITS, 128>;
  return nullptr;
}

template <bool MV, int DT>
typed_fn pick_bits(int bits, int gs) {
  if constexpr (DT != LISAQ_DTYPE_BF16) {
    if (bits == 2) return pick_gs<MV, DT, 2>(gs);
    if (bits == 4) return pick_gs<MV, DT, 4>(gs);
  }
  if (bits == 8) return pick_gs<MV, DT, 8>(gs);
  return nullptr;
}

template <bool MV>
typed_fn pick(int dtype, int bits, int gs) {
  if (dtype == LISAQ_DTYPE_BF16) return pick_bits<MV, 0>(bits, gs);
  if (dtype == LISAQ_DTYPE_F32) return pick_bits<MV, 1>(bits, gs);
  if (dtype == LISAQ_DTYPE_F16) return pick_bits<MV, 2>(bits, gs);
  return nullptr;
}

}  // namespace

int launch_typed_mm(hipStream_t st, bool matvec, const void* x, const uint32_t* w, const void* s, const void* b,
                    void* y, int64_t M, int64_t N, int64_t K, int gs, int bits, int dtype) {
  typed_fn fn = matvec ? pick<true>(dtype, bits, gs) : pick<false>(dtype, bits, gs);
  // 16-bit compute dtypes: the matrix-core matmul (x 16-byte aligned), in
  // 128 x 128 tiles where those make at least 512 workgroups (measured, f16
  // 4-bit: 512 x 17408 x 5120, 544 tiles, 397 vs 242 TFLOP/s for 64 x 64;
  // bf16 8-bit 1024 x 4096 x 4096, 256 tiles, 264 vs 331)
  int tile = 64;
  if (!matvec && fn && reinterpret_cast<uintptr_t>(x) % 16 == 0 && tune_int("LISAQ_TYPED_MFMA", 1) != 0 &&
      (dtype == LISAQ_DTYPE_BF16 || dtype == LISAQ_DTYPE_F16)) {
    const bool wide = ((M + 127) / 128) * ((N + 127) / 128) >= 512 && tune_int("LISAQ_TYPED_TB", 2) == 2;
    if (dtype == LISAQ_DTYPE_BF16) fn = wide ? pick_mfma<0, 2>(bits, gs) : pick_mfma<0, 1>(bits, gs);
    else fn = wide ? pick_mfma<2, 2>(bits, gs) : pick_mfma<2, 1>(bits, gs);
    if (wide) tile = 128;
  }
  // f32: the matrix-core matmul (x 16-byte aligned), in 64 x 64 tiles where
  // those make a workgroup per compute unit, else 32 x 32 with K over the waves
  // (4-bit, 64- / 32-row tiles: 64 x 4096 x 4096, 64 tiles, 99.8 / 39.8 us; 16 x
  // 9728 x 2560, 152 tiles, 63 / 41; 256 x 4096 x 4096, 256 tiles, 100 / 126; 40 x
  // 17408 x 2560, 272 tiles, 106 / 99; 900 x 2048 x 2048, 480 tiles, 87 / 125)
  if (!matvec && fn && dtype == LISAQ_DTYPE_F32 && reinterpret_cast<uintptr_t>(x) % 16 == 0 && (M + 31) / 32 <= 65535) {
    const bool ks = ((M + 63) / 64) * ((N + 63) / 64) < 256;
    fn = ks ? pick_f32<true>(bits, gs) : pick_f32<false>(bits, gs);
    tile = ks ? 32 : 64;
  }
  if (!fn) return set_error(LISAQ_EUNSUPPORTED, "quantized_matmul_typed: dtype=%d bits=%d gs=%d", dtype, bits, gs);
  // grid.y carries the 64-row tiles of M (at most 65535 of them)
  if (!matvec && (M + 63) / 64 > 65535)
    return set_error(LISAQ_EINVAL_SHAPE, "quantized_matmul_typed: M=%lld exceeds %d rows", (long long)M, 65535 * 64);
  // Matvec, x and W 16-byte aligned and a row of x fits the LDS: the rows
  // kernel.  Rows of x per workgroup (MR): four save re-reading a large W where
  // they take at most 48 KB of LDS (f16 8-bit 17408 x 5120 4 rows 30.5 us, two
  // at a time 37.2; 12 rows 71 / 90), else two up to 48 KB, and of 16-bit types up
  // to 80 KB (bf16 8-bit 5120 x 17408 4 rows 38 us, one at a time 51; 12 rows 86 /
  // 147; but 4-bit 3 rows 38.7 / 35.4; f32 4-bit 2560 x 9728 3 rows 18.9 / 14.6), else one.
  // Rows of W per wave (RW): one row of x two, one below 4096 rows (f32 1000 x
  // 8192 RW 2 6.0 us, RW 4 7.6); else four where that makes a workgroup per
  // compute unit, of 16-bit pairs of rows 400 (bf16 8-bit 2 rows of 4096 x 4096, 256
  // with four rows, 8.2 us, with two 6.5; 6 rows of 2560 x 9728, 480, 15.0 / 18.9), and
  // one where two leave compute units without a workgroup.
  const bool al16 = reinterpret_cast<uintptr_t>(x) % 16 == 0 && reinterpret_cast<uintptr_t>(w) % 16 == 0;
  if (matvec && M == 1 && dtype == LISAQ_DTYPE_F16 && bits == 4 && al16 && N <= 4096) {
    const typed_fn dot = gs == 32 ? qmv_f16_dot_kernel<32> : gs == 64 ? qmv_f16_dot_kernel<64> : qmv_f16_dot_kernel<128>;
    hipLaunchKernelGGL(dot, dim3((unsigned)((N + 3) / 4)), dim3(256), 0, st, x, w, s, b, y, 1, (int)N, (int)K);
    return check_launch("quantized_matmul_typed");
  }
  const int P = bits == 8 ? 16 : 32;
  const int64_t per_row = K * (dtype == LISAQ_DTYPE_F32 ? 4 : 2) + K / P * 4;
  if (matvec && al16 && per_row <= 160 * 1024) {
    const int64_t room = 48 * 1024;
    const bool half = dtype != LISAQ_DTYPE_F32;
    const int MR = M >= 3 && N * K * bits / 8 >= ((int64_t)32 << 20) && 4 * per_row <= room ? 4
                   : M >= 2 && 2 * per_row <= (half && M != 3 ? 80 * 1024 : room)           ? 2
                                                                                            : 1;
    const int64_t groups = (M + MR - 1) / MR;
    const auto blocks_of = [&](int rw) { return (N + 4 * rw - 1) / (4 * rw) * groups; };
    const int RW = M == 1                                              ? (N >= 4096 ? 2 : 1)
                   : blocks_of(4) >= (MR == 2 && half ? 400 : 256)     ? 4
                   : blocks_of(2) >= 256 || MR == 4                    ? 2
                                                                       : 1;
    const TypedRows k = pick_rows(dtype, bits, gs, MR, RW);
    if (k.fn) {
      const int lds = (int)(MR * per_row);
      if (int rc = allow_dyn_lds((const void*)k.fn, lds, "quantized_matmul_typed")) return rc;
      // as many workgroups as the chip holds (each stages x once), at most 8 per compute unit
      const int64_t blocks = (N + 4 * k.rw - 1) / (4 * k.rw), per_cu = (160 * 1024) / lds < 8 ? (160 * 1024) / lds : 8;
      const int64_t cap = 256 * per_cu;
      hipLaunchKernelGGL(k.fn, dim3((unsigned)(blocks < cap ? blocks : cap), (unsigned)groups), dim3(256), lds, st, x,
                         w, s, b, y, (int)M, (int)N, (int)K);
      return check_launch("quantized_matmul_typed");
    }
  }
  if (matvec)
    hipLaunchKernelGGL(fn, dim3((unsigned)((N + 3) / 4)), dim3(256), 0, st, x, w, s, b, y, (int)M, (int)N, (int)K);
  else
    hipLaunchKernelGGL(fn, dim3((unsigned)((N + tile - 1) / tile), (unsigned)((M + tile - 1) / tile)), dim3(256), 0,
                       st, x, w, s, b, y, (int)M, (int)N, (int)K);
  return check_launch("quantized_matmul_typed");
}

}  // namespace lisaq
