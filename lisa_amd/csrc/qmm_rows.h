// Matmul of few rows (13-64: batched decode, short prompts) on gfx950.
//
// Arithmetic contract of qmm_kernel.h: every weight T(scale * q + bias) from
// an f32 fma, f32 accumulation on v_mfma_f32_32x32x16, one rounding to T.
//
// What bounds it: W has to be read once (51 MB at 17408 x 5120 4-bit, 10.4 us at
// the rate of a large copy), and dequantizing a code takes ~9 cycles of a
// SIMD whatever the number of rows it serves (measured per wave instruction:
// v_fma_mix, v_perm and v_cvt_pk 4.2 cycles, and / shift / add / mul / fma 2.5),
// 5.6 us of all SIMDs for that matrix.  qmm_kernel.h's tall tiles hide both
// under matrix work; with few rows its two waves per SIMD wait for memory in
// every 64-code step.  Here a workgroup's sixteen waves (four per SIMD) share a
// ring of chunks of 128 or 256 codes, NB - 1 of them (64-96 KB per compute unit)
// in flight, with one barrier per chunk.  Measured with the reduction launch,
// qmm_kernel.h -> here: 4-bit 17408 x 5120 24 rows 31.2 -> 22.7 us, 64 rows 36.1
// -> 30.1; 5120 x 17408 16 rows 31.8 -> 21.8; 2560 x 9728 32 rows 17.6 -> 14.6;
// 8-bit 9728 x 2560 24 rows 14.5 -> 12.0.  Left: ~6 us of launch, first copies
// and sums, 4 us of the reduction launch, and the dequantization (7 us of VALU
// cycles at 17408 x 5120 on the 204 of 256 units that three parts of 68 tiles
// use).  Eight waves with the next
// chunk's LDS reads issued a chunk ahead: the same times.
//
// Workgroup: 256 columns by all 32 * MT rows of one K part.  Wave w takes the
// 32 columns w % 8 and the chunk's K-steps w / 8, w / 8 + 2, ...; the two waves of a
// column group add their sums through LDS at the end.  All global reads are
// direct-to-LDS copies.  x: CK columns of every row per chunk, as K-steps of 64
// ([32 * MT rows][128 B] each, swizzled as in qmm_kernel.h).  W: 32 rows per
// column group, CK * BITS / 8 contiguous bytes of each.  Scales/biases: the
// group's 32 rows x 16 bytes (8 groups) of both in one copy per 8 groups.
#pragma once
#include "qmm_kernel.h"

namespace lisaq {

// K-steps of 64 codes per chunk.  256 codes are 64 (2 bits) or 128 bytes (4 bits)
// of a row per copy; 4 bits with 33-64 rows or groups of 32 (whose scale blocks
// hold 256 codes) take 128: the ring would be three chunks or none.
constexpr int rows_chunk_steps(int bits, int gs, int mt) {
  return bits == 2 || (bits == 4 && mt == 1 && gs > 32) ? 4 : 2;
}

template <int BITS, int GS, int MT>
struct RowsGeo {
  static constexpr int BM = 32 * MT, NG = 8, BN = 32 * NG, NW = 2 * NG;  // column groups, waves
  static constexpr int CK = 64 * rows_chunk_steps(BITS, GS, MT);  // codes of a row per chunk
  static constexpr int KS = CK / 64;                // K-steps of 64 per chunk (two waves of a group share them)
  static constexpr int X = BM * CK * 2;             // x bytes of a chunk
  static constexpr int RBW = CK * BITS / 8;         // W bytes of a row per chunk
  static constexpr int WW = 32 * RBW;               // W bytes of a column group per chunk
  static constexpr int W = NG * WW;
  static constexpr int BC = 8 * GS;                 // codes per scale/bias block
  static constexpr int sbn(int nb) { return ((nb - 1) * CK + BC - 1) / BC + 1; }
  static constexpr int total(int nb) { return nb * (X + W) + sbn(nb) * NG * 1024; }
  static constexpr int kMax = 160 * 1024;
  // ring depth: as deep as the 160 KB of LDS allow, at most 5
  static constexpr int NB = total(5) <= kMax ? 5 : total(4) <= kMax ? 4 : 3;
  static constexpr int SBN = sbn(NB);  // scale/bias blocks that NB chunks can touch
  static constexpr int TOTAL = total(NB);
  static constexpr bool OK = TOTAL <= kMax;
  static constexpr int XB = X / NW;                       // x bytes per wave and chunk
  static constexpr int XI = XB >= 1024 ? XB / 1024 : 1;   // x copies per wave and chunk
  static constexpr int XL = XB >= 1024 ? 64 : XB / 16;    // lanes of an x copy
  static constexpr int WI = W / NW / 1024;                // W copies per wave and chunk (1 KB each)
  static_assert(W % (NW * 1024) == 0 && (XB % 1024 == 0 || XB == 512), "ring geometry");
};

// swizzle of the 16-byte pieces of a W row in LDS (by its bytes per chunk): the
// 32 rows' reads of one piece hit distinct banks, see x_swz / w_swz2
template <int RBW>
__device__ __forceinline__ int rows_w_swz(int row) {
  return RBW == 128 ? x_swz(row) : RBW == 64 ? w_swz2(row) : 0;
}

template <int BITS, int GS, int MT, int CT>
__global__ __launch_bounds__(1024) void qmm_rows_kernel(QmmParams p) {
  using R = RowsGeo<BITS, GS, MT>;
  using C = Ct<CT>;
  constexpr int WPL = MGeo<BITS>::WPL;  // code words of a lane per K-step
  extern __shared__ __attribute__((aligned(16))) unsigned char smem[];
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int cg = wave % R::NG, kh = wave / R::NG;  // column group, first K-step
  const int col = lane & 31, h = lane >> 5;
  const int gn = (p.N + R::BN - 1) / R::BN;
  const int nt0 = (blockIdx.x % gn) * R::BN, split = blockIdx.x / gn;
  const int n0 = nt0 + cg * 32;  // the wave's first column
  // chunks [c0, c1) of this K part; the last one of a row may be partial
  const int nks = p.K / 64, nc = (nks + R::KS - 1) / R::KS, per = (nc + p.ksplit - 1) / p.ksplit;
  const int c0 = split * per, c1 = c0 + per < nc ? c0 + per : nc;

  unsigned char* const xl = smem;
  unsigned char* const wl = smem + R::NB * R::X + cg * R::WW;
  unsigned char* const sl = smem + R::NB * (R::X + R::W) + cg * 1024;

  // ---- copies (rows past the matrices clamped to the last: never stored)
  const __amdgpu_buffer_rsrc_t rx = lds_rsrc(p.x, (uint32_t)p.M * (uint32_t)p.K * 2u);
  uint32_t xvo[R::XI];
#pragma unroll
  for (int i = 0; i < R::XI; ++i) {
    const int off = wave * R::XB + i * 1024 + lane * 16;          // byte of the chunk's image
    const int t = off / (R::BM * 128), row = off / 128 % R::BM;  // K-step, row
    const int chunk = (lane & 7) ^ x_swz(row);
    xvo[i] = ((uint32_t)(row < p.M ? row : p.M - 1) * (uint32_t)p.K + (uint32_t)(t * 64 + chunk * 8)) * 2u;
  }
  const uint32_t rowbytes = (uint32_t)p.K * BITS / 8;
  const __amdgpu_buffer_rsrc_t rw = lds_rsrc(p.w, (uint32_t)p.N * rowbytes);
  uint32_t wvo[R::WI];
#pragma unroll
  for (int i = 0; i < R::WI; ++i) {
    const int off = (kh * R::WI + i) * 1024 + lane * 16, row = off / R::RBW;
    const int n = n0 + row < p.N ? n0 + row : p.N - 1;
    wvo[i] = (uint32_t)n * rowbytes + (uint32_t)((off % R::RBW) ^ (rows_w_swz<R::RBW>(row) << 4));
  }
  // scales (lanes 0-31) and biases (32-63) of the group's rows: 16 bytes of a
  // row per block; a block that would end past the array is read from its last
  // 16 bytes, and its groups are then found that much further on
  const int sn = n0 + col < p.N ? n0 + col : p.N - 1;
  const int srow = sn * p.G * 2, send = p.N * p.G * 2;
  const unsigned char* const sbase = reinterpret_cast<const unsigned char*>(h ? p.b : p.s);
  auto sb_shift = [&](int blk) {
    const int over = srow + blk * 16 + 16 - send;
    return over > 0 ? over : 0;
  };
  auto issue = [&](int c) {
    const int slot = (c - c0) % R::NB;
    // (a scale/bias block with the part's first chunk and with each chunk that starts one)
    if (kh == 0 && (c == c0 || c * R::CK % R::BC == 0)) {
      const int blk = c * R::CK / R::BC;
      load_lds16(sbase + srow + blk * 16 - sb_shift(blk), sl + (blk % R::SBN) * (R::NG * 1024));
    }
#pragma unroll
    for (int i = 0; i < R::WI; ++i)
      buf_lds16(rw, wvo[i], (uint32_t)c * R::RBW, wl + slot * R::W + (kh * R::WI + i) * 1024);
#pragma unroll
    for (int i = 0; i < R::XI; ++i)
      if (R::XL == 64 || lane < R::XL)
        buf_lds16(rx, xvo[i], (uint32_t)c * (R::CK * 2), xl + slot * R::X + wave * R::XB + i * 1024);
  };

  f32x16 acc[MT];
#pragma unroll
  for (int mt = 0; mt < MT; ++mt) acc[mt] = f32x16{};
  constexpr int PC = R::XI + R::WI;  // copies per chunk (scale/bias blocks beside: waits count them as later ones)
#pragma unroll
  for (int i = 0; i < R::NB - 1; ++i)
    if (c0 + i < c1) issue(c0 + i);
  for (int c = c0; c < c1; ++c) {
    // this chunk landed (the chunks after it may be in flight), for every wave
    const int later = c1 - 1 - c;
    if (later >= R::NB - 2) wait_vm<(R::NB - 2) * PC>();
    else if (R::NB > 4 && later == 2) wait_vm<2 * PC>();
    else if (R::NB > 3 && later == 1) wait_vm<PC>();
    else wait_vm<0>();
    block_sync();
    // (its ring slot's last readers are behind the barrier)
    if (c + R::NB - 1 < c1) issue(c + R::NB - 1);
    const int slot = (c - c0) % R::NB, left = nks - c * R::KS;  // K-steps of the row from here on
    const unsigned char* const ws = wl + slot * R::W + col * R::RBW;
#pragma unroll
    for (int tt = 0; tt < R::KS; tt += 2) {
      const int t = tt + kh;
      if (t >= left) break;
      // group of the lane's 32 codes (gs 32: one per half-wave)
      const int g = (c * R::CK + t * 64 + (GS == 32 ? 32 * h : 0)) / GS, blk = g >> 3;
      const unsigned char* const sb = sl + (blk % R::SBN) * (R::NG * 1024) + col * 16 + (g & 7) * 2 + sb_shift(blk);
      const uint16_t sv = *reinterpret_cast<const uint16_t*>(sb), bv = *reinterpret_cast<const uint16_t*>(sb + 512);
      uint32_t wv[WPL];
      if constexpr (BITS == 2) {
        const int off = t * 16 + 8 * h;
        const u32x2 v = *reinterpret_cast<const u32x2*>(ws + ((off & ~15) ^ (rows_w_swz<R::RBW>(col) << 4)) + (off & 15));
        wv[0] = v[0];
        wv[1] = v[1];
      } else {
#pragma unroll
        for (int q = 0; q < WPL / 4; ++q) {
          const int off = t * (8 * BITS) + h * (4 * BITS) + q * 16;
          const u32x4 v = *reinterpret_cast<const u32x4*>(ws + (off ^ (rows_w_swz<R::RBW>(col) << 4)));
#pragma unroll
          for (int e = 0; e < 4; ++e) wv[4 * q + e] = v[e];
        }
      }
      // (every LDS read before the dequantization, which hides them)
      const unsigned char* const xs = xl + slot * R::X + t * (R::BM * 128);
      u32x4 av[4][MT];
#pragma unroll
      for (int j = 0; j < 4; ++j)
#pragma unroll
        for (int mt = 0; mt < MT; ++mt)
          av[j][mt] = *reinterpret_cast<const u32x4*>(xs + x_lds_off(mt * 32 + col, 4 * h + j));
      __builtin_amdgcn_sched_barrier(0);
      const float s_ = deq_scale<BITS, CT>(C::f(sv)), bs = C::f(bv);
      uint32_t bop[16];
      static_for<WPL>([&](auto JI) {
        constexpr int j = decltype(JI)::value;
        deq_word<BITS, CT>(wv[j], s_, bs, &bop[j * (16 / WPL)]);
      });
#pragma unroll
      for (int j = 0; j < 4; ++j)
#pragma unroll
        for (int mt = 0; mt < MT; ++mt)
          acc[mt] = C::mfma(u32x4{bop[4 * j], bop[4 * j + 1], bop[4 * j + 2], bop[4 * j + 3]}, av[j][mt], acc[mt]);
    }
  }

  // the second wave of a column group hands its sums to the first (every copy
  // has landed: the last chunk waited for all)
  static_assert(R::NG * MT * 4096 <= R::TOTAL, "sums fit the ring");
  block_sync();
  f32x4* const ex = reinterpret_cast<f32x4*>(smem) + cg * (MT * 256) + lane;
  if (kh == 1) {
#pragma unroll
    for (int mt = 0; mt < MT; ++mt)
#pragma unroll
      for (int g = 0; g < 4; ++g)
        ex[mt * 256 + g * 64] = f32x4{acc[mt][4 * g], acc[mt][4 * g + 1], acc[mt][4 * g + 2], acc[mt][4 * g + 3]};
  }
  wait_lgkm0();
  block_sync();
  if (kh == 1) return;
  // the accumulator is y^T: lane holds row 32 mt + col and columns 8 g + 4 h .. + 3
  const bool vec = (p.N & 3) == 0;
  float* const part = p.partial + (int64_t)split * p.M * p.N;
#pragma unroll
  for (int mt = 0; mt < MT; ++mt) {
    const int m = mt * 32 + col;
    if (m >= p.M) continue;
#pragma unroll
    for (int g = 0; g < 4; ++g) {
      const int n = n0 + 8 * g + 4 * h;
      const int64_t at = (int64_t)m * p.N + n;
      const f32x4 v = f32x4{acc[mt][4 * g], acc[mt][4 * g + 1], acc[mt][4 * g + 2], acc[mt][4 * g + 3]} +
                      ex[mt * 256 + g * 64];
      if (vec && n + 3 < p.N) {
        if (p.ksplit > 1) *reinterpret_cast<f32x4*>(part + at) = v;
        else *reinterpret_cast<u32x2*>(p.y + at) = u32x2{C::pk(v[0], v[1]), C::pk(v[2], v[3])};
      } else {
#pragma unroll
        for (int e = 0; e < 4; ++e)
          if (n + e < p.N) {
            if (p.ksplit > 1) part[at + e] = v[e];
            else p.y[at + e] = C::one(v[e]);
          }
      }
    }
  }
}

// Kernel of one (bits, compute type): qmm_rows_*.hip instantiate them.
// *lds = dynamic LDS bytes; null for a tile height that is not built.
template <int BITS, int CT>
qmm_fn qmm_rows_get(int gs, int MT, int* lds);

template <int BITS, int CT>
qmm_fn qmm_rows_get_impl(int gs, int MT, int* lds) {
  auto one = [&](auto mt) -> qmm_fn {
    constexpr int M_ = decltype(mt)::value;
    auto pick = [&](auto g) -> qmm_fn {
      using R = RowsGeo<BITS, decltype(g)::value, M_>;
      *lds = R::TOTAL;
      if constexpr (R::OK) return qmm_rows_kernel<BITS, decltype(g)::value, M_, CT>;
      else return nullptr;
    };
    if (gs == 32) return pick(std::integral_constant<int, 32>{});
    if (gs == 64) return pick(std::integral_constant<int, 64>{});
    if (gs == 128) return pick(std::integral_constant<int, 128>{});
    return nullptr;
  };
  if (MT == 1) return one(std::integral_constant<int, 1>{});
  if (MT == 2) return one(std::integral_constant<int, 2>{});
  return nullptr;
}

}  // namespace lisaq
