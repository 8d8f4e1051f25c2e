// Block-FP8 GEMM tiles of 256 weight rows x up to 128 activation rows for gfx950:
// the linears above 64 rows and the routed experts' larger groups.
//
// y[m, n] = sum_k x[m, k] w[n, k] scale_inv[n/128, k/128], w e4m3fn converted
// exactly to bf16 in registers, 32x32x16 bf16 MFMAs, fp32 sums.
#include <algorithm>
#include <type_traits>

#include "amla_common.h"
#include "amla_internal.h"
#include "gemm_epilogue.h"

namespace amla {

// A workgroup is four waves on two 128-row weight segments: wave w multiplies
// rows 32w .. +31 of both by all activation rows (NJ groups of 32), so a weight
// byte is converted by one wave only, and with gate rows as segment 0 and up
// rows as segment 1 the lane that holds a gate output holds the same up output:
// silu(gate) * up needs no exchange.  A tile costs MFMAs for its own rows
// rounded up to 32, and two workgroups share a CU (80 KB of LDS, at most 256
// VGPRs), one computing while the other waits for its copies.
//
// What bounds it: with few rows per expert the weight stream from HBM (64 rows
// are 128 FLOP per weight byte), above about 128 rows the MFMAs.  MI355X, 256
// R1 experts, top 8: 300 tokens (9 rows per expert) [gate | up] with silu * up
// 1.27 ms (5.9 TB/s), down 0.68 ms, where the skinny GEMM with fp32 K parts and
// finishing passes took 1.55 + 0.82 ms; 2000 tokens (62 rows) 1.59 + 0.87 ms
// against 2.75 + 1.62 for that and 256 x 256 tiles for groups above 64 rows;
// 8000 tokens (250 rows) 4.4 + 2.2 ms against 5.6 + 2.9.  Gathering and
// scattering the rows here saved two more passes (0.14 ms at 2000 tokens).
//
// Above 64 rows (TileHalves): two K stages of 64 in LDS, fp8 weight rows (64 B,
// chunk c of row r at c ^ ((r >> 2) & 3)) and bf16 activation rows (128 B,
// chunk c of row r at c ^ ((r >> 1) & 7)): the 16 lanes of each fragment-read
// pass hit distinct banks.  Up to 64 rows: TileLines below.
constexpr int T_BK = 64;
constexpr int T_WBYTES = 256 * T_BK;             // weight part of a stage
constexpr int T_XROW = T_BK * 2;                 // activation row of a stage
constexpr int T_LDS = 80 * 1024;
constexpr int T_ZERO = T_LDS - 16;               // weight fragments of a block whose scale is zero
constexpr int T_PITCH_H = 128 * 2 + 16;          // epilogue rows in LDS: 128 or 256 bf16 outputs
constexpr int T_PITCH_Y = 256 * 2 + 16;
static_assert(128 * T_PITCH_Y <= T_ZERO, "staged output tile exceeds LDS");
static_assert(2 * (T_WBYTES + 128 * T_XROW) <= T_ZERO, "stages exceed LDS");

// x row strides (bf16) up to which the byte offsets of 128 rows fit 32 bits;
// weight rows are half as far apart
constexpr int T_MAX_LD = (int)((UINT32_MAX - T_XROW) / (2 * 127));

struct TileArgs {
  const uint8_t *w[2];   // first row of each segment
  const float *s[2];     // scale row (K / 128) of each segment
  int wrows[2];          // rows of each segment (128, fewer at the end of a matrix: the last one is repeated)
  const uint16_t *x;     // activation rows
  const int32_t *xrow;   // row of x for tile row r, or null: row r
  uint16_t *y;           // outputs, column 0 of the tile
  const int32_t *yrow;   // row of y for tile row r, or null: row r
  int ldx, ldy, K, rows;
  int kb0, kb1;          // 128-wide K blocks
  bool two;              // segment 1 is stored (always multiplied)
  bool wide;             // byte offsets of the tile's x rows may not fit 32 bits
};

// A block scale that is zero, or below 2^-64 of the largest of the tile's K range
// so far, counts as zero (some quantisers give a block of zeros the smallest
// float): rescaling the sums to units that small would overflow them.  Scales are
// compared as bits without the sign, on the scalar unit: `floor`, the smallest
// that counts, grows with each block.  (All scales read ahead of the loop instead,
// by the lanes: 1.5 us more per launch.)
AMLA_DEV int scale_bits(float s) { return (int)(__float_as_uint(s) & 0x7fffffffu); }
AMLA_DEV int scale_floor(int bits) { return max(bits - (64 << 23), 1); }

// A tile's sums: acc[segment][row group of 32], in units of s_run[segment].
template <int NJ>
struct TileSums {
  f32x16 acc[2][NJ];
  float s_run[2];
};

// WIDE: nor do those of its weight rows
template <int NJ, bool WIDE>
struct TileHalves {
  static AMLA_DEV void run(const TileArgs &a, TileSums<NJ> &sums) {
  auto &acc = sums.acc;
  auto &s_run = sums.s_run;
  extern __shared__ __align__(16) uint8_t tsm[];
  constexpr int STAGE = T_WBYTES + 32 * NJ * T_XROW;
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int j32 = lane & 31, hh = lane >> 5;

  // copies: the wave's own 2 x 32 weight rows (16 rows of 64 B each) and its
  // quarter of the activation rows (8 rows of 128 B each), as scalar bases that
  // advance with the stage plus 32-bit lane offsets
  uint32_t woff[2][2], xoff[NJ];
#pragma unroll
  for (int g = 0; g < 2; ++g)
#pragma unroll
    for (int c = 0; c < 2; ++c)
    {
      const uint32_t wr = min(32 * wave + 16 * c + (lane >> 2), a.wrows[g] - 1);
      // a.wide, WIDE: the row index only, the offset is formed per copy
      woff[g][c] = WIDE ? wr : wr * (uint32_t)a.K + 16 * ((lane & 3) ^ ((lane >> 4) & 3));
    }
#pragma unroll
  for (int c = 0; c < NJ; ++c) {
    const int r = 8 * (NJ * wave + c) + (lane >> 3);
    const int rc = min(r, a.rows - 1);  // rows past the tile repeat its last row (not stored)
    const uint32_t xr = a.xrow ? a.xrow[rc] : rc;
    xoff[c] = a.wide ? xr : xr * ((uint32_t)a.ldx * 2) + 16 * ((lane & 7) ^ ((r >> 1) & 7));
  }
  auto dma = [&](int it, int stg) {
    uint8_t *st = tsm + stg * STAGE;
    // (scalar base + 32-bit lane offset per copy: with the bases or the offsets'
    // extension visible outside the loop, each copy costs a 64-bit vector add)
    auto opaque = [](uint32_t v) {
      asm volatile("" : "+v"(v));
      return v;
    };
    typedef const __attribute__((address_space(1))) uint8_t *gptr;
    gptr wb[2] = {(gptr)(a.w[0] + it * T_BK), (gptr)(a.w[1] + it * T_BK)};
    gptr xb = (gptr)(reinterpret_cast<const uint8_t *>(a.x) + it * T_XROW);
    asm volatile("" : "+s"(wb[0]));
    asm volatile("" : "+s"(wb[1]));
    asm volatile("" : "+s"(xb));
    if constexpr (!WIDE) {
#pragma unroll
      for (int g = 0; g < 2; ++g)
#pragma unroll
        for (int c = 0; c < 2; ++c)
          __builtin_amdgcn_global_load_lds(wb[g] + opaque(woff[g][c]), LDS_PTR(st + (128 * g + 32 * wave + 16 * c) * T_BK), 16, 0, 0);
    } else {
#pragma unroll
      for (int g = 0; g < 2; ++g)
#pragma unroll
        for (int c = 0; c < 2; ++c)
          __builtin_amdgcn_global_load_lds(wb[g] + (size_t)woff[g][c] * a.K + 16 * ((lane & 3) ^ ((lane >> 4) & 3)),
                                           LDS_PTR(st + (128 * g + 32 * wave + 16 * c) * T_BK), 16, 0, 0);
    }
    if (!a.wide) {
#pragma unroll
      for (int c = 0; c < NJ; ++c)
        __builtin_amdgcn_global_load_lds(xb + opaque(xoff[c]), LDS_PTR(st + T_WBYTES + 8 * (NJ * wave + c) * T_XROW), 16, 0, 0);
    } else {
#pragma unroll
      for (int c = 0; c < NJ; ++c)
        __builtin_amdgcn_global_load_lds(
            xb + (size_t)xoff[c] * a.ldx * 2 + 16 * ((lane & 7) ^ ((4 * (NJ * wave + c) + (lane >> 4)) & 7)),
            LDS_PTR(st + T_WBYTES + 8 * (NJ * wave + c) * T_XROW), 16, 0, 0);
    }
  };

  uint32_t aoff[2], boff[2][2];
#pragma unroll
  for (int pr = 0; pr < 2; ++pr) {
    aoff[pr] = (32 * wave + j32) * T_BK + 16 * ((2 * pr + hh) ^ ((j32 >> 2) & 3));
#pragma unroll
    for (int s2 = 0; s2 < 2; ++s2)
      boff[pr][s2] = T_WBYTES + j32 * T_XROW + 16 * ((4 * pr + 2 * hh + s2) ^ ((j32 >> 1) & 7));
  }
  const __attribute__((address_space(4))) float *srow[2];
#pragma unroll
  for (int g = 0; g < 2; ++g) srow[g] = (const __attribute__((address_space(4))) float *)(a.s[g]);

#pragma unroll
  for (int g = 0; g < 2; ++g)
#pragma unroll
    for (int j = 0; j < NJ; ++j)
#pragma unroll
      for (int r = 0; r < 16; ++r) acc[g][j][r] = 0.f;
  // The accumulators are kept in units of the current K block's scale: acc *=
  // s_prev / s_cur between two blocks, * s_last at the end (fp32 rounding of
  // the ratios, ~1e-5 relative over 128 blocks).  A zero scale (below sfloor, scale_floor)
  // dequantises to zeros: the segment's fragments of that block are read from 16
  // zeroed bytes instead and the units stay.
#pragma unroll
  for (int g = 0; g < 2; ++g) s_run[g] = srow[g][a.kb0];
  if (tid < 4) *reinterpret_cast<uint32_t *>(tsm + T_ZERO + 4 * tid) = 0;  // visible after the first barrier
  asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");

  int sfloor[2] = {scale_floor(scale_bits(s_run[0])), scale_floor(scale_bits(s_run[1]))};
  bool zero[2] = {s_run[0] == 0.f, s_run[1] == 0.f};

  const int it0 = 2 * a.kb0, iters = 2 * a.kb1;
  dma(it0, 0);
  // One stage of 64: four sub-steps of 16 (K 32 pr + 16 hh + 8 s2 .. +7 of each
  // half-wave).  While a sub-step multiplies, the fragments of the next are
  // read and converted between its MFMAs.  The rescaling between two blocks
  // (16 multiplies per 32 x 32 tile) runs between the last sub-step's MFMAs
  // from the third on, while the next stage's first fragments are read, and
  // between its first MFMAs.  Scheduling barriers keep the order: left to
  // itself the compiler issues the multiplies and the LDS waits in runs.
  constexpr int NT = 2 * NJ;           // tiles, in the order of their MFMAs
  constexpr int LATE = 2;              // tiles rescaled between the next block's first MFMAs
  auto rescale = [&](int half, const float *r) {  // half tiles in MFMA order
    const int g = (half >> 1) / NJ, j = (half >> 1) % NJ;
#pragma unroll
    for (int e = 0; e < 8; ++e) acc[g][j][8 * (half & 1) + e] *= r[g];
  };
  auto stage = [&](int it, auto odd_c, const float *r) {
    constexpr bool ODD = decltype(odd_c)::value;
    constexpr int stg = ODD ? 1 : 0;
    wait_vmcnt<0>();
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
    if (it + 1 < iters) dma(it + 1, 1 - stg);
    const uint8_t *st = tsm + stg * STAGE;
    const uint8_t *sa[2];
#pragma unroll
    for (int g = 0; g < 2; ++g) sa[g] = zero[g] ? tsm + T_ZERO : st + g * 128 * T_BK;
    u32x4 araw[2][2], bx[2][NJ];
    bf16x8 av[2][2];
    auto read_a = [&](int pr) {
#pragma unroll
      for (int g = 0; g < 2; ++g) araw[pr][g] = *reinterpret_cast<const u32x4 *>(sa[g] + (zero[g] ? 0 : aoff[pr]));
    };
    auto read_b = [&](int q) {
#pragma unroll
      for (int j = 0; j < NJ; ++j)
        bx[q & 1][j] = *reinterpret_cast<const u32x4 *>(st + boff[q >> 1][q & 1] + j * 32 * T_XROW);
    };
    auto cvt = [&](int q, int g) {
      typedef __bf16 bf16x2_t __attribute__((ext_vector_type(2)));
      const uint32_t w0 = araw[q >> 1][g][2 * (q & 1)], w1 = araw[q >> 1][g][2 * (q & 1) + 1];
      const bf16x2_t c0 = __builtin_amdgcn_cvt_scalef32_pk_bf16_fp8(w0, 1.f, false);
      const bf16x2_t c1 = __builtin_amdgcn_cvt_scalef32_pk_bf16_fp8(w0, 1.f, true);
      const bf16x2_t c2 = __builtin_amdgcn_cvt_scalef32_pk_bf16_fp8(w1, 1.f, false);
      const bf16x2_t c3 = __builtin_amdgcn_cvt_scalef32_pk_bf16_fp8(w1, 1.f, true);
      av[q & 1][g] = bf16x8{c0[0], c0[1], c1[0], c1[1], c2[0], c2[1], c3[0], c3[1]};
    };
    read_a(0);
    read_b(0);
    __builtin_amdgcn_sched_barrier(0);
    if (!ODD) {
#pragma unroll
      for (int h = NT - 2; h < 2 * (NT - LATE); ++h) rescale(h, r);
      __builtin_amdgcn_sched_barrier(0);
    }
    cvt(0, 0);
    cvt(0, 1);
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int q = 0; q < 4; ++q) {
#pragma unroll
      for (int g = 0; g < 2; ++g)
#pragma unroll
        for (int j = 0; j < NJ; ++j) {
          const int i = g * NJ + j;
          acc[g][j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(av[q & 1][g], as_bf16x8(bx[q & 1][j]), acc[g][j], 0, 0, 0);
          // (the reads go out behind the first MFMA: the wait before it covers
          // every LDS read in flight)
          if (i == 0 && q == 0) read_a(1);
          if (i == 0 && q < 3) read_b(q + 1);
          if (!ODD && q == 0 && i < 2 * LATE) rescale(2 * (NT - LATE) + i, r);
          if (ODD && q == 3 && i >= 2) rescale(i - 2, r);
          if (q < 3 && i == NT - 2) cvt(q + 1, 0);
          if (q < 3 && i == NT - 1) cvt(q + 1, 1);
          __builtin_amdgcn_sched_barrier(0);
        }
    }
  };
  float r[2] = {1.f, 1.f};
  for (int kb = a.kb0; kb < a.kb1; ++kb) {
    float sn[2];
#pragma unroll
    for (int g = 0; g < 2; ++g) sn[g] = srow[g][min(kb + 1, a.kb1 - 1)];
    stage(2 * kb, std::false_type{}, r);
#pragma unroll
    for (int g = 0; g < 2; ++g)
      r[g] = s_run[g] == 0.f || scale_bits(sn[g]) < sfloor[g] ? 1.f : __fdiv_rn(s_run[g], sn[g]);
    stage(2 * kb + 1, std::true_type{}, r);
    if (kb + 1 < a.kb1) {
#pragma unroll
      for (int g = 0; g < 2; ++g) {
        zero[g] = scale_bits(sn[g]) < sfloor[g];
        if (!zero[g]) s_run[g] = sn[g];
        sfloor[g] = max(sfloor[g], scale_floor(scale_bits(sn[g])));
      }
    }
  }
  // the tiles rescaled after the last block were so by s / s = 1
}
};

// Up to 64 rows, where the weight stream is the bound: the stages are whole 128 B
// lines of the weights, one segment of a K block at a time (16 KB: 128 rows x 128 B,
// three in the ring, two ahead), the activation rows a K block at a time (two
// buffers).  With stages of 64 K values of both segments every line was fetched
// in two halves: [gate | up] of 256 experts at 300 tokens took 1344 us against
// 1252, at 1000 tokens 1409 / 1317.
//
// LDS: weight row 128 B, chunk c of row r at c ^ ((r >> 1) & 7); activation row
// 256 B, chunk c of row r at c ^ (r & 15): the 16 lanes of a fragment-read pass
// hit distinct banks.  At 64 rows this is all of the 80 KB: the fragments of a
// block whose scale is zero are masked in registers.
constexpr int T_WSEG = 128 * 128;  // one segment of a K block
constexpr int T_XBLK = 256;        // activation row of a K block
static_assert(3 * T_WSEG + 2 * 64 * T_XBLK <= T_LDS, "stages exceed LDS");

template <int NJ, bool WIDE>
struct TileLines {
  static AMLA_DEV void run(const TileArgs &a, TileSums<NJ> &sums) {
  auto &acc = sums.acc;
  auto &s_run = sums.s_run;
  extern __shared__ __align__(16) uint8_t tsm[];
  constexpr int WC = 4, XC = 2 * NJ;  // copies per wave: a segment, the activation rows of a block
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int j32 = lane & 31, hh = lane >> 5;

  // copies: the wave's own 32 weight rows (8 rows of 128 B each) and its quarter
  // of the activation rows (4 rows of 256 B each), scalar bases plus lane offsets
  uint32_t woff[2][WC], xoff[XC];
  auto wchunk = [&](int c) { return 16 * ((lane & 7) ^ ((4 * c + (lane >> 4)) & 7)); };
#pragma unroll
  for (int g = 0; g < 2; ++g)
#pragma unroll
    for (int c = 0; c < WC; ++c)
    {
      const uint32_t wr = min(32 * wave + 8 * c + (lane >> 3), a.wrows[g] - 1);
      // a.wide, WIDE: the row index only, the offset is formed per copy
      woff[g][c] = WIDE ? wr : wr * (uint32_t)a.K + wchunk(c);
    }
  auto xchunk = [&](int c) { return 16 * ((lane & 15) ^ ((8 * NJ * wave + 4 * c + (lane >> 4)) & 15)); };
#pragma unroll
  for (int c = 0; c < XC; ++c) {
    const int rc = min(8 * NJ * wave + 4 * c + (lane >> 4), a.rows - 1);  // rows past the tile repeat its last row (not stored)
    const uint32_t xr = a.xrow ? a.xrow[rc] : rc;
    xoff[c] = a.wide ? xr : xr * ((uint32_t)a.ldx * 2) + xchunk(c);
  }
  typedef const __attribute__((address_space(1))) uint8_t *gptr;
  auto opaque = [](uint32_t v) {  // (keeps the copies on scalar bases, as above)
    asm volatile("" : "+v"(v));
    return v;
  };
  auto dma_w = [&](int kb, int g, int slot) {
    gptr wb = (gptr)(a.w[g] + (size_t)kb * 128);
    asm volatile("" : "+s"(wb));
    if constexpr (!WIDE) {
#pragma unroll
      for (int c = 0; c < WC; ++c)
        __builtin_amdgcn_global_load_lds(wb + opaque(woff[g][c]), LDS_PTR(tsm + slot * T_WSEG + (32 * wave + 8 * c) * 128), 16, 0, 0);
    } else {
#pragma unroll
      for (int c = 0; c < WC; ++c)
        __builtin_amdgcn_global_load_lds(wb + (size_t)woff[g][c] * a.K + wchunk(c),
                                         LDS_PTR(tsm + slot * T_WSEG + (32 * wave + 8 * c) * 128), 16, 0, 0);
    }
  };
  auto dma_x = [&](int kb, int buf) {
    gptr xb = (gptr)(reinterpret_cast<const uint8_t *>(a.x) + (size_t)kb * T_XBLK);
    asm volatile("" : "+s"(xb));
    uint8_t *dst = tsm + 3 * T_WSEG + (buf * 32 * NJ + 8 * NJ * wave) * T_XBLK;
    if (!a.wide) {
#pragma unroll
      for (int c = 0; c < XC; ++c)
        __builtin_amdgcn_global_load_lds(xb + opaque(xoff[c]), LDS_PTR(dst + 4 * c * T_XBLK), 16, 0, 0);
    } else {
#pragma unroll
      for (int c = 0; c < XC; ++c)
        __builtin_amdgcn_global_load_lds(xb + (size_t)xoff[c] * a.ldx * 2 + xchunk(c), LDS_PTR(dst + 4 * c * T_XBLK), 16, 0, 0);
    }
  };

  const __attribute__((address_space(4))) float *srow[2];
#pragma unroll
  for (int g = 0; g < 2; ++g) srow[g] = (const __attribute__((address_space(4))) float *)(a.s[g]);
#pragma unroll
  for (int g = 0; g < 2; ++g)
#pragma unroll
    for (int j = 0; j < NJ; ++j)
#pragma unroll
      for (int r = 0; r < 16; ++r) acc[g][j][r] = 0.f;
  // (units of the accumulators: as in TileHalves)
#pragma unroll
  for (int g = 0; g < 2; ++g) s_run[g] = srow[g][a.kb0];
  asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");

  dma_w(a.kb0, 0, 0);
  dma_x(a.kb0, 0);
  dma_w(a.kb0, 1, 1);
  int sfloor[2] = {scale_floor(scale_bits(s_run[0])), scale_floor(scale_bits(s_run[1]))};
  uint32_t keep[2] = {s_run[0] == 0.f ? 0u : ~0u, s_run[1] == 0.f ? 0u : ~0u};
  int slot = 0, buf = 0;
  // One segment of a K block: eight sub-steps of 16 (K 32 pr + 16 hh + 8 s2 ..
  // +7 of each half-wave).  `other`: the other segment's sums change their units
  // by r meanwhile (segment 0's to the next block, segment 1's to this one).
  auto stage = [&](int kb, auto g_c, float r) {
    constexpr int G = decltype(g_c)::value;
    const bool more = kb + 1 < a.kb1;
    // issued after what this stage reads: segment 1 of this block; then, of the
    // next block, segment 0 and the activation rows
    if (G == 0) wait_vmcnt<WC>();
    else if (more) wait_vmcnt<WC + XC>();
    else wait_vmcnt<0>();
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
    if (more) {
      dma_w(kb + 1, G, slot == 0 ? 2 : slot - 1);
      if (G == 0) dma_x(kb + 1, buf ^ 1);
    }
    const uint8_t *sw = tsm + slot * T_WSEG + (32 * wave + j32) * 128;
    const uint8_t *sx = tsm + 3 * T_WSEG + (buf * 32 * NJ + j32) * T_XBLK;
    u32x4 aw[4], bx[8][NJ];
#pragma unroll
    for (int q = 0; q < 8; ++q) {
      if ((q & 1) == 0) aw[q >> 1] = *reinterpret_cast<const u32x4 *>(sw + 16 * ((q + hh) ^ ((j32 >> 1) & 7)));
#pragma unroll
      for (int j = 0; j < NJ; ++j)
        bx[q][j] = *reinterpret_cast<const u32x4 *>(sx + j * 32 * T_XBLK + 16 * ((4 * (q >> 1) + 2 * hh + (q & 1)) ^ (j32 & 15)));
    }
#pragma unroll
    for (int q = 0; q < 8; ++q) {
      typedef __bf16 bf16x2_t __attribute__((ext_vector_type(2)));
      const uint32_t w0 = aw[q >> 1][2 * (q & 1)] & keep[G], w1 = aw[q >> 1][2 * (q & 1) + 1] & keep[G];
      const bf16x2_t c0 = __builtin_amdgcn_cvt_scalef32_pk_bf16_fp8(w0, 1.f, false);
      const bf16x2_t c1 = __builtin_amdgcn_cvt_scalef32_pk_bf16_fp8(w0, 1.f, true);
      const bf16x2_t c2 = __builtin_amdgcn_cvt_scalef32_pk_bf16_fp8(w1, 1.f, false);
      const bf16x2_t c3 = __builtin_amdgcn_cvt_scalef32_pk_bf16_fp8(w1, 1.f, true);
      const bf16x8 av = bf16x8{c0[0], c0[1], c1[0], c1[1], c2[0], c2[1], c3[0], c3[1]};
#pragma unroll
      for (int j = 0; j < NJ; ++j) {
        acc[G][j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(av, as_bf16x8(bx[q][j]), acc[G][j], 0, 0, 0);
#pragma unroll
        for (int e = 0; e < 2; ++e) acc[1 - G][j][2 * q + e] *= r;
      }
    }
    slot = slot == 2 ? 0 : slot + 1;
  };
  float r1 = 1.f;
  for (int kb = a.kb0; kb < a.kb1; ++kb) {
    float sn[2], r[2];
#pragma unroll
    for (int g = 0; g < 2; ++g) sn[g] = srow[g][min(kb + 1, a.kb1 - 1)];
    stage(kb, std::integral_constant<int, 0>{}, r1);
#pragma unroll
    for (int g = 0; g < 2; ++g)
      r[g] = s_run[g] == 0.f || scale_bits(sn[g]) < sfloor[g] ? 1.f : __fdiv_rn(s_run[g], sn[g]);
    stage(kb, std::integral_constant<int, 1>{}, r[0]);
    r1 = r[1];
    buf ^= 1;
    if (kb + 1 < a.kb1) {
#pragma unroll
      for (int g = 0; g < 2; ++g) {
        keep[g] = scale_bits(sn[g]) < sfloor[g] ? 0u : ~0u;
        if (keep[g]) s_run[g] = sn[g];
        sfloor[g] = max(sfloor[g], scale_floor(scale_bits(sn[g])));
      }
    }
  }
  // segment 0's sums were rescaled after the last block by s / s = 1
  asm volatile("" ::: "memory");
}
};

template <int NJ, bool WIDE>
using TileMain = std::conditional_t<(NJ <= 2), TileLines<NJ, WIDE>, TileHalves<NJ, WIDE>>;

// Stores a tile.  SILU: y = bf16(silu(segment 0)) * segment 1, 128 columns;
// else y = both segments, 256 columns.
template <int NJ, bool SILU>
AMLA_DEV void tile_store(const TileArgs &a, const TileSums<NJ> &ts) {
  extern __shared__ __align__(16) uint8_t tsm[];
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int j32 = lane & 31, hh = lane >> 5;
  auto &acc = ts.acc;
  auto &s_run = ts.s_run;

  // Lane holds row 32 j + j32, columns 32 wave + 8 q + 4 hh .. +3 of each
  // segment.  The outputs go through LDS so that every store is 16 bytes of
  // one output row.
  __builtin_amdgcn_s_barrier();  // every wave is past its last fragment read
  asm volatile("" ::: "memory");
#pragma unroll
  for (int j = 0; j < NJ; ++j)
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      f32x4 v[2];
#pragma unroll
      for (int g = 0; g < 2; ++g)
        v[g] = f32x4{acc[g][j][4 * q], acc[g][j][4 * q + 1], acc[g][j][4 * q + 2], acc[g][j][4 * q + 3]} * s_run[g];
      const int col = 32 * wave + 8 * q + 4 * hh;
      if constexpr (SILU) {
        uint8_t *dst = tsm + (32 * j + j32) * T_PITCH_H + col * 2;
        float o[4];
#pragma unroll
        for (int i = 0; i < 4; ++i) o[i] = silu_bf16(round_bf16(v[0][i])) * round_bf16(v[1][i]);
        *reinterpret_cast<u32x2 *>(dst) = u32x2{pack_bf16(o[0], o[1]), pack_bf16(o[2], o[3])};
      } else {
        uint8_t *dst = tsm + (32 * j + j32) * T_PITCH_Y + col * 2;
#pragma unroll
        for (int g = 0; g < 2; ++g)
          *reinterpret_cast<u32x2 *>(dst + g * 256) = u32x2{pack_bf16(v[g].x, v[g].y), pack_bf16(v[g].z, v[g].w)};
      }
    }
  asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
  __builtin_amdgcn_s_barrier();
  asm volatile("" ::: "memory");
  constexpr int CPR = SILU ? 16 : 32;  // 16-byte chunks per row
  constexpr int PITCH = SILU ? T_PITCH_H : T_PITCH_Y;
  const int c = tid % CPR;
  if (SILU || a.two || c < 16) {
    for (int r = tid / CPR; r < a.rows; r += 256 / CPR) {
      const u32x4 v = *reinterpret_cast<const u32x4 *>(tsm + r * PITCH + c * 16);
      const int64_t yr = a.yrow ? a.yrow[r] : r;
      *reinterpret_cast<u32x4 *>(a.y + yr * a.ldy + 8 * c) = v;
    }
  }
}

// ---------------------------------------------------------------- linears of many rows

// The GEMM of launch_gemm (GemvMode epilogues): tiles of 256 weight rows x 128
// activation rows.  Workgroup i runs on XCD i % 8: each XCD takes a contiguous
// run of the tiles in panels of 8 column tiles, row tiles within a panel, so
// the 64 tiles it holds at a time share 8 + 8 tile operands through its L2;
// with up to 8 row tiles the row tiles of a column tile come together (the
// weights are then the larger operand).
constexpr int TL_PANEL = 8;

AMLA_DEV void tile_coords(int t, int n_tiles, int m_tiles, int &nt, int &mt) {
  if (m_tiles <= TL_PANEL) {
    nt = t / m_tiles;
    mt = t - nt * m_tiles;
    return;
  }
  const int per = TL_PANEL * m_tiles, p = t / per, r = t - p * per;
  const int width = min(TL_PANEL, n_tiles - p * TL_PANEL);
  mt = r / width;
  nt = p * TL_PANEL + r - mt * width;
}
// logical index of workgroup i of n (or -1): a contiguous run per XCD
AMLA_DEV int xcd_run(int i, int n) {
  const int run = (n + 7) >> 3, l = (i & 7) * run + (i >> 3);
  return (i >> 3) < run && l < n ? l : -1;
}

template <int MODE, int NJ, bool WIDE>
AMLA_DEV void tile_linear_body(const GemvParams &p, const TileArgs &a, int n0, int n1, int m0, bool staged,
                               float *partial) {
  extern __shared__ __align__(16) uint8_t tsm[];
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int j32 = lane & 31, hh = lane >> 5;
  TileSums<NJ> ts;
  TileMain<NJ, WIDE>::run(a, ts);
  auto &acc = ts.acc;
  auto &s_run = ts.s_run;
  auto sums = [&](int g, int j, int q) {
    return f32x4{acc[g][j][4 * q], acc[g][j][4 * q + 1], acc[g][j][4 * q + 2], acc[g][j][4 * q + 3]} * s_run[g];
  };
  if (partial) {
    // [g][j][wave][q][lane] f32x4: every store is 1 KB contiguous per wave
    f32x4 *dst = reinterpret_cast<f32x4 *>(partial);
#pragma unroll
    for (int g = 0; g < 2; ++g)
#pragma unroll
      for (int j = 0; j < NJ; ++j)
#pragma unroll
        for (int q = 0; q < 4; ++q) dst[(((g * 4 + j) * 4 + wave) * 4 + q) * 64 + lane] = sums(g, j, q);
    return;
  }
  if (MODE == GEMV_F32 || (MODE != GEMV_SILU && !staged)) {
    // fp32 rows, or rows without 16-byte alignment: four outputs per store straight from the accumulators
#pragma unroll
    for (int j = 0; j < NJ; ++j) {
      const int r = 32 * j + j32;
      if (r >= a.rows) continue;
#pragma unroll
      for (int g = 0; g < 2; ++g)
#pragma unroll
        for (int q = 0; q < 4; ++q) {
          const int c = 32 * wave + 8 * q + 4 * hh;
          if (c < a.wrows[g] && (g == 0 || a.two)) pstore4<MODE == GEMV_SILU ? GEMV_PLAIN : MODE>(p, m0 + r, (g ? n1 : n0) + c, sums(g, j, q));
        }
    }
    return;
  }
  if constexpr (MODE == GEMV_SILU) {
    tile_store<NJ, true>(a, ts);
    return;
  }
  __builtin_amdgcn_s_barrier();  // every wave is past its last fragment read
  asm volatile("" ::: "memory");
#pragma unroll
  for (int j = 0; j < NJ; ++j)
#pragma unroll
    for (int q = 0; q < 4; ++q)
#pragma unroll
      for (int g = 0; g < 2; ++g) {
        const f32x4 v = sums(g, j, q);
        *reinterpret_cast<u32x2 *>(tsm + (32 * j + j32) * T_PITCH_Y + g * 256 + (32 * wave + 8 * q + 4 * hh) * 2) =
            u32x2{pack_bf16(v.x, v.y), pack_bf16(v.z, v.w)};
      }
  asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
  __builtin_amdgcn_s_barrier();
  asm volatile("" ::: "memory");
  const int g = (tid >> 4) & 1, c = 8 * (tid & 15);
  const int n = (g ? n1 : n0) + c;
  if (c < (g ? a.wrows[1] : a.wrows[0]) && (g == 0 || a.two))
    for (int r = tid >> 5; r < a.rows; r += 8)
      pstore8<MODE == GEMV_SILU ? GEMV_PLAIN : MODE>(
          p, m0 + r, n, *reinterpret_cast<const u32x4 *>(tsm + r * T_PITCH_Y + (tid & 31) * 16));
}

// Workgroups [0, full): whole tiles; then K part (i - full) % parts of tile full + (i - full) / parts.
// WIDE: x or weight rows whose byte offsets from the tile's first row do not
// fit 32 bits, each formed in 64 per copy (a kernel of its own: with the choice
// made inside, 4096 x 7168 x 18432 took 4 % longer).
template <int MODE, bool WIDE>
__global__ __launch_bounds__(256, 2) void tile_linear_kernel(GemvParams p, bool staged, GemmSplit sp) {
  const int KB = p.K >> 7;
  int t, kb0 = 0, kb1 = KB;
  float *partial = nullptr;
  if ((int)blockIdx.x < sp.full_blocks) {
    t = xcd_run(blockIdx.x, sp.full);
    if (t < 0) return;
  } else {
    const int l = xcd_run(blockIdx.x - sp.full_blocks, sp.rest * sp.parts);
    if (l < 0) return;
    // K part q of `group` tiles at a time: the row tiles of a column tile read
    // the same weights
    const int per = sp.group * sp.parts, g = l / per, r = l - g * per;
    const int q = r / sp.group, st = g * sp.group + r - q * sp.group;
    t = sp.full + st;
    kb0 = q * KB / sp.parts;
    kb1 = (q + 1) * KB / sp.parts;
    partial = sp.partial + (size_t)(st * sp.parts + q) * TILE_PART_F32;
  }
  int nt, mt;
  tile_coords(t, sp.n_tiles, sp.m_tiles, nt, mt);
  TileArgs a;
  const int m0 = mt * TILE_ROWS;
  a.rows = min(TILE_ROWS, p.M - m0);
  a.K = p.K;
  a.ldx = p.ldx;
  a.kb0 = kb0;
  a.kb1 = kb1;
  a.x = p.x + (size_t)m0 * p.ldx;
  a.xrow = nullptr;
  a.wide = WIDE;
  // segment = a run of up to 128 rows of one weight: the first weight's
  // segments come before the second's (n_split % 128 == 0)
  int n0[2];
  a.two = true;
  if constexpr (MODE == GEMV_SILU) {
#pragma unroll
    for (int g = 0; g < 2; ++g) {
      n0[g] = nt * 128;
      a.w[g] = (g ? p.w1 : p.w0) + (size_t)n0[g] * p.K;
      a.s[g] = (g ? p.s1 : p.s0) + (size_t)nt * KB;
      a.wrows[g] = 128;
    }
    a.y = p.y + (size_t)m0 * p.ldy + n0[0];
    a.yrow = nullptr;
    a.ldy = p.ldy;
  } else
#pragma unroll
  for (int g = 0; g < 2; ++g) {
    int n = nt * 256 + g * 128;
    if (g == 1) {
      a.two = n < p.N;
      if (!a.two) n = nt * 256;  // no second segment: the first is multiplied twice
    }
    n0[g] = n;
    const bool second = p.w1 && n >= p.n_split;
    const int nl = second ? n - p.n_split : n;
    a.w[g] = (second ? p.w1 : p.w0) + (size_t)nl * p.K;
    a.s[g] = (second ? p.s1 : p.s0) + (size_t)(nl >> 7) * KB;
    a.wrows[g] = min(128, (p.w1 && !second ? p.n_split : p.N) - n);
  }
  switch ((a.rows + 31) >> 5) {
    case 1: tile_linear_body<MODE, 1, WIDE>(p, a, n0[0], n0[1], m0, staged, partial); break;
    case 2: tile_linear_body<MODE, 2, WIDE>(p, a, n0[0], n0[1], m0, staged, partial); break;
    case 3: tile_linear_body<MODE, 3, WIDE>(p, a, n0[0], n0[1], m0, staged, partial); break;
    default: tile_linear_body<MODE, 4, WIDE>(p, a, n0[0], n0[1], m0, staged, partial); break;
  }
}

// Sums the K parts of the split tiles in part order and applies the epilogue.
// Workgroup = 32 rows x 128 columns (row group j of segment g, or of both for
// SILU) of one split tile: the parts are read in the lane order they were
// written, summed in part order, staged in LDS as rows, and stored 8 outputs
// per thread through the same epilogue as the staged tiles.
template <int MODE>
__global__ __launch_bounds__(256) void tile_finish_kernel(GemvParams p, GemmSplit sp) {
  constexpr bool SILU = MODE == GEMV_SILU;
  constexpr int SEGS = SILU ? 2 : 1;
  __shared__ float rows[32][128 + 4];
  const int tid = threadIdx.x;
  const int st = blockIdx.x >> (SILU ? 2 : 3), g = SILU ? 0 : (blockIdx.x >> 2) & 1, j = blockIdx.x & 3;
  int nt, mt;
  tile_coords(sp.full + st, sp.n_tiles, sp.m_tiles, nt, mt);
  const int m0 = mt * TILE_ROWS + 32 * j, n0 = SILU ? nt * 128 : nt * 256 + g * 128;
  if (m0 >= p.M || n0 >= p.N) return;
  const f32x4 *src = reinterpret_cast<const f32x4 *>(sp.partial + (size_t)st * sp.parts * TILE_PART_F32) +
                     (g * 4 + j) * 1024 + (tid >> 6) * 256 + (tid & 63);
  f32x4 sum[SEGS][4];
#pragma unroll
  for (int s = 0; s < SEGS; ++s)
#pragma unroll
    for (int q = 0; q < 4; ++q) sum[s][q] = src[s * 4096 + q * 64];
#pragma unroll 4
  for (int k = 1; k < sp.parts; ++k)
#pragma unroll
    for (int s = 0; s < SEGS; ++s)
#pragma unroll
      for (int q = 0; q < 4; ++q) sum[s][q] += src[(size_t)k * (TILE_PART_F32 / 4) + s * 4096 + q * 64];
#pragma unroll
  for (int q = 0; q < 4; ++q) {
    f32x4 v = sum[0][q];
    if constexpr (SILU)
#pragma unroll
      for (int i = 0; i < 4; ++i) v[i] = silu_bf16(round_bf16(v[i])) * round_bf16(sum[SEGS - 1][q][i]);
    *reinterpret_cast<f32x4 *>(&rows[tid & 31][32 * (tid >> 6) + 8 * q + 4 * ((tid >> 5) & 1)]) = v;
  }
  __syncthreads();
#pragma unroll
  for (int k = 0; k < 2; ++k) {
    const int r = (tid >> 4) + 16 * k, c = (tid & 15) * 8;
    if (m0 + r >= p.M || n0 + c >= p.N) continue;
    const float *v = &rows[r][c];
    if constexpr (MODE == GEMV_F32) {
      pstore4<MODE>(p, m0 + r, n0 + c, f32x4{v[0], v[1], v[2], v[3]});
      pstore4<MODE>(p, m0 + r, n0 + c + 4, f32x4{v[4], v[5], v[6], v[7]});
    } else {
      pstore8<SILU ? GEMV_PLAIN : MODE>(
          p, m0 + r, n0 + c,
          u32x4{pack_bf16(v[0], v[1]), pack_bf16(v[2], v[3]), pack_bf16(v[4], v[5]), pack_bf16(v[6], v[7])});
    }
  }
}

// ---------------------------------------------------------------- routed experts

template <int NJ, bool SILU>
AMLA_DEV void tile_body(const TileArgs &a) {
  TileSums<NJ> ts;
  TileMain<NJ, false>::run(a, ts);
  tile_store<NJ, SILU>(a, ts);
}

template <bool SILU>
AMLA_DEV void tile_dispatch(const TileArgs &a) {
  switch ((a.rows + 31) >> 5) {
    case 1: tile_body<1, SILU>(a); break;
    case 2: tile_body<2, SILU>(a); break;
    case 3: tile_body<3, SILU>(a); break;
    default: tile_body<4, SILU>(a); break;
  }
}

// Column tile nt of the rows g.first .. of one expert.
//   GATEUP: h (first + r, n) = bf16(silu(gate)) * up of x row xrow[r]
//   else:   y row yrow[r] = down projection of h row (first + r)
// (null row lists: row first + r).
template <bool GATEUP>
AMLA_DEV void moe_tile(const MoeTileParams &p, const TileGroup &g, int nt, const int32_t *xrow, const int32_t *yrow) {
  TileArgs a;
  a.rows = g.rows;
  a.K = p.K;
  a.ldx = p.ldx;
  a.ldy = p.ldy;
  const int KB = p.K >> 7;
  a.x = xrow ? p.x : p.x + (size_t)g.first * p.ldx;
  a.wide = xrow && p.wide;
  a.xrow = xrow;
  a.y = (yrow ? p.y : p.y + (size_t)g.first * p.ldy) + nt * (GATEUP ? 128 : 256);
  a.yrow = yrow;
  a.kb0 = 0;
  a.kb1 = KB;
  a.wrows[0] = a.wrows[1] = 128;
  a.two = GATEUP || nt * 256 + 128 < p.N;  // N % 256 == 128: the last tile multiplies its one segment twice
  a.w[0] = static_cast<const uint8_t *>(g.w0) + (size_t)nt * (GATEUP ? 128 : 256) * p.K;
  a.s[0] = g.s0 + (size_t)nt * (GATEUP ? 1 : 2) * KB;
  if constexpr (GATEUP) {
    a.w[1] = static_cast<const uint8_t *>(g.w1) + (size_t)nt * 128 * p.K;
    a.s[1] = g.s1 + (size_t)nt * KB;
  } else {
    a.w[1] = a.two ? a.w[0] + (size_t)128 * p.K : a.w[0];
    a.s[1] = a.two ? a.s[0] + KB : a.s[0];
  }
  tile_dispatch<GATEUP>(a);
}

// Tiles of the routed experts from a device schedule.  Workgroup i runs on XCD
// i % 8 (round-robin dispatch): entry t is computed by XCD t % 8, its column
// tiles one after another, so the group's activation rows are read from that
// XCD's L2.  Entries past the count return at once.
template <bool GATEUP>
__global__ __launch_bounds__(256, 2) void tile_sched_kernel(MoeTileParams p, MoeSched s) {
  const int xcd = blockIdx.x & 7, k = blockIdx.x >> 3;
  const int t = (k / p.ntiles) * 8 + xcd, nt = k % p.ntiles;
  if (t >= *s.count) return;
  const int32_t *en = s.ent + 4 * t;
  const int e = en[0], r0 = en[1];
  const void *const *wt = s.wtab + (GATEUP ? 0 : 4) * s.E;
  TileGroup g;
  g.w0 = wt[e];
  g.s0 = static_cast<const float *>(wt[s.E + e]);
  g.w1 = GATEUP ? wt[2 * s.E + e] : nullptr;
  g.s1 = GATEUP ? static_cast<const float *>(wt[3 * s.E + e]) : nullptr;
  g.first = r0;
  g.rows = en[2];
  moe_tile<GATEUP>(p, g, nt, GATEUP ? s.rowmap + r0 : nullptr, GATEUP ? nullptr : s.rowmap + r0);
}

// The same tiles from a host list (rows by position on both sides).
template <bool GATEUP>
__global__ __launch_bounds__(256, 2) void tile_grouped_kernel(MoeTileParams p, TileGroups gr) {
  const int xcd = blockIdx.x & 7, k = blockIdx.x >> 3;
  const int t = (k / p.ntiles) * 8 + xcd, nt = k % p.ntiles;
  if (t >= gr.n) return;
  moe_tile<GATEUP>(p, gr.g[t], nt, nullptr, nullptr);
}

static int check_tiles(const MoeTileParams &p) {
  if (p.K % 128 || p.N % 128 || p.ldx % 8 || p.ldy % 8 || !aligned16(p.x) || !aligned16(p.y) || p.K > T_MAX_LD ||
      p.ldx > T_MAX_LD)
    return fail(AMLA_EUNSUPPORTED,
                "expert fp8 tiles need K %% 128 == 0, N %% 128 == 0, 16-byte aligned rows and K, ldx <= %d", T_MAX_LD);
  return AMLA_OK;
}

static int tile_lds(const void *fn) {  // dynamic LDS above 64 KB
  const hipError_t e = hipFuncSetAttribute(fn, hipFuncAttributeMaxDynamicSharedMemorySize, T_LDS);
  return e == hipSuccess ? AMLA_OK : fail((int)e, "expert fp8 tiles: LDS size: %s", hipGetErrorString(e));
}

int launch_tile_sched(const MoeTileParams &p0, const MoeSched &s, int max_entries, hipStream_t st) {
  if (max_entries <= 0) return AMLA_OK;
  MoeTileParams p = p0;
  int rc = check_tiles(p);
  if (rc) return rc;
  p.ntiles = s.down ? (p.N + 255) / 256 : p.N / 128;
  const int64_t blocks = (int64_t)((max_entries + 7) / 8) * 8 * p.ntiles;
  if (blocks > INT32_MAX) return fail(AMLA_EUNSUPPORTED, "scheduled fp8 tiles: %d entries", max_entries);
  if ((rc = tile_lds(s.down ? (const void *)tile_sched_kernel<false> : (const void *)tile_sched_kernel<true>))) return rc;
  if (s.down) tile_sched_kernel<false><<<dim3((unsigned)blocks), 256, T_LDS, st>>>(p, s);
  else tile_sched_kernel<true><<<dim3((unsigned)blocks), 256, T_LDS, st>>>(p, s);
  return check_launch("scheduled fp8 tiles");
}

int launch_tile_grouped(const MoeTileParams &p0, const TileGroups &gr, bool down, hipStream_t st) {
  if (gr.n <= 0) return AMLA_OK;
  MoeTileParams p = p0;
  int rc = check_tiles(p);
  if (rc) return rc;
  p.ntiles = down ? (p.N + 255) / 256 : p.N / 128;
  const int64_t blocks = (int64_t)((gr.n + 7) / 8) * 8 * p.ntiles;
  if (blocks > INT32_MAX) return fail(AMLA_EUNSUPPORTED, "grouped fp8 tiles: N = %d", p.N);
  if ((rc = tile_lds(down ? (const void *)tile_grouped_kernel<false> : (const void *)tile_grouped_kernel<true>))) return rc;
  if (down) tile_grouped_kernel<false><<<dim3((unsigned)blocks), 256, T_LDS, st>>>(p, gr);
  else tile_grouped_kernel<true><<<dim3((unsigned)blocks), 256, T_LDS, st>>>(p, gr);
  return check_launch("grouped fp8 tiles");
}

// Workgroups: 512 run at a time (two per CU).  Tiles past the last full round
// are cut into K parts where that shortens the launch.  Measured on MI355X, a
// 128-wide K block of a 128-row tile takes 3.7 us with two workgroups per CU
// and 2.1 us with one; writing and reading a part's sums (128 KB) adds about
// 0.03 us each, the finishing pass 5 us of its own.  Against every part count
// from 1 to 16 at N = 576, 4096, 7168, 24576 and 100-1000 rows the plan is
// within 5 % of the best (7168 x 16384: 100 rows 50 us in 9 parts, 228 in one;
// 333 rows 106 in 3; 1000 rows 242 in 2, 267 in one).
//
// More than 256 tiles past the last full round: 256 of them run whole, one per
// CU, and the K parts of the others share the CUs with them at first (two per
// CU for `kb` blocks, then one).  The parts end long before the launch does,
// but their finish is not hidden (8 us with the disturbance measured).
// 7168 x 16384 at 1400 rows 381 -> 350 us; q_a | kv_a at 4096 rows (288 tiles)
// 177 -> 159, finish included; o_proj at 4096 rows 882 -> 838; 24576 x 1536 at
// 333 rows (288 tiles of 12 blocks) 47 either way, left whole.
GemmSplit plan_gemm_split(int M, int N, int K, int mode) {
  GemmSplit sp = {};
  const int cols = mode == GEMV_SILU ? 128 : 256;
  sp.n_tiles = (N + cols - 1) / cols;
  sp.m_tiles = (M + TILE_ROWS - 1) / TILE_ROWS;
  const int tiles = sp.n_tiles * sp.m_tiles;
  const int KB = K / 128;
  const int full = tiles / 512 * 512, rest = tiles - full;
  const double nj = (std::min(M, TILE_ROWS) + 31) / 32;
  const double one = 0.9 + 0.3 * nj, two = std::max(1.3, 0.925 * nj);  // us per K block
  auto cost_of = [&](int parts) {
    const int items = rest * parts, last = items % 512;
    const double kb = (KB + parts - 1) / parts;
    const double rounds = items / 512 * two + (last == 0 ? 0.0 : last <= 256 ? one : two);
    return rounds * kb + (parts > 1 ? 5.0 + items * 0.03 * nj / 4 : 0.0);
  };
  int best = 1;
  double best_cost = rest ? cost_of(1) : 0.0;
  for (int s = 2; s <= std::min(GEMM_MAX_PARTS, KB) && rest; ++s) {
    const double cost = cost_of(s);
    if (cost < best_cost * 0.97) {
      best_cost = cost;
      best = s;
    }
  }
  sp.full = best > 1 ? full : tiles;
  if (rest > 256) {
    const int whole = sp.m_tiles <= TL_PANEL ? (full + 256) / sp.m_tiles * sp.m_tiles : full + 256;
    const int over = tiles - whole, s = std::min({256 / std::max(1, over), GEMM_MAX_PARTS, KB});
    if (s > 1) {
      const int kb = (KB + s - 1) / s;
      const double cost = kb * two + (KB - kb) * one + 8.0 + over * s * 0.03 * nj / 4;
      if (cost < best_cost * 0.97) {
        best = s;
        sp.full = whole;
      }
    }
  }
  sp.rest = tiles - sp.full;
  sp.parts = best;
  sp.group = sp.m_tiles <= TL_PANEL && sp.full % sp.m_tiles == 0 ? sp.m_tiles : 1;
  sp.full_blocks = (sp.full + 7) / 8 * 8;
  sp.bytes = (size_t)sp.rest * (best > 1 ? best : 0) * TILE_PART_F32 * 4;
  return sp;
}

size_t gemm_ws_bytes(int M, int N, int K, int mode) { return plan_gemm_split(M, N, K, mode).bytes; }

template <int MODE>
static int launch_tile_linear(const GemvParams &p, bool staged, const GemmSplit &sp, hipStream_t st) {
  // the epilogue modes' rows are packed: only x of the plain ones has a stride of its own
  constexpr bool STRIDED = MODE == GEMV_PLAIN || MODE == GEMV_F32;
  const bool wide = p.ldx > T_MAX_LD || p.K > T_MAX_LD;
  if (wide && !STRIDED) return fail(AMLA_EUNSUPPORTED, "fp8 GEMM: rows of %d elements in epilogue mode %d", p.ldx, MODE);
  const auto kernel = wide ? tile_linear_kernel<MODE, STRIDED> : tile_linear_kernel<MODE, false>;
  int rc = tile_lds((const void *)kernel);
  if (rc) return rc;
  const unsigned blocks = (unsigned)(sp.full_blocks + (sp.rest * sp.parts + 7) / 8 * 8);
  kernel<<<dim3(blocks), 256, T_LDS, st>>>(p, staged, sp);
  if ((rc = check_launch("fp8 GEMM")) || !sp.rest) return rc;
  tile_finish_kernel<MODE><<<dim3((unsigned)sp.rest * (MODE == GEMV_SILU ? 4 : 8)), 256, 0, st>>>(p, sp);
  return check_launch("fp8 GEMM K-part finish");
}

int launch_gemm(const GemvParams &p, int mode, hipStream_t st, float *split_ws, size_t split_ws_bytes) {
  if (p.K % 128 || p.N % 4) return fail(AMLA_EUNSUPPORTED, "fp8 GEMM needs K %% 128 == 0 and N %% 4 == 0");
  if (p.ldx % 8) return fail(AMLA_EUNSUPPORTED, "fp8 GEMM needs 16-byte aligned activation rows");
  if ((mode == GEMV_QKVA && p.max_rows <= 0) || (mode == GEMV_QROPE && p.rope_rows <= 0))
    return fail(AMLA_EINVAL, "fp8 GEMM: cache rows / rope rows of the epilogue not set");
  if (mode == GEMV_SILU && (p.N % 128 || p.ldy % 8 || !aligned16(p.y) || !p.w1))
    return fail(AMLA_EUNSUPPORTED, "fp8 GEMM: silu * up needs two weights of N %% 128 == 0 rows and 16-byte aligned rows");
  if (mode != GEMV_SILU && p.w1 && p.n_split % 128)
    return fail(AMLA_EUNSUPPORTED, "fp8 GEMM: the first weight segment must be a multiple of 128 rows");
  // 16-byte output stores need N, the row strides and the bases of every
  // output (and of the residual) on 8-element boundaries
  bool staged = p.N % 8 == 0 && p.ldy % 8 == 0 && aligned16(p.y);
  if (mode == GEMV_RESID) staged = staged && p.ldr % 8 == 0 && aligned16(p.res);
  if (mode == GEMV_QKVA)
    staged = staged && aligned16(p.ckv) && aligned16(p.kpe) && p.kv_lora % 8 == 0 && p.rope % 8 == 0 &&
             p.ckv_bstride % 8 == 0 && p.kpe_bstride % 8 == 0;
  if (mode == GEMV_QROPE) staged = staged && p.head_dim % 8 == 0 && p.nope % 8 == 0;
  if (mode == GEMV_F32) staged = p.N % 8 == 0 && p.ldy % 4 == 0 && aligned16(p.y);
  GemmSplit sp = plan_gemm_split(p.M, p.N, p.K, mode);
  if (sp.rest && (!staged || !split_ws || split_ws_bytes < sp.bytes || !aligned16(split_ws))) {
    // no room for the partial sums (or outputs without 16-byte stores): whole tiles
    sp.full = sp.n_tiles * sp.m_tiles;
    sp.rest = 0;
    sp.parts = 1;
    sp.full_blocks = (sp.full + 7) / 8 * 8;
  }
  sp.partial = split_ws;
  switch (mode) {
    case GEMV_PLAIN: return launch_tile_linear<GEMV_PLAIN>(p, staged, sp, st);
    case GEMV_RESID: return launch_tile_linear<GEMV_RESID>(p, staged, sp, st);
    case GEMV_QKVA: return launch_tile_linear<GEMV_QKVA>(p, staged, sp, st);
    case GEMV_QROPE: return launch_tile_linear<GEMV_QROPE>(p, staged, sp, st);
    case GEMV_F32: return launch_tile_linear<GEMV_F32>(p, staged, sp, st);
    case GEMV_SILU: return launch_tile_linear<GEMV_SILU>(p, staged, sp, st);
    default: return fail(AMLA_EINVAL, "fp8 GEMM: unknown epilogue mode %d", mode);
  }
}

}  // namespace amla
