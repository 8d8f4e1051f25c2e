// Block-FP8 GEMM tiles of 256 weight rows x up to 128 activation rows for gfx950:
// the routed experts' groups of more than 16 rows (amla_moe_experts_dev).
//
// y[m, n] = sum_k x[m, k] w[n, k] scale_inv[n/128, k/128], w e4m3fn converted
// exactly to bf16 in registers, 32x32x16 bf16 MFMAs, fp32 sums.
#include <type_traits>

#include "amla_common.h"
#include "amla_internal.h"

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
// 1.28 ms (5.9 TB/s), down 0.66 ms, where the skinny GEMM with fp32 K parts and
// finishing passes took 1.55 + 0.82 ms; 2000 tokens (62 rows) 1.66 + 0.89 ms
// against 2.75 + 1.62 for that and 256 x 256 tiles for groups above 64 rows;
// 8000 tokens (250 rows) 4.8 + 2.4 ms against 5.6 + 2.9.  Gathering and
// scattering the rows here saved two more passes (0.14 ms at 2000 tokens).
//
// K stages of 64 in LDS: fp8 weight rows (64 B, chunk c of row r at
// c ^ ((r >> 2) & 3)), bf16 activation rows (128 B, chunk c of row r at
// c ^ ((r >> 1) & 7)): the 16 lanes of each fragment-read pass hit distinct
// banks.  Three stages for up to 64 rows, two above (80 KB).
constexpr int T_BK = 64;
constexpr int T_WBYTES = 256 * T_BK;             // weight part of a stage
constexpr int T_XROW = T_BK * 2;                 // activation row of a stage
constexpr int T_LDS = 80 * 1024;
constexpr int T_ZERO = T_LDS - 16;               // weight fragments of a block whose scale is zero
constexpr int T_PITCH_H = 128 * 2 + 16;          // epilogue rows in LDS: 128 or 256 bf16 outputs
constexpr int T_PITCH_Y = 256 * 2 + 16;
static_assert(128 * T_PITCH_Y <= T_ZERO, "staged output tile exceeds LDS");
constexpr int tile_stages(int nj) { return nj <= 2 ? 3 : 2; }
static_assert(tile_stages(2) * (T_WBYTES + 64 * T_XROW) <= T_ZERO && tile_stages(4) * (T_WBYTES + 128 * T_XROW) <= T_ZERO,
              "stages exceed LDS");

struct TileArgs {
  const uint8_t *w[2];   // first row of each segment
  const float *s[2];     // scale row (K / 128) of each segment
  const uint16_t *x;     // activation rows
  const int32_t *xrow;   // row of x for tile row r, or null: row r
  uint16_t *y;           // outputs, column 0 of the tile
  const int32_t *yrow;   // row of y for tile row r, or null: row r
  int ldx, ldy, K, rows;
  bool two;              // segment 1 is stored (PLAIN; always multiplied)
};

template <int NJ, bool SILU>
AMLA_DEV void tile_body(const TileArgs &a) {
  extern __shared__ __align__(16) uint8_t tsm[];
  constexpr int NST = tile_stages(NJ);
  constexpr int STAGE = T_WBYTES + 32 * NJ * T_XROW;
  constexpr int COPIES = 4 + NJ;  // per wave and stage
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int j32 = lane & 31, hh = lane >> 5;
  const int KB = a.K >> 7;

  // copies: the wave's own 2 x 32 weight rows (16 rows of 64 B each) and its
  // quarter of the activation rows (8 rows of 128 B each)
  const uint32_t wlane = (uint32_t)(lane >> 2) * a.K + 16 * ((lane & 3) ^ ((lane >> 4) & 3));
  const uint8_t *wsrc[2];
#pragma unroll
  for (int g = 0; g < 2; ++g) wsrc[g] = a.w[g] + (size_t)(32 * wave) * a.K;
  const uint8_t *xsrc[NJ];
#pragma unroll
  for (int c = 0; c < NJ; ++c) {
    const int r = 8 * (NJ * wave + c) + (lane >> 3);
    const int rc = min(r, a.rows - 1);  // rows past the tile repeat its last row (not stored)
    const int64_t xr = a.xrow ? a.xrow[rc] : rc;
    xsrc[c] = reinterpret_cast<const uint8_t *>(a.x + xr * a.ldx) + 16 * ((lane & 7) ^ ((r >> 1) & 7));
  }
  auto dma = [&](int it, int stg) {
    uint8_t *st = tsm + stg * STAGE;
#pragma unroll
    for (int g = 0; g < 2; ++g)
#pragma unroll
      for (int c = 0; c < 2; ++c)
        __builtin_amdgcn_global_load_lds(wsrc[g] + (size_t)(16 * c) * a.K + it * T_BK + wlane,
                                         LDS_PTR(st + (128 * g + 32 * wave + 16 * c) * T_BK), 16, 0, 0);
#pragma unroll
    for (int c = 0; c < NJ; ++c)
      __builtin_amdgcn_global_load_lds(xsrc[c] + it * T_XROW, LDS_PTR(st + T_WBYTES + 8 * (NJ * wave + c) * T_XROW),
                                       16, 0, 0);
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

  f32x16 acc[2][NJ];
#pragma unroll
  for (int g = 0; g < 2; ++g)
#pragma unroll
    for (int j = 0; j < NJ; ++j)
#pragma unroll
      for (int r = 0; r < 16; ++r) acc[g][j][r] = 0.f;
  // The accumulators are kept in units of the current K block's scale, as in
  // the 256 x 256 GEMM: acc *= s_prev / s_cur on entering a block, * s_last at
  // the end (fp32 rounding of the ratios, ~1e-5 relative over 128 blocks).  A
  // zero scale dequantises to zeros: the segment's fragments of that block are
  // read from 16 zeroed bytes instead.
  float s_run[2] = {0.f, 0.f};
  bool skip[2] = {false, false};

  if (tid < 4) *reinterpret_cast<uint32_t *>(tsm + T_ZERO + 4 * tid) = 0;  // visible after the first barrier
  asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");

  const int iters = 2 * KB;
#pragma unroll
  for (int i = 0; i < NST - 1; ++i) dma(i, i);  // iters >= 2 >= NST - 1
  int stg = 0;
  for (int it = 0; it < iters; ++it) {
    if (NST == 3 && it + 1 < iters) wait_vmcnt<COPIES>();
    else wait_vmcnt<0>();
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
    if (it + NST - 1 < iters) dma(it + NST - 1, stg == 0 ? NST - 1 : stg - 1);
    if ((it & 1) == 0) {
#pragma unroll
      for (int g = 0; g < 2; ++g) {
        const float sk = srow[g][it >> 1];
        skip[g] = sk == 0.f;
        if (!skip[g]) {
          if (s_run[g] != 0.f) {
            const float r = __fdiv_rn(s_run[g], sk);
#pragma unroll
            for (int j = 0; j < NJ; ++j) acc[g][j] *= r;
          }
          s_run[g] = sk;
        }
      }
    }
    // Four sub-steps of 16 (K 32 pr + 16 hh + 8 s2 .. +7 of each half-wave);
    // the fragments of the next one are read while the current one multiplies.
    const uint8_t *st = tsm + stg * STAGE;
    const uint8_t *sa[2];
#pragma unroll
    for (int g = 0; g < 2; ++g) sa[g] = skip[g] ? tsm + T_ZERO : st + g * 128 * T_BK;
    u32x4 araw[2][2], bx[2][NJ];
    auto read_a = [&](int pr) {
#pragma unroll
      for (int g = 0; g < 2; ++g) araw[pr][g] = *reinterpret_cast<const u32x4 *>(sa[g] + (skip[g] ? 0 : aoff[pr]));
    };
    auto read_b = [&](int q) {
#pragma unroll
      for (int j = 0; j < NJ; ++j)
        bx[q & 1][j] = *reinterpret_cast<const u32x4 *>(st + boff[q >> 1][q & 1] + j * 32 * T_XROW);
    };
    read_a(0);
    read_b(0);
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      if (q < 3) read_b(q + 1);
      if (q == 1) read_a(1);
      __builtin_amdgcn_sched_barrier(0);
      typedef __bf16 bf16x2_t __attribute__((ext_vector_type(2)));
#pragma unroll
      for (int g = 0; g < 2; ++g) {
        const uint32_t w0 = araw[q >> 1][g][2 * (q & 1)], w1 = araw[q >> 1][g][2 * (q & 1) + 1];
        const bf16x2_t c0 = __builtin_amdgcn_cvt_scalef32_pk_bf16_fp8(w0, 1.f, false);
        const bf16x2_t c1 = __builtin_amdgcn_cvt_scalef32_pk_bf16_fp8(w0, 1.f, true);
        const bf16x2_t c2 = __builtin_amdgcn_cvt_scalef32_pk_bf16_fp8(w1, 1.f, false);
        const bf16x2_t c3 = __builtin_amdgcn_cvt_scalef32_pk_bf16_fp8(w1, 1.f, true);
        const bf16x8 av = {c0[0], c0[1], c1[0], c1[1], c2[0], c2[1], c3[0], c3[1]};
#pragma unroll
        for (int j = 0; j < NJ; ++j)
          acc[g][j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(av, as_bf16x8(bx[q & 1][j]), acc[g][j], 0, 0, 0);
      }
      __builtin_amdgcn_sched_barrier(0);
    }
    stg = stg == NST - 1 ? 0 : stg + 1;
  }

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
  a.xrow = xrow;
  a.y = (yrow ? p.y : p.y + (size_t)g.first * p.ldy) + nt * (GATEUP ? 128 : 256);
  a.yrow = yrow;
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
  if (p.K % 128 || p.N % 128 || p.ldx % 8 || p.ldy % 8 || !aligned16(p.x) || !aligned16(p.y))
    return fail(AMLA_EUNSUPPORTED, "expert fp8 tiles need K %% 128 == 0, N %% 128 == 0 and 16-byte aligned rows");
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

}  // namespace amla
