// Epilogues of the large-M fp8 GEMM kernels (the modes of GemvMode; the skinny
// GEMM's own are in fp8_linear.hip, same contract).
#pragma once

#include "amla_common.h"
#include "amla_internal.h"

namespace amla {

AMLA_DEV int prow_position(const GemvParams &p, int m) { return p.pos[m / p.seq_len] + m % p.seq_len; }

template <int MODE>
AMLA_DEV void pstore4(const GemvParams &p, int m, int n, f32x4 v) {
  if (MODE == GEMV_PLAIN) {
    u32x2 o = {pack_bf16(v.x, v.y), pack_bf16(v.z, v.w)};
    *reinterpret_cast<u32x2 *>(p.y + (size_t)m * p.ldy + n) = o;
  } else if (MODE == GEMV_F32) {
    *reinterpret_cast<f32x4 *>(reinterpret_cast<float *>(p.y) + (size_t)m * p.ldy + n) = v;
  } else if (MODE == GEMV_RESID) {
    const u32x2 r = *reinterpret_cast<const u32x2 *>(p.res + (size_t)m * p.ldr + n);
    u32x2 o = {pack_bf16(lo_bf(r.x) + round_bf16(v.x), hi_bf(r.x) + round_bf16(v.y)),
               pack_bf16(lo_bf(r.y) + round_bf16(v.z), hi_bf(r.y) + round_bf16(v.w))};
    *reinterpret_cast<u32x2 *>(p.y + (size_t)m * p.ldy + n) = o;
  } else if (MODE == GEMV_QKVA) {
    u32x2 o = {pack_bf16(v.x, v.y), pack_bf16(v.z, v.w)};
    if (n < p.n_split) {
      *reinterpret_cast<u32x2 *>(p.y + (size_t)m * p.ldy + n) = o;
    } else {
      const int b = m / p.seq_len;
      const int64_t row = prow_position(p, m);
      if (row >= p.max_rows) return;  // a device position past the cache: nothing is written
      const int nn = n - p.n_split;
      uint16_t *dst = nn < p.kv_lora ? p.ckv + b * p.ckv_bstride + row * p.kv_lora + nn
                                     : p.kpe + b * p.kpe_bstride + row * p.rope + (nn - p.kv_lora);
      *reinterpret_cast<u32x2 *>(dst) = o;
    }
  } else {
    float a0 = round_bf16(v.x), a1 = round_bf16(v.y), a2 = round_bf16(v.z), a3 = round_bf16(v.w);
    const int d = n % p.head_dim;
    if (d >= p.nope) {
      const int i = (d - p.nope) >> 1;
      const int64_t row = min(prow_position(p, m), p.rope_rows - 1);  // in bounds for any device position
      const f32x4 cs = *reinterpret_cast<const f32x4 *>(p.rope_table + (row * (p.rope >> 1) + i) * 2);
      const float r0 = __fsub_rn(__fmul_rn(a0, cs.x), __fmul_rn(a1, cs.y));
      const float r1 = __fadd_rn(__fmul_rn(a0, cs.y), __fmul_rn(a1, cs.x));
      const float r2 = __fsub_rn(__fmul_rn(a2, cs.z), __fmul_rn(a3, cs.w));
      const float r3 = __fadd_rn(__fmul_rn(a2, cs.w), __fmul_rn(a3, cs.z));
      a0 = r0; a1 = r1; a2 = r2; a3 = r3;
    }
    u32x2 o = {pack_bf16(a0, a1), pack_bf16(a2, a3)};
    *reinterpret_cast<u32x2 *>(p.y + (size_t)m * p.ldy + n) = o;
  }
}

// Eight consecutive outputs n .. n+7 (n % 8 == 0) already rounded to bf16.
template <int MODE>
AMLA_DEV void pstore8(const GemvParams &p, int m, int n, u32x4 v) {
  if (MODE == GEMV_F32) {
    // not reached: fp32 outputs take the unstaged epilogue (launch_gemm)
  } else if (MODE == GEMV_PLAIN) {
    *reinterpret_cast<u32x4 *>(p.y + (size_t)m * p.ldy + n) = v;
  } else if (MODE == GEMV_RESID) {
    const u32x4 r = *reinterpret_cast<const u32x4 *>(p.res + (size_t)m * p.ldr + n);
    u32x4 o;
#pragma unroll
    for (int i = 0; i < 4; ++i) o[i] = pack_bf16(lo_bf(r[i]) + lo_bf(v[i]), hi_bf(r[i]) + hi_bf(v[i]));
    *reinterpret_cast<u32x4 *>(p.y + (size_t)m * p.ldy + n) = o;
  } else if (MODE == GEMV_QKVA) {
    if (n < p.n_split) {
      *reinterpret_cast<u32x4 *>(p.y + (size_t)m * p.ldy + n) = v;
    } else {
      const int b = m / p.seq_len;
      const int64_t row = prow_position(p, m);
      if (row >= p.max_rows) return;  // a device position past the cache: nothing is written
      const int nn = n - p.n_split;
      uint16_t *dst = nn < p.kv_lora ? p.ckv + b * p.ckv_bstride + row * p.kv_lora + nn
                                     : p.kpe + b * p.kpe_bstride + row * p.rope + (nn - p.kv_lora);
      *reinterpret_cast<u32x4 *>(dst) = v;
    }
  } else {
    const int d = n % p.head_dim;
    u32x4 o = v;
    if (d >= p.nope) {
      const int64_t row = min(prow_position(p, m), p.rope_rows - 1);  // in bounds for any device position
      const float *tab = p.rope_table + (row * (p.rope >> 1) + ((d - p.nope) >> 1)) * 2;
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const float a0 = lo_bf(v[i]), a1 = hi_bf(v[i]);
        const float c = tab[2 * i], s = tab[2 * i + 1];
        o[i] = pack_bf16(__fsub_rn(__fmul_rn(a0, c), __fmul_rn(a1, s)), __fadd_rn(__fmul_rn(a0, s), __fmul_rn(a1, c)));
      }
    }
    *reinterpret_cast<u32x4 *>(p.y + (size_t)m * p.ldy + n) = o;
  }
}

}  // namespace amla
