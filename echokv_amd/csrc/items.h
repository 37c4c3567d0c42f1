// Items of the kernels that dequantize stored tokens into registers or LDS (prefill.hip,
// decode_any.hip): four consecutive keys of one block, chunk and K group x eight
// channels of a head, loaded whole and converted later.
#pragma once

#include "args.h"

namespace ek {

__device__ __forceinline__ h2_t u2h(uint32_t u) { return __builtin_bit_cast(h2_t, u); }

// Eight codes, `sh` bits into the 8 bytes w, as fp16 pairs (exact). A byte b < 16 read as
// E4M3 is b * 2^-9, so the fp8 conversion with scale 2^9 gives INT4 / INT2 codes; INT8
// codes take the exponent of 1024.
template <int BITS>
__device__ __forceinline__ void code_pairs(uint2 w, int sh, h2_t c[4]) {
  if constexpr (BITS == 8) {
    const uint32_t m = 0x64646464u;
    const h2_t k = {(_Float16)1024.0f, (_Float16)1024.0f};
    c[0] = u2h(__builtin_amdgcn_perm(m, w.x, 0x04010400u)) - k;
    c[1] = u2h(__builtin_amdgcn_perm(m, w.x, 0x04030402u)) - k;
    c[2] = u2h(__builtin_amdgcn_perm(m, w.y, 0x04010400u)) - k;
    c[3] = u2h(__builtin_amdgcn_perm(m, w.y, 0x04030402u)) - k;
  } else {
    const uint32_t x = (uint32_t)(((uint64_t)w.y << 32 | w.x) >> sh);
    uint32_t a, b;  // channels 0..3, 4..7, a byte each
    if constexpr (BITS == 4) {
      const uint32_t lo = x & 0x0f0f0f0fu, hi = (x >> 4) & 0x0f0f0f0fu;  // even / odd channels
      a = __builtin_amdgcn_perm(hi, lo, 0x05010400u);
      b = __builtin_amdgcn_perm(hi, lo, 0x07030602u);
    } else {
      const uint32_t y0 = x & 0x03030303u, y1 = (x >> 2) & 0x03030303u;  // byte b of y_k: channel 4b + k
      const uint32_t y2 = (x >> 4) & 0x03030303u, y3 = (x >> 6) & 0x03030303u;
      const uint32_t p = __builtin_amdgcn_perm(y1, y0, 0x05010400u), q = __builtin_amdgcn_perm(y3, y2, 0x05010400u);
      a = __builtin_amdgcn_perm(q, p, 0x05040100u);
      b = __builtin_amdgcn_perm(q, p, 0x07060302u);
    }
    c[0] = __builtin_amdgcn_cvt_scalef32_pk_f16_fp8(a, 512.0f, false);
    c[1] = __builtin_amdgcn_cvt_scalef32_pk_f16_fp8(a, 512.0f, true);
    c[2] = __builtin_amdgcn_cvt_scalef32_pk_f16_fp8(b, 512.0f, false);
    c[3] = __builtin_amdgcn_cvt_scalef32_pk_f16_fp8(b, 512.0f, true);
  }
}

// The item of a layout whose items can straddle groups or chunks (block sizes or K groups
// that are not powers of two, V groups that are not multiples of 8, head sizes with half
// an octet): channels [ch, ch + 8) of head h of the keys (KEY) or values at offsets
// [off, off + 4) of a block, the first `live` of them (others, chunks out of range and
// channels past the head: zeros). Runs of four channels (head sizes are multiples of
// 4) take one load each, and nothing is used before all of the item is requested.
template <bool KEY>
__device__ __forceinline__ void item_general(const Lay& L, const uint8_t* pages, const Res& res, long blk,
                                             const Hdr& hd, long rs, int rg, int off, int bits, int live, int h, int ch,
                                             float (*y)[8]) {
  typedef _Float16 h4_any_t __attribute__((ext_vector_type(4), aligned(2)));
  const uint8_t* pg = pages + blk * L.stride;
  const int D = L.D, G = D / L.VG;
  const uint8_t* p[4][2];
  bool ok[4][2];
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const long rb = i < live ? row_base_h(L, blk, hd, off + i, bits) : -1;
    const uint8_t* row = pages + rb + ((KEY ? 0 : L.H * D) + h * D) * bits / 8;
#pragma unroll
    for (int r = 0; r < 2; ++r) {
      ok[i][r] = rb >= 0 && ch + 4 * r < D;
      p[i][r] = ok[i][r] ? row + (ch + 4 * r) * bits / 8 : pg;
    }
  }
  uint32_t c[4][2];
  auto codes = [&](auto word) {
    using W = decltype(word);
#pragma unroll
    for (int i = 0; i < 4; ++i)
#pragma unroll
      for (int r = 0; r < 2; ++r) c[i][r] = *(const W*)p[i][r];
  };
  if (bits == 4) codes(uint16_t{});
  else if (bits == 2) codes(uint8_t{});
  else codes(uint32_t{});
  const uint32_t mask = (1u << bits) - 1u;
  auto put = [&](int i, int r, const float* s, const float* m) {
#pragma unroll
    for (int e = 0; e < 4; ++e)
      y[i][4 * r + e] = ok[i][r] ? __builtin_fmaf((float)((c[i][r] >> (e * bits)) & mask), s[e], m[e]) : 0.f;
  };
  if constexpr (KEY) {
    const bool one = L.KG % 4 == 0;  // the four keys share a K group (offsets are multiples of 4)
    h4_any_t s4[2], m4[2];
    auto stats = [&](int i) {
#pragma unroll
      for (int r = 0; r < 2; ++r) {
        const long se = ((long)((off + i) / L.KG) * L.H + h) * D + (ch + 4 * r < D ? ch + 4 * r : 0);
        s4[r] = *(const h4_any_t*)(pg + L.o_ks + 2 * se);
        m4[r] = *(const h4_any_t*)(pg + L.o_km + 2 * se);
      }
    };
    stats(0);
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      if (i > 0 && !one && i < live) stats(i);
#pragma unroll
      for (int r = 0; r < 2; ++r) {
        float s[4], m[4];
#pragma unroll
        for (int e = 0; e < 4; ++e) s[e] = (float)s4[r][e], m[e] = (float)m4[r][e];
        put(i, r, s, m);
      }
    }
    if ((unsigned long)rs < (unsigned long)res.rows) {  // the block's open K group
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        if (rg != (off + i) / L.KG) continue;
#pragma unroll
        for (int r = 0; r < 2; ++r)
          if (ok[i][r])
            ld4(res.ptr, res.dtype, rs * res.s0 + (long)((off + i) % L.KG) * res.s1 + h * res.s2 + ch + 4 * r, &y[i][4 * r]);
      }
    }
  } else if (L.VG % 4 == 0) {  // a run is in one V group
    float s[4][2], m[4][2];
#pragma unroll
    for (int i = 0; i < 4; ++i)
#pragma unroll
      for (int r = 0; r < 2; ++r) {
        const long ve = ((long)(off + i) * L.H + h) * G + (ch + 4 * r < D ? ch + 4 * r : 0) / L.VG;
        s[i][r] = (float)*f16p(pages, blk * L.stride + L.o_vs + 2 * ve);
        m[i][r] = (float)*f16p(pages, blk * L.stride + L.o_vm + 2 * ve);
      }
#pragma unroll
    for (int i = 0; i < 4; ++i)
#pragma unroll
      for (int r = 0; r < 2; ++r) {
        const float s4[4] = {s[i][r], s[i][r], s[i][r], s[i][r]}, m4[4] = {m[i][r], m[i][r], m[i][r], m[i][r]};
        put(i, r, s4, m4);
      }
  } else {
#pragma unroll
    for (int i = 0; i < 4; ++i)
#pragma unroll
      for (int r = 0; r < 2; ++r) {
        float s[4], m[4];
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          const long ve = ((long)(off + i) * L.H + h) * G + (ch + 4 * r < D ? ch + 4 * r + e : 0) / L.VG;
          s[e] = (float)*f16p(pages, blk * L.stride + L.o_vs + 2 * ve);
          m[e] = (float)*f16p(pages, blk * L.stride + L.o_vm + 2 * ve);
        }
        put(i, r, s, m);
      }
  }
}

}  // namespace ek
