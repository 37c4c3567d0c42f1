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

}  // namespace ek
