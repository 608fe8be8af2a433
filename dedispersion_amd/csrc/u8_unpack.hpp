// u8_unpack.hpp -- unpacking of packed rows (inputBits 1, 2 or 4,
// include/Dedispersion.hpp:92-103) to one byte per sample, shared by the
// staged kernels over byte rows.
#pragma once

#include "staged_common.hpp"

namespace ddamd {
namespace staged {

// The 16 samples of window group m (one byte each, 4 dwords u) and the 4
// after them (`next`) from the packed dwords d[0..2], which start at the
// dword holding packed byte 16m >> LF; LF = log2 of samples per byte (1..3).
// Samples are the fields of each byte from the least significant bit up.
template <int LF>
__device__ __forceinline__ void unpack_group(const u32x4 &d, uint32_t m, uint32_t (&u)[4], uint32_t &next) {
  if constexpr (LF == 1) {
    // 4-bit fields, 64 bits from d[0] and d[1] (the next 4 samples in the low
    // half of d[2]): even fields to the bytes of `lo`, odd fields to those
    // of `hi`, interleaved
#pragma unroll
    for (int e = 0; e < 3; ++e) {
      const uint32_t lo = d[e] & 0x0F0F0F0Fu, hi = (d[e] >> 4) & 0x0F0F0F0Fu;
      const uint32_t a = __builtin_amdgcn_perm(hi, lo, 0x05010400u);
      if (e < 2) {
        u[2 * e] = a;
        u[2 * e + 1] = __builtin_amdgcn_perm(hi, lo, 0x07030602u);
      } else {
        next = a;
      }
    }
  } else if constexpr (LF == 2) {
    // 2-bit fields, 32 bits from d[0] (the next 4 samples in the low byte of
    // d[1]): m_j byte k = sample 4k + j; two rounds of byte interleave
    const uint32_t x = d[0];
    const uint32_t m0 = x & 0x03030303u, m1 = (x >> 2) & 0x03030303u;
    const uint32_t m2 = (x >> 4) & 0x03030303u, m3 = (x >> 6) & 0x03030303u;
    const uint32_t a01 = __builtin_amdgcn_perm(m1, m0, 0x05010400u);  // s0 s1 s4 s5
    const uint32_t a23 = __builtin_amdgcn_perm(m3, m2, 0x05010400u);  // s2 s3 s6 s7
    const uint32_t b01 = __builtin_amdgcn_perm(m1, m0, 0x07030602u);  // s8 s9 s12 s13
    const uint32_t b23 = __builtin_amdgcn_perm(m3, m2, 0x07030602u);  // s10 s11 s14 s15
    u[0] = __builtin_amdgcn_perm(a23, a01, 0x05040100u);
    u[1] = __builtin_amdgcn_perm(a23, a01, 0x07060302u);
    u[2] = __builtin_amdgcn_perm(b23, b01, 0x05040100u);
    u[3] = __builtin_amdgcn_perm(b23, b01, 0x07060302u);
    const uint32_t y = d[1];
    const uint32_t c01 = __builtin_amdgcn_perm((y >> 2) & 0x03030303u, y & 0x03030303u, 0x05010400u);
    const uint32_t c23 = __builtin_amdgcn_perm((y >> 6) & 0x03030303u, (y >> 4) & 0x03030303u, 0x05010400u);
    next = __builtin_amdgcn_perm(c23, c01, 0x05040100u);
  } else {
    // 1-bit fields, 16 bits from bit 16 (m & 1) of d[0]: a nibble n spread to
    // bytes by n * (1 + 2^7 + 2^14 + 2^21), whose four shifted copies do not
    // overlap, then bit 0 of each byte kept
    const uint32_t x = __builtin_amdgcn_alignbit(d[1], d[0], 16 * (m & 1));
#pragma unroll
    for (int q = 0; q < 4; ++q) u[q] = (((x >> (4 * q)) & 0xFu) * 0x204081u) & 0x01010101u;
    next = (((x >> 16) & 0xFu) * 0x204081u) & 0x01010101u;
  }
}

} // namespace staged
} // namespace ddamd
