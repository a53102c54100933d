// Block sizes of the quantized formats and the workspace form of Q8_K blocks,
// shared by the projection kernels.
#pragma once

#include "common.h"

namespace q35 {

constexpr int QK = 256;
constexpr int Q4K_BYTES = 144, Q6K_BYTES = 210, Q5K_BYTES = 176, IQ4XS_BYTES = 136, Q2_BYTES = 130, STQ_BYTES = 42;
// Workspace form of a Q8_K block, 304 bytes (19 x 16): dword 0 d, dwords 4..67
// qs (16-byte aligned), dwords 68..75 bsums; dwords 1..3 unused.
constexpr int Q8K_WORDS = 76;
constexpr int Q8K_QS = 4, Q8K_BS = 68;

typedef int i32x4 __attribute__((ext_vector_type(4)));
typedef float f32x4 __attribute__((ext_vector_type(4)));

__device__ __forceinline__ float half_bits_to_float(uint32_t h) {
    return static_cast<float>(__builtin_bit_cast(_Float16, static_cast<uint16_t>(h)));
}

typedef short s16x2 __attribute__((ext_vector_type(2)));

// Four unsigned 6-bit values given doubled (bytes of v2 = 2 v) times sc, as
// the low (& 127) and high (>> 7, two's complement) int8 planes of the
// products sc v.  The doubled 16-bit products 2 sc v are formed in pairs:
// the high plane is their high bytes, the low plane bits 1-7 of their low
// bytes.
__device__ __forceinline__ void q6k_split(uint32_t v2, int sc, uint32_t& lo, uint32_t& hi) {
    const s16x2 s2 = {(short)sc, (short)sc};
    const uint32_t a = __builtin_bit_cast(uint32_t, __builtin_bit_cast(s16x2, __builtin_amdgcn_perm(0u, v2, 0x0c010c00u)) * s2);
    const uint32_t b = __builtin_bit_cast(uint32_t, __builtin_bit_cast(s16x2, __builtin_amdgcn_perm(0u, v2, 0x0c030c02u)) * s2);
    lo = (__builtin_amdgcn_perm(b, a, 0x06040200u) >> 1) & 0x7f7f7f7fu;
    hi = __builtin_amdgcn_perm(b, a, 0x07050301u);
}

// Four IQ4_XS grid values (IQ4XS.cs:15-18) of four 4-bit indices, one a byte:
// two byte permutes (entries 0-7 and 8-15) and a select on the index's bit 3.
__device__ __forceinline__ uint32_t iq4_grid(uint32_t idx) {
    // grid bytes: -127 -104 -83 -65 | -49 -35 -22 -10 | 1 13 25 38 | 53 69 89 113
    const uint32_t g0 = 0xBFAD9881u, g1 = 0xF6EADDCFu, g2 = 0x26190D01u, g3 = 0x71594535u;
    const uint32_t sel = idx & 0x07070707u;
    const uint32_t m = ((idx >> 3) & 0x01010101u) * 0xffu;
    const uint32_t lo = __builtin_amdgcn_perm(g1, g0, sel), hi = __builtin_amdgcn_perm(g3, g2, sel);
    return (lo & ~m) | (hi & m);
}

// The four-lane patterns of four STQ1_0 groups, one a byte: h the groups' 4-bit
// slots, s4 their signs.  The slots spread to bytes are looked up in the two
// 16-byte codebook halves (STQ1_0.Codebook, entries 0-15 for sign 0 and 16-31
// for sign 1, 4 a dword), the half chosen per byte by the sign.
__device__ __forceinline__ uint32_t stq_patterns(uint32_t h, uint32_t s4) {
    constexpr uint32_t L0 = 0x092989A9u, L1 = 0x062686A6u, L2 = 0x121A929Au, L3 = 0x424A626Au;
    constexpr uint32_t H0 = 0xA1812101u, H1 = 0xA4842404u, H2 = 0x98901810u, H3 = 0x68604840u;
    const uint32_t idx = (h & 0xfu) | ((h & 0xf0u) << 4) | ((h & 0xf00u) << 8) | ((h & 0xf000u) << 12);
    const uint32_t sel = idx & 0x07070707u;
    const uint32_t hib = ((idx >> 3) & 0x01010101u) * 0xffu;
    const uint32_t lo = (__builtin_amdgcn_perm(L1, L0, sel) & ~hib) | (__builtin_amdgcn_perm(L3, L2, sel) & hib);
    const uint32_t hi = (__builtin_amdgcn_perm(H1, H0, sel) & ~hib) | (__builtin_amdgcn_perm(H3, H2, sel) & hib);
    const uint32_t neg = ((s4 * 0x00204081u) & 0x01010101u) * 0xffu;
    return (lo & ~neg) | (hi & neg);
}

}  // namespace q35
