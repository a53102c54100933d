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

}  // namespace q35
