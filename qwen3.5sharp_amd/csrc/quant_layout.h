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

}  // namespace q35
