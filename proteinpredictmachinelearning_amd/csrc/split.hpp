// Binary32 numbers as two halves under a power of two (see gemm_f16x2.hip for what the arithmetic is and what it costs).
#pragma once
#include "common.hpp"

namespace ppmlhip {

typedef _Float16 v8h __attribute__((ext_vector_type(8)));

// two halves of four consecutive elements times s
__device__ __forceinline__ void split4_f16(const v4f& x, float s, uint2 (&out)[2]) {
    typedef _Float16 v4h __attribute__((ext_vector_type(4)));
    v4h h, l;
#pragma unroll
    for (int c = 0; c < 4; ++c) {
        h[c] = static_cast<_Float16>(__builtin_fmaf(x[c], s, 0.0f));
        l[c] = static_cast<_Float16>(__builtin_fmaf(x[c], s, -static_cast<float>(h[c])));       // (the difference is exact)
    }
    out[0] = __builtin_bit_cast(uint2, h);
    out[1] = __builtin_bit_cast(uint2, l);
}

}  // namespace ppmlhip
