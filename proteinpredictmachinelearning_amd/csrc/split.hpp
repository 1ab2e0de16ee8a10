// Binary32 numbers as two halves under a power of two (see gemm_f16x2.hip for what the arithmetic is and what it costs).
#pragma once
#include "common.hpp"

namespace ppmlhip {

typedef _Float16 v8h __attribute__((ext_vector_type(8)));
typedef short v4s __attribute__((ext_vector_type(4)));

constexpr int SPLIT16_TERMS[3][2] = {{1, 0}, {0, 1}, {0, 0}};      // (part of a, part of b), smallest first
constexpr int SPLIT16_MOST = 126;                                  // the largest power of two an operand is scaled by
// A fragment of 32 rows x 16 columns in LDS: two halves (columns 0 .. 7 and 8 .. 15) of 32 rows x 16 bytes, 576 bytes apart:
// row reads, transposing reads and eight-byte writes then touch every bank once.
constexpr int SPLIT16_HALF = 576, SPLIT16_FRAG = 2 * SPLIT16_HALF;

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

__device__ __forceinline__ v8h pack_halves(const uint2& lo, const uint2& hi) {
    return __builtin_bit_cast(v8h, v4i{static_cast<int>(lo.x), static_cast<int>(lo.y), static_cast<int>(hi.x), static_cast<int>(hi.y)});
}

// 2^e; zero below the normal numbers (e at most 127)
__device__ __forceinline__ float power_of_two(int e) { return __uint_as_float(static_cast<uint32_t>(e < -127 ? 0 : e + 127) << 23); }

// the largest finite magnitude
__device__ __forceinline__ float max_finite4(float m, const v4f& x) {
#pragma unroll
    for (int c = 0; c < 4; ++c) {
        const float a = __builtin_fabsf(x[c]);
        m = fmaxf(m, a < INFINITY ? a : 0.0f);
    }
    return m;
}

// the exponent of the power of two that brings a largest magnitude (its bits) to 2^14 .. 2^15; SPLIT16_MOST for zero and for tiny ones
__device__ __forceinline__ int split16_exponent(uint32_t top) {
    const int e = 141 - static_cast<int>(top >> 23);
    return e > SPLIT16_MOST ? SPLIT16_MOST : e;
}

// over lanes l and l ^ 32
__device__ __forceinline__ uint32_t max_across_halves(uint32_t v) {
    const uint32_t o = __shfl_xor(v, 32, 64);
    return o > v ? o : v;
}

// over all 64 lanes
__device__ __forceinline__ uint32_t max_across_wave(uint32_t v) {
#if defined(__HIP_DEVICE_COMPILE__)
    const auto meet = [&](uint32_t o) { v = o > v ? o : v; };
    meet(__builtin_amdgcn_update_dpp(0, v, 0x128, 0xf, 0xf, true));      // row_ror:8
    meet(__builtin_amdgcn_update_dpp(0, v, 0x124, 0xf, 0xf, true));      // row_ror:4
    meet(__builtin_amdgcn_update_dpp(0, v, 0x4e, 0xf, 0xf, true));
    meet(__builtin_amdgcn_update_dpp(0, v, 0xb1, 0xf, 0xf, true));
    meet(__shfl_xor(v, 16, 64));
    meet(__shfl_xor(v, 32, 64));
#endif
    return v;
}

// eight 16-bit elements of this lane's column, four rows at `at` and four at `at + step`, each piece transposed on the
// way (a group of sixteen lanes names four rows of sixteen columns, four columns per lane)
__device__ __forceinline__ v8h read_transposed16(const uint8_t* at, int step) {
#if defined(__HIP_DEVICE_COMPILE__)
    typedef __attribute__((address_space(3))) v4s* lds_v4s;
    const v4s lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_v4s)(at));
    const v4s hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_v4s)(at + step));
    return __builtin_bit_cast(v8h, __builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7));
#else
    return v8h{};
#endif
}

}  // namespace ppmlhip
