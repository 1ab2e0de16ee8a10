// What the binary32 contractions of this library share: the description of a contraction, the reference's own loop for
// outputs whose operands a split cannot carry, and the stores of compound outputs.
#pragma once
#include "split.hpp"

namespace ppmlhip {

struct GemmParams {
    const float* A;       // rows m: A(m,k) = A[m*a_rs + k*a_ks]
    const float* B;       // cols n: B(n,k) = B[n*b_rs + k*b_ks]
    float* C;
    const float* bias;    // [N] or null
    int M, N, K;
    int64_t a_rs, a_ks, b_rs, b_ks;
    // planes: p = p3*np2 + p2
    int np2, np3;
    int64_t a_p2, a_p3, b_p2, b_p3, c_p2, c_p3;
    int b_div2, b_div3;   // B-side plane index = p / div (out_prod's src0 broadcast)
    float alpha;
    // C(m,n) = C[(m/c_lm)*c_mo + (m%c_lm)*c_mi + (n/c_ln)*c_no + (n%c_ln)*c_ni]
    int c_lm, c_ln;
    int64_t c_mo, c_mi, c_no, c_ni;
    int tiles_m, tiles_n;
    int stream_c;         // output larger than the last-level cache: write it with streaming stores
    uint32_t c_span;      // compound output: bytes from C to behind a plane's last element where buffer addressing reaches them, else 0
    int f16_in;           // A and B hold IEEE halves (k contiguous); products and sums are binary32
    int clamp;            // finite guard in the epilogue (triangle multiplication)
    // LOAD_SPLIT_A: both indices of A are compound, A(m,k) = A[(m/a_lm)*a_mo + (m%a_lm)*a_mi + (k/a_lk)*a_ko + (k%a_lk)*a_ki]
    int a_lm, a_lk;
    int64_t a_mo, a_mi, a_ko, a_ki;
    // the sums over k of A's rows, which the forms with K slices leave beside the product (a linear layer's bias gradient, whose
    // terms its weight gradient reads anyway); null where nobody wants them, and again once they are taken care of
    float* row_sums;
};

// What reduce_slices_kernel adds up besides: partial[part][pad] of `rows` sums, parts in their order
struct RowSumParts {
    const float* partial;
    float* out;
    int rows, parts, pad;
};

// Workspace of a contraction: the pool's, or out of the array that the caller brings (`fixed`, of `cap` bytes: the pool is then
// never touched); null where there is none.  Given back by workspace_give either way.
inline Workspace workspace_take(size_t bytes, hipStream_t stream, uint8_t* fixed, size_t cap) {
    if (!fixed) return workspace_take(bytes, stream);
    Workspace ws;
    ws.ptr = bytes <= cap ? fixed : nullptr;
    return ws;
}

// gemm_f16x2.hip: a large single-plane contraction in two f16 parts; -1 when the contraction is not of the kind that form is
// for or no workspace is to be had.  `fixed_ws` / `fixed_cap`: a workspace the caller brings.
// sums_done: set where p.row_sums has been seen to.
int try_f16x2(const GemmParams& p, hipStream_t stream, const char* what, uint8_t* fixed_ws, size_t fixed_cap, bool& sums_done);
// f32_gemm.hip: C = alpha * (bias + sum over the slices of partial[slice][ma_pad][nb_pad]), NaN sums redone the reference's way
int launch_reduce_slices(const GemmParams& p, hipStream_t stream, const char* what, const float* partial, int slices, int ma_pad, int nb_pad,
                         const RowSumParts& sums);
int launch_reduce_slices_pair(const GemmParams& a, const GemmParams& b, hipStream_t stream, const char* what, const float* partial_a, const float* partial_b,
                              int slices, int ma_pad, int nb_pad);
// gemm_f16x2.hip: both gradients of an outer-product-mean, in shared launches; -1 as above, `wanted` where either by itself would take
// that form all the same
int try_f16x2_pair(const GemmParams& a, const GemmParams& b, hipStream_t stream, const char* what, bool& wanted);
// How many K slices make `groups` output tiles come out even over the CUs (f32_gemm.hip)
int even_slices(int groups, int chunks, int most_slices, int least_chunks);

namespace {

// Lanes outside the matrix carry this byte offset, which no buffer resource reaches (planes below 2 GiB).
constexpr uint32_t OUTSIDE = 0x80000000u;

// One output the reference's way (src/backend/CPUKernels.cpp:763-771, 836-884, 1006-1028): from the bias (or zero),
// one product at a time, k ascending, every product and every sum rounded to binary32 on its own (this file is
// compiled without contraction).  A and B are the plane's bases.
__device__ __forceinline__ float plain_dot(const GemmParams& p, const float* __restrict__ A, const float* __restrict__ B, int m, int n) {
    float s = p.bias ? p.bias[n] : 0.0f;
    const int64_t ra = p.a_lm > 0 ? static_cast<int64_t>(m / p.a_lm) * p.a_mo + static_cast<int64_t>(m % p.a_lm) * p.a_mi
                                  : static_cast<int64_t>(m) * p.a_rs;
    const float* b = B + static_cast<int64_t>(n) * p.b_rs;
    for (int k = 0; k < p.K; ++k) {
        const float a = p.a_lm > 0 ? A[ra + static_cast<int64_t>(k / p.a_lk) * p.a_ko + static_cast<int64_t>(k % p.a_lk) * p.a_ki]
                                   : A[ra + static_cast<int64_t>(k) * p.a_ks];
        const float prod = a * b[static_cast<int64_t>(k) * p.b_ks];
        s = s + prod;
    }
    return s;
}

// A whole tile of the output (rows x cols from (m0, n0) of the plane whose bases are A, B, C) by plain_dot, written
// straight to C with the contraction's own output addressing: what a work-group does INSTEAD of storing its
// accumulators when a SplitGuard fired for the tile.  One loop, no use of the accumulators: the ordinary path pays
// nothing for it but the test.
__device__ __forceinline__ void plain_tile(const GemmParams& p, const float* __restrict__ A, const float* __restrict__ B,
                                           float* __restrict__ C, int m0, int n0, int rows, int cols, int tid, int step = 256) {
    for (int e = tid; e < rows * cols; e += step) {
        const int m = m0 + e / cols, n = n0 + e % cols;
        if (m >= p.M || n >= p.N) continue;
        const float v = plain_dot(p, A, B, m, n) * p.alpha;
        C[static_cast<int64_t>(m / p.c_lm) * p.c_mo + static_cast<int64_t>(m % p.c_lm) * p.c_mi +
          static_cast<int64_t>(n / p.c_ln) * p.c_no + static_cast<int64_t>(n % p.c_ln) * p.c_ni] = v;
    }
}

// SPLIT_C of the kernels below: how the output is addressed.  The two compound forms are instances of their own: with both
// stores in one kernel, chosen by p.c_span as it ran, the general one cost 1 to 2.5 us more per launch (32 features x 24
// residues x 8 sequences 14.0 -> 16.5 us, the value form at 8 x 8 x 33 13.5 -> 15.6).
constexpr int C_DENSE = 0, C_COMPOUND = 1, C_COMPOUND_BUFFER = 2;

// The same for an output with compound addressing whose planes 32-bit byte offsets reach (p.c_span, set by the launcher:
// below 2 GiB, row runs of at least 32).  The general form above spends 36 vector instructions per stored register on
// 64-bit addresses, carries and bounds, in a phase without matrix work (a third of all issue cycles of the contraction of
// 12288 x 12288 outputs over 256).  Here a tile of 32 rows that stays within one run and inside the matrix -- known per
// wave -- takes its row steps from scalar registers: a product and a store.  Other tiles pick the run per row.  Measured,
// with both gradients: 384 residues x 32 features x 256 sequences 1342 -> 1239 us, 103 residues 152 -> 145.
// One tile row, rows from m_base (a multiple of 32, the same for the wave), columns from n_base:
template <bool STREAM_C, int TJ>
__device__ __forceinline__ void store_tile_compound_buffer(const GemmParams& p, float* __restrict__ C, const v16f (&acc)[TJ],
                                                           int m_base, int n_base, int lane) {
    constexpr int AUX = STREAM_C ? 3 : 0;
    const __amdgpu_buffer_rsrc_t rsrc = __builtin_amdgcn_make_buffer_rsrc(C, 0, static_cast<int>(p.c_span), 0x00020000);
    const int m0 = __builtin_amdgcn_readfirstlane(m_base);
    const uint32_t mi_bytes = static_cast<uint32_t>(p.c_mi) * 4u;
    const uint32_t carry = static_cast<uint32_t>(p.c_mo - p.c_lm * p.c_mi) * 4u;      // (modulo 2^32: only the sum has to be an offset)
    const int q = m0 / p.c_lm, rem = m0 - q * p.c_lm;
    const uint32_t row0 = static_cast<uint32_t>(q * p.c_mo + rem * p.c_mi) * 4u;
    const bool whole = rem + 32 <= p.c_lm && m0 + 32 <= p.M;
    const int own = 4 * (lane >> 5);                   // this lane's first row of the tile
#pragma unroll
    for (int tj = 0; tj < TJ; ++tj) {
        const int n = n_base + tj * 32 + (lane & 31);
        if (n >= p.N) continue;
        const int nq = n / p.c_ln;
        const uint32_t base = row0 + own * mi_bytes + static_cast<uint32_t>(nq * p.c_no + (n - nq * p.c_ln) * p.c_ni) * 4u;
        if (whole) {
#pragma unroll
            for (int r = 0; r < 16; ++r)
                __builtin_amdgcn_raw_buffer_store_b32(__builtin_bit_cast(uint32_t, acc[tj][r] * p.alpha), rsrc, base,
                                                      (8 * (r >> 2) + (r & 3)) * mi_bytes, AUX);
        } else {
#pragma unroll
            for (int r = 0; r < 16; ++r) {
                const int step = 8 * (r >> 2) + (r & 3);
                uint32_t at = base + step * mi_bytes;
                if (rem + own + step >= p.c_lm) at += carry;                          // (at most one: the run is 32 or longer)
                if (m0 + own + step < p.M)
                    __builtin_amdgcn_raw_buffer_store_b32(__builtin_bit_cast(uint32_t, acc[tj][r] * p.alpha), rsrc, at, 0, AUX);
            }
        }
    }
}

// Any compound output, 64-bit addresses
template <int TJ>
__device__ __forceinline__ void store_tile_compound(const GemmParams& p, float* __restrict__ C, const v16f (&acc)[TJ], int m_base, int n_base, int lane) {
#pragma unroll
    for (int tj = 0; tj < TJ; ++tj) {
        const int n = n_base + tj * 32 + (lane & 31);
        if (n >= p.N) continue;
        float* const col = C + static_cast<int64_t>(n / p.c_ln) * p.c_no + static_cast<int64_t>(n % p.c_ln) * p.c_ni;
#pragma unroll
        for (int r = 0; r < 16; ++r) {
            const int m = m_base + mfma32_row(r, lane);
            if (m < p.M) col[static_cast<int64_t>(m / p.c_lm) * p.c_mo + static_cast<int64_t>(m % p.c_lm) * p.c_mi] = acc[tj][r] * p.alpha;
        }
    }
}

template <bool STREAM_C, int TI>
__device__ __forceinline__ void store_acc_compound_buffer(const GemmParams& p, float* __restrict__ C, const v16f (&acc)[TI][2],
                                                          int m_base, int n_base, int lane) {
#pragma unroll
    for (int ti = 0; ti < TI; ++ti) store_tile_compound_buffer<STREAM_C, 2>(p, C, acc[ti], m_base + ti * 32, n_base, lane);
}

}  // namespace
}  // namespace ppmlhip
