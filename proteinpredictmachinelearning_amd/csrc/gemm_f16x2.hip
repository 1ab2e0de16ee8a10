// Large binary32 contractions on the f16 matrix pipe.
//
// A binary32 number times a power of two that brings the largest element of its row near 2^12 .. 2^15 is the sum of two
// halves, h = f16(x), l = f16(x - h), to within 2^-23 of itself.  Three products -- h h, h l, l h -- are kept (l l lies below
// 2^-22 of |a||b|); the matrix pipe forms each exactly and adds it into a binary32 accumulator, and the powers of two leave
// again by ldexp, exactly.  Together: 2^-21 of |a||b| at worst, for operands of one constant each; random ones measure half the error
// of the exact split into three bf16 parts with its six products (gemm_bf16x3_kernel), whose sums take twice as many
// additions.  Against that form it is half the matrix work, a third less LDS traffic and less than half the vector work (two
// v_fma_mixlo/hi per element).
//
// What it asks for is the scale: a half has five bits of exponent.  One power of two per ROW of either operand and K slice -- not
// per operand, whose rows may differ by anything -- carries what lies within 2^-14 (A) or 2^-16 (B) of its row's largest
// element.  A smaller one, below 2^-2 once scaled, is kept to a fixed 2^-25 instead of a share of itself, which is as good as lost where the
// row's large elements meet zeros (an outlier against a zero weight, a spike of a gradient against a token that a mask made
// zero).  So those elements are counted, n per row of A and c per row of B: what they cost an output is at most (n + c) 2^-10 in scaled
// units (the partner lies below 2^15).  An output that is not 2^21 times that -- so that it could lose more than the 2^-21 above
// -- is computed again, with the tile of 32 x 32 that it lies in, by the exact split (redo_tiles).  The test is against the output itself, or
// against what its sum was halfway through K: neither is larger than sum |a||b|, so no output gets past it by luck.  Of
// normal operands one lane in 2^11 fails with one of the two, next to none with both, and the test costs a minimum over the
// accumulators.  With the counting, us without / with: 384 residues x 32 features x 256 sequences 294 / 301 forward, 518 / 525
// backward, 103 residues 41.9 / 42.3 and 79.3 / 83.1, 26368 x 256 -> 768 53.0 / 54.4, its weight gradient 57.5 / 58.3.  Operands of wide
// range throughout are contracted twice: 12288 x 256 x 12288 with spikes of 10^9 in one column or log-normal with sigma 3
// 1.5 ms (0.47 by the exact split alone), 26368 x 256 -> 768 0.29.
//
// B (the smaller operand as a rule: a weight, an alignment's projection) is split ahead by split_f16x2_kernel, which sees a
// whole row of the slice and knows its maximum.  A is split in the tile loop by the loading waves, whose scale
// follows the data: a row starts at the scale of its first nonzero stage with three bits of room, and a stage with a larger element moves it
// and leaves a factor by which the contracting waves multiply what they hold (a branch that is taken once in a row's life
// as a rule).
//
// Infinities and NaN are noticed with the maxima (v_maximum3_f32 passes NaN on), and the outputs concerned are redone in plain
// binary32 arithmetic, one product at a time (plain_dot), as everywhere in this library.
#include "gemm.hpp"
#include "split.hpp"

#include <algorithm>

namespace ppmlhip {
namespace {

constexpr int HX_M = 128;                          // rows of A per tile
constexpr int HX_K = 32;                           // k per stage
// A stage of A in LDS: 32 rows x 16 k of one part are two halves (k 0 .. 7, 8 .. 15) of 32 rows x 16 bytes, as the MFMA reads
// them.  The paddings put the eight-byte pieces that sixteen lanes write (two rows, 32 k) into sixteen different banks' pairs.
constexpr int HX_HALF = 576, HX_FRAG = 2 * HX_HALF, HX_STEP = 4 * HX_FRAG + 32, HX_PART = 2 * HX_STEP, HX_STAGE = 2 * HX_PART;
constexpr int HX_BUFS = 3;                         // stages in LDS: one being written, one contracted, one peeked into
constexpr int HX_AHEAD = 3;                        // stages a loading wave has in flight
constexpr int HX_EXPS = 4;                         // items whose row exponents are kept (see lds_exp)
constexpr int HX_BAD = 511;                        // exponent of a row that holds an infinity or a NaN (others: -115 .. 127) ...
constexpr int HX_ANY_BAD = 300;                    // ... and what no sum of two others reaches
constexpr float HX_SMALL = 0.25f;                  // scaled elements below this keep 2^-25, those above it 2^-23 of themselves
constexpr float HX_LOST = 2048.0f;                 // 2^21 times the 2^-10 that such an element may cost an output
constexpr float HX_ZEROS = -1e9f;                  // small elements of a row of zeros: it costs nothing, whatever its partner
constexpr uint32_t HX_PLAIN = 0xffffffffu;         // of a wave's note on an item: all of it, one product at a time
constexpr uint32_t HX_FIRST_SCALE = (127u + 126u) << 23;      // before a row's first nonzero element: 2^126
constexpr int HX_KC = 0, HX_RC = 1, HX_KRUN = 2, HX_RRUN = 3; // how A lies: contiguous in k / in its rows; compound indices with runs along k / the rows
constexpr int HX_PARTIAL = 0, HX_DENSE = 1, HX_COMPOUND = 2;  // where the sums go: the slices' workspace, a dense C, a compound C

struct F16x2Job {
    const uint8_t* wb;        // B's fragments: [stage][part][16-k step][tile of 32 columns][1 KB]
    const uint32_t* eb;       // [slice][nb_pad]: of B's column in the slice, the exponent (ten bits, signed) and its small elements (22 bits, all set: zeros)
    float* partial;           // [slice][ma_pad][nb_pad]
    uint64_t* notes;          // [work-group][contracting wave][most_items]: item and, a bit each, its tiles of 32 x 32 to redo
    int most_items;           // items of a work-group at most
    int nb_pad, ma_pad;
    int chunks, slice_chunks; // stages in all and per slice: even numbers
    int slices, items;
    int wgs;                  // work-groups of this contraction: a multiple of eight
    uint32_t a_span;          // bytes of A from its base to behind its last element
    float* a_sums;            // [slice][ma_pad]: the sums over k of A's rows, or null
};

// the largest magnitude, NaN if there is one
__device__ __forceinline__ float max4(float m, const v4f& x) {
#if defined(__HIP_DEVICE_COMPILE__)
    m = __builtin_elementwise_maximum(__builtin_elementwise_maximum(m, __builtin_fabsf(x[0])), __builtin_fabsf(x[1]));
    return __builtin_elementwise_maximum(__builtin_elementwise_maximum(m, __builtin_fabsf(x[2])), __builtin_fabsf(x[3]));
#else
    return m + x[0];
#endif
}

// the smallest magnitude (a NaN: the row is a bad one, whatever comes of it)
__device__ __forceinline__ float min4(float m, const v4f& x) {
#if defined(__HIP_DEVICE_COMPILE__)
    m = __builtin_elementwise_minimum(__builtin_elementwise_minimum(m, __builtin_fabsf(x[0])), __builtin_fabsf(x[1]));
    return __builtin_elementwise_minimum(__builtin_elementwise_minimum(m, __builtin_fabsf(x[2])), __builtin_fabsf(x[3]));
#else
    return m + x[0];
#endif
}

__device__ __forceinline__ float sum8(const v4f (&x)[2]) {
    const v4f s = x[0] + x[1];
    return (s[0] + s[1]) + (s[2] + s[3]);
}

// how many of four elements are small ones under this scale (a power of two from 2^-115 to 2^127): not zero, below 2^-2 of it
__device__ __forceinline__ int count_small4(const v4f& x, float scale) {
    const float limit = ldexpf(HX_SMALL, 127 - static_cast<int>(__float_as_uint(scale) >> 23));
    const uint32_t below = (__float_as_uint(limit) << 1) - 1;       // (zeros wrap round to the largest number)
    int n = 0;
#pragma unroll
    for (int c = 0; c < 4; ++c) n += (__float_as_uint(x[c]) << 1) - 1 < below ? 1 : 0;
    return n;
}

// ------------------------------------------------------------------------------------------------------------
// B ahead of the contraction.  A work-group takes 32 rows of B (columns of the product) and one slice of K: maxima, scale,
// parts.  A round covers 256 k; a slice of up to eight rounds stays in registers between the two passes.
constexpr int HX_SPLIT_ROUNDS = 8;
struct F16x2Split {
    const float* src;
    uint8_t* dst;
    uint32_t* exps;
    int rows, rows_pad, K, chunks, slice_chunks;
    int64_t rs, ks;
    int64_t span;             // elements from src to behind the last one: below 2^29, any 32 rows' offsets too
    float* sums;              // [slice][rows_pad]: the rows' sums, or null
};

template <bool KS1>
__device__ __forceinline__ void split_f16x2(const F16x2Split& jb) {
    __shared__ uint32_t lds_max[32][33];
    __shared__ int lds_small[32];
    const int tid = threadIdx.x;
    if (tid < 32) lds_small[tid] = 0;
    // (row of the 32, octet of k within a round): lanes along k or along the rows, as the operand lies
    const int row = KS1 ? tid >> 5 : tid & 31, oct = KS1 ? tid & 31 : tid >> 5;
    const int r = blockIdx.x * 32 + row;
    const int c_begin = blockIdx.y * jb.slice_chunks;
    const int c_end = c_begin + jb.slice_chunks < jb.chunks ? c_begin + jb.slice_chunks : jb.chunks;
    const int k_begin = c_begin * HX_K, k_end = c_end * HX_K;
    const int rounds = (k_end - k_begin + 255) / 256;
    // through a buffer resource from the work-group's first row on (outside: zero): loads under conditions are waited for one
    // after the other (256 columns x 12288 14.2 us, this way 11.4; 256 x 26368 13.6 / 12.7, 768 x 256 5.6 / 5.3)
    const int64_t span = jb.span - static_cast<int64_t>(blockIdx.x) * 32 * jb.rs;       // elements from there to the operand's end
    const __amdgpu_buffer_rsrc_t rsrc = __builtin_amdgcn_make_buffer_rsrc(const_cast<float*>(jb.src + static_cast<int64_t>(blockIdx.x) * 32 * jb.rs), 0,
                                                                          static_cast<int>(span > 0 ? span * 4 : 0), 0x00020000);
    const uint32_t row_at = r < jb.rows ? static_cast<uint32_t>(row * jb.rs) * 4u : OUTSIDE;
    const uint32_t k_step = static_cast<uint32_t>(KS1 ? 1 : jb.ks) * 4u;
    const auto load = [&](int i, v4f (&v)[2]) {
        const int kb = k_begin + i * 256 + oct * 8;
        const uint32_t at = row_at + static_cast<uint32_t>(kb) * k_step;
        const int k_last = k_end < jb.K ? k_end : jb.K;
        if (KS1 && k_begin + (i + 1) * 256 <= k_last) {          // (the same for the work-group)
#pragma unroll
            for (int h = 0; h < 2; ++h) v[h] = __builtin_bit_cast(v4f, __builtin_amdgcn_raw_buffer_load_b128(rsrc, at + 16u * h, 0, 0));
        } else {
#pragma unroll
            for (int c = 0; c < 8; ++c)
                v[c >> 2][c & 3] = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(rsrc, kb + c < k_last ? at + c * k_step : OUTSIDE, 0, 0));
        }
    };
    const bool kept = rounds <= HX_SPLIT_ROUNDS;
    v4f held[HX_SPLIT_ROUNDS][2];
    uint32_t top = 0;
    float sum = 0.0f;
    const auto see = [&](const v4f (&v)[2]) {
        if (jb.sums) sum += sum8(v);
        const uint32_t b = __float_as_uint(max4(max4(0.0f, v[0]), v[1]));
        top = b > top ? b : top;
    };
    if (kept) {
#pragma unroll
        for (int i = 0; i < HX_SPLIT_ROUNDS; ++i) if (i < rounds) load(i, held[i]);
#pragma unroll
        for (int i = 0; i < HX_SPLIT_ROUNDS; ++i) if (i < rounds) see(held[i]);
    } else {
        for (int i = 0; i < rounds; i += 2) {
            v4f a[2], b[2];
            load(i, a);
            load(i + 1, b);
            see(a);
            see(b);
        }
    }
    lds_max[row][oct] = top;
    __syncthreads();
#pragma unroll
    for (int i = 0; i < 32; ++i) { const uint32_t o = lds_max[row][i]; top = o > top ? o : top; }
    if (jb.sums) {                                      // (the maxima's places, once they have been read)
        __syncthreads();
        lds_max[row][oct] = __float_as_uint(sum);
        __syncthreads();
        if (oct == 0) {
            float s[4] = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
            for (int i = 0; i < 32; ++i) s[i & 3] += __uint_as_float(lds_max[row][i]);
            jb.sums[static_cast<int64_t>(blockIdx.y) * jb.rows_pad + r] = (s[0] + s[1]) + (s[2] + s[3]);
        }
    }
    // the largest element goes to 2^14 .. 2^15, or as near as 2^127 brings it; an all-zero row needs no scale
    const int e = static_cast<int>(top >> 23) & 0xff;
    const bool bad = top >= 0x7f800000u;
    const int scale_exp = top == 0 || bad ? 127 : e >= 14 ? 268 - e : 254;          // biased exponent of the scale
    const float scale = __uint_as_float(static_cast<uint32_t>(scale_exp) << 23);
    int small = 0;
    const auto put = [&](int i, const v4f (&v)[2]) {
        const int kb = k_begin + i * 256 + oct * 8;
        if (kb >= k_end) return;
        if (min4(min4(__builtin_inff(), v[0]), v[1]) * scale < HX_SMALL) small += count_small4(v[0], scale) + count_small4(v[1], scale);
        uint2 lo[2], hi[2];
        split4_f16(v[0], scale, lo);
        split4_f16(v[1], scale, hi);
        // [stage][part][16-k step][tile][half][row]
        uint8_t* dst = jb.dst + ((static_cast<int64_t>(kb >> 5) * 2 * 2 + ((kb >> 4) & 1)) * jb.rows_pad + blockIdx.x * 32) * 32 + ((kb >> 3) & 1) * 512 + row * 16;
        const int64_t part = static_cast<int64_t>(jb.rows_pad) * 64;
        *reinterpret_cast<uint4*>(dst) = uint4{lo[0].x, lo[0].y, hi[0].x, hi[0].y};
        *reinterpret_cast<uint4*>(dst + part) = uint4{lo[1].x, lo[1].y, hi[1].x, hi[1].y};
    };
    if (kept) {
#pragma unroll
        for (int i = 0; i < HX_SPLIT_ROUNDS; ++i) put(i, held[i]);
    } else {
        for (int i = 0; i < rounds; i += 2) {
            v4f a[2], b[2];
            load(i, a);
            load(i + 1, b);
            put(i, a);
            put(i + 1, b);
        }
    }
    if (small != 0) atomicAdd(&lds_small[row], small);
    __syncthreads();
    if (oct == 0) {
        const uint32_t n = static_cast<uint32_t>(lds_small[row]);
        jb.exps[static_cast<int64_t>(blockIdx.y) * jb.rows_pad + r] =
            (static_cast<uint32_t>(bad ? HX_BAD : scale_exp - 127) & 1023u) | (top == 0 ? 0x3fffffu : n < 0x3ffffeu ? n : 0x3ffffeu) << 10;
    }
}

template <bool KS1>
__global__ __launch_bounds__(1024) void split_f16x2_kernel(const F16x2Split jb) { split_f16x2<KS1>(jb); }
// two operands of the same sizes, contiguous in their rows
__global__ __launch_bounds__(1024) void split_f16x2_pair_kernel(const F16x2Split ja, const F16x2Split jb) { split_f16x2<false>(blockIdx.z == 0 ? ja : jb); }

// A work-group's items: first, first + step, ...; an XCD's are consecutive ones
template <int TJ>
struct Items {
    struct Item { int m0, n0, slice, c_begin, nch; };
    const GemmParams& p;
    const F16x2Job& jb;
    int first, step, mine;
    __device__ __forceinline__ Items(const GemmParams& p_, const F16x2Job& jb_, int block) : p(p_), jb(jb_) {
        const int xcd = block & 7;
        step = jb.wgs >> 3;
        const int lo = static_cast<int>(static_cast<int64_t>(jb.items) * xcd / 8);
        const int hi = static_cast<int>(static_cast<int64_t>(jb.items) * (xcd + 1) / 8);
        first = lo + (block >> 3);
        mine = first < hi ? (hi - first + step - 1) / step : 0;
    }
    __device__ __forceinline__ Item at(int i) const {
        Item it;
        const int tiles = p.tiles_m * p.tiles_n;
        int t = first + i * step;
        it.slice = t / tiles;
        t -= it.slice * tiles;
        const int band_rows = 8;
        const int band = t / (band_rows * p.tiles_n);
        t -= band * band_rows * p.tiles_n;
        const int rows_here = (p.tiles_m - band * band_rows) < band_rows ? (p.tiles_m - band * band_rows) : band_rows;
        it.m0 = (band * band_rows + t % rows_here) * HX_M;
        it.n0 = (t / rows_here) * (128 * TJ);
        it.c_begin = it.slice * jb.slice_chunks;
        it.nch = jb.chunks - it.c_begin < jb.slice_chunks ? jb.chunks - it.c_begin : jb.slice_chunks;
        return it;
    }
};

// ------------------------------------------------------------------------------------------------------------
// Outputs that the scaled parts did not carry, again, by the exact split into three bf16 parts and over the k of a slice: tiles
// of 32 x 32 from (m0, n0) and from (m0 + 32, n0) on, a bit of `which` each; by one wave, straight from memory.
template <int OUT, int AHEAD>
__device__ __forceinline__ void redo_tiles(const GemmParams& p, const F16x2Job& jb, int m0, int n0, int slice, uint32_t which, int lane) {
    const int k0 = slice * jb.slice_chunks * HX_K;
    const int k1 = OUT == HX_PARTIAL && k0 + jb.slice_chunks * HX_K < p.K ? k0 + jb.slice_chunks * HX_K : p.K;
    const bool runs = p.a_lm > 0;
    const int j = lane & 31, hh = lane >> 5;
    // both operands by 32-bit byte offsets, as in the tile loop (outside: zero)
    const int64_t b_span = (static_cast<int64_t>(p.N - 1) * p.b_rs + static_cast<int64_t>(p.K - 1) * p.b_ks + 1) * 4;
    const __amdgpu_buffer_rsrc_t ra = __builtin_amdgcn_make_buffer_rsrc(const_cast<float*>(p.A), 0, static_cast<int>(jb.a_span), 0x00020000);
    const __amdgpu_buffer_rsrc_t rb = __builtin_amdgcn_make_buffer_rsrc(const_cast<float*>(p.B), 0, static_cast<int>(b_span), 0x00020000);
    const uint32_t a_step = static_cast<uint32_t>(runs ? p.a_ki : p.a_ks) * 4u, b_step = static_cast<uint32_t>(p.b_ks) * 4u;
    const uint32_t carry = runs ? static_cast<uint32_t>(p.a_ko - p.a_lk * p.a_ki) * 4u : 0;      // from behind a run to the next one's start
    uint32_t a_at[2], b_at;
#pragma unroll
    for (int u = 0; u < 2; ++u) {
        const int m = m0 + 32 * u + j;
        const int64_t el = runs ? static_cast<int64_t>(m / p.a_lm) * p.a_mo + static_cast<int64_t>(m % p.a_lm) * p.a_mi : static_cast<int64_t>(m) * p.a_rs;
        a_at[u] = m < p.M ? static_cast<uint32_t>(el) * 4u + 8 * hh * a_step : OUTSIDE;
    }
    b_at = n0 + j < p.N ? static_cast<uint32_t>((n0 + j) * p.b_rs) * 4u + 8 * hh * b_step : OUTSIDE;
    // eight consecutive k from byte offset `at` on, of which `left` are there; from the `turn`-th on they lie in the next run
    const auto load8 = [](const __amdgpu_buffer_rsrc_t r, uint32_t at, uint32_t step, bool whole, int left, int turn, uint32_t carry_, v4f (&x)[2]) {
        if (step == 4u && whole) {
#pragma unroll
            for (int h = 0; h < 2; ++h) x[h] = __builtin_bit_cast(v4f, __builtin_amdgcn_raw_buffer_load_b128(r, at + 16u * h, 0, 0));
        } else {
#pragma unroll
            for (int i = 0; i < 8; ++i)
                x[i >> 2][i & 3] = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(r, i < left ? at + i * step + (i < turn ? 0u : carry_) : OUTSIDE, 0, 0));
        }
    };
    const auto load = [&](int k, v4f (&xa)[2][2], v4f (&xb)[2]) {
        const int kd = runs ? k / p.a_lk : 0, kr = runs ? k - kd * p.a_lk : k;
        const uint32_t off = runs ? static_cast<uint32_t>(kd * p.a_ko + kr * p.a_ki) * 4u : static_cast<uint32_t>(k) * a_step;
        const int turn = runs ? p.a_lk - kr : 16;       // (a run is at least a stage long)
        const bool in = k + 16 <= k1, whole = in && turn >= 16;
        const int left = k1 - k - 8 * hh;
#pragma unroll
        for (int u = 0; u < 2; ++u) load8(ra, a_at[u] + off, a_step, whole, left, turn - 8 * hh, carry, xa[u]);
        load8(rb, b_at + static_cast<uint32_t>(k) * b_step, b_step, in, left, 8, 0u, xb);
    };
    v16f acc[2];
#pragma unroll
    for (int u = 0; u < 2; ++u)
#pragma unroll
        for (int r = 0; r < 16; ++r) acc[u][r] = 0.0f;
    SplitGuard guard;
    v4f xa[AHEAD][2][2], xb[AHEAD][2];                  // steps of 16 k in flight (behind k1: zeros)
#pragma unroll
    for (int d = 0; d < AHEAD; ++d) load(k0 + 16 * d, xa[d], xb[d]);
#pragma unroll 1
    for (int k = k0; k < k1; k += 16 * AHEAD) {
#pragma unroll
        for (int d = 0; d < AHEAD; ++d) {
            v8bf fa[2][3], fb[3];
            split8(xa[d][0], fa[0], guard);
            split8(xa[d][1], fa[1], guard);
            split8(xb[d], fb, guard);
            if (k + 16 * AHEAD < k1) load(k + 16 * (AHEAD + d), xa[d], xb[d]);
#pragma unroll
            for (int q = 0; q < 6; ++q)
#pragma unroll
                for (int u = 0; u < 2; ++u) acc[u] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(fa[u][SPLIT_TERMS[q][0]], fb[SPLIT_TERMS[q][1]], acc[u], 0, 0, 0);
        }
    }
    const bool fired = __builtin_amdgcn_ballot_w64(guard.fired()) != 0;
#pragma unroll
    for (int u = 0; u < 2; ++u) {
        if ((which >> u & 1) == 0) continue;
        if (OUT != HX_PARTIAL && fired) {               // bits below the exact split's own range
            plain_tile(p, p.A, p.B, p.C, m0 + 32 * u, n0, 32, 32, lane, 64);
            continue;
        }
#pragma unroll
        for (int r = 0; r < 16; ++r) {
            const int m = m0 + 32 * u + mfma32_row(r, lane), n = n0 + j;
            if (m >= p.M || n >= p.N) continue;
            float v = fired ? __builtin_nanf("") : acc[u][r];       // (NaN: reduce_slices_kernel redoes it)
            if (OUT == HX_PARTIAL) {
                jb.partial[(static_cast<size_t>(slice) * jb.ma_pad + m) * jb.nb_pad + n] = v;
            } else {
                if (p.bias) v += p.bias[n];
                p.C[static_cast<int64_t>(m / p.c_lm) * p.c_mo + static_cast<int64_t>(m % p.c_lm) * p.c_mi +
                    static_cast<int64_t>(n / p.c_ln) * p.c_no + static_cast<int64_t>(n % p.c_ln) * p.c_ni] = v * p.alpha;
            }
        }
    }
}

// ------------------------------------------------------------------------------------------------------------
// The contraction.  One work-group of eight waves per CU walks a list of items (128 x 128 TJ tiles, times the slices of K).
// Waves 4 .. 7 load A three stages ahead, find the rows' maxima, scale, split and write the stage to LDS; they run on into
// the next item while waves 0 .. 3 store the finished one.  A contracting wave takes all 128 rows and 32 TJ columns: B's
// fragments belong to it alone and come straight from memory (L2), two stages ahead; A's come from LDS one step ahead of
// their six MFMAs.  Barrier i + 1 says "stages up to i + 1 are in LDS" and "stage i - 1 has been read".
struct F16x2Lds {
    __attribute__((aligned(16))) uint8_t a[HX_BUFS * HX_STAGE];
    __attribute__((aligned(16))) float factor[HX_BUFS][HX_M];
    __attribute__((aligned(16))) int mark[HX_BUFS][4];
    // exponents of the rows' scales, per item: written with an item's last stage, read behind it, by when the loading waves
    // are at most two stages (two items, were an item one stage) further
    __attribute__((aligned(16))) int exp[HX_EXPS][HX_M];
    __attribute__((aligned(16))) float small[HX_EXPS][HX_M];      // their small elements, HX_ZEROS for a row of zeros ...
    __attribute__((aligned(16))) float most[HX_EXPS][4];          // ... and the most of them in a row, per loading wave
    int noted[4];
};
template <int AMODE, bool GEN, int TJ, int OUT, bool STREAM>
__device__ __forceinline__ void f16x2_items(const GemmParams& p, const F16x2Job& jb, F16x2Lds& lds, int block) {
    constexpr bool KLOAD = AMODE == HX_KC || AMODE == HX_KRUN;
    constexpr bool RUNS = AMODE == HX_KRUN || AMODE == HX_RRUN;
    constexpr int NR = KLOAD ? 4 : 1;                  // rows of A a loading lane has a share of
    uint8_t (&lds_a)[HX_BUFS * HX_STAGE] = lds.a;
    float (&lds_factor)[HX_BUFS][HX_M] = lds.factor;
    int (&lds_mark)[HX_BUFS][4] = lds.mark;
    int (&lds_exp)[HX_EXPS][HX_M] = lds.exp;
    float (&lds_small)[HX_EXPS][HX_M] = lds.small;
    float (&lds_most)[HX_EXPS][4] = lds.most;
    int (&lds_noted)[4] = lds.noted;

    const int tid = threadIdx.x;
    const int lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);

    const Items<TJ> items(p, jb, block);
    const int my_items = items.mine;
    const auto item_at = [&](int i) { return items.at(i); };
    if (my_items == 0) return;                          // (the whole work-group: no barrier is left behind)
    int total = 0;                                      // stages of this work-group
    for (int i = 0; i < my_items; ++i) total += item_at(i).nch;
    const int padded = (total + HX_AHEAD - 1) / HX_AHEAD * HX_AHEAD;

    if (wave >= 4) {
        const int w = wave - 4;                         // this wave's 32 rows
        const __amdgpu_buffer_rsrc_t rsrc = __builtin_amdgcn_make_buffer_rsrc(const_cast<float*>(p.A), 0, static_cast<int>(jb.a_span), 0x00020000);
        // (A with runs of whole stages is read once, by one column of tiles as a rule, and is larger than the caches: it goes past
        // L2, where B's fragments stay; 384 residues x 32 features x 256 sequences, one gradient: 262 -> 254 us.  Stages that
        // begin inside a line share it with the next one's: those stay in L2, 211 residues 115 us past it)
        constexpr int AUX = RUNS && !GEN ? 2 : 0;
        const auto load4 = [&](uint32_t at) { return __builtin_bit_cast(v4f, __builtin_amdgcn_raw_buffer_load_b128(rsrc, at, 0, AUX)); };
        const auto load1 = [&](uint32_t at) { return __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(rsrc, at, 0, AUX)); };
        // KLOAD: rows 8 i + r0, four k from u0 on; otherwise row r0, sixteen k from u0 on
        const int r0 = KLOAD ? lane >> 3 : lane & 31;
        const int u0 = KLOAD ? (lane & 7) * 4 : (lane >> 5) * 16;
        const uint32_t k_step = static_cast<uint32_t>(RUNS ? p.a_ki : p.a_ks) * 4u;        // bytes from k to k + 1
        uint32_t roff[NR];
        typename Items<TJ>::Item load_item = item_at(0);
        int li = 0, lc = 0, kd = 0, kr = 0;
        const auto open = [&]() {
#pragma unroll
            for (int i = 0; i < NR; ++i) {
                const int row = load_item.m0 + w * 32 + 8 * i + r0;
                const int64_t el = RUNS ? static_cast<int64_t>(row / p.a_lm) * p.a_mo + static_cast<int64_t>(row % p.a_lm) * p.a_mi
                                        : static_cast<int64_t>(row) * p.a_rs;
                roff[i] = row < p.M ? static_cast<uint32_t>(el) * 4u + u0 * k_step : OUTSIDE;
            }
            if (RUNS) { kd = load_item.c_begin * HX_K / p.a_lk; kr = load_item.c_begin * HX_K - kd * p.a_lk; }
        };
        open();
        const int nruns = RUNS ? p.K / p.a_lk : 0;
        // requests the next stage; past the last item every offset is outside (the loads are still made: the count of loads
        // in flight that the wait for a stage names is then the same in every iteration)
        const auto request = [&](v4f (&x)[4]) {
            const bool live = li < my_items;
            const int k0 = (load_item.c_begin + lc) * HX_K;
            if (AMODE == HX_KC) {
                const uint32_t koff = static_cast<uint32_t>(k0) * 4u;
                if (!GEN) {                             // K a multiple of four: a piece lies inside its row or behind it
                    const bool in = live && k0 + u0 < p.K;
#pragma unroll
                    for (int i = 0; i < 4; ++i) x[i] = load4(in ? roff[i] + koff : OUTSIDE);
                } else if (live && k0 + HX_K <= p.K) {
#pragma unroll
                    for (int i = 0; i < 4; ++i) x[i] = load4(roff[i] + koff);
                } else {
#pragma unroll
                    for (int i = 0; i < 4; ++i)
#pragma unroll
                        for (int c = 0; c < 4; ++c) x[i][c] = load1(live && k0 + u0 + c < p.K ? roff[i] + koff + 4u * c : OUTSIDE);
                }
            } else if (AMODE == HX_RC) {                // (k behind K: behind the end of the plane)
                const uint32_t base = (live ? roff[0] : OUTSIDE) + static_cast<uint32_t>(k0) * k_step;
#pragma unroll
                for (int c = 0; c < 16; ++c) x[c >> 2][c & 3] = load1(base + c * k_step);
            } else if (!GEN) {                          // runs of whole stages
                const bool in = live && kd < nruns;
                const uint32_t koff = static_cast<uint32_t>(static_cast<int64_t>(kd) * p.a_ko + static_cast<int64_t>(kr) * p.a_ki) * 4u;
                if (KLOAD) {
#pragma unroll
                    for (int i = 0; i < 4; ++i) x[i] = load4(in ? roff[i] + koff : OUTSIDE);
                } else {
                    const uint32_t base = in ? roff[0] + koff : OUTSIDE;
#pragma unroll
                    for (int c = 0; c < 16; ++c) x[c >> 2][c & 3] = load1(base + c * k_step);
                }
            } else {
                // element u places behind the stage's first k lies in this run while kr + u < run length, else in the next one
                // (a run is at least a stage long: the launcher's rule); a run behind the last one is outside: 2^30, which with
                // the operand's span (at most 2^30 bytes in this form) and with a row's 2^31 stays outside
                constexpr uint32_t NO_RUN = 0x40000000u;
                const uint32_t here = live && kd < nruns ? static_cast<uint32_t>(static_cast<int64_t>(kd) * p.a_ko + static_cast<int64_t>(kr) * p.a_ki) * 4u : NO_RUN;
                const uint32_t next = live && kd + 1 < nruns ? static_cast<uint32_t>(static_cast<int64_t>(kd + 1) * p.a_ko + static_cast<int64_t>(kr - p.a_lk) * p.a_ki) * 4u : NO_RUN;
                const int left = p.a_lk - kr;
                if (KLOAD && left >= HX_K) {            // a stage inside one run
#pragma unroll
                    for (int i = 0; i < 4; ++i) x[i] = load4(roff[i] + here);
                } else if (KLOAD) {
#pragma unroll
                    for (int i = 0; i < 4; ++i)
#pragma unroll
                        for (int c = 0; c < 4; ++c) x[i][c] = load1(roff[i] + (u0 + c < left ? here : next) + 4u * c);
                } else {
#pragma unroll
                    for (int c = 0; c < 16; ++c) x[c >> 2][c & 3] = load1(roff[0] + (u0 + c < left ? here : next) + c * k_step);
                }
            }
            if (RUNS) { kr += HX_K; if (kr >= p.a_lk) { kr -= p.a_lk; ++kd; } }
            if (++lc == load_item.nch) {
                lc = 0;
                if (++li < my_items) { load_item = item_at(li); open(); }
            }
        };

        float scale[NR];
        uint32_t seen[NR];                              // OR of the maxima's bits; the sign bit: infinite or NaN
        int small[NR];                                  // this lane's share of the row's small elements
        float sum = 0.0f;                               // ... and, where they are asked for, of its sum (HX_RC)
        int pi = 0, pc = 0, p_nch = load_item.nch, buf = 0;
        // splits the next stage into LDS
        const auto place = [&](const v4f (&x)[4]) {
            if (pc == 0) {
#pragma unroll
                for (int i = 0; i < NR; ++i) { scale[i] = __uint_as_float(HX_FIRST_SCALE); seen[i] = 0; small[i] = 0; }
                sum = 0.0f;
            }
            if (AMODE == HX_RC && OUT == HX_PARTIAL && jb.a_sums) sum += sum8({x[0], x[1]}) + sum8({x[2], x[3]});
            uint32_t top[NR], before[NR];
            bool over = false;
#pragma unroll
            for (int i = 0; i < NR; ++i) {
                float m = max4(0.0f, x[i]);
                if (!KLOAD) m = max4(max4(max4(m, x[1]), x[2]), x[3]);
                uint32_t b = __float_as_uint(m);
                const auto meet = [&](uint32_t o) { b = o > b ? o : b; };
                if (KLOAD) {                            // the eight lanes of the row: neighbours, pairs, then the other four
                    meet(__builtin_amdgcn_mov_dpp(b, 0xB1, 0xf, 0xf, true));
                    meet(__builtin_amdgcn_mov_dpp(b, 0x4E, 0xf, 0xf, true));
                    meet(__builtin_amdgcn_mov_dpp(b, 0x141, 0xf, 0xf, true));
                } else {
                    meet(__shfl_xor(b, 32, 64));
                }
                top[i] = b;
                before[i] = seen[i];
                seen[i] |= b;
                over |= !(__uint_as_float(b) * scale[i] < 32768.0f);
            }
            int mark = 0;
            if (__builtin_amdgcn_ballot_w64(over) != 0) {
#pragma unroll
                for (int i = 0; i < NR; ++i) {
                    float factor = 1.0f;
                    if (!(__uint_as_float(top[i]) * scale[i] < 32768.0f)) {
                        if (top[i] >= 0x7f800000u) {
                            seen[i] |= 0x80000000u;
                        } else {
                            const int e = static_cast<int>(top[i] >> 23);                    // (at least 16: the first scale is 2^126)
                            const int was = static_cast<int>(__float_as_uint(scale[i]) >> 23), now = 266 - e;
                            const int f = now - was + 127;
                            factor = f > 0 ? __uint_as_float(static_cast<uint32_t>(f) << 23) : 0.0f;
                            scale[i] = __uint_as_float(static_cast<uint32_t>(now) << 23);
                            // (what the sums hold may leave binary32's range on this way: less than a small element's share)
                            if (before[i] != 0 && u0 == 0) ++small[i];
                        }
                    }
                    if (u0 == 0) lds_factor[buf][w * 32 + 8 * i + r0] = factor;
                }
                mark = 1;
            }
            if (lane == 0) lds_mark[buf][w] = mark;
            // (zeros pass this test too: an ordinary stage of nonzero elements pays for a minimum, one with zeros or small ones for the count)
            bool few = false;
#pragma unroll
            for (int i = 0; i < NR; ++i) {
                float m = min4(__builtin_inff(), x[i]);
                if (!KLOAD) m = min4(min4(min4(m, x[1]), x[2]), x[3]);
                few |= m * scale[i] < HX_SMALL;
            }
            if (__builtin_amdgcn_ballot_w64(few) != 0) {
#pragma unroll
                for (int i = 0; i < 4; ++i) small[i % NR] += count_small4(x[i], scale[i % NR]);
            }
            uint8_t* const stage = lds_a + buf * HX_STAGE + w * HX_FRAG;
            if (KLOAD) {
                uint8_t* const dst = stage + (u0 >> 4) * HX_STEP + ((u0 >> 3) & 1) * HX_HALF + ((u0 >> 2) & 1) * 8 + r0 * 16;
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                    uint2 parts[2];
                    split4_f16(x[i], scale[i % NR], parts);
                    *reinterpret_cast<uint2*>(dst + i * 128) = parts[0];
                    *reinterpret_cast<uint2*>(dst + HX_PART + i * 128) = parts[1];
                }
            } else {
                uint8_t* const dst = stage + (u0 >> 4) * HX_STEP + r0 * 16;
#pragma unroll
                for (int h = 0; h < 2; ++h) {
                    uint2 a[2], b[2];
                    split4_f16(x[2 * h], scale[0], a);
                    split4_f16(x[2 * h + 1], scale[0], b);
                    *reinterpret_cast<uint4*>(dst + h * HX_HALF) = uint4{a[0].x, a[0].y, b[0].x, b[0].y};
                    *reinterpret_cast<uint4*>(dst + HX_PART + h * HX_HALF) = uint4{a[1].x, a[1].y, b[1].x, b[1].y};
                }
            }
            if (++pc == p_nch) {
                if (pi < my_items) {
                    int most = 0;
#pragma unroll
                    for (int i = 0; i < NR; ++i) {
                        int n = small[i];               // (the lanes of the row, as with the maxima)
                        if (KLOAD) {
                            n += __builtin_amdgcn_mov_dpp(n, 0xB1, 0xf, 0xf, true);
                            n += __builtin_amdgcn_mov_dpp(n, 0x4E, 0xf, 0xf, true);
                            n += __builtin_amdgcn_mov_dpp(n, 0x141, 0xf, 0xf, true);
                        } else {
                            n += __shfl_xor(n, 32, 64);
                        }
                        most = n > most ? n : most;
                        if (u0 != 0) continue;
                        lds_exp[pi & (HX_EXPS - 1)][w * 32 + 8 * i + r0] = (seen[i] & 0x80000000u) != 0 ? HX_BAD : seen[i] == 0 ? 0 : static_cast<int>(__float_as_uint(scale[i]) >> 23) - 127;
                        lds_small[pi & (HX_EXPS - 1)][w * 32 + 8 * i + r0] = seen[i] == 0 ? HX_ZEROS : static_cast<float>(n);
                    }
                    const float m = wave_max(static_cast<float>(most));
                    if (lane == 0) lds_most[pi & (HX_EXPS - 1)][w] = m;
                    if (AMODE == HX_RC && OUT == HX_PARTIAL && jb.a_sums) {
                        sum += __shfl_xor(sum, 32, 64);
                        const typename Items<TJ>::Item it = item_at(pi);
                        // (the tiles of one column of tiles see every row of A once)
                        if (it.n0 == 0 && lane < 32) jb.a_sums[static_cast<size_t>(it.slice) * jb.ma_pad + it.m0 + w * 32 + r0] = sum;
                    }
                }
                pc = 0;
                if (++pi < my_items) p_nch = item_at(pi).nch;
            }
            buf = buf == HX_BUFS - 1 ? 0 : buf + 1;
        };

        v4f x[HX_AHEAD][4];
#pragma unroll
        for (int d = 0; d < HX_AHEAD; ++d) { request(x[d]); __builtin_amdgcn_sched_barrier(0); }
        for (int g = 0; g < padded; g += HX_AHEAD) {
#pragma unroll
            for (int d = 0; d < HX_AHEAD; ++d) {
                place(x[d]);
                request(x[d]);
                __syncthreads();
            }
        }
        __syncthreads();
        return;
    }

    // ---- contracting waves
    const int j = lane & 31, hh = lane >> 5;
    const int wn = wave * 32 * TJ;
    v8h fb[2][TJ][2][2];                                // [stage parity][tile column][16-k step][part]
    typename Items<TJ>::Item b_item = item_at(0);
    int bi = 0, bc = 0;
    const size_t b_unit = static_cast<size_t>(jb.nb_pad) * 32;
    // the fragments of the next stage of the sequence (behind the last item: of that item's first stages again)
    const auto load_b = [&](v8h (&f)[TJ][2][2]) {
        const uint8_t* src = jb.wb + static_cast<size_t>(b_item.c_begin + bc) * 4 * b_unit + static_cast<size_t>(b_item.n0 + wn) * 32 + lane * 16;
#pragma unroll
        for (int part = 0; part < 2; ++part)
#pragma unroll
            for (int ks = 0; ks < 2; ++ks)
#pragma unroll
                for (int tj = 0; tj < TJ; ++tj) f[tj][ks][part] = *reinterpret_cast<const v8h*>(src + (part * 2 + ks) * b_unit + tj * 1024);
        if (++bc == b_item.nch) {
            bc = 0;
            if (bi + 1 < my_items) b_item = item_at(++bi);
        }
    };
    load_b(fb[0]);
    load_b(fb[1]);
    const uint8_t* const frag = lds_a + hh * HX_HALF + j * 16;
    v8h fa[2][2];                                       // the step at hand and the next
    int buf = 0;
    __syncthreads();
    __syncthreads();                                    // stages 0 and 1 are in LDS
#pragma unroll
    for (int part = 0; part < 2; ++part) fa[0][part] = *reinterpret_cast<const v8h*>(frag + part * HX_PART);
    v4i mark = *reinterpret_cast<const v4i*>(lds_mark[0]);
    v16f acc[4][TJ];
    int g = 0;
    uint64_t* const notes = jb.notes + static_cast<size_t>(block * 4 + wave) * jb.most_items;
    int noted = 0;                                      // items with outputs to redo
    // the smallest of this lane's sums in a tile row
    const auto least = [&](int ti) {
        float m = __builtin_inff();
#pragma unroll
        for (int tj = 0; tj < TJ; ++tj)
#pragma unroll
            for (int r = 0; r < 16; ++r) m = __builtin_elementwise_minimum(m, __builtin_fabsf(acc[ti][tj][r]));
        return m;
    };
    for (int i = 0; i < my_items; ++i) {
        const typename Items<TJ>::Item it = item_at(i);
        uint32_t of_b[TJ];
#pragma unroll
        for (int tj = 0; tj < TJ; ++tj) of_b[tj] = jb.eb[static_cast<size_t>(it.slice) * jb.nb_pad + it.n0 + wn + tj * 32 + j];
#pragma unroll
        for (int ti = 0; ti < 4; ++ti)
#pragma unroll
            for (int tj = 0; tj < TJ; ++tj)
#pragma unroll
                for (int r = 0; r < 16; ++r) acc[ti][tj][r] = 0.0f;
        // this lane's smallest sum halfway through K: no sum of |a||b| is smaller than that of a part of it, so a lane that passes the
        // test below with either need not be looked at
        float halfway = 0.0f;
        const auto chunk = [&](v8h (&f)[TJ][2][2], int k0, bool fresh) {
            if (!fresh && __builtin_amdgcn_readfirstlane(mark[0] | mark[1] | mark[2] | mark[3]) != 0) {
                // some rows' scales have moved: what their sums hold so far moves with them
                halfway = 0.0f;
#pragma unroll
                for (int ti = 0; ti < 4; ++ti) {
                    if (__builtin_amdgcn_readfirstlane(mark[ti]) == 0) continue;
#pragma unroll
                    for (int q = 0; q < 4; ++q) {
                        const v4f fac = *reinterpret_cast<const v4f*>(&lds_factor[buf][ti * 32 + 8 * q + 4 * hh]);
#pragma unroll
                        for (int tj = 0; tj < TJ; ++tj)
#pragma unroll
                            for (int c = 0; c < 4; ++c) acc[ti][tj][4 * q + c] *= fac[c];
                    }
                }
            }
            const uint8_t* const here = frag + buf * HX_STAGE;
            buf = buf == HX_BUFS - 1 ? 0 : buf + 1;
            const uint8_t* const next = frag + buf * HX_STAGE;
            // (16-k steps behind K are left out: K padded to whole pairs of stages would be contracted in full)
            const int steps = (p.K - k0 + 15) / 16;
#pragma unroll
            for (int ks = 0; ks < 2; ++ks) {
                if (ks >= steps) {
                    if (ks == 0 || steps == 1) {
#pragma unroll
                        for (int part = 0; part < 2; ++part) fa[0][part] = *reinterpret_cast<const v8h*>(next + part * HX_PART);
                    }
                    break;
                }
#pragma unroll
                for (int ti = 0; ti < 4; ++ti) {
                    const int s = ks * 4 + ti;
                    const uint8_t* const at = s < 7 ? here + ((s + 1) >> 2) * HX_STEP + ((s + 1) & 3) * HX_FRAG : next;
                    fa[(s + 1) & 1][0] = *reinterpret_cast<const v8h*>(at);
                    fa[(s + 1) & 1][1] = *reinterpret_cast<const v8h*>(at + HX_PART);
                    __builtin_amdgcn_sched_barrier(0);  // (left to itself the scheduler reads a fragment where it is needed)
                    const v8h (&a)[2] = fa[s & 1];
                    // smallest first: l h, h l, h h
#pragma unroll
                    for (int tj = 0; tj < TJ; ++tj) acc[ti][tj] = __builtin_amdgcn_mfma_f32_32x32x16_f16(a[1], f[tj][ks][0], acc[ti][tj], 0, 0, 0);
#pragma unroll
                    for (int tj = 0; tj < TJ; ++tj) acc[ti][tj] = __builtin_amdgcn_mfma_f32_32x32x16_f16(a[0], f[tj][ks][1], acc[ti][tj], 0, 0, 0);
#pragma unroll
                    for (int tj = 0; tj < TJ; ++tj) acc[ti][tj] = __builtin_amdgcn_mfma_f32_32x32x16_f16(a[0], f[tj][ks][0], acc[ti][tj], 0, 0, 0);
                    __builtin_amdgcn_sched_barrier(0);
                }
            }
            mark = *reinterpret_cast<const v4i*>(lds_mark[buf]);
            load_b(f);
            ++g;
            if (g < total) __syncthreads();             // stage g - 1 has been read; stage g + 1 is in LDS
        };
        for (int c = 0; c < it.nch; c += 2) {
            if (c == it.nch / 4 * 2 && c != 0) {
                halfway = __builtin_inff();
#pragma unroll
                for (int ti = 0; ti < 4; ++ti)          // (tile rows past the matrix hold zeros)
                    if (it.m0 + ti * 32 < p.M) halfway = __builtin_elementwise_minimum(halfway, least(ti));
            }
            chunk(fb[0], (it.c_begin + c) * HX_K, c == 0);
            chunk(fb[1], (it.c_begin + c + 1) * HX_K, false);
        }

        // ---- the scales leave, the sums go out
        const int (&ea)[HX_M] = lds_exp[i & (HX_EXPS - 1)];
        int eb[TJ], worst = ea[lane] > ea[lane + 64] ? ea[lane] : ea[lane + 64];
        float cb[TJ], bound = 0.0f;
#pragma unroll
        for (int tj = 0; tj < TJ; ++tj) {
            eb[tj] = static_cast<int>(of_b[tj] << 22) >> 22;
            worst = eb[tj] > worst ? eb[tj] : worst;
            cb[tj] = of_b[tj] >> 10 == 0x3fffffu ? HX_ZEROS : static_cast<float>(of_b[tj] >> 10);
            bound = fmaxf(bound, cb[tj]);
        }
        const bool any_bad = __builtin_amdgcn_ballot_w64(worst >= HX_ANY_BAD) != 0;
        if (OUT != HX_PARTIAL && any_bad) {
            // infinities or NaN in this wave's tile: all of it again, the reference's way
            if (lane == 0) notes[noted] = static_cast<uint64_t>(i) << 32 | HX_PLAIN;
            ++noted;
            continue;
        }
        // outputs that the small elements of their rows may have cost more than the products' own error (see above): by the most of
        // them in a row first, which all but a few tiles pass, then row by row; the tiles of 32 x 32 that fail are noted
        const v4f most = *reinterpret_cast<const v4f*>(lds_most[i & (HX_EXPS - 1)]);
        bound = HX_LOST * (bound + fmaxf(fmaxf(most[0], most[1]), fmaxf(most[2], most[3])));
        if (__builtin_amdgcn_ballot_w64(!(halfway >= bound)) != 0) {
            const float (&na)[HX_M] = lds_small[i & (HX_EXPS - 1)];
            uint32_t which = 0;
#pragma unroll
            for (int ti = 0; ti < 4; ++ti) {
                const uint64_t open = __builtin_amdgcn_ballot_w64(!(halfway >= bound) && !(least(ti) >= bound));
                if (it.m0 + ti * 32 >= p.M || open == 0) continue;
                uint64_t lost[TJ] = {};
#pragma unroll
                for (int q = 0; q < 4; ++q) {
                    const v4f n4 = *reinterpret_cast<const v4f*>(&na[ti * 32 + 8 * q + 4 * hh]);
#pragma unroll
                    for (int tj = 0; tj < TJ; ++tj)
#pragma unroll
                        for (int c = 0; c < 4; ++c)     // (a NaN comes from a row that is a bad one)
                            lost[tj] |= __builtin_amdgcn_ballot_w64(__builtin_fabsf(acc[ti][tj][4 * q + c]) < HX_LOST * (n4[c] + cb[tj]));
                }
#pragma unroll
                for (int tj = 0; tj < TJ; ++tj) which |= (lost[tj] & open) != 0 ? 1u << (ti * TJ + tj) : 0u;
            }
            if (which != 0) {
                if (lane == 0) notes[noted] = static_cast<uint64_t>(i) << 32 | which;
                ++noted;
            }
        }
        if (OUT == HX_PARTIAL && any_bad) {             // NaN: reduce_slices_kernel redoes those
#pragma unroll
            for (int ti = 0; ti < 4; ++ti)
#pragma unroll
                for (int r = 0; r < 16; ++r)
#pragma unroll
                    for (int tj = 0; tj < TJ; ++tj)
                        if (ea[ti * 32 + 8 * (r >> 2) + 4 * hh + (r & 3)] + eb[tj] >= HX_ANY_BAD) acc[ti][tj][r] = __builtin_nanf("");
        }
        // (one tile row at a time: with all sixty-four exponents read ahead the kernel spills)
        const auto unscale = [&](int ti) {
            __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (int q = 0; q < 4; ++q) {
                const v4i e4 = *reinterpret_cast<const v4i*>(&ea[ti * 32 + 8 * q + 4 * hh]);
#pragma unroll
                for (int tj = 0; tj < TJ; ++tj)
#pragma unroll
                    for (int c = 0; c < 4; ++c) acc[ti][tj][4 * q + c] = ldexpf(acc[ti][tj][4 * q + c], -(e4[c] + eb[tj]));
            }
        };
        if constexpr (OUT == HX_COMPOUND) {
#pragma unroll
            for (int ti = 0; ti < 4; ++ti) {
                unscale(ti);
                store_tile_compound_buffer<STREAM, TJ>(p, p.C, acc[ti], it.m0 + ti * 32, it.n0 + wn, lane);
            }
        } else {
            constexpr bool part = OUT == HX_PARTIAL;
            const uint32_t ld = part ? static_cast<uint32_t>(jb.nb_pad) * 4u : static_cast<uint32_t>(p.c_mi) * 4u;
            float* const base = part ? jb.partial + static_cast<size_t>(it.slice) * jb.ma_pad * jb.nb_pad : p.C;
            // rows past the matrix fall outside the plane by themselves
            const __amdgpu_buffer_rsrc_t rsrc_c = __builtin_amdgcn_make_buffer_rsrc(base, 0, static_cast<int>((part ? jb.ma_pad : p.M) * ld), 0x00020000);
            float tail[TJ];
            uint32_t col[TJ];
#pragma unroll
            for (int tj = 0; tj < TJ; ++tj) {
                const int n = it.n0 + wn + tj * 32 + j;
                tail[tj] = !part && p.bias && n < p.N ? p.bias[n] : 0.0f;
                col[tj] = part || n < p.N ? static_cast<uint32_t>(n) * 4u : OUTSIDE;
            }
            uint32_t row = static_cast<uint32_t>(it.m0 + 4 * hh) * ld;
#pragma unroll
            for (int ti = 0; ti < 4; ++ti) {
                unscale(ti);
#pragma unroll
                for (int r = 0; r < 16; ++r) {
#pragma unroll
                    for (int tj = 0; tj < TJ; ++tj) {
                        float v = acc[ti][tj][r];
                        if (!part) v = (v + tail[tj]) * p.alpha;
                        __builtin_amdgcn_raw_buffer_store_b32(__builtin_bit_cast(uint32_t, v), rsrc_c, row + col[tj], 0, STREAM ? 3 : 0);
                    }
                    // to the next row (opaque: one offset that moves on, not sixty-four at once)
                    row += (r & 3) == 3 ? 5 * ld : ld;
                    asm volatile("" : "+v"(row));
                }
            }
        }
    }
    for (; g < padded; ++g) __syncthreads();
    if (lane == 0) lds_noted[wave] = noted;
}

// (kernarg_at: where the parameters lie in the kernel's arguments)
template <int AMODE, bool GEN, int TJ, int OUT, bool STREAM>
__device__ __forceinline__ void f16x2_contract(const GemmParams& p, const F16x2Job& jb, F16x2Lds& lds, int block, size_t kernarg_at) {
    if (threadIdx.x < 4) lds.noted[threadIdx.x] = 0;    // (a work-group without items leaves them so)
    f16x2_items<AMODE, GEN, TJ, OUT, STREAM>(p, jb, lds, block);
    // What the items left to redo, by all eight waves.  Behind the last item, where nothing else is held in registers (among the items the
    // two-to-a-CU form spilled its fragments), and with the parameters read again, which the items then need not hold either.
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");    // (the notes, and the stores of the outputs concerned, have landed)
    __syncthreads();
    int counts[4], any = 0;
#pragma unroll
    for (int w = 0; w < 4; ++w) { counts[w] = __builtin_amdgcn_readfirstlane(lds.noted[w]); any |= counts[w]; }
    if (any == 0) return;
    typedef const __attribute__((address_space(4))) GemmParams* KernargPtr;
    typedef const __attribute__((address_space(4))) uint8_t* KernargBytes;
    KernargPtr again = (KernargPtr)((KernargBytes)__builtin_amdgcn_kernarg_segment_ptr() + kernarg_at);
    asm volatile("" : "+s"(again));
    const GemmParams pr = *(const GemmParams*)again;
    const Items<TJ> items(pr, jb, block);
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    int unit = 0;
#pragma unroll 1
    for (int w = 0; w < 4; ++w) {
        const int count = w == 0 ? counts[0] : w == 1 ? counts[1] : w == 2 ? counts[2] : counts[3];
#pragma unroll 1
        for (int u = 0; u < count * 2 * TJ; ++u) {      // (64 rows x 32 columns each)
            if ((unit++ & 7) != wave) continue;
            const uint64_t note = jb.notes[static_cast<size_t>(block * 4 + w) * jb.most_items + u / (2 * TJ)];
            const auto it = items.at(__builtin_amdgcn_readfirstlane(static_cast<int>(note >> 32)));
            const uint32_t which = __builtin_amdgcn_readfirstlane(static_cast<uint32_t>(note));
            const int ti = u / TJ % 2 * 2, tj = u % TJ;
            const int m0 = it.m0 + ti * 32, n0 = it.n0 + (w * TJ + tj) * 32;
            if (OUT != HX_PARTIAL && which == HX_PLAIN) {
                plain_tile(pr, pr.A, pr.B, pr.C, m0, n0, 64, 32, lane, 64);
                continue;
            }
            const uint32_t these = (which >> (ti * TJ + tj) & 1) | (which >> ((ti + 1) * TJ + tj) & 1) << 1;
            if (these != 0) redo_tiles<OUT, TJ>(pr, jb, m0, n0, it.slice, these, lane);
        }
    }
}

template <int AMODE, bool GEN, int TJ, int OUT, bool STREAM>
__global__ __launch_bounds__(512, TJ == 1 ? 4 : 2) void gemm_f16x2_kernel(const GemmParams p, const F16x2Job jb) {
    __shared__ F16x2Lds lds;
    f16x2_contract<AMODE, GEN, TJ, OUT, STREAM>(p, jb, lds, static_cast<int>(blockIdx.x), 0);
}

// Both gradients of an outer-product-mean in one launch, each by half of the work-groups: the same tiles, and bits, as in two, without the
// second's start, and with the splits ahead and the sums of the slices in one launch each too.  Forward and both gradients, in two / this way, us:
// 103 residues x 32 features x 256 sequences 124 / 109, 384 residues 853 / 841.
struct F16x2Pair { GemmParams pa, pb; F16x2Job ja, jb; };
template <bool GEN, int TJ>
__global__ __launch_bounds__(512, TJ == 1 ? 4 : 2) void gemm_f16x2_pair_kernel(const F16x2Pair pair) {
    __shared__ F16x2Lds lds;
    const int block = static_cast<int>(blockIdx.x);
    if (block < pair.ja.wgs) f16x2_contract<HX_KRUN, GEN, TJ, HX_PARTIAL, false>(pair.pa, pair.ja, lds, block, offsetof(F16x2Pair, pa));
    else f16x2_contract<HX_RRUN, GEN, TJ, HX_PARTIAL, false>(pair.pb, pair.jb, lds, block - pair.ja.wgs, offsetof(F16x2Pair, pb));
}

// How one contraction goes: what try_f16x2 settles before it has memory
struct F16x2Plan {
    GemmParams p;
    F16x2Job jb;
    int amode, tj, out, sum_pad;
    bool gen, partial, swapped, sums, compound;
    int64_t b_span;
    size_t b_bytes, e_bytes, n_bytes, part_bytes, sum_bytes;
    size_t bytes() const { return b_bytes + e_bytes + n_bytes + part_bytes + sum_bytes; }
    float* sum_partial(uint8_t* ws) const { return sums ? reinterpret_cast<float*>(ws + b_bytes + e_bytes + n_bytes + part_bytes) : nullptr; }
    F16x2Job job(uint8_t* ws) const {
        F16x2Job j = jb;
        j.wb = ws;
        j.eb = reinterpret_cast<uint32_t*>(ws + b_bytes);
        j.notes = reinterpret_cast<uint64_t*>(ws + b_bytes + e_bytes);
        j.partial = reinterpret_cast<float*>(ws + b_bytes + e_bytes + n_bytes);
        j.a_sums = swapped ? nullptr : sum_partial(ws);
        return j;
    }
    F16x2Split split(uint8_t* ws) const {
        return {p.B, ws, reinterpret_cast<uint32_t*>(ws + b_bytes), p.N, jb.nb_pad, p.K, jb.chunks, jb.slice_chunks, p.b_rs, p.b_ks, b_span, swapped ? sum_partial(ws) : nullptr};
    }
    dim3 split_grid(int operands = 1) const { return dim3(jb.nb_pad / 32, jb.slices, operands); }
};

// cu_share: the part of the CUs this contraction is to have (a half where two go side by side)
bool plan_f16x2(const GemmParams& p0, F16x2Plan& pl, int cu_share = 1) {
    GemmParams& p = pl.p;
    p = p0;
    if (p.np2 * p.np3 != 1 || p.clamp || p.f16_in) return false;
    if (p.K < 64 || p.N <= 32) return false;
    const bool compound = !(p.c_lm >= p.M && p.c_ln >= p.N);
    const int cus = device_cu_count() / 8 * 8;
    // matrix work: 16-k steps of 128 x 128 tiles per CU
    const int64_t tiles128 = static_cast<int64_t>((p.M + 127) / 128) * ((p.N + 127) / 128);
    const int64_t load = tiles128 * ((p.K + 15) / 16) / cus;
    // few tiles under a long K (a LinearLayer's weight gradient): slices of K, and the smaller operand is split ahead
    const bool sliced = !compound && p.a_lm == 0 && tiles128 * 2 <= cus;
    bool swapped = false;
    if (sliced && p.M < p.N && !p.bias) {
        swapped = true;
        std::swap(p.A, p.B);
        std::swap(p.M, p.N);
        std::swap(p.a_rs, p.b_rs);
        std::swap(p.a_ks, p.b_ks);
        std::swap(p.c_mi, p.c_ni);
    }
    if (p.M < 128) return false;
    // how A lies, and 32-bit byte offsets into it
    int amode;
    bool gen = false;
    int64_t span;
    if (p.a_lm > 0) {
        if (p.a_lk < HX_K || p.K % p.a_lk != 0 || p.a_mo < 0 || p.a_mi < 0 || p.a_ko < 0 || p.a_ki < 0) return false;
        amode = p.a_ki == 1 ? HX_KRUN : p.a_mi == 1 ? HX_RRUN : -1;
        gen = p.a_lk % HX_K != 0;
        span = static_cast<int64_t>((p.M - 1) / p.a_lm) * p.a_mo + static_cast<int64_t>(std::min(p.a_lm, p.M) - 1) * p.a_mi +
               static_cast<int64_t>((p.K - 1) / p.a_lk) * p.a_ko + static_cast<int64_t>(p.a_lk - 1) * p.a_ki + 1;
        if (gen && span * 4 > (1LL << 30)) return false;
    } else if (p.a_ks == 1) {
        amode = HX_KC;
        gen = p.K % 4 != 0;
        span = static_cast<int64_t>(p.M - 1) * p.a_rs + p.K;
        if (p.a_rs < p.K) return false;
    } else if (p.a_rs == 1) {
        amode = HX_RC;
        span = static_cast<int64_t>(p.K) * p.a_ks;
        if (p.a_ks < p.M || (span + 128 * p.a_ks) * 4 >= (1LL << 31)) return false;
    } else {
        return false;
    }
    if (amode < 0 || span * 4 >= (1LL << 31) - 65536) return false;
    // B by 32-bit byte offsets as well
    const int64_t b_span = static_cast<int64_t>(p.N - 1) * p.b_rs + static_cast<int64_t>(p.K - 1) * p.b_ks + 1;
    if (p.b_rs <= 0 || p.b_ks <= 0 || b_span * 4 >= (1LL << 31) || (static_cast<int64_t>(p.K) + 64) * p.b_ks * 4 + 32 * p.b_rs * 4 >= (1LL << 31)) return false;
    // the output (slices: any strides)
    if (compound ? p.c_span == 0 : (p.c_ni != 1 && !sliced) || static_cast<int64_t>(p.M + HX_M) * p.c_mi * 4 >= (1LL << 31)) return false;

    // Where the lines lie (us, the other forms / this one; `load` in steps).  The split ahead and a deeper pipeline cost 5 us
    // before the first tile, so the contraction has to be worth it:
    //   * compound A (outer-product-mean backward), one gradient: 2480 x 2480 x 245 (load 24) 34 / 32, 1984 x 1984 x 241 (15)
    //     30 / 33, 4000 x 4000 x 135 56 / 42, 12288 x 12288 x 256 412 / 245;
    //   * compound C (its forward): 3136 x 106 x 3136 (17) 25 / 32, 4464 x 123 x 4464 (38) 59 / 43, 7808 x 202 x 7808 242 / 165;
    //   * slices: 888 x 3490 x 504 (24) 29 / 29, 832 x 8990 x 304 (46) 42 / 38, 768 x 26368 x 256 (77) 61 / 52; with few rows the
    //     split of the other operand weighs more: 464 x 12651 x 392 (49) 42 / 43, 564 x 26377 x 197 (64) 51 / 52;
    //   * otherwise, from more than a tile per CU on (2601 x 512 -> 1024, 168 tiles, 22.4 / 33.4, 10609 x 448 -> 288, 249 tiles, 22.5
    //     / 25.0, 10609 x 328 -> 420, 332 tiles, 28.9 / 26.8): 10609 x 176 -> 532 (15) 20 / 21, 26368 x 256 -> 256 (26) 25 / 21, 26368 x 512 -> 1024 (206) 189 / 101.
    //     a tile of few stages has less to hide the split ahead behind: 20000 x 197 -> 400 (23) 31.5 / 35.7, 9040 x 221 -> 832 (25)
    //     25.8 / 28.1, 12000 x 223 -> 800 (32) 32.7 / 34.2, 26368 x 223 -> 512 (45) 47.1 / 39.2; 9040 x 333 -> 600 (27) 34.4 / 29.7.
    // A K below 128 stays with the form that splits in the tile loop at any size (the bits of a contraction that is cut
    // out of a larger one then do not depend on the size).
    if (p.a_lm > 0) { if (load < 22) return false; }
    else if (compound) { if (load < 30) return false; }
    else if (sliced) { if (load < 42 || (p.M < 700 && load < 66) || p.K < 128) return false; }
    else if (p.K < 128 || tiles128 <= cus || static_cast<double>(p.M) * p.N * p.K < (p.K < 256 ? 40.0 : 20.0) * 128 * 128 * 16 * cus) return false;      // (without the padding: 30001 x 131 -> 260 25.8 / 29.7)
    // Tiles of 128 x 256 by one work-group per CU, or of 128 x 128 by two, which store while the other contracts but read A
    // twice as often: where 256 columns would be half empty, where the wide tiles' last round leaves more than half of the CUs idle (26368 x 256 -> 768: 51.4
    // / 48.8 us; 32768 x 512 -> 1024, whole rounds, 110 / 118), and for compound rows that are not whole lines, whose stores
    // take as long as the products (7808 x 202 x 7808: 196 / 165; 12288 x 256 x 12288, whole lines, 288 / 314).
    const int tn = (p.N + 127) / 128;
    int tj = 2;
    if (compound) {
        if (p.c_lm % 32 != 0 || tn == 1) tj = 1;
    } else if (tn == 1 || (tn == 3 && p.a_lm == 0)) {
        tj = 1;
    } else if (p.a_lm == 0 && !sliced) {
        const int64_t wide = static_cast<int64_t>((p.M + HX_M - 1) / HX_M) * ((tn + 1) / 2);
        if (wide > cus && wide % cus != 0 && wide % cus * 2 < cus) tj = 1;
    }
    const int nt = 128 * tj;
    p.tiles_m = (p.M + HX_M - 1) / HX_M;
    p.tiles_n = (p.N + nt - 1) / nt;
    const int64_t tiles = static_cast<int64_t>(p.tiles_m) * p.tiles_n;
    const int chunks = ((p.K + HX_K - 1) / HX_K + 1) / 2 * 2;
    int slices = 1;
    if (!compound && tiles * 4 < 3 * cus) {
        slices = even_slices(static_cast<int>(tiles), chunks / 2, 128, 4);      // (whole pairs of stages, at least 256 k)
    }
    if (tiles > (1 << 24) || tiles * slices < 32 || (compound && p.c_ni <= 0)) return false;
    const int slice_chunks = (chunks / 2 + slices - 1) / slices * 2;
    slices = (chunks + slice_chunks - 1) / slice_chunks;
    const int ma_pad = p.tiles_m * HX_M, nb_pad = p.tiles_n * nt;
    const size_t b_bytes = static_cast<size_t>(chunks) * 128 * nb_pad;
    const size_t e_bytes = (static_cast<size_t>(slices) * nb_pad * 4 + 255) / 256 * 256;
    const bool partial = slices > 1 || p.a_lm > 0 || p.c_ni != 1;     // (no direct instances for a compound A)
    const size_t part_bytes = partial ? static_cast<size_t>(slices) * ma_pad * nb_pad * 4 : 0;
    if (static_cast<size_t>(ma_pad) * nb_pad * 4 >= (1ull << 31) && partial) return false;
    const int wgs = std::min<int64_t>((tiles * slices + 7) / 8 * 8, std::max((tj == 1 ? 2 * cus : cus) / cu_share / 8 * 8, 8));
    const int most_items = static_cast<int>(((tiles * slices + 7) / 8 + wgs / 8 - 1) / (wgs / 8));
    pl.b_bytes = b_bytes;
    pl.e_bytes = e_bytes;
    pl.n_bytes = (static_cast<size_t>(wgs) * 4 * most_items * 8 + 255) / 256 * 256;
    pl.part_bytes = part_bytes;
    // row sums: of the operand split ahead, or of the other one by its loading waves
    pl.sums = p.row_sums && partial && (swapped || amode == HX_RC);
    pl.sum_pad = swapped ? nb_pad : ma_pad;
    pl.sum_bytes = pl.sums ? static_cast<size_t>(slices) * pl.sum_pad * 4 : 0;
    pl.amode = amode; pl.tj = tj; pl.gen = gen; pl.partial = partial; pl.swapped = swapped; pl.compound = compound; pl.b_span = b_span;
    pl.out = partial ? HX_PARTIAL : compound ? HX_COMPOUND : HX_DENSE;
    F16x2Job& jb = pl.jb;
    jb = F16x2Job{};
    jb.most_items = most_items;
    jb.nb_pad = nb_pad; jb.ma_pad = ma_pad;
    jb.chunks = chunks; jb.slice_chunks = slice_chunks; jb.slices = slices;
    jb.items = static_cast<int>(tiles) * slices;
    jb.wgs = wgs;
    jb.a_span = static_cast<uint32_t>(span * 4);
    return true;
}

}  // namespace

int try_f16x2(const GemmParams& p0, hipStream_t stream, const char* what, uint8_t* fixed_ws, size_t fixed_cap, bool& sums_done) {
    F16x2Plan pl;
    if (!plan_f16x2(p0, pl)) return -1;
    const Workspace held = workspace_take(pl.bytes(), stream, fixed_ws, fixed_cap);
    uint8_t* const ws = held.ptr;
    if (!ws) return -1;
    const GemmParams& p = pl.p;
    const F16x2Job jb = pl.job(ws);
    const int amode = pl.amode, tj = pl.tj, out = pl.out, wgs = jb.wgs;
    const bool gen = pl.gen;
    const F16x2Split sp = pl.split(ws);
    if (p.b_ks == 1) hipLaunchKernelGGL((split_f16x2_kernel<true>), pl.split_grid(), dim3(1024), 0, stream, sp);
    else             hipLaunchKernelGGL((split_f16x2_kernel<false>), pl.split_grid(), dim3(1024), 0, stream, sp);
    int rc = check_launch(what);
    if (rc == RC_OK) {
        const bool stream_c = p.stream_c && !pl.partial;
#define PPML_HX(A_, G_, T_, O_, S_) hipLaunchKernelGGL((gemm_f16x2_kernel<A_, G_, T_, O_, S_>), dim3(wgs), dim3(512), 0, stream, p, jb)
#define PPML_HX_T(A_, G_, O_, S_) do { if (tj == 1) PPML_HX(A_, G_, 1, O_, S_); else PPML_HX(A_, G_, 2, O_, S_); } while (0)
#define PPML_HX_O(A_, G_)                                                                                         \
    do {                                                                                                          \
        if (out == HX_PARTIAL) PPML_HX_T(A_, G_, HX_PARTIAL, false);                                              \
        else if (stream_c) PPML_HX_T(A_, G_, HX_DENSE, true);                                                     \
        else PPML_HX_T(A_, G_, HX_DENSE, false);                                                                  \
    } while (0)
#define PPML_HX_C(A_, G_) do { if (stream_c) PPML_HX_T(A_, G_, HX_COMPOUND, true); else PPML_HX_T(A_, G_, HX_COMPOUND, false); } while (0)
        if (out == HX_COMPOUND) {
            if (amode == HX_KC) { if (gen) PPML_HX_C(HX_KC, true); else PPML_HX_C(HX_KC, false); }
            else                PPML_HX_C(HX_RC, false);
        }
        else if (amode == HX_KC)   { if (gen) PPML_HX_O(HX_KC, true); else PPML_HX_O(HX_KC, false); }
        else if (amode == HX_RC)   PPML_HX_O(HX_RC, false);
        else if (amode == HX_KRUN) { if (gen) PPML_HX_T(HX_KRUN, true, HX_PARTIAL, false); else PPML_HX_T(HX_KRUN, false, HX_PARTIAL, false); }
        else                       { if (gen) PPML_HX_T(HX_RRUN, true, HX_PARTIAL, false); else PPML_HX_T(HX_RRUN, false, HX_PARTIAL, false); }
#undef PPML_HX_C
#undef PPML_HX_O
#undef PPML_HX_T
#undef PPML_HX
        rc = check_launch(what);
    }
    if (rc == RC_OK && pl.partial)
        rc = launch_reduce_slices(p, stream, what, jb.partial, jb.slices, jb.ma_pad, jb.nb_pad,
                                  RowSumParts{pl.sum_partial(ws), p.row_sums, pl.swapped ? p.N : p.M, jb.slices, pl.sum_pad});
    workspace_give(held, stream);
    sums_done = pl.sums;
    return rc;
}

int try_f16x2_pair(const GemmParams& a, const GemmParams& b, hipStream_t stream, const char* what, bool& wanted) {
    F16x2Plan pa, pb;
    const bool fa = plan_f16x2(a, pa, 2), fb = plan_f16x2(b, pb, 2);
    wanted = fa || fb;
    if (!fa || !fb || pa.amode != HX_KRUN || pb.amode != HX_RRUN || pa.gen != pb.gen || pa.tj != pb.tj || !pa.partial || !pb.partial) return -1;
    if (a.M != b.M || a.N != b.N || a.K != b.K || pa.jb.slices != pb.jb.slices || a.b_ks == 1 || b.b_ks == 1) return -1;
    const size_t need_a = (pa.bytes() + 255) / 256 * 256;
    const Workspace held = workspace_take(need_a + pb.bytes(), stream);
    uint8_t* const ws = held.ptr;
    if (!ws) return -1;
    StatsScope stat("hip/outer_prod_mean_back_pair", a.M, a.K, a.N, stream);
    const F16x2Pair pair{pa.p, pb.p, pa.job(ws), pb.job(ws + need_a)};
    hipLaunchKernelGGL(split_f16x2_pair_kernel, pa.split_grid(2), dim3(1024), 0, stream, pa.split(ws), pb.split(ws + need_a));
    int rc = check_launch(what);
    if (rc == RC_OK) {
        const dim3 grid(pair.ja.wgs + pair.jb.wgs);
#define PPML_HX_PAIR(G_, T_) hipLaunchKernelGGL((gemm_f16x2_pair_kernel<G_, T_>), grid, dim3(512), 0, stream, pair)
        if (pa.tj == 1) { if (pa.gen) PPML_HX_PAIR(true, 1); else PPML_HX_PAIR(false, 1); }
        else            { if (pa.gen) PPML_HX_PAIR(true, 2); else PPML_HX_PAIR(false, 2); }
#undef PPML_HX_PAIR
        rc = check_launch(what);
    }
    if (rc == RC_OK) rc = launch_reduce_slices_pair(pa.p, pb.p, stream, what, pair.ja.partial, pair.jb.partial, pair.ja.slices, pair.ja.ma_pad, pair.ja.nb_pad);
    workspace_give(held, stream);
    return rc;
}

}  // namespace ppmlhip
