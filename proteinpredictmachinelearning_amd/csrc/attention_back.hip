// Fused attention backward for gfx950: the twin of the reference's flash_attn_backward_cuda
// (include/ppml/FlashAttn.h:97-101, declared src/backend/CUDAKernels.cpp:176-179, called from
// kernel_flash_attn_back_cuda, 905-924) with the mathematics of flash_attn_backward_cpu
// (src/ops/FlashAttn.cpp:140-210):
//     P = exp(S - LSE)          S = scale * Q K^T + bias           D_i = sum_d dO_id O_id
//     dS = P * (dO V^T - D)     dQ = scale * dS K     dK = scale * dS^T Q     dV = P^T dO     dbias = dS
// Nothing is stored between forward and backward but O and LSE; P is recomputed per 32 x 32 tile.
//
// For head dimensions up to 32 one kernel makes all four gradients in one pass over the score planes
// (flash_attn_back_fused_kernel, below).  Larger heads, long sequences in few planes (a work-group of that kernel takes a
// whole plane) and calls for dQ and dbias or for dK and dV alone go in two kernels, each the forward kernel's arrangement (see attention.hip) with one side held
// in registers:
//   * rows kernel  (dQ, dbias): a wave owns 32 queries; scores and dO V^T are computed transposed, so a lane
//     holds 16 keys of ITS query: D_i and LSE_i are per-lane scalars, dS is ready as the B operand of
//     dQ^T += K^T dS, and dbias is written from the registers;
//   * columns kernel (dK, dV): a wave owns 32 keys; scores and dO V^T are computed un-transposed, so a lane
//     holds 16 queries of ITS key: P and dS are ready as the B operands of dV^T += dO^T P and
//     dK^T += Q^T dS; LSE and D of the tile's queries come from LDS.
// All five contractions run on the bf16 matrix pipe at binary32 accuracy (exact three-way split of every
// operand, six partial products per 16 contracted elements; common.hpp): the streamed side lies in LDS as ready
// MFMA fragments of its rows (for S and dO V^T), which transposing reads also serve as those of its columns (for the gradients), the
// held side and the freshly computed P / dS are split in registers.
// Measured, us, forward and all gradients, with a second arrangement of the streamed side in LDS (two-byte writes) and one work-group per
// CU in the columns kernel / this way: 64 features, bias, 412 planes of 103 122 / 86, of 160 278 / 184, 824 of 256 778 / 584, without 669 /
// 468; 52 of 52 37.7 / 30.3; 32 features, 40 planes of 384 98 / 88.
// No atomics and no scratch memory: every output element has one owner, so the results do not depend on
// scheduling (the reference's CUDA path accumulates dK and dV with atomicAdd).
#include "common.hpp"

#include <cmath>
#include <type_traits>

namespace ppmlhip {
namespace {

constexpr float LOG2E = 1.44269504088896340736f;

struct AttnBackParams {
    const float* Q; const float* K; const float* V; const float* bias;
    const float* O; const float* dO; const float* LSE;
    float* dQ; float* dK; float* dV; float* dbias;
    int planes, L, d;
    int causal;
    float scale;
    int stage_rows;      // rows of the streamed side staged in LDS at a time (a multiple of 32)
};

__device__ __forceinline__ float lane_xor32(float x) { return __shfl_xor(x, 32, 64); }

// Loads through a buffer resource return zero for an offset that is outside; under conditions of the lane they were waited for one after
// the other.
constexpr uint32_t OUTSIDE = 0x80000000u;
__device__ __forceinline__ __amdgpu_buffer_rsrc_t buffer_of(const float* base, int64_t elements) {
    return __builtin_amdgcn_make_buffer_rsrc(const_cast<float*>(base), 0, elements * 4 < 0x7fffffff ? static_cast<int>(elements * 4) : 0x7fffffff, 0x00020000);
}
__device__ __forceinline__ v4f buffer_load4(const __amdgpu_buffer_rsrc_t r, uint32_t at) { return __builtin_bit_cast(v4f, __builtin_amdgcn_raw_buffer_load_b128(r, at, 0, 0)); }
__device__ __forceinline__ float buffer_load1(const __amdgpu_buffer_rsrc_t r, uint32_t at) { return __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(r, at, 0, 0)); }

template <int DP> struct BackTiling {
    static constexpr int NC = DP / 16;                // 16-feature chunks of a contraction over the features
    static constexpr int NB = DP / 32;                // 32-feature blocks of a transposed gradient
    // A 32-row tile of a streamed matrix in LDS, as MFMA operand fragments, one per (chunk, part): features 8 half .. + 7 of
    // the chunk, sixteen bytes per row, the two halves 576 bytes apart (the transposing reads and, of heads of up to 32, the staging writes then touch every bank
    // once; of wider ones, chunks two apart share banks).  The same fragments serve the contraction over the tile's rows: ds_read_b64_tr_b16 hands them out transposed
    // (read_transposed), in the order in which the accumulator registers 8 ch .. 8 ch + 7 of a 32 x 32 product hold the rows.
    static constexpr int HALF = 576, FRAG = 2 * HALF, CHUNK = 3 * FRAG;
    static constexpr int TILE = NC * CHUNK;
    static constexpr int CH_ROWS = 64;                // rows staged at a time by the rows kernel
    // ... by the columns kernel.  Wide heads: its loads' registers beside the held slices and sums have to leave room for a second wave per
    // SIMD (64 rows at a time: 45 registers spilled, 412 planes of 103 91 us against 86)
    static constexpr int CH_COLS = DP <= 32 ? 96 : 32;
};

// this lane's place in a tile: its row's half chunk, and what it names of the transposed reads of 32 features
template <int DP> __device__ __forceinline__ int row_place(int lane) { return (lane & 31) * 16 + (lane >> 5) * BackTiling<DP>::HALF; }
template <int DP> __device__ __forceinline__ int column_place(int lane) {
    using T = BackTiling<DP>;
    const int grp = lane & 15;
    return ((lane >> 4) & 1) * T::CHUNK + ((grp >> 1) & 1) * T::HALF + (4 * (lane >> 5) + (grp >> 2)) * 16 + (grp & 1) * 8;
}

__device__ __forceinline__ v8bf pack_parts(const uint2& lo, const uint2& hi) {
    return __builtin_bit_cast(v8bf, v4i{static_cast<int>(lo.x), static_cast<int>(lo.y), static_cast<int>(hi.x), static_cast<int>(hi.y)});
}

// This lane's slice of row `first` + j of a [L][d] matrix, as the B operand of a contraction over the features: chunk c holds features
// 16 c + 8 half .. + 7 (zero past d and past L).  `first` is the same for the wave and below L.
template <int DP>
__device__ __forceinline__ void load_slice(const float* base, int first, int j, int L, int d, int half, v4f (&x)[DP / 16][2]) {
    const int rows = L - first < 32 ? L - first : 32;
    const __amdgpu_buffer_rsrc_t r = buffer_of(base + static_cast<int64_t>(first) * d, rows * d);
#pragma unroll
    for (int c = 0; c < DP / 16; ++c)
#pragma unroll
        for (int h = 0; h < 2; ++h) {
            const int e = 16 * c + 8 * half + 4 * h;
            x[c][h] = buffer_load4(r, j < rows && e < d ? static_cast<uint32_t>(j * d + e) * 4u : OUTSIDE);
        }
}

// ... times `factor`, split into three bf16 parts
template <int DP>
__device__ __forceinline__ void slice_parts(const v4f (&x)[DP / 16][2], float factor, v8bf (&out)[DP / 16][3]) {
#pragma unroll
    for (int c = 0; c < DP / 16; ++c) {
        uint2 lo[3], hi[3];
        split4(x[c][0] * factor, lo);
        split4(x[c][1] * factor, hi);
#pragma unroll
        for (int part = 0; part < 3; ++part) out[c][part] = pack_parts(lo[part], hi[part]);
    }
}

// Writes features c .. c+3 of row `row` of a staged matrix into its tiles: eight bytes of each part's fragment.
template <int DP>
__device__ __forceinline__ void put_fragments(const v4f& x, int row, int c, uint8_t* tiles) {
    using T = BackTiling<DP>;
    uint2 parts[3];
    split4(x, parts);
    uint8_t* dst = tiles + (row >> 5) * T::TILE + (c >> 4) * T::CHUNK + ((c >> 3) & 1) * T::HALF + (row & 31) * 16 + ((c >> 2) & 1) * 8;
#pragma unroll
    for (int part = 0; part < 3; ++part) *reinterpret_cast<uint2*>(dst + part * T::FRAG) = parts[part];
}

// Stages rows r0 .. r0+rows-1 (at most MAXROWS) of two [L][d] matrices into LDS as fragments (zeros past `valid`
// rows and past d); SCALED: the first one times a_factor at `a_lds`, and as it is at `a_plain`.  Every load of the stage is issued before the first value is used: a work-group waits for
// one memory round trip per stage, not one per loop iteration.
template <int DP, int NT, int MAXROWS, bool SCALED>
__device__ __forceinline__ void stage_two(const float* a, uint8_t* a_lds, uint8_t* a_plain, float a_factor, const float* b, uint8_t* b_lds,
                                          int r0, int rows, int valid, int d, int tid) {
    constexpr int NI = (MAXROWS * (DP / 4) + NT - 1) / NT;
    const __amdgpu_buffer_rsrc_t ra = buffer_of(a + static_cast<int64_t>(r0) * d, valid * d), rb = buffer_of(b + static_cast<int64_t>(r0) * d, valid * d);
    v4f xa[NI], xb[NI];
#pragma unroll
    for (int i = 0; i < NI; ++i) {
        const int idx = tid + i * NT;
        const int row = idx / (DP / 4), c = (idx % (DP / 4)) * 4;
        const uint32_t at = row < valid && c < d ? static_cast<uint32_t>(row * d + c) * 4u : OUTSIDE;
        xa[i] = buffer_load4(ra, at);
        xb[i] = buffer_load4(rb, at);
    }
#pragma unroll
    for (int i = 0; i < NI; ++i) {
        const int idx = tid + i * NT;
        const int row = idx / (DP / 4), c = (idx % (DP / 4)) * 4;
        if (row < rows) {
            put_fragments<DP>(SCALED ? xa[i] * a_factor : xa[i], row, c, a_lds);
            if (SCALED) put_fragments<DP>(xa[i], row, c, a_plain);
            put_fragments<DP>(xb[i], row, c, b_lds);
        }
    }
}

// acc(32 x 32) = tile(32 rows x DP in LDS, rows = accumulator rows) . slice^T (this lane's column);
// `frags` points at this lane's place in the tile (row_place).  SWAP: the partial products in the order of the
// transposed product (the bits of slice . tile^T)
template <int DP, bool SWAP = false>
__device__ __forceinline__ v16f tile_times_slice(const uint8_t* frags, const v8bf (&slice)[DP / 16][3]) {
    v16f acc;
#pragma unroll
    for (int c = 0; c < DP / 16; ++c) {
        v8bf a[3];
#pragma unroll
        for (int part = 0; part < 3; ++part) a[part] = *reinterpret_cast<const v8bf*>(frags + c * BackTiling<DP>::CHUNK + part * BackTiling<DP>::FRAG);
#pragma unroll
        for (int t = 0; t < 6; ++t) {
            // the first product starts from the constant zero: no registers to clear
            const v16f zero = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
            acc = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a[SPLIT_TERMS[t][SWAP]], slice[c][SPLIT_TERMS[t][!SWAP]], (c == 0 && t == 0) ? zero : acc, 0, 0, 0);
        }
    }
    return acc;
}

// out^T(DP features x 32 columns) += tile^T . w, contracting the 32 rows of the tile in the order in which the
// accumulator registers of `w` hold them; `frags` points at this lane's place in the tile (column_place).
// FROM_ZERO: without what `out` held (the constant zero as the first product's addend: no registers to clear).
template <int DP, bool FROM_ZERO = false>
__device__ __forceinline__ void accumulate_transposed(v16f (&out)[DP / 32], const uint8_t* frags, const v16f& w) {
#pragma unroll
    for (int ch = 0; ch < 2; ++ch) {
        uint2 lo[3], hi[3];
        split4(v4f{w[8 * ch], w[8 * ch + 1], w[8 * ch + 2], w[8 * ch + 3]}, lo);
        split4(v4f{w[8 * ch + 4], w[8 * ch + 5], w[8 * ch + 6], w[8 * ch + 7]}, hi);
        v8bf wb[3];
#pragma unroll
        for (int part = 0; part < 3; ++part) wb[part] = pack_parts(lo[part], hi[part]);
#pragma unroll
        for (int b = 0; b < DP / 32; ++b) {
            v8bf a[3];
#pragma unroll
            for (int part = 0; part < 3; ++part) a[part] = read_transposed(frags + b * 2 * BackTiling<DP>::CHUNK + part * BackTiling<DP>::FRAG + ch * 256, 128);
#pragma unroll
            for (int t = 0; t < 6; ++t)
                out[b] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a[SPLIT_TERMS[t][0]], wb[SPLIT_TERMS[t][1]], FROM_ZERO && ch == 0 && t == 0 ? v16f{} : out[b], 0, 0, 0);
        }
    }
}

constexpr int TWIN_KEYS = 256;                        // keys whose shares of dQ are added up before the scale (eight waves' of the one-pass kernel)

// ------------------------------------------------------------------------------------------------------------
// dQ and dbias: a wave owns 32 queries and walks over the keys.
// TWIN (one block of features): the bits of the one-pass kernel, for calls whose full set of gradients goes there.  K
// carries the scale of the scores, the partial products come in the un-transposed order, D is summed as a butterfly over
// the eight quads of features, and dQ is the sum of its tiles' shares, 256 keys at a time.  The price is a second split of
// K and sixteen additions per tile that wait for their products; LATE adds a tile's share behind the next tile's products
// instead, in sixteen more registers.  Against the form that owes nobody its bits, us: dQ of 8 planes of 256 without bias
// 17.1 / 17.0 (18.3 not late), of 824 planes 76 / 77; with bias, 412 planes of 192, dQ and dbias 51.2 / 52.0 (54.4 not late).
// BIAS: a compile-time property for the registers of its prefetch.
template <int DP, int NW, bool TWIN, bool BIAS, bool LATE>
__global__ __launch_bounds__(NW * 64, !TWIN ? 1 : BIAS && LATE ? 2 : 3) void flash_attn_back_rows_kernel(const AttnBackParams p) {
    using T = BackTiling<DP>;
    constexpr int NB = T::NB, NC = T::NC;
    static_assert(TWIN ? (NB == 1 && NC == 2) : !LATE, "the one-pass kernel's features");
    extern __shared__ __attribute__((aligned(16))) uint8_t back_lds[];
    const int tiles_staged = p.stage_rows / 32;
    uint8_t* const lds_v = back_lds;                                // V: (dO V^T)^T = V . dO^T
    uint8_t* const lds_k = lds_v + tiles_staged * T::TILE;          // K: S^T = K . Q^T and, transposed,
    uint8_t* const lds_kt = TWIN ? lds_k + tiles_staged * T::TILE : lds_k;      // dQ^T += K^T . dS (without the scale)
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int j = lane & 31, half = lane >> 5;
    const int row_at = row_place<DP>(lane), col_at = column_place<DP>(lane);
    const int plane = blockIdx.y, L = p.L, d = p.d;
    const int q0 = (blockIdx.x * NW + wave) * 32, q = q0 + j;
    const bool wave_active = q0 < L;
    const int64_t po = static_cast<int64_t>(plane) * L * d;

    v8bf qb[NC][3], dob[NC][3];
    // D_i = sum_d dO_id * O_id: this lane's half of the features, then the other half from lane j + 32
    float D_i = 0.0f, D_c[NC] = {}, lse = -INFINITY;
    if (wave_active) {
        v4f xq[NC][2], xdo[NC][2], xo[NC][2];
        load_slice<DP>(p.Q + po, q0, j, L, d, half, xq);
        load_slice<DP>(p.dO + po, q0, j, L, d, half, xdo);
        load_slice<DP>(p.O + po, q0, j, L, d, half, xo);
        if (q < L) lse = p.LSE[static_cast<int64_t>(plane) * L + q];
        slice_parts<DP>(xq, TWIN ? 1.0f : p.scale * LOG2E, qb);
        slice_parts<DP>(xdo, 1.0f, dob);
#pragma unroll
        for (int c = 0; c < NC; ++c)
#pragma unroll
            for (int h = 0; h < 2; ++h) {
                const v4f a = xdo[c][h], o = xo[c][h];
                const float quad = a[0] * o[0] + a[1] * o[1] + a[2] * o[2] + a[3] * o[3];
                if (16 * c + 8 * half + 4 * h >= d) continue;
                D_i += quad;
                D_c[c] += quad;
            }
    }
    if (TWIN) {
        D_i = D_c[0] + lane_xor32(D_c[0]);
        if (NC > 1) D_i += D_c[NC - 1] + lane_xor32(D_c[NC - 1]);
    } else {
        D_i += lane_xor32(D_i);
    }
    // a row without any visible key (LSE = -inf) has no gradient: +inf makes every probability exp2(-inf) = 0
    const float lse2 = lse > -INFINITY ? lse * LOG2E : INFINITY;
    const int row_keys = p.causal ? (q + 1 < L ? q + 1 : L) : L;
    const int wave_keys = p.causal ? (q0 + 32 < L ? q0 + 32 : L) : L;
    const bool has_bias = BIAS && p.bias;
    const int wave_rows = !wave_active ? 0 : L - q0 < 32 ? L - q0 : 32;
    const __amdgpu_buffer_rsrc_t rbias = buffer_of(has_bias && wave_active ? p.bias + (static_cast<int64_t>(plane) * L + q0) * L : p.Q,
                                                   has_bias ? static_cast<int64_t>(wave_rows) * L : 0);
    const uint32_t bias_at = static_cast<uint32_t>(j * L + 4 * half) * 4u;
    float* dbias_row = p.dbias ? p.dbias + (static_cast<int64_t>(plane) * L + (q < L ? q : L - 1)) * L : nullptr;

    v16f acc_q[NB];
#pragma unroll
    for (int b = 0; b < NB; ++b)
#pragma unroll
        for (int r = 0; r < 16; ++r) acc_q[b][r] = 0.0f;
    v16f late = {};                                    // LATE: the last tile's share of dQ, not yet in acc_q
    // acc_q times the scale to this lane's query, or added to what it stored there before
    const auto store_dq = [&](bool add) {
        if (q >= L || !p.dQ) return;
        float* row = p.dQ + po + static_cast<int64_t>(q) * d;
#pragma unroll
        for (int b = 0; b < NB; ++b)
#pragma unroll
            for (int g = 0; g < 4; ++g) {
                const int dd = b * 32 + 8 * g + 4 * half;
                if (dd >= d) continue;
                v4f* const dst = reinterpret_cast<v4f*>(row + dd);
                v4f x = v4f{acc_q[b][4 * g], acc_q[b][4 * g + 1], acc_q[b][4 * g + 2], acc_q[b][4 * g + 3]} * p.scale;
                if (add) x += *dst;
                *dst = x;
            }
    };

    // Bias of this lane's 16 keys of the tile that starts at key0, 16 bytes at a time (what lies behind a row's end is masked with
    // the probabilities).
    float bv[16];
    const auto load_bias = [&](int key0) {
        if (!BIAS || !has_bias) return;
#pragma unroll
        for (int g = 0; g < 4; ++g) {
            const v4f x = buffer_load4(rbias, bias_at + static_cast<uint32_t>(key0 + 8 * g) * 4u);
#pragma unroll
            for (int i = 0; i < 4; ++i) bv[4 * g + i] = x[i];
        }
    };
    if (wave_active) load_bias(0);

    const int stage = p.stage_rows;
    for (int c0 = 0; c0 < L; c0 += stage) {
        __syncthreads();
        const int ckeys = L - c0 < stage ? L - c0 : stage;
        const int rows = (ckeys + 31) / 32 * 32;
        stage_two<DP, NW * 64, T::CH_ROWS, TWIN>(p.K + po, lds_k, lds_kt, p.scale * LOG2E, p.V + po, lds_v, c0, rows, ckeys, d, tid);
        __syncthreads();
        if (!wave_active) continue;
        for (int kt = 0; kt < rows / 32; ++kt) {
            const int key0 = c0 + kt * 32;
            // ---- probabilities of this lane's query for its 16 keys of the tile (their bias was requested a
            // tile ago, see below)
            v16f st = tile_times_slice<DP, TWIN>(lds_k + kt * T::TILE + row_at, qb);
            v16f dp = tile_times_slice<DP, TWIN>(lds_v + kt * T::TILE + row_at, dob);
#pragma unroll
            for (int r = 0; r < 16; ++r) {
                const int key = key0 + 8 * (r >> 2) + 4 * half + (r & 3);
                float s2 = st[r];
                if (BIAS && has_bias) s2 = __builtin_fmaf(bv[r], LOG2E, s2);
                // dS (chosen behind the product: 0 * NaN is not 0)
                st[r] = key < row_keys ? __builtin_amdgcn_exp2f(s2 - lse2) * (dp[r] - D_i) : 0.0f;
            }
            // the bias registers are free again: the next tile's values travel during the rest of this tile
            // and the first contractions of the next (the tiles follow each other across the stages)
            if (key0 + 32 < L) load_bias(key0 + 32);
            // ---- dbias = dS (zeros where the key is masked; every position of a valid row is written)
            if (dbias_row && q < L) {
#pragma unroll
                for (int g = 0; g < 4; ++g) {
                    const int key = key0 + 8 * g + 4 * half;
                    if (key + 3 < L) {
                        *reinterpret_cast<v4f_u*>(dbias_row + key) = v4f{st[4 * g], st[4 * g + 1], st[4 * g + 2], st[4 * g + 3]};
                    } else {
#pragma unroll
                        for (int i = 0; i < 4; ++i) if (key + i < L) dbias_row[key + i] = st[4 * g + i];
                    }
                }
            }
            if (key0 >= wave_keys) continue;           // causal: no query of the wave sees this tile (dS = 0)
            // ---- dQ^T += K^T . dS
            if (!p.dQ) continue;
            if (TWIN) {
                if (key0 > 0 && key0 % TWIN_KEYS == 0) {
                    if (LATE) acc_q[0] += late;
                    store_dq(key0 > TWIN_KEYS);
                    acc_q[0] = late = v16f{};
                }
                v16f share[NB];
                if (LATE) acc_q[0] += late;
                accumulate_transposed<DP, true>(share, lds_kt + kt * T::TILE + col_at, st);
                if (LATE) late = share[0];
                else acc_q[0] += share[0];
            } else {
                accumulate_transposed<DP>(acc_q, lds_kt + kt * T::TILE + col_at, st);
            }
        }
    }
    if (!wave_active) return;
    if (LATE) acc_q[0] += late;
    store_dq(TWIN && wave_keys > TWIN_KEYS);
}

// ------------------------------------------------------------------------------------------------------------
// dK and dV: a wave owns 32 keys and walks over the queries.
template <int DP, int NW>
__global__ __launch_bounds__(NW * 64, 2) void flash_attn_back_cols_kernel(const AttnBackParams p) {
    using T = BackTiling<DP>;
    constexpr int NB = T::NB, NC = T::NC;
    extern __shared__ __attribute__((aligned(16))) uint8_t back_lds[];
    const int tiles_staged = p.stage_rows / 32;
    uint8_t* const lds_q = back_lds;                                 // Q: S = Q . K^T and, transposed, dK^T += Q^T . dS
    uint8_t* const lds_do = lds_q + tiles_staged * T::TILE;          // dO: dO . V^T and, transposed, dV^T += dO^T . P
    float* lds_lse = reinterpret_cast<float*>(lds_do + tiles_staged * T::TILE);       // LSE * log2(e) of the staged queries (+inf for dead rows)
    float* lds_D = lds_lse + p.stage_rows;             // D of the staged queries
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int j = lane & 31, half = lane >> 5;
    const int row_at = row_place<DP>(lane), col_at = column_place<DP>(lane);
    const int plane = blockIdx.y, L = p.L, d = p.d;
    const int k0w = (blockIdx.x * NW + wave) * 32, key = k0w + j;       // this lane's key
    const bool wave_active = k0w < L;
    const int64_t po = static_cast<int64_t>(plane) * L * d;

    v8bf kb[NC][3], vb[NC][3];
    if (wave_active) {
        v4f xk[NC][2], xv[NC][2];
        load_slice<DP>(p.K + po, k0w, j, L, d, half, xk);
        load_slice<DP>(p.V + po, k0w, j, L, d, half, xv);
        slice_parts<DP>(xk, p.scale * LOG2E, kb);
        slice_parts<DP>(xv, 1.0f, vb);
    }
    const float* bias_plane = p.bias ? p.bias + static_cast<int64_t>(plane) * L * L : nullptr;

    v16f acc_k[NB], acc_v[NB];
#pragma unroll
    for (int b = 0; b < NB; ++b)
#pragma unroll
        for (int r = 0; r < 16; ++r) { acc_k[b][r] = 0.0f; acc_v[b][r] = 0.0f; }

    const int stage = p.stage_rows;
    // causal: queries before the wave's first key see none of its keys
    const int first_chunk = p.causal ? (k0w / stage) * stage : 0;
    for (int c0 = 0; c0 < L; c0 += stage) {
        __syncthreads();
        const int cq = L - c0 < stage ? L - c0 : stage;
        const int rows = (cq + 31) / 32 * 32;
        // Q and dO as fragments, and LSE and D = sum_d dO * O of the staged queries, from one batch of loads: a
        // thread holds four features of a row, the eight threads of a row add up their parts of D.
        {
            constexpr int NT = NW * 64, NI = (T::CH_COLS * (DP / 4) + NT - 1) / NT;
            static_assert(DP / 4 == 8 || DP / 4 == 16, "eight or sixteen threads per staged row");
            const int64_t from = po + static_cast<int64_t>(c0) * d;
            const __amdgpu_buffer_rsrc_t rq = buffer_of(p.Q + from, cq * d), rdo = buffer_of(p.dO + from, cq * d), ro = buffer_of(p.O + from, cq * d),
                                         rlse = buffer_of(p.LSE + static_cast<int64_t>(plane) * L + c0, cq);
            v4f xq[NI], xdo[NI], xo[NI];
            float lse_in[NI];
#pragma unroll
            for (int i = 0; i < NI; ++i) {
                const int idx = tid + i * NT;
                const int row = idx / (DP / 4), c = (idx % (DP / 4)) * 4;
                const uint32_t at = row < cq && c < d ? static_cast<uint32_t>(row * d + c) * 4u : OUTSIDE;
                xq[i] = buffer_load4(rq, at);
                xdo[i] = buffer_load4(rdo, at);
                xo[i] = buffer_load4(ro, at);
                lse_in[i] = buffer_load1(rlse, static_cast<uint32_t>(row) * 4u);
            }
#pragma unroll
            for (int i = 0; i < NI; ++i) {
                const int idx = tid + i * NT;
                const int row = idx / (DP / 4), c = (idx % (DP / 4)) * 4;
                float sum = xdo[i][0] * xo[i][0] + xdo[i][1] * xo[i][1] + xdo[i][2] * xo[i][2] + xdo[i][3] * xo[i][3];
                sum += __shfl_xor(sum, 1, 64);
                sum += __shfl_xor(sum, 2, 64);
                sum += __shfl_xor(sum, 4, 64);
                if (DP / 4 == 16) sum += __shfl_xor(sum, 8, 64);
                if (row < rows) {
                    put_fragments<DP>(xq[i], row, c, lds_q);
                    put_fragments<DP>(xdo[i], row, c, lds_do);
                    if (c == 0) {
                        lds_lse[row] = row < cq && lse_in[i] > -INFINITY ? lse_in[i] * LOG2E : INFINITY;
                        lds_D[row] = sum;
                    }
                }
            }
        }
        __syncthreads();
        if (!wave_active || c0 < first_chunk) continue;
        for (int qt = 0; qt < rows / 32; ++qt) {
            const int qbase = c0 + qt * 32;
            if (p.causal && qbase + 32 <= k0w) continue;           // every query of the tile precedes every key of the wave
            // bias of this lane's key for its 16 queries of the tile, requested before the matrix work
            float bv[16];
            if (bias_plane) {
                // (from the tile's first row on: 32-bit offsets whatever the length; rows and keys past the matrix: zero, and masked below)
                const __amdgpu_buffer_rsrc_t rbias = buffer_of(bias_plane + static_cast<int64_t>(qbase) * L, static_cast<int64_t>(L - qbase < 32 ? L - qbase : 32) * L);
                const uint32_t row_bytes = static_cast<uint32_t>(L) * 4u;
                uint32_t at = key < L ? static_cast<uint32_t>(key) * 4u + 4u * half * row_bytes : OUTSIDE;
#pragma unroll
                for (int r = 0; r < 16; ++r) {
                    bv[r] = buffer_load1(rbias, at);
                    // (opaque: one offset that moves on, not sixteen at once)
                    at += (r & 3) == 3 ? 5 * row_bytes : row_bytes;
                    asm volatile("" : "+v"(at));
                }
            }
            // ---- S[query][key], un-transposed: this lane's key, 16 of the tile's queries
            // (heads wider than one block of features: one phase after the other, the held slices and sums leave no registers for two)
            const auto phase = [] { if (DP > 32) __builtin_amdgcn_sched_barrier(0); };
            v16f st = tile_times_slice<DP>(lds_q + qt * T::TILE + row_at, kb), dp;
            phase();
            if (DP <= 32) dp = tile_times_slice<DP>(lds_do + qt * T::TILE + row_at, vb);
            const auto seen = [&](int r) {
                const int qq = qbase + 8 * (r >> 2) + 4 * half + (r & 3);
                return qq < L && (!p.causal || key <= qq);
            };
#pragma unroll
            for (int g = 0; g < 4; ++g) {
                const v4f lse4 = *reinterpret_cast<const v4f*>(lds_lse + qt * 32 + 8 * g + 4 * half);
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                    const int r = 4 * g + i;
                    float s2 = st[r];
                    if (bias_plane) s2 = __builtin_fmaf(bv[r], LOG2E, s2);
                    st[r] = seen(r) ? __builtin_amdgcn_exp2f(s2 - lse4[i]) : 0.0f;      // P
                }
            }
            phase();
            // ---- dV^T += dO^T . P,  dO V^T,  dS = P (dO V^T - D),  dK^T += Q^T . dS
            if (p.dV) accumulate_transposed<DP>(acc_v, lds_do + qt * T::TILE + col_at, st);
            phase();
            if (!p.dK) continue;
            if (DP > 32) dp = tile_times_slice<DP>(lds_do + qt * T::TILE + row_at, vb);
            phase();
#pragma unroll
            for (int g = 0; g < 4; ++g) {
                const v4f D4 = *reinterpret_cast<const v4f*>(lds_D + qt * 32 + 8 * g + 4 * half);
#pragma unroll
                for (int i = 0; i < 4; ++i) st[4 * g + i] *= dp[4 * g + i] - D4[i];
            }
            phase();
            accumulate_transposed<DP>(acc_k, lds_q + qt * T::TILE + col_at, st);
        }
    }
    if (!wave_active || key >= L) return;
#pragma unroll
    for (int b = 0; b < NB; ++b)
#pragma unroll
        for (int g = 0; g < 4; ++g) {
            const int dd = b * 32 + 8 * g + 4 * half;
            if (dd >= d) continue;
            const int64_t off = po + static_cast<int64_t>(key) * d + dd;
            if (p.dK) *reinterpret_cast<v4f*>(p.dK + off) = v4f{acc_k[b][4 * g] * p.scale, acc_k[b][4 * g + 1] * p.scale,
                                                                acc_k[b][4 * g + 2] * p.scale, acc_k[b][4 * g + 3] * p.scale};
            if (p.dV) *reinterpret_cast<v4f*>(p.dV + off) = v4f{acc_v[b][4 * g], acc_v[b][4 * g + 1], acc_v[b][4 * g + 2], acc_v[b][4 * g + 3]};
        }
}

// ------------------------------------------------------------------------------------------------------------
// All four gradients in one pass over the score planes (d <= 32).  A work-group takes whole planes, one after the other,
// each of its NW waves 32 keys of a plane (NW * 32 keys at a time, longer planes in several rounds), and all waves walk
// over the query tiles together.  The columns kernel's arrangement -- S and dO V^T un-transposed, a lane holds 16 queries
// of ITS key -- gives P and dS as B operands of dV^T and dK^T as they stand and reads the bias / writes dbias in whole
// 128-byte row pieces; what it lacks is dQ^T += K^T dS^T, whose B operand wants a lane per QUERY.  dS, split once for dK,
// goes through LDS as bf16 parts and comes back transposed by ds_read_b64_tr_b16; the waves' partial dQ tiles meet in LDS
// and are added in wave order (no atomics: results do not depend on scheduling).  The same instruction reads Q and dO for
// the gradients out of their row fragments, so no second arrangement of them is staged.  Against the two kernels above, S,
// P and dO V^T are computed once instead of twice (60 MFMAs per 32 x 32 tile instead of 84) and the bias is read once.
// One barrier per query tile: the next tile is staged into the other half of a double buffer from loads issued two tiles
// ahead (across planes too), the partial tiles alternate between two regions.
// A step is five phases of twelve MFMAs -- S, dO V^T, dV, dK, dQ -- each with the vector work that does not depend on it
// placed between its MFMAs, and the fragments of a phase read during the one before: eight waves fill the registers and
// the LDS of a CU, so nothing else hides that work.  Per-wave time stamps: a step takes 8200 cycles for the two waves of a
// SIMD, 3840 of them MFMAs; what is left is the 32 accesses to bias and dbias (20 cycles each), LDS reads behind the
// barrier, and a clock of 1.7 GHz.  Registers decide: a variant with one more fragment set or with a second copy of the
// step (keys past the matrix handled apart) spilled inside the loop, and every reload waits for all stores in flight
// (370 us instead of 162).
// Measured, us, against the two kernels (dQ + dbias, dK + dV): 824 planes of 256 x 256, d 32, with bias 291 -> 162 (648 MB:
// 4.0 TB/s), 412 of 103 x 103 46 -> 25, 824 of 64 x 64 40 -> 25, 16 of 256 x 256 47 -> 33.
// Causal: a wave none of whose keys the tile's queries see leaves the five phases out (staging, zeros for dbias and dQ, and
// the barrier remain), and a round starts at its first visible tile; the tiles before it only have their dbias cleared.
// With all tiles contracted and P = 0 at masked pairs, one NaN behind a query reached its gradients as 0 * NaN.  With bias,
// us, contracted / left out / the two kernels: 412 planes of 256 72 / 67 / 152, 412 of 192 54 / 47 / 101, 412 of 257
// 162 / 101 / 208, 128 of 640 238 / 148 / 260; of 103, where every wave has a diagonal tile, 24.6 / 23.0 / 41.
template <int NW> struct FusedBack {
    // Row fragments of 32 rows x 32 features as in BackTiling, but with the halves (features 8 .. 15 of a chunk) 576 bytes
    // apart: the transposing reads and the staging writes then touch every bank once.
    static constexpr int HALF = 576, FRAG = 2 * HALF, CHUNK = 3 * FRAG;
    static constexpr int TILE = 2 * CHUNK;
    static constexpr int STAGE = 2 * TILE + 512;          // Q, dO, then LSE * log2(e) and D of the 32 queries, then 256 bytes nobody reads
    static constexpr int NO_KEY = 256;                     // what a lane whose key lies past the matrix reads instead of those: +inf and 0
    // A wave's dS parts ([key][query] of bf16, 64 bytes per key, its eight-byte pieces exchanged by key / 4 so that the
    // writes of sixteen keys meet every bank once), then its partial dQ tile ([query][36] floats)
    static constexpr int PART = 32 * 64;
    static constexpr int REGION = 3 * PART;
    static constexpr int QP = 36;
    static constexpr size_t LDS = 2 * STAGE + 2 * NW * static_cast<size_t>(REGION) + NO_KEY;
    static_assert(32 * QP * 4 <= REGION, "the partial tile takes the place of the parts");
};

// DB: dbias not wanted / ordinary stores / streaming stores (rows of whole 128-byte lines)
constexpr int DB_NONE = 0, DB_ORDINARY = 1, DB_STREAM = 2;

// One MFMA, then up to `valu` vector instructions, `count` times over: a wave issues in order, so vector work hides behind
// its own matrix work only where the two alternate in the program.
template <int count, int valu> __device__ __forceinline__ void interleave() {
#pragma unroll
    for (int i = 0; i < count; ++i) {
        __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
        __builtin_amdgcn_sched_group_barrier(0x002, valu, 0);
    }
}

template <int NW, bool BIAS, int DB, bool CAUSAL>
__global__ __launch_bounds__(NW * 64, 2) void flash_attn_back_fused_kernel(const AttnBackParams p) {
    using F = FusedBack<NW>;
    extern __shared__ __attribute__((aligned(16))) uint8_t back_lds[];
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int j = lane & 31, half = lane >> 5;
    const int L = p.L, d = p.d;
    const int tiles = (L + 31) / 32;
    uint8_t* const regions = back_lds + 2 * F::STAGE;
    uint8_t* const no_key_lds = regions + 2 * NW * F::REGION;
    if (tid < 64) reinterpret_cast<float*>(no_key_lds)[tid] = tid < 32 ? INFINITY : 0.0f;   // (read behind the first barrier)

    const int64_t mat = static_cast<int64_t>(L) * d, square = static_cast<int64_t>(L) * L;
    const uint32_t mat_bytes = static_cast<uint32_t>(L) * d * 4u, square_bytes = static_cast<uint32_t>(L) * L * 4u;
    const auto rsrc = [](const float* base, uint32_t bytes) {
        return __builtin_amdgcn_make_buffer_rsrc(const_cast<float*>(base), 0, static_cast<int>(bytes), 0x00020000);
    };
    const auto load4 = [](__amdgpu_buffer_rsrc_t r, uint32_t at) { return __builtin_bit_cast(v4f, __builtin_amdgcn_raw_buffer_load_b128(r, at, 0, 0)); };
    const auto load1 = [](__amdgpu_buffer_rsrc_t r, uint32_t at) { return __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(r, at, 0, 0)); };
    constexpr uint32_t OUT = 0x80000000u;

    // The work-group's sequence of steps: its planes, per plane the rounds of NW * 32 keys, per round the query tiles
    // (causal: from the first one that sees a key of the round).  Loads run ahead of the computation along this sequence,
    // across rounds and planes.
    struct Step { int plane, g0, t; };
    const auto advance = [&](Step& s) {
        if (++s.t < tiles) return;
        s.t = 0;
        s.g0 += NW * 32;
        if (CAUSAL && s.g0 < L) s.t = s.g0 / 32;
        if (s.g0 < L) return;
        s.g0 = 0;
        s.plane += static_cast<int>(gridDim.x);
    };
    // Causal: no query of the tile sees a key of this wave (or it has none).  Such a wave contracts nothing: P = 0 there,
    // but 0 * NaN is not, and what lies behind a query has no part in its gradients.
    const auto hidden = [&](const Step& s) {
        const int k0 = s.g0 + wave * 32;
        return CAUSAL && (s.t * 32 + 31 < k0 || k0 >= L);
    };

    // ---- staging of a query tile: 256 items (row, four features) of Q and 256 of dO (with O, for D), shared out over
    // the threads; rows and features past the matrix, and everything past the last plane, read as zeros
    constexpr int NT = NW * 64, ITEMS = (512 + NT - 1) / NT;
    v4f xs[ITEMS], xo[ITEMS];
    float xl[ITEMS];
    Step ahead{static_cast<int>(blockIdx.x), 0, 0};        // the tile whose loads are next (two steps ahead of the computation)
    const auto stage_load = [&]() {
        const bool there = ahead.plane < p.planes;
        const int64_t po = there ? ahead.plane * mat : 0;
        const uint32_t bytes = there ? mat_bytes : 0;
        const __amdgpu_buffer_rsrc_t rlse = rsrc(p.LSE + (there ? static_cast<int64_t>(ahead.plane) * L : 0), there ? static_cast<uint32_t>(L) * 4u : 0);
        const __amdgpu_buffer_rsrc_t ro = rsrc(p.O + po, bytes);
#pragma unroll
        for (int i = 0; i < ITEMS; ++i) {
            const bool is_do = (wave * 64 + i * NT) >= 256;          // (items of one kind per wave and turn)
            const __amdgpu_buffer_rsrc_t rx = rsrc((is_do ? p.dO : p.Q) + po, bytes);
            const int e = (tid + i * NT) & 255;
            const int row = ahead.t * 32 + (e >> 3), c = (e & 7) * 4;
            const uint32_t at = row < L && c < d ? (static_cast<uint32_t>(row) * d + c) * 4u : OUT;
            xs[i] = load4(rx, at);
            if (NT >= 512 || is_do) {
                xo[i] = load4(ro, is_do ? at : OUT);
                // (a row past the matrix: log of a sum of zero, which makes its probabilities zero)
                xl[i] = load1(rlse, is_do && row < L ? static_cast<uint32_t>(row) * 4u : OUT);
                xl[i] = row < L ? xl[i] : -INFINITY;
            }
        }
        advance(ahead);
    };
    const auto stage_put = [&](int n) {
        uint8_t* const stage = back_lds + (n & 1) * F::STAGE;
#pragma unroll
        for (int i = 0; i < ITEMS; ++i) {
            const bool is_do = (wave * 64 + i * NT) >= 256;
            const int e = (tid + i * NT) & 255;
            const int row = e >> 3, c = (e & 7) * 4;
            uint2 parts[3];
            split4(xs[i], parts);
            uint8_t* const dst = stage + (is_do ? F::TILE : 0) + (c >> 4) * F::CHUNK + ((c >> 3) & 1) * F::HALF + row * 16 + ((c >> 2) & 1) * 8;
#pragma unroll
            for (int part = 0; part < 3; ++part) *reinterpret_cast<uint2*>(dst + part * F::FRAG) = parts[part];
            if (NT >= 512 || is_do) {
                float sum = xs[i][0] * xo[i][0] + xs[i][1] * xo[i][1] + xs[i][2] * xo[i][2] + xs[i][3] * xo[i][3];
                // the eight lanes of the row: neighbours, pairs, then the other four
                sum += __builtin_bit_cast(float, __builtin_amdgcn_mov_dpp(__builtin_bit_cast(int, sum), 0xB1, 0xf, 0xf, true));
                sum += __builtin_bit_cast(float, __builtin_amdgcn_mov_dpp(__builtin_bit_cast(int, sum), 0x4E, 0xf, 0xf, true));
                sum += __builtin_bit_cast(float, __builtin_amdgcn_mov_dpp(__builtin_bit_cast(int, sum), 0x141, 0xf, 0xf, true));
                // A row without any visible key (LSE = -inf) has no gradient: +inf makes every probability exp2(-inf) = 0.
                // (Lanes that have nothing to write write where nobody reads: a branch here would cut the block in which
                // this work hides behind the matrix pipe.)
                float* const lse_at = reinterpret_cast<float*>(stage + 2 * F::TILE) + (c == 0 && is_do ? row : 64 + (lane & 31));
                lse_at[0] = xl[i] > -INFINITY ? xl[i] * LOG2E : INFINITY;
                lse_at[c == 0 && is_do ? 32 : 0] = sum;
            }
        }
    };

    // dQ of a tile: the waves' shares, in wave order
    const auto add_shares = [&](const Step& s, int n) {
        constexpr int W = NT >= 512 ? 2 : 4;               // floats per thread and turn
        typedef float vw __attribute__((ext_vector_type(W)));
#pragma unroll
        for (int i = 0; i < (1024 / W + NT - 1) / NT; ++i) {
            const int e = tid + i * NT;
            const int row = s.t * 32 + e / (32 / W), c = e % (32 / W) * W;
            if (row >= L || c >= d) continue;
            const float* src = reinterpret_cast<const float*>(regions + (n & 1) * NW * F::REGION) + e / (32 / W) * F::QP + c;
            vw x[NW];
#pragma unroll
            for (int w = 0; w < NW; ++w) x[w] = *reinterpret_cast<const vw*>(src + w * (F::REGION / 4));
            vw sum = x[0];
#pragma unroll
            for (int w = 1; w < NW; ++w) sum += x[w];
            vw* const dst = reinterpret_cast<vw*>(p.dQ + s.plane * mat + static_cast<int64_t>(row) * d + c);
            sum *= p.scale;
            if (s.g0 > 0) sum += *dst;                     // (this thread wrote it in the round before)
            *dst = sum;
        }
    };

    // ---- The bias of this lane's key for its 16 queries of a tile (requested a step ahead) and dbias; rows and keys past
    // the matrix fall outside the plane.
    float bv[16];
    const uint32_t row_bytes = static_cast<uint32_t>(L) * 4u;
    const auto square_at = [&](const Step& s) {
        const int key = s.g0 + wave * 32 + j;
        return key < L ? static_cast<uint32_t>(key) * 4u + (static_cast<uint32_t>(s.t) * 32u + 4u * half) * row_bytes : OUT;
    };
    // from the row of accumulator register r to that of the next one; opaque, so that the sixteen offsets of a tile
    // follow each other through one register instead of taking one each
    const auto next_row = [&](uint32_t& at, int r) {
        at += (r & 3) == 3 ? 5 * row_bytes : row_bytes;
        asm volatile("" : "+v"(at));
    };
    const auto load_bias = [&](const Step& s) {
        if (!BIAS) return;
        const bool there = s.plane < p.planes;
        const __amdgpu_buffer_rsrc_t rbias = rsrc(p.bias + (there ? s.plane * square : 0), there ? square_bytes : 0);
        uint32_t at = hidden(s) ? OUT : square_at(s);
#pragma unroll
        for (int r = 0; r < 16; ++r) {
            bv[r] = load1(rbias, at);
            next_row(at, r);
        }
    };
    const auto store_dbias = [&](const Step& s, const v16f& x) {
        if (DB == DB_NONE) return;
        const __amdgpu_buffer_rsrc_t rdb = rsrc(p.dbias + s.plane * square, square_bytes);
        uint32_t at = square_at(s);
#pragma unroll
        for (int r = 0; r < 16; ++r) {
            const float v = x[r];
            __builtin_amdgcn_raw_buffer_store_b32(__float_as_uint(v), rdb, at, 0, DB == DB_STREAM ? 3 : 0);
            next_row(at, r);
        }
    };

    // this lane's place in the fragments: row reads; transposing reads (see read_transposed) of staged rows and of dS parts
    const int grp = lane & 15;
    const int row_at = (lane & 31) * 16 + half * F::HALF;
    const int tr = ((lane >> 4) & 1) * F::CHUNK + ((grp >> 1) & 1) * F::HALF + (4 * half + (grp >> 2)) * 16 + (grp & 1) * 8;
    const auto read_rows = [&](const uint8_t* tile, v8bf (&a)[2][3]) {
#pragma unroll
        for (int c = 0; c < 2; ++c)
#pragma unroll
            for (int part = 0; part < 3; ++part) a[c][part] = *reinterpret_cast<const v8bf*>(tile + row_at + c * F::CHUNK + part * F::FRAG);
    };
    const auto read_columns = [&](const uint8_t* tile, v8bf (&a)[2][3]) {
#pragma unroll
        for (int ch = 0; ch < 2; ++ch)
#pragma unroll
            for (int part = 0; part < 3; ++part) a[ch][part] = read_transposed(tile + tr + part * F::FRAG + ch * 256, 128);
    };
    const auto contract = [](v16f& acc, const v8bf (&a)[2][3], const v8bf (&b)[2][3], bool from_zero) {
        const v16f zero = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int c = 0; c < 2; ++c)
#pragma unroll
            for (int q = 0; q < 6; ++q)
                acc = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a[c][SPLIT_TERMS[q][0]], b[c][SPLIT_TERMS[q][1]], from_zero && c == 0 && q == 0 ? zero : acc, 0, 0, 0);
    };
    const auto parts_of = [](const v4f& x0, const v4f& x1, v8bf (&out)[3]) {
        uint2 lo[3], hi[3];
        split4(x0, lo);
        split4(x1, hi);
#pragma unroll
        for (int part = 0; part < 3; ++part) out[part] = pack_parts(lo[part], hi[part]);
    };

    v8bf kb[2][3], vb[2][3], kt[2][3], fs[2][3];
    v16f acc_k, acc_v;

    // One step of this wave: 32 queries, its 32 keys.  Fragments are read a phase ahead of their MFMAs.
    const auto tile_step = [&](const Step& s, const Step& next, int n) {
        const uint8_t* const stage = back_lds + (n & 1) * F::STAGE;
        uint8_t* const region = regions + ((n & 1) * NW + wave) * F::REGION;
        if (hidden(s)) {
            float* const part_at = reinterpret_cast<float*>(region) + j * F::QP + 4 * half;
            stage_put(n + 1);
            stage_load();
            load_bias(next);
            store_dbias(s, v16f{});
#pragma unroll
            for (int g = 0; g < 4; ++g) *reinterpret_cast<v4f*>(part_at + 8 * g) = v4f{0.0f, 0.0f, 0.0f, 0.0f};
            return;
        }
        const bool no_key = s.g0 + wave * 32 + j >= L;
        const float* const lse_at = reinterpret_cast<const float*>(no_key ? no_key_lds : stage + 2 * F::TILE) + 4 * half;
        // ---- S[query][key]: this lane's key, 16 of the tile's queries; beside it, the next tile goes to LDS
        v16f st, ds;
        v8bf fd[2][3], fo[2][3], fq[2][3];
        contract(st, fs, kb, true);
        read_rows(stage + F::TILE, fd);
        stage_put(n + 1);
        stage_load();
        interleave<12, 6>();
        __builtin_amdgcn_sched_barrier(0);
        // ---- dO V^T; beside it, the probabilities and their parts
        contract(ds, fd, vb, true);
        read_columns(stage + F::TILE, fo);
        if (BIAS)
#pragma unroll
            for (int r = 0; r < 16; ++r) st[r] = __builtin_fmaf(bv[r], LOG2E, st[r]);
        // causal: accumulator register r holds a query that does not lie before this lane's key
        const int first = s.g0 + wave * 32 + j - s.t * 32 - 4 * half;
        const auto seen = [&](int r) { return !CAUSAL || 8 * (r >> 2) + (r & 3) >= first; };
        v8bf wp[2][3], wd[2][3];
#pragma unroll
        for (int ch = 0; ch < 2; ++ch) {
#pragma unroll
            for (int g = 2 * ch; g < 2 * ch + 2; ++g) {
                const v4f lse4 = *reinterpret_cast<const v4f*>(lse_at + 8 * g);
#pragma unroll
                for (int i = 0; i < 4; ++i) st[4 * g + i] = seen(4 * g + i) ? __builtin_amdgcn_exp2f(st[4 * g + i] - lse4[i]) : 0.0f;
            }
            parts_of(v4f{st[8 * ch], st[8 * ch + 1], st[8 * ch + 2], st[8 * ch + 3]}, v4f{st[8 * ch + 4], st[8 * ch + 5], st[8 * ch + 6], st[8 * ch + 7]}, wp[ch]);
        }
        interleave<12, 11>();
        __builtin_amdgcn_sched_barrier(0);
        // ---- dV^T += dO^T . P; beside it, dS and its parts, which also go to LDS to be transposed
        contract(acc_v, fo, wp, false);
        int put_at = j * 64 + ((half ^ (j >> 2)) & 7) * 8; // (opaque: the four pieces' places are formed from this one, not held)
        asm volatile("" : "+v"(put_at));
#pragma unroll
        for (int ch = 0; ch < 2; ++ch) {
#pragma unroll
            for (int g = 2 * ch; g < 2 * ch + 2; ++g) {
                const v4f D4 = *reinterpret_cast<const v4f*>(lse_at + 32 + 8 * g);
#pragma unroll
                for (int i = 0; i < 4; ++i) ds[4 * g + i] = seen(4 * g + i) ? st[4 * g + i] * (ds[4 * g + i] - D4[i]) : 0.0f;
            }
            parts_of(v4f{ds[8 * ch], ds[8 * ch + 1], ds[8 * ch + 2], ds[8 * ch + 3]}, v4f{ds[8 * ch + 4], ds[8 * ch + 5], ds[8 * ch + 6], ds[8 * ch + 7]}, wd[ch]);
            // piece of eight bytes: queries 4 u .. 4 u + 3, u = 4 ch + half and two further on
#pragma unroll
            for (int part = 0; part < 3; ++part) {
                const v4i x = __builtin_bit_cast(v4i, wd[ch][part]);
                *reinterpret_cast<uint2*>(region + part * F::PART + (put_at ^ (32 * ch))) = uint2{static_cast<uint32_t>(x[0]), static_cast<uint32_t>(x[1])};
                *reinterpret_cast<uint2*>(region + part * F::PART + (put_at ^ (32 * ch + 16))) = uint2{static_cast<uint32_t>(x[2]), static_cast<uint32_t>(x[3])};
            }
        }
        interleave<12, 10>();
        __builtin_amdgcn_sched_barrier(0);
        // ---- dK^T += Q^T . dS; beside it, dbias = dS and the next step's bias (into the registers read above)
        read_columns(stage, fq);
        contract(acc_k, fq, wd, false);
        v8bf w[2][3];
        // keys 16 ch + 4 half + grp / 4 and eight further on, pieces of four queries (queries from 16 * (lane / 16 % 2))
        int get_at = (4 * half + (grp >> 2)) * 64 + ((4 * ((lane >> 4) & 1) + (grp & 3)) ^ half) * 8;
        asm volatile("" : "+v"(get_at));
#pragma unroll
        for (int ch = 0; ch < 2; ++ch) {
#pragma unroll
            for (int part = 0; part < 3; ++part) {
                typedef __attribute__((address_space(3))) v4s* lds_v4s;
                const uint8_t* const at = region + part * F::PART + ch * 1024;
                const v4s lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_v4s)(at + (get_at ^ (32 * ch))));
                const v4s hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_v4s)(at + 512 + (get_at ^ (32 * ch + 16))));
                w[ch][part] = __builtin_bit_cast(v8bf, __builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7));
            }
        }
        load_bias(next);
        store_dbias(s, ds);
        __builtin_amdgcn_sched_barrier(0);
        // ---- this wave's share of dQ^T = K^T . dS^T: lane = query
        v16f dq;
        contract(dq, kt, w, true);
        float* const part_at = reinterpret_cast<float*>(region) + j * F::QP + 4 * half;
#pragma unroll
        for (int g = 0; g < 4; ++g) *reinterpret_cast<v4f*>(part_at + 8 * g) = v4f{dq[4 * g], dq[4 * g + 1], dq[4 * g + 2], dq[4 * g + 3]};
    };

    Step s{static_cast<int>(blockIdx.x), 0, 0};
    stage_load();
    load_bias(s);
    stage_put(0);
    stage_load();
    __syncthreads();
    read_rows(back_lds, fs);
    int n = 0;                                             // steps so far: which half of the double buffers a step uses
    while (s.plane < p.planes) {
        // ---- a round begins: this wave's slices of K and V as B operands over the features, K^T as the A operand of
        // dQ^T (lane = feature, its keys in the order of the transposed dS).  All loads before the first use: one round trip.
        {
            const __amdgpu_buffer_rsrc_t rk = rsrc(p.K + s.plane * mat, mat_bytes), rv = rsrc(p.V + s.plane * mat, mat_bytes);
            const int k0w = s.g0 + wave * 32, key = k0w + j;
            v4f xk[2][2], xv[2][2];
            float xt[16];
#pragma unroll
            for (int c = 0; c < 2; ++c)
#pragma unroll
                for (int i = 0; i < 2; ++i) {
                    const int e = 16 * c + 8 * half + 4 * i;
                    const uint32_t at = key < L && e < d ? (static_cast<uint32_t>(key) * d + e) * 4u : OUT;
                    xk[c][i] = load4(rk, at);
                    xv[c][i] = load4(rv, at);
                }
#pragma unroll
            for (int i = 0; i < 16; ++i) {
                const int kk = k0w + 8 * (i >> 2) + 4 * half + (i & 3);
                xt[i] = load1(rk, kk < L && j < d ? (static_cast<uint32_t>(kk) * d + j) * 4u : OUT);
            }
#pragma unroll
            for (int c = 0; c < 2; ++c) {
                parts_of(xk[c][0] * (p.scale * LOG2E), xk[c][1] * (p.scale * LOG2E), kb[c]);
                parts_of(xv[c][0], xv[c][1], vb[c]);
                parts_of(v4f{xt[8 * c], xt[8 * c + 1], xt[8 * c + 2], xt[8 * c + 3]}, v4f{xt[8 * c + 4], xt[8 * c + 5], xt[8 * c + 6], xt[8 * c + 7]}, kt[c]);
            }
        }
#pragma unroll
        for (int r = 0; r < 16; ++r) { acc_k[r] = 0.0f; acc_v[r] = 0.0f; }
        const Step round = s;
        if (CAUSAL)                                        // the tiles before the round's first one see none of its keys
            for (int t = 0; t < round.t; ++t) store_dbias(Step{round.plane, round.g0, t}, v16f{});
        for (int t = CAUSAL ? round.t : 0; t < tiles; ++t, ++n) {
            Step next = s;
            advance(next);
            tile_step(s, next, n);
            // the tile's shares are complete and the next tile is staged; the next write to this region is two steps away
            __syncthreads();
            read_rows(back_lds + ((n + 1) & 1) * F::STAGE, fs);
            if (p.dQ) add_shares(s, n);
            s = next;
        }
        const int key = round.g0 + wave * 32 + j;
        if (key < L) {
#pragma unroll
            for (int g = 0; g < 4; ++g) {
                const int dd = 8 * g + 4 * half;
                if (dd >= d) continue;
                const int64_t off = round.plane * mat + static_cast<int64_t>(key) * d + dd;
                if (p.dK) *reinterpret_cast<v4f*>(p.dK + off) = v4f{acc_k[4 * g] * p.scale, acc_k[4 * g + 1] * p.scale, acc_k[4 * g + 2] * p.scale, acc_k[4 * g + 3] * p.scale};
                if (p.dV) *reinterpret_cast<v4f*>(p.dV + off) = v4f{acc_v[4 * g], acc_v[4 * g + 1], acc_v[4 * g + 2], acc_v[4 * g + 3]};
            }
        }
    }
}

template <int NW, bool BIAS, int DB, bool CAUSAL>
int launch_fused(const AttnBackParams& p, hipStream_t stream) {
    using F = FusedBack<NW>;
    static LdsLimit limit;
    if (!limit.reserve(reinterpret_cast<const void*>(&flash_attn_back_fused_kernel<NW, BIAS, DB, CAUSAL>), F::LDS)) {
        set_error("flash_attn_backward_hip: cannot reserve the LDS of the one-pass kernel");
        return RC_LAUNCH;
    }
    const int resident = device_cu_count() * (NW >= 8 ? 1 : 2);
    hipLaunchKernelGGL((flash_attn_back_fused_kernel<NW, BIAS, DB, CAUSAL>), dim3(p.planes < resident ? p.planes : resident), dim3(NW * 64), F::LDS, stream, p);
    return check_launch("flash_attn_back_fused_kernel");
}

template <int DP, bool TWIN, bool BIAS, bool LATE>
int launch_rows(AttnBackParams p, hipStream_t stream) {
    using T = BackTiling<DP>;
    constexpr int NW = 4, MATRICES = TWIN ? 3 : 2;
    const int l32 = (p.L + 31) / 32 * 32;
    p.stage_rows = l32 < T::CH_ROWS ? l32 : T::CH_ROWS;
    const size_t lds = static_cast<size_t>(p.stage_rows / 32) * MATRICES * T::TILE;
    static LdsLimit limit;
    if (!limit.reserve(reinterpret_cast<const void*>(&flash_attn_back_rows_kernel<DP, NW, TWIN, BIAS, LATE>),
                       (T::CH_ROWS / 32) * MATRICES * T::TILE)) {
        set_error("flash_attn_backward_hip: cannot reserve the LDS of the rows kernel");
        return RC_LAUNCH;
    }
    hipLaunchKernelGGL((flash_attn_back_rows_kernel<DP, NW, TWIN, BIAS, LATE>), dim3((p.L + 32 * NW - 1) / (32 * NW), p.planes), dim3(NW * 64), lds, stream, p);
    return check_launch("flash_attn_back_rows_kernel");
}

template <int DP, bool TWIN>
int launch_back(AttnBackParams p, hipStream_t stream) {
    using T = BackTiling<DP>;
    constexpr int NW = 4;
    const int l32 = (p.L + 31) / 32 * 32;
    if (p.dQ || p.dbias) {
        int rc;
        if constexpr (TWIN) {
            // With a bias the late form's registers leave room for two work-groups per CU instead of three: taken where its
            // rounds over the chip still come no dearer.  dQ and dbias, us, late / not: 8 planes of 256 20.8 / 22.9, 412 of
            // 192 51.2 / 54.4, 412 of 103 21.1 / 22.4; 300 of 256 (600 work-groups) 55.8 / 49.4.
            const int64_t groups = static_cast<int64_t>((p.L + 127) / 128) * p.planes, cus = device_cu_count();
            const bool late = (groups + 2 * cus - 1) / (2 * cus) * 2 <= (groups + 3 * cus - 1) / (3 * cus) * 3;
            rc = !p.bias ? launch_rows<DP, true, false, true>(p, stream)
                 : late  ? launch_rows<DP, true, true, true>(p, stream)
                         : launch_rows<DP, true, true, false>(p, stream);
        } else {
            rc = launch_rows<DP, false, true, false>(p, stream);
        }
        if (rc != RC_OK) return rc;
    }
    if (p.dK || p.dV) {
        p.stage_rows = l32 < T::CH_COLS ? l32 : T::CH_COLS;
        const size_t lds = static_cast<size_t>(p.stage_rows / 32) * 2 * T::TILE +
                           static_cast<size_t>(p.stage_rows) * 2 * sizeof(float);
        static LdsLimit limit;
        if (!limit.reserve(reinterpret_cast<const void*>(&flash_attn_back_cols_kernel<DP, NW>),
                           (T::CH_COLS / 32) * 2 * T::TILE + T::CH_COLS * 8)) {
            set_error("flash_attn_backward_hip: cannot reserve the LDS of the columns kernel");
            return RC_LAUNCH;
        }
        hipLaunchKernelGGL((flash_attn_back_cols_kernel<DP, NW>), dim3((p.L + 32 * NW - 1) / (32 * NW), p.planes), dim3(NW * 64), lds, stream, p);
        return check_launch("flash_attn_back_cols_kernel");
    }
    return RC_OK;
}

}  // namespace
}  // namespace ppmlhip

using namespace ppmlhip;

extern "C" int flash_attn_backward_hip(int B, int h, int L, int d, int causal, float scale,
                                       const float* Q, const float* K, const float* V, const float* bias,
                                       const float* O, const float* dO, const float* LSE,
                                       float* dQ, float* dK, float* dV, float* dbias, ppml_hip_stream_t stream) {
    if (!Q || !K || !V || !O || !dO || !LSE || (!dQ && !dK && !dV && !dbias) || B <= 0 || h <= 0 || L <= 0 || d <= 0) {
        set_error("flash_attn_backward_hip: bad arguments (B=%d h=%d L=%d d=%d)", B, h, L, d);
        return RC_BAD_ARGS;
    }
    if (d > 64 || (d & 3) != 0) {
        set_error("flash_attn_backward_hip: head dimension %d not supported (multiple of 4, at most 64)", d);
        return RC_BAD_ARGS;
    }
    const auto misaligned = [](const void* ptr) { return ptr && (reinterpret_cast<uintptr_t>(ptr) & 15) != 0; };
    if (misaligned(Q) || misaligned(K) || misaligned(V) || misaligned(O) || misaligned(dO) || misaligned(dQ) || misaligned(dK) || misaligned(dV)) {
        set_error("flash_attn_backward_hip: Q, K, V, O, dO and the gradients must be 16-byte aligned");
        return RC_BAD_ARGS;
    }
    const int64_t planes = static_cast<int64_t>(B) * h;
    if (planes > 65535) {
        set_error("flash_attn_backward_hip: %lld planes exceed the grid limit of 65535", static_cast<long long>(planes));
        return RC_BAD_ARGS;
    }
    AttnBackParams p;
    p.Q = Q; p.K = K; p.V = V; p.bias = bias; p.O = O; p.dO = dO; p.LSE = LSE;
    p.dQ = dQ; p.dK = dK; p.dV = dV; p.dbias = dbias;
    p.planes = static_cast<int>(planes); p.L = L; p.d = d;
    p.causal = causal ? 1 : 0;
    p.scale = scale > 0.0f ? scale : 1.0f / std::sqrt(static_cast<float>(d));   // FlashAttn.cpp:153
    p.stage_rows = 0;
    StatsScope stat("hip/flash_attn_back", static_cast<int64_t>(planes) * L, d, L, static_cast<hipStream_t>(stream));
    hipStream_t s = static_cast<hipStream_t>(stream);
    // One pass or two kernels, for head dimensions of one feature block (all figures us, one pass / two kernels).
    // A call that wants gradients on both sides (dQ or dbias, dK or dV): one pass up to 256 rows.  Beyond, a work-group walks
    // over a plane in rounds while the two kernels have one per 128 rows, and the planes alone have to occupy the chip -- from
    // 3/8 of the CUs on if causal (96 planes of 384 62 / 90) or, up to 512 rows, with a bias (of 384 90 / 101; 64 planes
    // 89 / 72), half of them with a bias beyond (128 of 640 245 / 295, 96 of them 220 / 198), and without either only where the
    // rounds over the chip are 3/5 full (160 of 512 113 / 160, 128 of 320 73 / 73, 300 of them 144 / 133).
    // A call that wants one side only would have the one-pass kernel contract for the other as well; for it the two kernels'
    // half is the rule (8 planes of 256, dQ 29 / 17, dK and dV 29 / 23; 128 of 640, dbias 215 / 149), and the exceptions need
    // rounds 3/4 full and a side's pair (dbias with the bias its kernel would read a lane per row): causal from 129 rows on
    // (412 of 256, dQ and dbias 62 / 83), not causal from 129 to 256 rows in at most two rounds (256 of 160, dK and dV 22 / 26),
    // or with a bias from 385 to 512 (200 of 448, dQ and dbias 117 / 142).
    // dQ on the memory of Q, dO or O, which such a call may have (the rows kernel reads a query's row before it writes it),
    // rules out rounds: they read those again.
    // Either way the bits are the same: where the whole set goes in one pass, the two kernels compute as it does.
    const int64_t cus = device_cu_count(), slots = (planes + cus - 1) / cus * cus;
    const bool rows = dQ || dbias, cols = dK || dV;
    const bool whole = d <= 32 && L < 16384 &&
                       (L <= 256 || (causal || (bias && L <= 512) ? 8 * planes >= 3 * cus : bias ? 2 * planes >= cus : 5 * planes >= 3 * slots));
    const bool pair = (dK && dV) || (dbias && bias);
    const bool in_place = dQ && (dQ == Q || dQ == dO || dQ == O);
    const bool one_side = pair && L > 128 && !(in_place && L > 256) && 4 * planes >= 3 * slots &&
                          (causal ? bias || planes <= 2 * cus
                                  : L <= 256 ? planes <= 2 * cus && (cols || dQ) : bias && L > 384 && L <= 512);
    if (whole && ((rows && cols) || one_side)) {
        const bool streaming = L % 32 == 0 && (reinterpret_cast<uintptr_t>(dbias) & 127) == 0;
        const int db = !dbias ? DB_NONE : streaming ? DB_STREAM : DB_ORDINARY;
        const int kt = (L + 31) / 32;
#define PPML_BACK_DB(NW_, BIAS_, C_) (db == DB_NONE ? launch_fused<NW_, BIAS_, DB_NONE, C_>(p, s) : db == DB_STREAM ? launch_fused<NW_, BIAS_, DB_STREAM, C_>(p, s) : launch_fused<NW_, BIAS_, DB_ORDINARY, C_>(p, s))
#define PPML_BACK_B(NW_, C_) (bias ? PPML_BACK_DB(NW_, true, C_) : PPML_BACK_DB(NW_, false, C_))
#define PPML_BACK(NW_) (causal ? PPML_BACK_B(NW_, true) : PPML_BACK_B(NW_, false))
        return kt <= 4 ? PPML_BACK(4) : PPML_BACK(8);
#undef PPML_BACK
#undef PPML_BACK_B
#undef PPML_BACK_DB
    }
    return d > 32 ? launch_back<64, false>(p, s) : whole ? launch_back<32, true>(p, s) : launch_back<32, false>(p, s);
}
