// The reference's default attention (src/modules/Attention.cpp:264-281) from its graph tensors in one launch:
//     out_prod(K, Q) -> scale -> [add bias] -> softmax -> out_prod(softmax^T, V^T),   Q, K, V, result [B][h][d][L]
// with the bits of the three launches the executor otherwise makes of it (out_prod_scaled, softmax_add, out_prod_tt): the same
// partial products in the same order (gemm_bf16x3_shortk_kernel, gemm_bf16x3_pc_narrow_kernel), the elements of a row on the
// same lanes and its sums in the same order (softmax_rows_kernel).  What goes is the memory between them: the scores were written, read,
// written again as probabilities and read again, four times the bytes of the bias.
//
// One work-group per plane of up to 128 rows, two waves per 32 queries.  K and V are split once per work-group and lie in
// LDS as MFMA fragments; a wave's scores (every other tile of 32 keys) stay in registers until every wave is done with K, then take K's place in LDS
// as whole rows, become probabilities there (sixteen rows per wave), and are split as they are read for the second contraction.  Rows of 103:
// 80 KB, two work-groups per CU.  What bounds it is the vector work of
// the softmax (thirteen instructions per exponential; with each row's two reductions and its division by itself, and an LDS round trip
// in the reductions, 412 planes of 103 took 23.8 us) and, with one work-group per CU, the chain of loads, split, scores,
// softmax and sum: 12.8 us for 256 planes, which a second work-group on the CU half hides (18.4 for 412).
// Measured, us, three launches / this, with bias: 412 planes of 103 31.1 / 18.4, 256 25.6 / 12.8, 824 of 51 27.6 / 13.6, 824 of 128 65 / 56,
// 32 of 24 11.0 / 8.8, of 80 11.9 / 12.2.  Rows of a multiple of four lie four elements a lane, as that kernel has them, and
// leave half of the lanes without any: 412 planes of 104 21.0.
#include "common.hpp"

namespace ppmlhip {
namespace {

constexpr int CHAIN_ROWS = 128, CHAIN_FEATURES = 32;

struct ChainParams {
    const float* Q; const float* K; const float* V; const float* bias;
    float* O;
    int planes, L, d;
    float scale;
    int pitch;           // floats per row of scores in LDS
};

// VEC: rows of whole 16-byte pieces (L a multiple of four), four elements per lane; otherwise PIECES single ones
template <bool VEC, int PIECES, bool HAS_BIAS>
__global__ __launch_bounds__(512, 4) void attention_chain_kernel(const ChainParams p) {
    constexpr int W = VEC ? 4 : 1, E = PIECES * W, ROWS = 4;
    extern __shared__ __attribute__((aligned(16))) uint8_t chain_lds[];
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6), tiles = blockDim.x >> 7;
    const int side = wave & 1;                          // which of the two waves of its 32 queries
    const int j = lane & 31, hh = lane >> 5;
    const int L = p.L, d = p.d, chunks = (L + 15) / 16;
    const int64_t plane = blockIdx.x;
    const float* const Q = p.Q + plane * d * L;
    const float* const K = p.K + plane * d * L;
    const float* const V = p.V + plane * d * L;
    uint8_t* const lds_v = chain_lds;                                        // [16 keys][part][1 KB]
    uint8_t* const lds_k = chain_lds + chunks * 3072;                        // [32 keys][16 features][part][1 KB], then the scores
    float* const rows = reinterpret_cast<float*>(lds_k) + (wave >> 1) * 32 * p.pitch;   // this wave's queries
    const int q0 = (wave >> 1) * 32;

    // ---- the operands: sixteen features of a tile of 32 keys, a chunk of sixteen keys of V, this wave's queries (lane: one
    // key / feature / query, eight features / keys)
    SplitGuard guard_s, guard_v;
    v4f kx[2], qx[2][2], vx[2];
    // through buffer resources over the plane's operands (outside: zero): a load under a condition is waited for where the
    // condition ends, one memory round trip after the other (412 planes of 103: 24.0 us)
    constexpr uint32_t OUT = 0x80000000u;
    const auto over_plane = [&](const float* base) {
        return __builtin_amdgcn_make_buffer_rsrc(const_cast<float*>(base), 0, d * L * 4, 0x00020000);
    };
    const __amdgpu_buffer_rsrc_t rk = over_plane(K), rq = over_plane(Q), rv = over_plane(V);
    const uint32_t col = q0 + j < L ? static_cast<uint32_t>(q0 + j) * 4u : OUT;
    const auto load_column = [&](const __amdgpu_buffer_rsrc_t r, int c, v4f (&x)[2]) {          // (features past the last: behind the plane)
#pragma unroll
        for (int i = 0; i < 8; ++i)
            x[i >> 2][i & 3] = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(r, col + static_cast<uint32_t>((16 * c + 8 * hh + i) * L) * 4u, 0, 0));
    };
    load_column(rk, side, kx);
    load_column(rq, 0, qx[0]);
    load_column(rq, 1, qx[1]);
    {
        const int key = wave * 16 + 8 * hh;
        const uint32_t at = j < d ? static_cast<uint32_t>(j * L + key) * 4u : OUT;
        if (wave * 16 + 16 <= L) {                      // (the same for the wave)
#pragma unroll
            for (int h = 0; h < 2; ++h) vx[h] = __builtin_bit_cast(v4f, __builtin_amdgcn_raw_buffer_load_b128(rv, at + 16u * h, 0, 0));
        } else {
#pragma unroll
            for (int i = 0; i < 8; ++i)
                vx[i >> 2][i & 3] = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(rv, key + i < L ? at + 4u * i : OUT, 0, 0));
        }
    }
    // the bias of the first rows travels meanwhile (lanes past a row's end read its last elements, rows past the plane its last)
    float vb[ROWS][HAS_BIAS ? E : 1];
    const auto load_bias = [&](int r0) {
        if (!HAS_BIAS) return;
#pragma unroll
        for (int r = 0; r < ROWS; ++r) {
            const int row = q0 + r0 + r < L ? q0 + r0 + r : L - 1;
            const float* b = p.bias + (plane * L + row) * L;
#pragma unroll
            for (int u = 0; u < PIECES; ++u) {
                const int want = (lane + 64 * u) * W, at = want < L ? want : L - W;
                if (VEC) {
                    const v4f t = *reinterpret_cast<const v4f_u*>(b + at);
#pragma unroll
                    for (int c = 0; c < 4; ++c) vb[r][u * W + c % W] = t[c];
                } else {
                    vb[r][u] = b[at];
                }
            }
        }
    };
    load_bias(16 * side);

    v8bf qf[2][3];
    {
        v8bf f[3];
        split8(kx, f, guard_s);
#pragma unroll
        for (int s = 0; s < 3; ++s) *reinterpret_cast<v8bf*>(lds_k + (wave * 3 + s) * 1024 + lane * 16) = f[s];
        split8(qx[0], qf[0], guard_s);
        split8(qx[1], qf[1], guard_s);
        split8(vx, f, guard_v);
        if (wave < chunks) {
#pragma unroll
            for (int s = 0; s < 3; ++s) *reinterpret_cast<v8bf*>(lds_v + (wave * 3 + s) * 1024 + lane * 16) = f[s];
        }
    }
    // operands that the split cannot carry: those contractions the reference's way (a whole work-group's at once)
    const bool plain_scores = __syncthreads_or(guard_s.fired() ? 1 : 0) != 0;
    const bool plain_v = __syncthreads_or(guard_v.fired() ? 1 : 0) != 0;

    // ---- scores, rows = queries: tiles `side` and `side` + 2
    v16f acc[2];
#pragma unroll
    for (int u = 0; u < 2; ++u)
#pragma unroll
        for (int r = 0; r < 16; ++r) acc[u][r] = 0.0f;
#pragma unroll
    for (int c = 0; c < 2; ++c) {
        v8bf kf[2][3];
#pragma unroll
        for (int u = 0; u < 2; ++u)                     // (a tile past the last: the first again, not stored)
#pragma unroll
            for (int s = 0; s < 3; ++s)
                kf[u][s] = *reinterpret_cast<const v8bf*>(lds_k + (((side + 2 * u < tiles ? side + 2 * u : 0) * 2 + c) * 3 + s) * 1024 + lane * 16);
#pragma unroll
        for (int q = 0; q < 6; ++q)
#pragma unroll
            for (int u = 0; u < 2; ++u)
                acc[u] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(qf[c][SPLIT_TERMS[q][0]], kf[u][SPLIT_TERMS[q][1]], acc[u], 0, 0, 0);
    }
    __syncthreads();                                    // K has been read: the rows take its place
    const int width = chunks * 16;                      // (columns past L: zeros, as the second contraction wants them)
    if (!plain_scores) {
        const bool scaled = p.scale != 1.0f;
#pragma unroll
        for (int u = 0; u < 2; ++u) {
            const int col0 = (side + 2 * u) * 32 + j;
            if (col0 >= width) continue;
#pragma unroll
            for (int r = 0; r < 16; ++r) rows[mfma32_row(r, lane) * p.pitch + col0] = scaled ? acc[u][r] * p.scale : acc[u][r];
        }
    } else {
        for (int e = side * 64 + lane; e < 32 * width; e += 128) {
            const int row = e / width, col = e - row * width;
            float s = 0.0f;
            if (q0 + row < L && col < L)
                for (int f = 0; f < d; ++f) {
                    const float prod = Q[static_cast<int64_t>(f) * L + q0 + row] * K[static_cast<int64_t>(f) * L + col];
                    s = s + prod;
                }
            rows[row * p.pitch + col] = s * p.scale;
        }
    }
    __syncthreads();

    // ---- softmax, four rows at a time: softmax_rows_kernel on rows in LDS
    for (int r0 = 16 * side; r0 < 16 * side + 16 && q0 + r0 < L; r0 += ROWS) {
        float v[ROWS][E], mx[ROWS], sum[ROWS];
#pragma unroll
        for (int r = 0; r < ROWS; ++r) {
            const float* const x = rows + (r0 + r) * p.pitch;
            mx[r] = -INFINITY;
#pragma unroll
            for (int u = 0; u < PIECES; ++u) {
                const int want = (lane + 64 * u) * W, at = want < L ? want : L - W;
                float t[W];
                if (VEC) {
                    const v4f y = *reinterpret_cast<const v4f*>(x + at);
#pragma unroll
                    for (int c = 0; c < W; ++c) t[c] = y[c];
                } else {
                    t[0] = x[at];
                }
#pragma unroll
                for (int c = 0; c < W; ++c) {
                    const float s = HAS_BIAS ? t[c] + vb[r][u * W + c] : t[c];
                    v[r][u * W + c] = want < L ? s : -INFINITY;
                    mx[r] = fmaxf(mx[r], v[r][u * W + c]);
                }
            }
        }
        if (r0 + ROWS < 16 * side + 16) load_bias(r0 + ROWS);
        // (a NaN that comes first stays the maximum of that kernel; here, as any NaN, it gets into the sum: the same row of NaN.
        // Elements past the row are -inf, and exp(-inf - maximum) is the zero that they are there.)
        const float top = wave_butterfly4(mx, [](float x, float y) { return fmaxf(x, y); });
#pragma unroll
        for (int r = 0; r < ROWS; ++r) {
            const float m = lane_value(top, FOLD4_LANE[r]);
            sum[r] = 0.0f;
#pragma unroll
            for (int e = 0; e < E; ++e) {
                v[r][e] = expf(v[r][e] - m);
                sum[r] += v[r][e];
            }
        }
        const float inv = 1.0f / (wave_butterfly4(sum, [](float x, float y) { return x + y; }) + 1e-9f);
        float f[ROWS];                                  // (read here, where every lane has computed its quotient)
#pragma unroll
        for (int r = 0; r < ROWS; ++r) f[r] = lane_value(inv, FOLD4_LANE[r]);
#pragma unroll
        for (int u = 0; u < PIECES; ++u) {
            const int at = (lane + 64 * u) * W;
            if (at >= L) continue;
#pragma unroll
            for (int r = 0; r < ROWS; ++r) {
                float* const y = rows + (r0 + r) * p.pitch;
                if (VEC) {
                    v4f t;
#pragma unroll
                    for (int c = 0; c < 4; ++c) t[c] = v[r][u * W + c % W] * f[r];
                    *reinterpret_cast<v4f*>(y + at) = t;
                } else {
                    y[at] = v[r][u] * f[r];
                }
            }
        }
    }
    __syncthreads();
    if (side != 0) return;

    // ---- the weighted sum, rows = features, this lane's query
    float* const O = p.O + plane * d * L;
    const int q = q0 + j;
    v16f out;
#pragma unroll
    for (int r = 0; r < 16; ++r) out[r] = 0.0f;
    SplitGuard guard_p;
    const float* const prob = rows + j * p.pitch + 8 * hh;
    for (int ch = 0; ch < chunks; ++ch) {
        v4f px[2] = {*reinterpret_cast<const v4f*>(prob + ch * 16), *reinterpret_cast<const v4f*>(prob + ch * 16 + 4)};
        if (q >= L) px[0] = px[1] = v4f{0.0f, 0.0f, 0.0f, 0.0f};          // (rows past the plane hold scores, not probabilities)
        v8bf pf[3], vf[3];
        split8(px, pf, guard_p);
#pragma unroll
        for (int s = 0; s < 3; ++s) vf[s] = *reinterpret_cast<const v8bf*>(lds_v + (ch * 3 + s) * 1024 + lane * 16);
#pragma unroll
        for (int t = 0; t < 6; ++t) out = __builtin_amdgcn_mfma_f32_32x32x16_bf16(vf[SPLIT_TERMS[t][0]], pf[SPLIT_TERMS[t][1]], out, 0, 0, 0);
    }
    if (plain_v || __builtin_amdgcn_ballot_w64(guard_p.fired()) != 0) {
        for (int e = lane; e < d * 32; e += 64) {
            const int f = e >> 5, row = e & 31;
            if (q0 + row >= L) continue;
            float s = 0.0f;
            for (int k = 0; k < L; ++k) {
                const float prod = V[static_cast<int64_t>(f) * L + k] * rows[row * p.pitch + k];
                s = s + prod;
            }
            O[static_cast<int64_t>(f) * L + q0 + row] = s;
        }
        return;
    }
    if (q >= L) return;
#pragma unroll
    for (int r = 0; r < 16; ++r) {
        const int f = mfma32_row(r, lane);
        if (f < d) O[static_cast<int64_t>(f) * L + q] = out[r];
    }
}

template <bool VEC, int PIECES, bool HAS_BIAS>
int launch_chain(const ChainParams& p, hipStream_t stream) {
    const auto kernel = &attention_chain_kernel<VEC, PIECES, HAS_BIAS>;
    const int chunks = (p.L + 15) / 16, tiles = (p.L + 31) / 32;
    const auto bytes = [](int chunks_, int tiles_, int pitch) {
        const int k = tiles_ * 6144, s = tiles_ * 32 * pitch * 4;
        return chunks_ * 3072 + (k > s ? k : s);
    };
    static LdsLimit limit;
    if (!limit.reserve(reinterpret_cast<const void*>(kernel), bytes(CHAIN_ROWS / 16, CHAIN_ROWS / 32, CHAIN_ROWS + 4))) {
        set_error("attention_chain: cannot reserve its LDS");
        return RC_LAUNCH;
    }
    hipLaunchKernelGGL(kernel, dim3(static_cast<unsigned>(p.planes)), dim3(tiles * 128), static_cast<size_t>(bytes(chunks, tiles, p.pitch)), stream, p);
    return check_launch("attention_chain_kernel");
}

}  // namespace

bool attention_chain_fits(int64_t planes, int64_t L, int64_t d) {
    return planes > 0 && planes <= 0x7fffffff && L > 0 && L <= CHAIN_ROWS && d > 0 && d <= CHAIN_FEATURES;
}

int attention_chain(const float* Q, const float* K, const float* V, const float* bias, float* O, int64_t planes, int L, int d, float scale,
                    hipStream_t stream) {
    if (!Q || !K || !V || !O || !attention_chain_fits(planes, L, d)) { set_error("attention_chain: bad arguments"); return RC_BAD_ARGS; }
    StatsScope stat("hip/attention_chain", planes * L, d, L, stream);
    ChainParams p{Q, K, V, bias, O, static_cast<int>(planes), L, d, scale, (L + 15) / 16 * 16 + 4};
    // (which lane holds which element decides the order of a row's sum: the softmax node's own choice)
    if (L % 4 == 0)  return bias ? launch_chain<true, 1, true>(p, stream) : launch_chain<true, 1, false>(p, stream);
    if (L <= 64)     return bias ? launch_chain<false, 1, true>(p, stream) : launch_chain<false, 1, false>(p, stream);
    return bias ? launch_chain<false, 2, true>(p, stream) : launch_chain<false, 2, false>(p, stream);
}

}  // namespace ppmlhip
