// tq_dense.hip -- attention over bf16 key / value rows for gfx950: the decoded rows of a packed
// layer (several query tokens at once) and the tokens kept dense.
//
// Reference: chunked_turboquant_attention (runtime/attention.py:215-304) and the dense-buffer
// merge of fused_attention (runtime/triton_kernels.py:338-366), which run fp32 matrix products
// and a dozen elementwise launches per chunk.
//
// Arithmetic: logits are fp32 sums of exact products (bf16 keys; a bf16 query as it is, an fp32
// query as three bf16 terms that add up to it), times the scale, plus the mask; the softmax
// weights stay fp32 and meet the bf16 values as three bf16 terms p = hi + mid + lo (8 + 8 + 8
// bits, exact down to weights of 2^-110 and within 2^-133 below), so no weight is rounded before its
// product.
//
// Layout.  A wave owns 32 query rows (query head x query token of one KV head) and walks its
// tokens in tiles of TK, all W waves of a workgroup on the same tile with different rows.
//   S^T = K Q^T   v_mfma_f32_32x32x16_bf16, A = 32 tokens x 16 dims, B = 16 dims x 32 rows: lane
//                 (r = l % 32, h = l / 32) ends with row r's scores of the tokens
//                 8 j + 4 h + (0..3) of each 32-token block
//   O^T = V^T P^T A = 32 dims x 16 tokens, B = 16 tokens x 32 rows.  The order of the 16 tokens
//                 along k is free, so it is chosen as the order the scores come back in: lane
//                 (r, h) holds tokens 4 h + (0..3), 8 + 4 h + (0..3), and its scores become its B
//                 operand with no exchange between lanes.  V is staged transposed in that order.
// A row's softmax is two lanes wide; the running maximum takes one exchange per tile.
//
// Bound: with a bf16 query and no fp32 mask a wave runs 32 MFMA (1024 cycles) and ~300 VALU (1200)
// per tile, half of them the weights' split into terms; with two waves per SIMD the two overlap
// little.  Measured at 256 query tokens, 32 query heads, 8 KV heads, 8192 tokens: 74 us without a
// mask, 84 us with a boolean one (34 GFLOP of products, 69 GFLOP of MFMA work); the torch operations
// it replaced took 1.65 ms.  The next tile's mask is read ahead of its rows: loads return in order,
// and a mask read after them waited for them in every tile (100 us).  Three waves per SIMD spill
// (119 us).  Splits over the tokens fill the chip when there are few rows; dense_merge_kernel adds
// them up: 4 query tokens against the same rows take 18 us with 43 splits, 33 us with 21.

#include <algorithm>
#include <type_traits>

#include "tq_common.h"

namespace {

constexpr int D = TQ_DIM;
constexpr int TK = 32;         // tokens per tile
constexpr int MAX_SPLIT = 64;   // partials a merge wave weighs with one lane each

typedef float f32x16 __attribute__((ext_vector_type(16)));
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
union Frag {
    uint32_t u[4];
    uint4 q;
    bf16x8 b;
};

__device__ __forceinline__ f32x16 mfma_32(const Frag& a, const Frag& b, f32x16 c) {
    return __builtin_amdgcn_mfma_f32_32x32x16_bf16(a.b, b.b, c, 0, 0, 0);
}

// bf16 terms of a pair of fp32 values, truncated: a - hi and (a - hi) - mid are exact, and what
// is left after two terms of 8 bits fits the third.
__device__ __forceinline__ uint32_t high_halves(float a, float b) {
    return __builtin_amdgcn_perm(__float_as_uint(b), __float_as_uint(a), 0x07060302u);
}
__device__ __forceinline__ float drop_high(float a) { return a - __uint_as_float(__float_as_uint(a) & 0xFFFF0000u); }

// The same for a query element, of which an infinity leaves nothing and a NaN stays one.
__device__ __forceinline__ float drop_high_query(float a) {
    return __builtin_fabsf(a) == __builtin_inff() ? 0.0f : drop_high(a);
}

// A weight of few bits has zero lower terms, and 0 x inf makes NaN of the infinity that its leading
// term's product with an infinite value gives.  Either leaves an output that is not finite, whatever
// follows, so a workgroup that ends with one walks its tokens a second time, with care: the leading terms
// meet the infinities and NaN alone, and then all terms the finite values.  Looking at the outputs once
// leaves a call of 4 query tokens over 8192 (32 query heads, 8 KV heads, boolean mask) at 23.6 us and one
// of 256 at 92.5; looking at each tile's values as it is staged took 25.5 and 94.2, no care at all 23.3.
// An fp32 query's terms meet the keys alike.

// All ones in the halves of a bf16 pair that are not finite.
__device__ __forceinline__ uint32_t special_mask(uint32_t p) {
    return ((p & 0x7FFFu) >= 0x7F80u ? 0x0000FFFFu : 0u) | ((p & 0x7FFF0000u) >= 0x7F800000u ? 0xFFFF0000u : 0u);
}

// 2^x (v_exp_f32, 1 ulp; 2^-inf = 0).
__device__ __forceinline__ float exp2_(float x) { return __builtin_amdgcn_exp2f(x); }
constexpr float LOG2E = 1.44269504f;

struct DenseArgs {
    const void* q;
    int q_heads, kv_heads, q_len;
    int64_t q_sb, q_sh, q_ss;
    const uint16_t* k;
    const uint16_t* v;
    int64_t tokens;
    int64_t k_sb, k_sh, k_st, v_sb, v_sh, v_st;
    const void* mask;
    int64_t mask_sb, mask_sh, mask_ss;
    const int32_t* starts;
    const int32_t* ends;
    int64_t pos0;
    float scale;
    int accumulate;
    int64_t rows;    // batch * q_heads * q_len
    float* part_o;   // [split][rows][D]
    float2* part_ms; // [split][rows] (running maximum, sum of weights)
};

enum { MASK_NONE = 0, MASK_BOOL = 1, MASK_F32 = 2 };

// LDS tiles: K [TK][128] with its 16-byte chunks xor-swizzled by the token (reads of one chunk
// column by 16 tokens hit 16 different chunk columns); V^T [128][TK] likewise by the dim, with the
// higher dim bits folded in so that the transposing writes, whose lanes differ in the higher bits,
// spread over the banks too.
__device__ __forceinline__ int v_swizzle(int dim) { return ((dim >> 2) ^ (dim >> 4)) & 3; }

template <int W, int QT, int MASK>
__global__ __launch_bounds__(64 * W, QT == 1 && W > 1 ? 2 : 1) void dense_attn_kernel(DenseArgs a) {
    constexpr int T = 64 * W;
    constexpr int KC = TK * 16 / T;     // 16-byte chunks of K a thread stages per tile
    constexpr int VP = TK / 2 * 16 / T; // (token pair, chunk) items of V
    __shared__ uint4 s_k[TK * 16];
    __shared__ uint32_t s_v[D * TK / 2];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int r = lane & 31, h = lane >> 5;
    const int b = blockIdx.z / a.kv_heads, kvh = blockIdx.z % a.kv_heads;
    const int group = a.q_heads / a.kv_heads;
    const int n_rows = group * a.q_len;
    const int row = (blockIdx.y * W + wave) * 32 + r;
    const bool live = row < n_rows;
    const int hq = live ? row / a.q_len : 0, sq = live ? row - hq * a.q_len : 0;

    // ---- this lane's query row: dims 16 s + 8 h + (0..7) for s = 0..7
    Frag q[QT][8];
    {
        const int64_t off = b * a.q_sb + (int64_t)(kvh * group + hq) * a.q_sh + sq * a.q_ss;
#pragma unroll
        for (int s = 0; s < 8; ++s) {
            if constexpr (QT == 1) {
                const uint4 w = reinterpret_cast<const uint4*>(static_cast<const uint16_t*>(a.q) + off)[2 * s + h];
                q[0][s].q = live ? w : make_uint4(0u, 0u, 0u, 0u);
            } else {
                const float4* p = reinterpret_cast<const float4*>(static_cast<const float*>(a.q) + off) + 4 * s + 2 * h;
                const float4 x = p[0], y = p[1];
                const float e[8] = {x.x, x.y, x.z, x.w, y.x, y.y, y.z, y.w};
#pragma unroll
                for (int k = 0; k < 4; ++k) {
                    float e0 = live ? e[2 * k] : 0.0f, e1 = live ? e[2 * k + 1] : 0.0f;
                    q[0][s].u[k] = high_halves(e0, e1);
                    e0 = drop_high_query(e0), e1 = drop_high_query(e1);
                    q[QT - 2][s].u[k] = high_halves(e0, e1);
                    q[QT - 1][s].u[k] = high_halves(drop_high(e0), drop_high(e1));
                }
            }
        }
    }

    // ---- token range of this split, whole tiles
    const int64_t tiles = (a.tokens + TK - 1) / TK;
    const int64_t per = (tiles + gridDim.x - 1) / gridDim.x;
    const int64_t t_begin = std::min<int64_t>((int64_t)blockIdx.x * per, tiles) * TK;
    const int64_t t_end = std::min<int64_t>(((int64_t)blockIdx.x + 1) * per * TK, a.tokens);
    const int64_t out_row = (int64_t)(b * a.q_heads + kvh * group) * a.q_len + row;
    const int64_t slot = (int64_t)blockIdx.x * a.rows + out_row;
    if (a.accumulate && t_begin >= t_end) return;  // uniform over the workgroup

    // attended positions of this batch row, relative to the first token
    int64_t lo = 0, hi = a.tokens;
    if (a.starts) lo = std::max<int64_t>(lo, a.starts[b] - a.pos0);
    if (a.ends) hi = std::min<int64_t>(hi, a.ends[b] - a.pos0);

    const uint16_t* kb = a.k + b * a.k_sb + kvh * a.k_sh;
    const uint16_t* vb = a.v + b * a.v_sb + kvh * a.v_sh;
    const uint8_t* mrow = nullptr;
    if constexpr (MASK != MASK_NONE)
        mrow = static_cast<const uint8_t*>(a.mask) +
               (b * a.mask_sb + (int64_t)(kvh * group + hq) * a.mask_sh + sq * a.mask_ss) * (MASK == MASK_F32 ? 4 : 1);

    // Without an fp32 mask a score's unit is the plain product q . k: its weight is
    // 2^((q . k) c - max c), c = scale log2(e), one fma and one exp2.  With one the score is the
    // logit itself (a mask of the type's lowest value would overflow in units of log2).
    constexpr bool LOGITS = MASK == MASK_F32;
    uint4 pk[KC], pv[VP][2];  // the next tile, on its way to LDS
    uint32_t next_mb[MASK == MASK_BOOL ? 4 : 1];  // and its mask at this lane's tokens 8 j + 4 h + (0..3)
    float next_add[LOGITS ? 16 : 1];
    auto load_tile = [&](int64_t t0) {
        const int left = (int)std::min<int64_t>(a.tokens - t0, TK);
        if constexpr (MASK == MASK_BOOL) {
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                const int tok = 8 * j + 4 * h;
                const uint8_t* p = mrow + t0 + tok;
                next_mb[j] = 0u;
                if (tok + 3 < left) {
                    __builtin_memcpy(&next_mb[j], p, 4);
                } else {
#pragma unroll
                    for (int e = 0; e < 4; ++e)
                        if (tok + e < left) next_mb[j] |= (uint32_t)p[e] << (8 * e);
                }
            }
        } else if constexpr (LOGITS) {
#pragma unroll
            for (int i = 0; i < 16; ++i) {
                const int tok = 8 * (i >> 2) + 4 * h + (i & 3);
                next_add[i] = tok < left ? reinterpret_cast<const float*>(mrow)[t0 + tok] : 0.0f;
            }
        }
        const uint16_t* k0 = kb + t0 * a.k_st;
        const uint16_t* v0 = vb + t0 * a.v_st;
#pragma unroll
        for (int i = 0; i < KC; ++i) {
            const int id = threadIdx.x + i * T, tok = id >> 4, c = id & 15;
            pk[i] = make_uint4(0u, 0u, 0u, 0u);
            if (tok < left) pk[i] = *reinterpret_cast<const uint4*>(k0 + tok * a.k_st + 8 * c);
        }
#pragma unroll
        for (int i = 0; i < VP; ++i) {
            const int id = threadIdx.x + i * T, tok = 2 * (id >> 4), c = id & 15;
#pragma unroll
            for (int e = 0; e < 2; ++e) {
                pv[i][e] = make_uint4(0u, 0u, 0u, 0u);
                if (tok + e < left) pv[i][e] = *reinterpret_cast<const uint4*>(v0 + (tok + e) * a.v_st + 8 * c);
            }
        }
    };
    auto store_tile = [&]() {
#pragma unroll
        for (int i = 0; i < KC; ++i) {
            const int id = threadIdx.x + i * T, tok = id >> 4, c = id & 15;
            s_k[tok * 16 + (c ^ (tok & 15))] = pk[i];
        }
#pragma unroll
        for (int i = 0; i < VP; ++i) {
            const int id = threadIdx.x + i * T, tok = 2 * (id >> 4), c = id & 15;
            // token tau of a 16-token block sits at k-slot 8 ((tau >> 2) & 1) + (tau & 3) + 4 (tau >> 3)
            const int chunk = 2 * (tok >> 4) + ((tok >> 2) & 1), pair = ((tok & 3) >> 1) + 2 * ((tok >> 3) & 1);
            const uint32_t x[4] = {pv[i][0].x, pv[i][0].y, pv[i][0].z, pv[i][0].w};
            const uint32_t y[4] = {pv[i][1].x, pv[i][1].y, pv[i][1].z, pv[i][1].w};
#pragma unroll
            for (int e = 0; e < 8; ++e) {
                const int dim = 8 * c + e;
                const uint32_t w = (e & 1) ? __builtin_amdgcn_perm(y[e >> 1], x[e >> 1], 0x07060302u)
                                           : __builtin_amdgcn_perm(y[e >> 1], x[e >> 1], 0x05040100u);
                s_v[dim * (TK / 2) + ((chunk ^ v_swizzle(dim)) << 2) + pair] = w;
            }
        }
    };

    // four waves hold the next tile's 6 KB of registers while they compute; with one or two waves
    // a thread's share would not fit beside the accumulators, and the tile is loaded when needed
    constexpr bool AHEAD = W == 4;
    const float c2 = a.scale * LOG2E;
    f32x16 o[4];
    float top, sum;  // running maximum in the scores' unit, sum of the weights
    auto walk = [&](auto careful) {
        float m = -__builtin_inff();  // of the logits
        sum = 0.0f;
#pragma unroll
        for (int d = 0; d < 4; ++d)
#pragma unroll
            for (int i = 0; i < 16; ++i) o[d][i] = 0.0f;
        if (a.accumulate && live) {
            const float2 ms = a.part_ms[slot];
            m = ms.x;
            sum = h == 0 ? ms.y : 0.0f;
#pragma unroll
            for (int d = 0; d < 4; ++d)
#pragma unroll
                for (int j = 0; j < 4; ++j) {
                    const float4 w = *reinterpret_cast<const float4*>(a.part_o + slot * D + 32 * d + 8 * j + 4 * h);
                    o[d][4 * j] = w.x, o[d][4 * j + 1] = w.y, o[d][4 * j + 2] = w.z, o[d][4 * j + 3] = w.w;
                }
        }
        top = LOGITS ? m : m / a.scale;
        if (AHEAD && t_begin < t_end) load_tile(t_begin);
        for (int64_t t0 = t_begin; t0 < t_end; t0 += TK) {
            if (t0 != t_begin) __syncthreads();  // every wave is done with the previous tile
            if (!AHEAD) load_tile(t0);
            store_tile();
            __syncthreads();

            // the tile's mask, before the next one's takes its place
            uint32_t mb[MASK == MASK_BOOL ? 4 : 1];
            float add[LOGITS ? 16 : 1];
            if constexpr (MASK == MASK_BOOL) {
#pragma unroll
                for (int j = 0; j < 4; ++j) mb[j] = next_mb[j];
            } else if constexpr (LOGITS) {
#pragma unroll
                for (int i = 0; i < 16; ++i) add[i] = next_add[i];
            }
            if (AHEAD && t0 + TK < t_end) load_tile(t0 + TK);

            // ---- scores
            f32x16 s;
#pragma unroll
            for (int i = 0; i < 16; ++i) s[i] = 0.0f;
#pragma unroll
            for (int ks = 0; ks < 8; ++ks) {
                Frag kf;
                kf.q = s_k[r * 16 + ((2 * ks + h) ^ (r & 15))];
                if constexpr (careful && QT > 1) {
                    Frag inf;
#pragma unroll
                    for (int k = 0; k < 4; ++k) {
                        inf.u[k] = kf.u[k] & special_mask(kf.u[k]);
                        kf.u[k] ^= inf.u[k];
                    }
                    // none: an infinite query element would make NaN of the zeros
                    if (__any((inf.u[0] | inf.u[1] | inf.u[2] | inf.u[3]) != 0u)) s = mfma_32(inf, q[0][ks], s);
                }
#pragma unroll
                for (int t = QT - 1; t >= 0; --t) s = mfma_32(kf, q[t][ks], s);
            }
            if constexpr (LOGITS) {
#pragma unroll
                for (int i = 0; i < 16; ++i) s[i] = s[i] * a.scale + add[i];
            }
            if constexpr (MASK == MASK_BOOL) {  // most tiles of a causal mask are attended whole
                const uint32_t all = mb[0] & mb[1] & mb[2] & mb[3];
                if (__any(all != 0x01010101u)) {
#pragma unroll
                    for (int i = 0; i < 16; ++i)
                        if (!((mb[i >> 2] >> (8 * (i & 3))) & 0xFFu)) s[i] = -__builtin_inff();
                }
            }
            if (t0 < lo || t0 + TK > hi) {  // uniform: some position is not attended
                const int lo_t = (int)std::min<int64_t>(std::max<int64_t>(lo - t0, 0), TK);
                const int hi_t = (int)std::min<int64_t>(std::max<int64_t>(hi - t0, 0), TK);
#pragma unroll
                for (int i = 0; i < 16; ++i) {
                    const int tok = 8 * (i >> 2) + 4 * h + (i & 3);
                    if (tok < lo_t || tok >= hi_t) s[i] = -__builtin_inff();
                }
            }
            float mx = top;
#pragma unroll
            for (int i = 0; i < 16; ++i) mx = fmaxf(mx, s[i]);
            mx = fmaxf(mx, __shfl_xor(mx, 32));
            const float safe = mx == -__builtin_inff() ? 0.0f : mx;  // nothing attended so far
            if (__any(mx > top)) {
                const float corr = LOGITS ? exp2_((top - safe) * LOG2E) : exp2_(__builtin_fmaf(top, c2, -safe * c2));
                sum *= corr;
#pragma unroll
                for (int d = 0; d < 4; ++d)
#pragma unroll
                    for (int i = 0; i < 16; ++i) o[d][i] *= corr;
            }
            top = mx;
            const float base = safe * c2;
#pragma unroll
            for (int i = 0; i < 16; ++i) {
                s[i] = LOGITS ? exp2_((s[i] - safe) * LOG2E) : exp2_(__builtin_fmaf(s[i], c2, -base));
                sum += s[i];
            }
            if constexpr (careful) {
#pragma unroll
                for (int kb16 = 0; kb16 < TK / 16; ++kb16) {
                    Frag p;
#pragma unroll
                    for (int k = 0; k < 4; ++k) p.u[k] = high_halves(s[8 * kb16 + 2 * k], s[8 * kb16 + 2 * k + 1]);
#pragma unroll
                    for (int d = 0; d < 4; ++d) {
                        const int dim = 32 * d + r;
                        Frag vf;
                        vf.q = reinterpret_cast<const uint4*>(s_v)[dim * (TK / 8) + ((2 * kb16 + h) ^ v_swizzle(dim))];
#pragma unroll
                        for (int k = 0; k < 4; ++k) vf.u[k] &= special_mask(vf.u[k]);
                        o[d] = mfma_32(vf, p, o[d]);
                    }
                }
                __syncthreads();
#pragma unroll 1
                for (int i = threadIdx.x; i < D * TK / 2; i += T) s_v[i] &= ~special_mask(s_v[i]);
                __syncthreads();
            }
            // ---- values: 16 tokens per step
#pragma unroll
            for (int kb16 = 0; kb16 < TK / 16; ++kb16) {
                Frag p[3];
#pragma unroll
                for (int k = 0; k < 4; ++k) {
                    float p0 = s[8 * kb16 + 2 * k], p1 = s[8 * kb16 + 2 * k + 1];
                    p[0].u[k] = high_halves(p0, p1);
                    p0 = drop_high(p0), p1 = drop_high(p1);
                    p[1].u[k] = high_halves(p0, p1);
                    p[2].u[k] = high_halves(drop_high(p0), drop_high(p1));
                }
#pragma unroll
                for (int d = 0; d < 4; ++d) {
                    Frag vf;
                    const int dim = 32 * d + r;
                    vf.q = reinterpret_cast<const uint4*>(s_v)[dim * (TK / 8) + ((2 * kb16 + h) ^ v_swizzle(dim))];
#pragma unroll
                    for (int t = 2; t >= 0; --t) o[d] = mfma_32(vf, p[t], o[d]);
                }
            }
        }
    };
    walk(std::false_type{});
    uint32_t largest = 0u;
#pragma unroll
    for (int d = 0; d < 4; ++d)
#pragma unroll
        for (int i = 0; i < 16; ++i) largest = max(largest, __float_as_uint(o[d][i]) & 0x7FFFFFFFu);
    if (__syncthreads_or(largest >= 0x7F800000u)) walk(std::true_type{});
    sum += __shfl_xor(sum, 32);
    if (!live) return;
    if (h == 0) a.part_ms[slot] = make_float2(LOGITS ? top : top * a.scale, sum);
#pragma unroll
    for (int d = 0; d < 4; ++d)
#pragma unroll
        for (int j = 0; j < 4; ++j)
            *reinterpret_cast<float4*>(a.part_o + slot * D + 32 * d + 8 * j + 4 * h) =
                make_float4(o[d][4 * j], o[d][4 * j + 1], o[d][4 * j + 2], o[d][4 * j + 3]);
}

// The slots' partials of a row (and a normalised part with its log-sum-exp, when given) weighted by
// their maxima; a row with nothing attended is 0.  Latency-bound (a row is n_split * 512 bytes that
// no other row shares), so a row's slots go round over GROUPS groups of 32 lanes, 4 dims a lane, with
// several loads in flight each: 48 slots of 128 rows 14 -> 5 us against one wave walking them in turn.
// With few slots a workgroup takes several rows instead.
template <int GROUPS>
__global__ __launch_bounds__(256) void dense_merge_kernel(const float* __restrict__ part_o,
                                                          const float2* __restrict__ part_ms, int n_split,
                                                          int64_t rows, const float* __restrict__ prev,
                                                          const float* __restrict__ prev_lse,
                                                          float* __restrict__ out_f32, uint16_t* __restrict__ out_bf16) {
    constexpr int ROWS = 8 / GROUPS;  // rows per workgroup
    __shared__ float4 s_o[8][32];
    __shared__ float s_w[4][MAX_SPLIT];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int l = threadIdx.x & 31, grp = threadIdx.x >> 5;
    const int rl = grp / GROUPS, part = grp % GROUPS;  // row of the workgroup, slots part, part + GROUPS, ...
    const int64_t row = (int64_t)blockIdx.x * ROWS + rl;
    const bool live = row < rows;
    // every wave weighs its row's slots, one lane each (GROUPS >= 2: a wave's lanes share a row)
    float2 ms = make_float2(-__builtin_inff(), 0.0f);
    if (live && lane < n_split) ms = part_ms[(int64_t)lane * rows + row];
    float top = ms.x;
#pragma unroll
    for (int k = 1; k < 64; k <<= 1) top = fmaxf(top, __shfl_xor(top, k));
    float pl = -__builtin_inff();
    if (live && prev) {
        pl = prev_lse[row];
        top = fmaxf(top, pl);
    }
    const float safe = top == -__builtin_inff() ? 0.0f : top;
    const float w = exp2_((ms.x - safe) * LOG2E);
    float den = w * ms.y;
#pragma unroll
    for (int k = 1; k < 64; k <<= 1) den += __shfl_xor(den, k);
    s_w[wave][lane] = w;
    __syncthreads();
    float4 o = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
    if (live) {
#pragma unroll 4
        for (int i = part; i < n_split; i += GROUPS) {
            const float wi = s_w[wave][i];
            const float4 p = reinterpret_cast<const float4*>(part_o + ((int64_t)i * rows + row) * D)[l];
            o.x = __builtin_fmaf(wi, p.x, o.x);
            o.y = __builtin_fmaf(wi, p.y, o.y);
            o.z = __builtin_fmaf(wi, p.z, o.z);
            o.w = __builtin_fmaf(wi, p.w, o.w);
        }
    }
    s_o[grp][l] = o;
    __syncthreads();
    if (part != 0 || !live) return;
#pragma unroll
    for (int g = 1; g < GROUPS; ++g) {
        const float4 p = s_o[grp + g][l];
        o.x += p.x, o.y += p.y, o.z += p.z, o.w += p.w;
    }
    if (prev) {
        const float wp = exp2_((pl - safe) * LOG2E);
        const float4 p = reinterpret_cast<const float4*>(prev + row * D)[l];
        o.x = __builtin_fmaf(wp, p.x, o.x);
        o.y = __builtin_fmaf(wp, p.y, o.y);
        o.z = __builtin_fmaf(wp, p.z, o.z);
        o.w = __builtin_fmaf(wp, p.w, o.w);
        den += wp;
    }
    den = den < 1e-30f ? 1e-30f : den;
    o.x /= den, o.y /= den, o.z /= den, o.w /= den;
    if (out_f32) reinterpret_cast<float4*>(out_f32 + row * D)[l] = o;
    if (out_bf16)
        reinterpret_cast<uint2*>(out_bf16 + row * D)[l] =
            make_uint2(tq::f32_to_bf16(o.x) | (tq::f32_to_bf16(o.y) << 16),
                       tq::f32_to_bf16(o.z) | (tq::f32_to_bf16(o.w) << 16));
}

bool aligned16(const void* p) { return (reinterpret_cast<uintptr_t>(p) & 15u) == 0; }

template <int W, int QT>
void launch_mask(const DenseArgs& a, int mask_type, dim3 grid, hipStream_t s) {
    if (mask_type == MASK_BOOL)
        hipLaunchKernelGGL((dense_attn_kernel<W, QT, MASK_BOOL>), grid, dim3(64 * W), 0, s, a);
    else if (mask_type == MASK_F32)
        hipLaunchKernelGGL((dense_attn_kernel<W, QT, MASK_F32>), grid, dim3(64 * W), 0, s, a);
    else
        hipLaunchKernelGGL((dense_attn_kernel<W, QT, MASK_NONE>), grid, dim3(64 * W), 0, s, a);
}

}  // namespace

extern "C" int tq_dense_attention(const void* q, int q_is_f32, int batch, int q_heads, int kv_heads, int q_len, int dim,
                                  int64_t q_sb, int64_t q_sh, int64_t q_ss, const uint16_t* k, const uint16_t* v,
                                  int64_t tokens, int64_t k_sb, int64_t k_sh, int64_t k_st, int64_t v_sb, int64_t v_sh,
                                  int64_t v_st, const void* mask, int mask_type, int64_t mask_sb, int64_t mask_sh,
                                  int64_t mask_ss, const int32_t* seq_starts, const int32_t* seq_ends, int64_t pos0,
                                  float scale, float* partials, int slots, int first_slot, int n_split, int accumulate,
                                  const float* prev, const float* prev_lse, float* out_f32, uint16_t* out_bf16,
                                  void* stream) {
    if (!q || !partials || batch < 1 || q_heads < 1 || kv_heads < 1 || q_len < 1 || tokens < 0 || q_heads % kv_heads ||
        slots < 1 || slots > MAX_SPLIT || n_split < 1 || first_slot < 0 || first_slot + n_split > slots ||
        mask_type < MASK_NONE || mask_type > MASK_F32 || (mask_type != MASK_NONE && !mask) || !(scale > 0.0f) ||
        (tokens > 0 && (!k || !v)) || (prev && !prev_lse))
        return TQ_ERR_INVALID_ARGUMENT;
    if (dim != D) return TQ_ERR_UNSUPPORTED;
    const int64_t qa = q_is_f32 ? 4 : 8;
    if (!aligned16(q) || q_sb % qa || q_sh % qa || q_ss % qa || !aligned16(k) || !aligned16(v) || k_sb % 8 || k_sh % 8 ||
        k_st % 8 || v_sb % 8 || v_sh % 8 || v_st % 8 || !aligned16(partials) ||
        (mask_type == MASK_F32 && (reinterpret_cast<uintptr_t>(mask) & 3u)))
        return TQ_ERR_UNSUPPORTED;
    const int64_t rows_per_head = (int64_t)(q_heads / kv_heads) * q_len;
    const int64_t heads = (int64_t)batch * kv_heads, rows = heads * rows_per_head;
    const int w = rows_per_head <= 32 ? 1 : rows_per_head <= 64 ? 2 : 4;
    const int64_t row_blocks = (rows_per_head + 32 * w - 1) / (32 * w);
    // the merge's launch of 256 threads to a row, or to four rows, holds fewer than 2^32
    const int64_t merge_blocks = slots > 8 ? rows : (rows + 3) / 4;
    if (heads > 65535 || row_blocks > 65535 || rows_per_head >= ((int64_t)1 << 31) - 128 ||
        merge_blocks >= (int64_t)1 << 24)
        return TQ_ERR_UNSUPPORTED;
    float* const part_o = partials + (int64_t)first_slot * rows * D;
    float2* const all_ms = reinterpret_cast<float2*>(partials + (int64_t)slots * rows * D);
    DenseArgs a{q, q_heads, kv_heads, q_len, q_sb, q_sh, q_ss, k, v, tokens, k_sb, k_sh, k_st, v_sb, v_sh, v_st,
                mask, mask_sb, mask_sh, mask_ss, seq_starts, seq_ends, pos0, scale, accumulate != 0,
                rows, part_o, all_ms + first_slot * rows};
    const dim3 grid((unsigned)n_split, (unsigned)row_blocks, (unsigned)heads);
    hipStream_t s = static_cast<hipStream_t>(stream);
    // few rows: one wave per workgroup, as many independent waves as there are splits; many rows:
    // the tile is staged once for four waves
    if (w == 1) {
        if (q_is_f32) launch_mask<1, 3>(a, mask_type, grid, s);
        else launch_mask<1, 1>(a, mask_type, grid, s);
    } else if (w == 2) {
        if (q_is_f32) launch_mask<2, 3>(a, mask_type, grid, s);
        else launch_mask<2, 1>(a, mask_type, grid, s);
    } else {
        if (q_is_f32) launch_mask<4, 3>(a, mask_type, grid, s);
        else launch_mask<4, 1>(a, mask_type, grid, s);
    }
    TQ_CHECK_LAUNCH();
    if (out_f32 || out_bf16) {
        if (slots > 8)
            hipLaunchKernelGGL(dense_merge_kernel<8>, dim3((unsigned)merge_blocks), dim3(256), 0, s, partials, all_ms, slots, rows,
                               prev, prev_lse, out_f32, out_bf16);
        else
            hipLaunchKernelGGL(dense_merge_kernel<2>, dim3((unsigned)merge_blocks), dim3(256), 0, s, partials, all_ms,
                               slots, rows, prev, prev_lse, out_f32, out_bf16);
        TQ_CHECK_LAUNCH();
    }
    return TQ_OK;
}
