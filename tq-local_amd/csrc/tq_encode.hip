// tq_encode.hip -- prefill encoders for gfx950: the fp32 encoder's bits from bf16 matrix products.
//
// The encoder's results are fixed by its fp32 evaluation order (tq_quantize.hip): a code is the
// bucket of an fma chain over 128 dims, a sign the sign of one.  Running those chains costs 32
// v_mfma_f32_16x16x4_f32 (1024 cycles) per 16 x 16 outputs, at the fp32 rate, and nothing else can
// use the SIMD meanwhile.  But a bucket only needs its chain when the value is close to a boundary.
// So the products run on the bf16 matrix cores (2 x 4 instructions of 16 cycles; the bf16 input is
// exact, the matrix enters as two bf16 terms), the value z' comes with a bound eps on its distance
// from the chain's z, and
//   |z' - b| >= eps for the one boundary b in reach:  the bucket of z' is the bucket of z;
//   otherwise (one output in 800 at 4 bits, in 1600 at 3): the chain itself is run for that output.
// The results are the chain's, bit for bit; only which outputs need it is decided by bounds.
//
// The bound, for rows of norm <= r and a vector of norm n (u = x / n has norm 1 up to 2^-20):
//   the chain: 128 roundings, each at most 2^-24 of a partial sum, which Cauchy-Schwarz keeps
//     below r: 7.63e-6 r, and u's own rounding 2^-24 r;
//   the matrix's terms (nearest even) leave 2^-18 of each entry: 3.8e-6 r;
//   z': the matrix instruction sums groups of 8 products aligned to the group's largest at 2^-24
//     of it, and rounds after each group (probed: products below that are cut off, the sum of a
//     group meets the accumulator with one rounding).  Over the groups of the leading term that is
//     7 * 2^-24 r + 16 * 2^-24 r, over the others less than 2^-7 of it: 1.4e-6 r, taken as 1.6e-6 r;
//   1 / n: the sum of squares is within 4e-6 of the exact one here and 7.7e-6 in the chain, half of
//     which (and 3e-7 of square root and reciprocal) scales z', and |z| is at most the largest
//     boundary's magnitude B where it matters: 6.3e-6 B;
//   the table's boundaries, whose low bits hold a code: 2^bits * 2^-23 B.
// r is measured when the matrix is staged; a matrix or vector outside the range where these
// hold (not finite, squares that under- or overflow, r below 1e-15: with n >= 1e-12 a second term or a
// product that is lost below 2^-126 is still 1e-3 of the slack left in 1.33e-5 r) takes the chain for
// every output, a zero vector too (0 x inf).  The fp16
// norm is handled alike: where the bound straddles a rounding boundary of fp16, the chain decides.
//
// Outputs that need their chain wait in a per-wave queue in LDS, their row of codes with them, and
// are run 64 at a time, one lane each, so that the chains' latency is shared.

#include <algorithm>
#include <atomic>

#include "tq_encode.h"

namespace {

using namespace tqmx;
using tqenc::EncodeArgs;
constexpr int D = TQ_DIM;
// Waves per workgroup of the codes kernel: 168 registers each, of which the variants of two tiles per wave
// spill 16-32 bytes a lane (channel groups up to 172).  16 waves spill more: 415 us against 300 at 2M vectors.
constexpr int CW = 12;
constexpr int CT = 64 * CW;
constexpr uint32_t NORM_ONLY = 255;

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
union Frag {
    uint32_t u[4];
    uint4 q;
    u32x4 w;
    bf16x8 b;
};
__device__ __forceinline__ f32x4 mfma_bf16(const Frag& a, const Frag& b, f32x4 c) {
    return __builtin_amdgcn_mfma_f32_16x16x32_bf16(a.b, b.b, c, 0, 0, 0);
}
// a.lo b.lo + a.hi b.hi + c over bf16 pairs; within 3 * 2^-24 of the sum (positive terms; probed).
__device__ __forceinline__ float dot2_bf16(uint32_t a, uint32_t b, float c) {
    typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
    return __builtin_amdgcn_fdot2_f32_bf16(__builtin_bit_cast(bf16x2, a), __builtin_bit_cast(bf16x2, b), c, false);
}

// The wave's LDS accesses complete in issue order; this keeps the compiler from moving them.
__device__ __forceinline__ void wave_lds_fence() {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// Largest row norm squared of an LDS-staged matrix: 16 neighbouring threads hold a row's partial
// sums of squares.  Norms compare as their bits; a NaN compares above every number.
__device__ __forceinline__ void row_norm_max(uint32_t* s_max, float part) {
#pragma unroll
    for (int k = 1; k < 16; k <<= 1) part += __shfl_xor(part, k);
    if ((threadIdx.x & 15) == 0) atomicMax(s_max, __float_as_uint(part));
}

// Folds a 64-lane predicate (lane 16 g + v) to one bit per vector v.
__device__ __forceinline__ uint32_t fold_vectors(uint64_t b) {
    const uint32_t h = (uint32_t)b | (uint32_t)(b >> 32);
    return (h | (h >> 16)) & 0xFFFFu;
}

__device__ __forceinline__ const uint16_t* row_of(const EncodeArgs& a, uint32_t vi, int64_t* slot) {
    const uint32_t gh = fdiv(vi, a.tok_div), t = vi - gh * (uint32_t)a.tokens;
    const uint32_t b = fdiv(gh, a.head_div), h = gh - b * (uint32_t)a.heads;
    *slot = (int64_t)gh * a.out_cap + a.out_offset + t;
    return a.x + (int64_t)b * a.x_sb + (int64_t)h * a.x_sh + (int64_t)t * a.x_st;
}

// Bits 16 (2 k), 16 (2 k + 1) of a group's channel mask as halves of a word: channels 2k, 2k + 1.
__device__ __forceinline__ uint32_t pair_mask(uint32_t m, int k) {
    return (((m >> (2 * k)) & 1u) ? 0x0000FFFFu : 0u) | (((m >> (2 * k + 1)) & 1u) ? 0xFFFF0000u : 0u);
}

// #{i : b_i < z} by binary search over the boundaries in LDS (the encoders' search).
__device__ __forceinline__ uint32_t bucket_lds(float z, const float* s_b, int bits) {
    uint32_t c = 0;
#pragma unroll 1
    for (uint32_t s = 1u << (bits - 1); s > 0; s >>= 1) c += (s_b[c + s - 1] < z) ? s : 0u;
    return c;
}

// ------------------------------------------------------------------ codes and norms
// Bucketize through a uniform grid.  Cells of width w = (smallest gap between neighbouring
// boundaries) / 4 start at e0 = b_0 - 2w; cell k holds c0 = #{i : b_i < e0 + (k - 1) w} and b_{c0}.
// z' goes to the cell k = clamp(floor(q)), q the quotient (z' - e0) / w, computed within 1/8 (rounded
// to quarters) + 1e-3 (|e0| / w and |b_NB-1| / w stay below 4096); z' is within w / 16 of z (eps < w / 16
// or the grid is not used).  So z lies in (e0 + (k - 0.2) w, e0 + (k + 1.2) w): every b_i below
// e0 + (k - 1) w is below z, b_{c0 + 1} >= b_{c0} + 4w is above it, and b_{c0} decides:
// code(z) = c0 + [b_{c0} < z].  The clamped ends: the first cell is 2w below b_0, the last more than w
// above b_NB-1, where b is a number above all z.  A cell is one word, the boundary with its low
// `bits` bits replaced by c0.
template <int BITS, bool GROUP, int NT>
__global__ __launch_bounds__(CT) void codes_kernel(EncodeArgs a) {
    constexpr int NB = (1 << BITS) - 1;
    constexpr int RW = 4 * BITS;  // dwords of a plain row; a queued row holds 32 codes per lane, BITS words
    constexpr uint32_t CMASK = NB;
    constexpr int LUT_MAX = BITS <= 6 ? 512 : 2048;  // cells of the bucketize grid
    // a wave's queue: vectors waiting, and single outputs; the next item may bring 16 NT and 64
    constexpr int QROWS = BITS <= 4 ? 96 : BITS <= 6 ? 64 : 48;
    constexpr int QPAIRS = 128;
    __shared__ struct {
        float lut[LUT_MAX];  // first, in reach of a read's immediate offset
        float bound[NB];
        uint32_t r_max;
        uint32_t row[CW][QROWS][RW];
        uint32_t vec[CW][QROWS];
        uint32_t pair[CW][QPAIRS];
        uint32_t all[CW][QROWS];
        uint4 img[8 * 4 * 2 * 64];  // [row tile][k-step][term][lane]
    } sh;

    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int v = lane & 15, g = lane >> 4;
    const int sub_dim = GROUP ? a.sub_dim : D;
    if (threadIdx.x == 0) sh.r_max = 0u;
    for (int i = threadIdx.x; i < NB; i += CT) sh.bound[i] = a.boundaries[i];
    __syncthreads();
    // ---- the matrix as two bf16 terms: index j = 32 q + 4 t + i is row 4 q + i of tile t, so that
    // lane 16 q + v ends with the codes [32 q, 32 q + 32) of its vector
    for (int idx = threadIdx.x; idx < D * D / 8; idx += CT) {
        const int j = idx >> 4, c = idx & 15;  // dims 8 c .. 8 c + 7
        float e[8];
        if (!GROUP || j < sub_dim) {
            const float4 p = reinterpret_cast<const float4*>(a.R)[j * (D / 4) + 2 * c];
            const float4 q = reinterpret_cast<const float4*>(a.R)[j * (D / 4) + 2 * c + 1];
            e[0] = p.x, e[1] = p.y, e[2] = p.z, e[3] = p.w, e[4] = q.x, e[5] = q.y, e[6] = q.z, e[7] = q.w;
        } else {
#pragma unroll
            for (int k = 0; k < 8; ++k) e[k] = 0.0f;
        }
        float part = 0.0f;
#pragma unroll
        for (int k = 0; k < 8; ++k) part = __builtin_fmaf(e[k], e[k], part);
        row_norm_max(&sh.r_max, part);
        const int t = (j >> 2) & 7, m = 4 * (j >> 5) + (j & 3), s = c >> 2, l = 16 * (c & 3) + m;
        uint32_t hi[4], lo[4];
#pragma unroll
        for (int k = 0; k < 4; ++k) {
            hi[k] = bf16_pair(e[2 * k], e[2 * k + 1]);
            lo[k] = bf16_pair(e[2 * k] - lo_half(hi[k]), e[2 * k + 1] - hi_half(hi[k]));
        }
        sh.img[((t * 4 + s) * 2 + 0) * 64 + l] = make_uint4(hi[0], hi[1], hi[2], hi[3]);
        sh.img[((t * 4 + s) * 2 + 1) * 64 + l] = make_uint4(lo[0], lo[1], lo[2], lo[3]);
    }
    // ---- bucket grid: one lane per gap between boundaries
    float gap = __builtin_inff(), b_max = 0.0f;
    bool sorted = true;
    for (int i = lane; i < NB; i += 64) {
        b_max = fmaxf(b_max, fabsf(sh.bound[i]));
        if (i > 0) {
            const float d = sh.bound[i] - sh.bound[i - 1];
            sorted = sorted && d > 0.0f;
            gap = fminf(gap, d);
        }
    }
    sorted = __all(sorted);
#pragma unroll
    for (int k = 1; k < 64; k <<= 1) {
        gap = fminf(gap, __shfl_xor(gap, k));
        b_max = fmaxf(b_max, __shfl_xor(b_max, k));
    }
    __syncthreads();
    const float r_norm = __builtin_sqrtf(__uint_as_float(sh.r_max)) * 1.0001f;
    const float eps = r_norm * 1.33e-5f + (b_max + 1e-4f * r_norm) * (6.5e-6f + (float)(1 << BITS) * 1.2e-7f);
    const float w = NB > 1 ? gap * 0.25f : 1.0f;
    const float e0 = sh.bound[0] - 2.0f * w;
    const float span = (sh.bound[NB - 1] - e0) / w;
    const float g_scale = 1.0f / w;
    const float g_off = -e0 * g_scale;
    // outside the bounds' range every output takes its chain
    const bool exact_all = !(r_norm < 1e18f) || !(r_norm > 1e-15f) || !(b_max < 1e18f);
    const bool use_grid = sorted && w > 16.0f * eps && span < (float)(LUT_MAX - 5) && fabsf(g_off) < 4096.0f &&
                          fabsf(sh.bound[NB - 1] * g_scale) < 4096.0f;
    const int cells = use_grid ? (int)ceilf(span) + 4 : 0;
    for (int k = threadIdx.x; k < cells; k += CT) {
        const float start = e0 + (float)(k - 1) * w;
        uint32_t c0 = 0;
        for (int i = 0; i < NB; ++i) c0 += sh.bound[i] < start ? 1u : 0u;
        const float b = c0 < NB ? sh.bound[c0] + 0.0f : 3e38f;
        sh.lut[k] = __uint_as_float((__float_as_uint(b) & ~CMASK) | c0);
    }
    __syncthreads();  // the last barrier: each wave then works on its own tiles

    // f = 4 * quotient + 2^23: one fma and one med3, and the low bits of f are the quotient's, in
    // quarters of a cell: without the last two, the byte offset of its word
    constexpr float MAGIC = 8388608.0f;
    const float q_scale = 4.0f * g_scale;
    const float f_off = 4.0f * g_off + MAGIC;
    const float f_top = MAGIC + (float)(4 * cells - 1);
    const float s_b0 = sh.bound[0];
    const uint32_t mw[4] = {a.mask[0], a.mask[1], a.mask[2], a.mask[3]};
    const int row_bytes = GROUP ? (sub_dim * BITS + 7) >> 3 : D * BITS / 8;
    // this lane's outputs 32 g + jj with jj < mine count
    const int mine = GROUP ? std::min(std::max(sub_dim - 32 * g, 0), 32) : 32;
    const int n_t = a.sub_dim < 32 ? (a.sub_dim + 3) >> 2 : 8;

    // this lane's fragments, all in reach of a read's immediate offset
    typedef __attribute__((address_space(3))) const u32x4* LdsFrags;
    LdsFrags img = (LdsFrags)(sh.img + lane);
    __asm__("" : "+v"(img));

    uint32_t q_rows = 0, q_pairs = 0, q_all = 0;  // wave-uniform
    auto store_row = [&](uint8_t* codes, const uint32_t* words) {  // this lane's BITS words of a row
        if constexpr (!GROUP) {
            uint32_t* dst = reinterpret_cast<uint32_t*>(codes) + BITS * g;
            if constexpr (BITS == 4) *reinterpret_cast<uint4*>(dst) = make_uint4(words[0], words[1], words[2], words[3]);
            else if constexpr (BITS == 2) *reinterpret_cast<uint2*>(dst) = make_uint2(words[0], words[1]);
            else
#pragma unroll
                for (int k = 0; k < BITS; ++k) dst[k] = words[k];
        } else {
            const int first = 4 * BITS * g;
#pragma unroll
            for (int k = 0; k < BITS; ++k) {
                const int left = row_bytes - (first + 4 * k);
                uint8_t* dst = codes + first + 4 * k;
                if (left >= 4) {
                    __builtin_memcpy(dst, &words[k], 4);
                } else {
#pragma unroll
                    for (int e = 0; e < 3; ++e)
                        if (e < left) dst[e] = (uint8_t)(words[k] >> (8 * e));
                }
            }
        }
    };
    // The queue's chains: 64 single outputs at a time, one lane each, then the vectors whose every output
    // is wanted, half a vector at a time; then the rows leave.
    auto run_queue = [&]() {
        wave_lds_fence();
        const uint32_t singles = (q_pairs + 63) >> 6, batches = singles + 2 * q_all;
        for (uint32_t batch = 0; batch < batches; ++batch) {
            const bool whole = batch >= singles;
            uint32_t qr = 0, j = 0;
            bool act;
            if (whole) {
                qr = sh.all[wave][(batch - singles) >> 1];
                j = 64 * ((batch - singles) & 1) + lane;
                act = !GROUP || (int)j < sub_dim;
            } else {
                act = 64 * batch + lane < q_pairs;
                const uint32_t e = act ? sh.pair[wave][64 * batch + lane] : 0u;
                qr = e >> 8, j = e & 255u;
            }
            if (act) {
                int64_t slot;
                const uint4* x4 = reinterpret_cast<const uint4*>(row_of(a, sh.vec[wave][qr], &slot));
                auto channels = [&](int c, float* o) {  // channels 8 c .. 8 c + 7, masked
                    const uint4 p = x4[c];
                    const uint32_t h[4] = {p.x, p.y, p.z, p.w};
#pragma unroll
                    for (int k = 0; k < 4; ++k) {
                        uint32_t hk = h[k];
                        if constexpr (GROUP) hk &= pair_mask(a.mask[c >> 2] >> (8 * (c & 3)), k);
                        o[2 * k] = lo_half(hk);
                        o[2 * k + 1] = hi_half(hk);
                    }
                };
                float ss = 0.0f;
#pragma unroll 8
                for (int c = 0; c < D / 8; ++c) {
                    float o[8];
                    channels(c, o);
#pragma unroll
                    for (int k = 0; k < 8; ++k) ss = __builtin_fmaf(o[k], o[k], ss);
                }
                float n = tq::sqrt_rn(ss);
                if (!(n > 0.0f)) n = 1.0f;
                if (j == NORM_ONLY || (whole && j == 0)) a.norms[slot] = (uint16_t)tq::f32_to_f16(n);
                if (j != NORM_ONLY) {
                    const float4* rj = reinterpret_cast<const float4*>(a.R) + j * (D / 4);
                    float z = 0.0f;
#pragma unroll 4
                    for (int c = 0; c < D / 8; ++c) {
                        float o[8];
                        channels(c, o);
                        const float4 p = rj[2 * c], q = rj[2 * c + 1];
                        const float rr[8] = {p.x, p.y, p.z, p.w, q.x, q.y, q.z, q.w};
#pragma unroll
                        for (int k = 0; k < 8; ++k) z = __builtin_fmaf(tq::div_rn(o[k], n), rr[k], z);
                    }
                    const uint32_t code = bucket_lds(z, sh.bound, BITS);
                    uint32_t* words = sh.row[wave][qr];
                    const uint32_t bit = j * BITS, wi = bit >> 5, at = bit & 31;
                    uint64_t old = words[wi];
                    if (at + BITS > 32) old |= (uint64_t)words[wi + 1] << 32;
                    const uint64_t diff = (uint64_t)(((uint32_t)(old >> at) & CMASK) ^ code) << at;
                    // other lanes may change other codes of the same word
                    if ((uint32_t)diff) atomicXor(&words[wi], (uint32_t)diff);
                    if ((uint32_t)(diff >> 32)) atomicXor(&words[wi + 1], (uint32_t)(diff >> 32));
                }
            }
        }
        wave_lds_fence();
        for (uint32_t r0 = 0; r0 < q_rows; r0 += 16) {
            const uint32_t qr = r0 + v;
            if (qr < q_rows) {
                int64_t slot;
                row_of(a, sh.vec[wave][qr], &slot);
                uint32_t words[BITS];
#pragma unroll
                for (int k = 0; k < BITS; ++k) words[k] = sh.row[wave][qr][BITS * g + k];
                store_row(a.codes + slot * row_bytes, words);
            }
        }
        q_rows = q_pairs = q_all = 0;
        wave_lds_fence();
    };

    const int64_t n_items = (a.n_vec + 16 * NT - 1) / (16 * NT);
    // NT tiles of 16 vectors: lane 16 g + v holds dims 32 s + 8 g + (0..7) of vector v, the B operand.
    // The next item's are read ahead: a wait for them does not wait for this item's stores.
    Frag ahead[NT][4];
    int64_t ahead_slot[NT];
    auto read_ahead = [&](int64_t item) {
#pragma unroll
        for (int n = 0; n < NT; ++n) {
            const uint32_t vi = (uint32_t)item * (16u * NT) + 16u * n + (uint32_t)v;  // n_vec < 2^31
            ahead_slot[n] = -1;
#pragma unroll
            for (int s = 0; s < 4; ++s) ahead[n][s].q = make_uint4(0u, 0u, 0u, 0u);
            if (item < n_items && vi < (uint64_t)a.n_vec) {
                const uint4* x4 = reinterpret_cast<const uint4*>(row_of(a, vi, &ahead_slot[n]));
#pragma unroll
                for (int s = 0; s < 4; ++s) ahead[n][s].q = x4[4 * s + g];
            }
        }
    };
    // items go round over the workgroups first, so that a small call uses every CU
    const int64_t stride = (int64_t)gridDim.x * CW;
    int64_t item = (int64_t)wave * gridDim.x + blockIdx.x;
    // stretches of items until the queue may not take the next one's, then the queue: nothing of an
    // item is live while the queue runs
    do {
        read_ahead(item);
        for (; item < n_items && q_rows + 16 * NT <= QROWS && q_pairs + 64 <= QPAIRS; item += stride) {
        Frag x[NT][4];
        int64_t slot[NT];
        float rn[NT], rg[NT], mg[NT];
        bool live[NT];
        uint32_t n_amb = 0, special = 0;  // per tile bit: the fp16 norm, or everything, needs the chain
#pragma unroll
        for (int n = 0; n < NT; ++n) {
            slot[n] = ahead_slot[n];
            live[n] = slot[n] >= 0;
#pragma unroll
            for (int s = 0; s < 4; ++s) x[n][s] = ahead[n][s];
        }
        read_ahead(item + stride);
#pragma unroll
        for (int n = 0; n < NT; ++n) {
            float ss = 0.0f;
            uint32_t any = 0u;
#pragma unroll
            for (int s = 0; s < 4; ++s)
#pragma unroll
                for (int k = 0; k < 4; ++k) {
                    if constexpr (GROUP) x[n][s].u[k] &= pair_mask(mw[s] >> (8 * g), k);
                    const uint32_t p = x[n][s].u[k];
                    ss = dot2_bf16(p, p, ss);
                    any |= p;
                }
            ss += __shfl_xor(ss, 16);
            ss += __shfl_xor(ss, 32);
            any &= 0x7FFF7FFFu;
            any |= (uint32_t)__shfl_xor((int)any, 16);
            any |= (uint32_t)__shfl_xor((int)any, 32);
            const bool zero = any == 0u;  // norm 1, every chain 0 (where the matrix is finite)
            const float n_ = zero ? 1.0f : __builtin_sqrtf(ss);
            rn[n] = __builtin_amdgcn_rcpf(n_);
            rg[n] = rn[n] * q_scale;
            mg[n] = zero ? -1.0f : eps;
            const bool bad = exact_all || (!zero && (!(ss > 1e-24f) || !(ss < 1e30f)));
            const uint32_t h0 = tq::f32_to_f16(n_ * (1.0f - 7e-6f)), h1 = tq::f32_to_f16(n_ * (1.0f + 7e-6f));
            if (bad || (h0 != h1 && !zero)) n_amb |= 1u << n;
            if (bad) special |= 1u << n;
            if (live[n] && g == 0 && !((n_amb >> n) & 1u)) a.norms[slot[n]] = (uint16_t)tq::f32_to_f16(n_);
        }

        // ---- products, codes; bit jj of amb: output 32 g + jj needs its chain
        uint32_t out[NT][BITS], amb[NT];
#pragma unroll
        for (int n = 0; n < NT; ++n) {
            amb[n] = 0u;
#pragma unroll
            for (int k = 0; k < BITS; ++k) out[n][k] = 0u;
        }
        auto products = [&](int t, f32x4* acc) {
#pragma unroll
            for (int n = 0; n < NT; ++n) acc[n] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
            for (int term = 1; term >= 0; --term)
#pragma unroll
                for (int s = 0; s < 4; ++s) {
                    Frag m;
                    m.w = img[((t * 4 + s) * 2 + term) * 64];
#pragma unroll
                    for (int n = 0; n < NT; ++n) acc[n] = mfma_bf16(m, x[n][s], acc[n]);
                }
        };
        // the boundary in reach of a product: its low bits hold c0, the code below it
        auto boundary = [&](int n, float acc) -> float {
            if constexpr (NB == 1) {
                return s_b0;
            }
            float f = __builtin_fmaf(acc, rg[n], f_off);
            f = __builtin_amdgcn_fmed3f(f, MAGIC, f_top);
            return *reinterpret_cast<const float*>(reinterpret_cast<const char*>(sh.lut) +
                                                   (__float_as_uint(f) & (4 * LUT_MAX - 4)));
        };
        if ((NB == 1 || use_grid) && n_t == 8) {
            // Products and buckets in turn, not interleaved: matrix and vector instructions of different
            // waves overlap (61% of the shorter one with four waves on a SIMD, groups of 4 and 16),
            // those of one wave hardly do (37% in groups of 1 and 4).
            uint32_t ch[NT];  // codes enter at the top, the first ends lowest
#pragma unroll
            for (int n = 0; n < NT; ++n) ch[n] = 0u;
#pragma unroll
            for (int t = 0; t < 8; ++t) {
                f32x4 acc[NT];
                products(t, acc);
                __builtin_amdgcn_sched_barrier(0);
                float b[NT][4];
#pragma unroll
                for (int n = 0; n < NT; ++n)
#pragma unroll
                    for (int i = 0; i < 4; ++i) b[n][i] = boundary(n, acc[n][i]);
#pragma unroll
                for (int n = 0; n < NT; ++n) {
#pragma unroll
                    for (int i = 0; i < 4; ++i) {
                        const float d = __builtin_fmaf(acc[n][i], rn[n], -b[n][i]);
                        const uint32_t code = (NB > 1 ? __float_as_uint(b[n][i]) : 0u) + (d > 0.0f ? 1u : 0u);
                        ch[n] = __builtin_amdgcn_alignbit(code, ch[n], BITS);
                        amb[n] |= fabsf(d) < mg[n] ? 1u << (4 * t + i) : 0u;
                    }
                    const int bit = 4 * t * BITS, wi = bit >> 5, at = bit & 31;  // 4 codes from here on
                    if constexpr (32 % BITS == 0) {
                        if (((bit + 4 * BITS) & 31) == 0) out[n][wi] = ch[n];
                    } else {
                        const uint32_t four = ch[n] >> (32 - 4 * BITS);
                        out[n][wi] |= four << at;
                        if (at + 4 * BITS > 32) out[n][wi + 1] |= four >> (32 - at);
                    }
                }
                __builtin_amdgcn_sched_barrier(0);
            }
        } else {
#pragma unroll
            for (int t = 0; t < 8; ++t) {
                if (t >= n_t) break;
                f32x4 acc[NT];
                products(t, acc);
#pragma unroll
                for (int n = 0; n < NT; ++n)
#pragma unroll
                    for (int i = 0; i < 4; ++i) {
                        uint32_t code;
                        float d;
                        if (NB == 1 || use_grid) {
                            const float b = boundary(n, acc[n][i]);
                            d = __builtin_fmaf(acc[n][i], rn[n], -b);
                            code = ((NB > 1 ? __float_as_uint(b) : 0u) + (d > 0.0f ? 1u : 0u)) & CMASK;
                        } else {  // no grid: the distance to the closest boundary
                            const float z = acc[n][i] * rn[n];
                            d = __builtin_inff();
#pragma unroll 1
                            for (int k = 0; k < NB; ++k) d = fminf(d, fabsf(z - sh.bound[k]));
                            code = bucket_lds(z, sh.bound, BITS);
                        }
                        amb[n] |= fabsf(d) < mg[n] ? 1u << (4 * t + i) : 0u;
                        const int bit = (4 * t + i) * BITS, wi = bit >> 5, at = bit & 31;
                        out[n][wi] |= code << at;
                        if (at + BITS > 32) out[n][wi + 1] |= code >> (32 - at);
                    }
                __builtin_amdgcn_sched_barrier(0);
            }
        }

        // ---- outputs beyond the group's rows are no outputs
        if constexpr (GROUP) {
#pragma unroll
            for (int k = 0; k < BITS; ++k) {
                const int left = mine * BITS - 32 * k;
                const uint32_t keep = left >= 32 ? 0xFFFFFFFFu : left <= 0 ? 0u : (1u << left) - 1u;
#pragma unroll
                for (int n = 0; n < NT; ++n) out[n][k] &= keep;
            }
        }
        const uint32_t valid = mine >= 32 ? 0xFFFFFFFFu : (1u << mine) - 1u;

        // ---- rows without a doubtful output leave; the others queue, with those outputs or, where the
        // item has more than the queue takes, with all of theirs
        uint32_t queued[NT], mine_q = 0u;
        bool any = false;
#pragma unroll
        for (int n = 0; n < NT; ++n) {
            if ((special >> n) & 1u) amb[n] = 0xFFFFFFFFu;
            amb[n] = live[n] ? amb[n] & valid : 0u;
            if (!live[n]) n_amb &= ~(1u << n);
            const bool norm = ((n_amb >> n) & 1u) && g == 0;
            mine_q += __popc(amb[n]) + (norm ? 1u : 0u);
            const uint32_t rows = fold_vectors(__builtin_amdgcn_ballot_w64(amb[n] != 0u));
            if (live[n] && !((rows >> v) & 1u)) store_row(a.codes + slot[n] * row_bytes, out[n]);
            queued[n] = rows | fold_vectors(__builtin_amdgcn_ballot_w64((n_amb >> n) & 1u));
            any = any || queued[n] != 0u;
        }
        if (any) {
#pragma unroll
            for (int k = 1; k < 64; k <<= 1) mine_q += (uint32_t)__shfl_xor((int)mine_q, k);
            const bool whole = mine_q > 64u;
#pragma unroll
            for (int n = 0; n < NT; ++n) {
                const uint32_t below = __popc(queued[n] & ((1u << v) - 1u)), qr = q_rows + below;
                if ((queued[n] >> v) & 1u) {
                    if (g == 0) {
                        sh.vec[wave][qr] = (uint32_t)item * (16u * NT) + 16u * n + (uint32_t)v;
                        if (whole) sh.all[wave][q_all + below] = qr;
                    }
#pragma unroll
                    for (int k = 0; k < BITS; ++k) sh.row[wave][qr][BITS * g + k] = out[n][k];
                }
                q_rows += __popc(queued[n]);
                if (whole) {
                    q_all += __popc(queued[n]);
                    continue;
                }
                for (;;) {
                    const bool norm = ((n_amb >> n) & 1u) && g == 0;
                    const bool p = norm || amb[n] != 0u;
                    const uint64_t who = __builtin_amdgcn_ballot_w64(p);
                    if (who == 0) break;
                    const uint32_t at = q_pairs + __builtin_amdgcn_mbcnt_hi((uint32_t)(who >> 32),
                                                                            __builtin_amdgcn_mbcnt_lo((uint32_t)who, 0));
                    const uint32_t jj = (uint32_t)__builtin_ctz(amb[n] | 0x80000000u);  // the first doubtful output
                    if (p) sh.pair[wave][at] = (qr << 8) | (norm ? NORM_ONLY : 32u * g + jj);
                    if (!norm) amb[n] &= ~(1u << jj);
                    n_amb &= ~(1u << n);
                    q_pairs += __popcll(who);
                }
            }
        }
        }
        if (q_rows) run_queue();
    } while (item < n_items);
}

// ------------------------------------------------------------------ residual sketch of Q_prod keys
// khat_d = bf16((fma chain j of C[code_j] R[j][d]) * f32(f16(n))) must be the chain itself: its bf16
// rounding has a boundary within the bound of one value in twenty.  So this product stays on the
// fp32 matrix cores (the decoder's image, tq_mfma.h; 8192 of a tile's ~12500 cycles), and the QJL
// projection, of which only signs are kept, runs on the bf16 ones: r = x - khat as two bf16
// terms (nearest even, r within 2^-18), S as two, three products.  With |r| factored out the bound is
// s (7.63e-6 chain + 3 * 2^-18 terms + 1.6e-6 + rounding) = 2.2e-5 s, s the largest row norm of S; a
// projection inside it, one in 4000, is run as the chain, with rhat from the division the chain uses.
template <int BITS, bool GROUP>
__global__ __launch_bounds__(MQ_THREADS) void residual_kernel(EncodeArgs a) {
    constexpr int RW = 4 * BITS;
    constexpr int GRW = RW + 2;  // staged dwords of a group row: a misaligned start, one spare
    __shared__ float4 s_img[D * D / 4];       // R^T, fp32
    __shared__ uint4 s_s[8 * 4 * 2 * 64];     // S, two bf16 terms: [row tile][k-step][term][lane]
    __shared__ float s_cent[1 << BITS];
    __shared__ uint32_t s_code[GROUP ? MQ_WAVES : 1][GROUP ? 16 : 1][GRW];
    __shared__ float4 s_r[MQ_WAVES][D / 4];
    __shared__ uint32_t s_max;
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int v = lane & 15, g = lane >> 4;
    const int sub_dim = GROUP ? a.sub_dim : D;
    const int pad = D - sub_dim;
    if (threadIdx.x == 0) s_max = 0u;
    __syncthreads();
    build_image_transposed(reinterpret_cast<float*>(s_img), a.R, sub_dim);
    for (int i = threadIdx.x; i < (1 << BITS); i += MQ_THREADS) s_cent[i] = a.centers[i];
    // lane 16 g + m of k-step s: dims 32 g + 8 s + (0..7), the dims in which lane 16 g + v holds r
    for (int idx = threadIdx.x; idx < D * D / 8; idx += MQ_THREADS) {
        const int j = idx >> 4, c = idx & 15;
        float e[8];
        if (!GROUP || j < sub_dim) {
            const float4 p = reinterpret_cast<const float4*>(a.S)[j * (D / 4) + 2 * c];
            const float4 q = reinterpret_cast<const float4*>(a.S)[j * (D / 4) + 2 * c + 1];
            e[0] = p.x, e[1] = p.y, e[2] = p.z, e[3] = p.w, e[4] = q.x, e[5] = q.y, e[6] = q.z, e[7] = q.w;
        } else {
#pragma unroll
            for (int k = 0; k < 8; ++k) e[k] = 0.0f;
        }
        float part = 0.0f;
#pragma unroll
        for (int k = 0; k < 8; ++k) part = __builtin_fmaf(e[k], e[k], part);
        row_norm_max(&s_max, part);
        const int t = (j >> 2) & 7, m = 4 * (j >> 5) + (j & 3), s = c & 3, l = 16 * (c >> 2) + m;
        uint32_t hi[4], lo[4];
#pragma unroll
        for (int k = 0; k < 4; ++k) {
            hi[k] = bf16_pair(e[2 * k], e[2 * k + 1]);
            lo[k] = bf16_pair(e[2 * k] - lo_half(hi[k]), e[2 * k + 1] - hi_half(hi[k]));
        }
        s_s[((t * 4 + s) * 2 + 0) * 64 + l] = make_uint4(hi[0], hi[1], hi[2], hi[3]);
        s_s[((t * 4 + s) * 2 + 1) * 64 + l] = make_uint4(lo[0], lo[1], lo[2], lo[3]);
    }
    __syncthreads();  // the last barrier: each wave then works on its own tiles
    const float s_norm = __builtin_sqrtf(__uint_as_float(s_max)) * 1.0001f;
    const float eps = s_norm * 2.25e-5f;
    const bool exact_all = !(s_norm < 1e15f) || !(s_norm > 1e-15f);
    const float4* a_img = s_img + (lane ^ g);
    const uint32_t mw = g == 0 ? a.mask[0] : g == 1 ? a.mask[1] : g == 2 ? a.mask[2] : a.mask[3];
    const int row_bytes = GROUP ? (sub_dim * BITS + 7) >> 3 : D * BITS / 8;
    const int sign_bytes = (sub_dim + 7) >> 3;
    const int mine = std::min(std::max(sub_dim - 32 * g, 0), 32);
    const uint32_t valid = mine >= 32 ? 0xFFFFFFFFu : (1u << mine) - 1u;
    const int n_t = sub_dim < 32 ? (sub_dim + 3) >> 2 : 8;

    const int64_t n_tiles = (a.n_vec + 15) / 16;
    for (int64_t tile = (int64_t)blockIdx.x * MQ_WAVES + wave; tile < n_tiles;
         tile += (int64_t)gridDim.x * MQ_WAVES) {
        const uint32_t vi = (uint32_t)tile * 16u + (uint32_t)v;
        const bool live = vi < (uint64_t)a.n_vec;
        int64_t slot = 0;
        uint4 xr[4];
        float nf = 0.0f;
#pragma unroll
        for (int c = 0; c < 4; ++c) xr[c] = make_uint4(0u, 0u, 0u, 0u);
        if (live) {
            const uint4* x4 = reinterpret_cast<const uint4*>(row_of(a, vi, &slot));
#pragma unroll
            for (int c = 0; c < 4; ++c) xr[c] = x4[4 * g + c];
            nf = tq::f16_to_f32(a.norms[slot]);
        }
        // ---- C[code] of index 4s + g (behind `pad` zeros for a group)
        float cv[32];
        if constexpr (!GROUP) {
            uint32_t w[RW + 1];
            const uint4* c4 = reinterpret_cast<const uint4*>(a.codes + slot * row_bytes);
#pragma unroll
            for (int c = 0; c < BITS; ++c) {
                uint4 q = make_uint4(0u, 0u, 0u, 0u);
                if (live) q = c4[c];
                w[4 * c] = q.x, w[4 * c + 1] = q.y, w[4 * c + 2] = q.z, w[4 * c + 3] = q.w;
            }
            w[RW] = 0u;
            centers_of<BITS>(w, g, s_cent, cv);
        } else {
            // the row byte by byte where it does not fill a dword, so nothing outside it is read
            uint32_t* row = s_code[wave][v];
            const uint8_t* src = a.codes + slot * row_bytes;
            for (int k = g; k < GRW; k += 4) {
                uint32_t w = 0u;
                if (live) {
                    if (4 * k + 4 <= row_bytes) {
                        __builtin_memcpy(&w, src + 4 * k, 4);
                    } else {
#pragma unroll
                        for (int e = 0; e < 3; ++e)
                            if (4 * k + e < row_bytes) w |= (uint32_t)src[4 * k + e] << (8 * e);
                    }
                }
                row[k] = w;
            }
            wave_lds_fence();
#pragma unroll
            for (int s = 0; s < 32; ++s) {
                const int j = 4 * s + g - pad;
                const uint32_t bit = (uint32_t)(j * BITS);
                cv[s] = 0.0f;
                if (j >= 0)
                    cv[s] = s_cent[__builtin_amdgcn_ubfe(
                        __builtin_amdgcn_alignbit(row[(bit >> 5) + 1], row[bit >> 5], bit & 31), 0, BITS)];
            }
            wave_lds_fence();
        }
        f32x4 acc[8];
        if constexpr (!GROUP) {
            image_products(a_img, cv, acc);
        } else {
            // a group's chains start behind `pad` zero products, which leave +0 as it is: whole blocks of
            // 16 of them are skipped (a group of 4 channels runs one block of eight)
#pragma unroll
            for (int t = 0; t < 8; ++t) acc[t] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
            for (int sb = 0; sb < 8; ++sb) {
                if (16 * sb + 16 <= pad) continue;
                float4 m[8];
#pragma unroll
                for (int t = 0; t < 8; ++t) m[t] = a_img[(t * 8 + sb) * 64];
#pragma unroll
                for (int e = 0; e < 4; ++e)
#pragma unroll
                    for (int t = 0; t < 8; ++t)
                        acc[t] = mfma_f32(e == 0 ? m[t].x : e == 1 ? m[t].y : e == 2 ? m[t].z : m[t].w, cv[4 * sb + e],
                                          acc[t]);
                __builtin_amdgcn_sched_barrier(0);
            }
        }
        // ---- r = x - bf16(khat), dims 32 g + (0..31)
        float r[32];
        float rs = 0.0f;
        const uint32_t xw[16] = {xr[0].x, xr[0].y, xr[0].z, xr[0].w, xr[1].x, xr[1].y, xr[1].z, xr[1].w,
                                 xr[2].x, xr[2].y, xr[2].z, xr[2].w, xr[3].x, xr[3].y, xr[3].z, xr[3].w};
#pragma unroll
        for (int p = 0; p < 16; ++p) {
            uint32_t xp = xw[p];
            if constexpr (GROUP) xp &= pair_mask(mw, p);
            const uint32_t kh = bf16_pair(acc[p >> 1][2 * (p & 1)] * nf, acc[p >> 1][2 * (p & 1) + 1] * nf);
            r[2 * p] = lo_half(xp) - lo_half(kh);
            r[2 * p + 1] = hi_half(xp) - hi_half(kh);
            rs = __builtin_fmaf(r[2 * p], r[2 * p], rs);
            rs = __builtin_fmaf(r[2 * p + 1], r[2 * p + 1], rs);
        }
        rs += __shfl_xor(rs, 16);
        rs += __shfl_xor(rs, 32);
        const bool bad = exact_all || (rs != 0.0f && (!(rs > 1e-24f) || !(rs < 1e30f)));
        // a sum of squares of 0 can hide residuals whose squares vanish; the chain's does as well
        const float rho = rs == 0.0f ? 1.0f : __builtin_sqrtf(rs);
        const uint32_t h0 = tq::f32_to_f16(rho * (1.0f - 7e-6f)), h1 = tq::f32_to_f16(rho * (1.0f + 7e-6f));
        const bool tiny = rs == 0.0f;
        bool rho_amb = bad || (h0 != h1 && !tiny);
        Frag rh[4], rl[4];
#pragma unroll
        for (int s = 0; s < 4; ++s)
#pragma unroll
            for (int k = 0; k < 4; ++k) {
                const float e0 = r[8 * s + 2 * k], e1 = r[8 * s + 2 * k + 1];
                rh[s].u[k] = bf16_pair(e0, e1);
                rl[s].u[k] = bf16_pair(e0 - lo_half(rh[s].u[k]), e1 - hi_half(rh[s].u[k]));
            }
        // ---- projections: lane g holds signs [32 g, 32 g + 32)
        f32x4 proj[8];
        uint32_t neg = 0u;  // sign bits, the first output's highest
        float closest = __builtin_inff();
#pragma unroll
        for (int t = 0; t < 8; ++t) {
            f32x4 p = {0.0f, 0.0f, 0.0f, 0.0f};
            proj[t] = p;
            if (GROUP && t >= n_t) {  // rows past the group's
                neg <<= 4;
                continue;
            }
            Frag m;
#pragma unroll
            for (int s = 0; s < 4; ++s) {
                m.q = s_s[((t * 4 + s) * 2 + 1) * 64 + lane];
                p = mfma_bf16(m, rh[s], p);
            }
#pragma unroll
            for (int s = 0; s < 4; ++s) {
                m.q = s_s[(t * 4 + s) * 2 * 64 + lane];
                p = mfma_bf16(m, rl[s], p);
                p = mfma_bf16(m, rh[s], p);
            }
            proj[t] = p;
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                neg = __builtin_amdgcn_alignbit(neg, __float_as_uint(p[i]), 31);
                if (!GROUP || 4 * t + i < mine) closest = fminf(closest, fabsf(p[i]));
            }
        }
        uint32_t sb = ~__brev(neg), amb = 0u;
        const float mg = eps * rho;
        if (__any(closest < mg)) {
#pragma unroll
            for (int t = 0; t < 8; ++t)
#pragma unroll
                for (int i = 0; i < 4; ++i) amb |= fabsf(proj[t][i]) < mg ? 1u << (4 * t + i) : 0u;
        }
        // every r of magnitude 0: the projections are +0 in the chain too.  Otherwise, with squares that
        // vanish, the chain decides.
        if (__any(tiny)) {
            uint32_t nz = 0u;
#pragma unroll
            for (int k = 0; k < 32; ++k) nz |= __float_as_uint(r[k]);
            nz &= 0x7FFFFFFFu;
            nz |= (uint32_t)__shfl_xor((int)nz, 16);
            nz |= (uint32_t)__shfl_xor((int)nz, 32);
            if (tiny) {
                amb = nz ? 0xFFFFFFFFu : 0u;
                if (!nz) sb = 0xFFFFFFFFu;
            }
        }
        if (bad) amb = 0xFFFFFFFFu;
        amb &= valid;
        if (!live) amb = 0u, rho_amb = false;

        uint32_t rho16 = tq::f32_to_f16(rho);
        if (__any(amb != 0u || rho_amb)) {
            // the tile's sums of squares as chains: lane group p runs dims [32 p, 32 p + 32) on from group p - 1
            float ss = 0.0f;
#pragma unroll
            for (int p = 0; p < 4; ++p) {
#pragma unroll
                for (int k = 0; k < 32; ++k) ss = __builtin_fmaf(r[k], r[k], ss);
                ss = __shfl(ss, 16 * p + v);
            }
            float rx = tq::sqrt_rn(ss);
            if (!(rx > 0.0f)) rx = 1.0f;
            rho16 = tq::f32_to_f16(rx);
            uint32_t todo = fold_vectors(__builtin_amdgcn_ballot_w64(amb != 0u));
            while (todo) {  // uniform: one vector at a time, its residual over rho in LDS
                const int vv = __builtin_ctz(todo);
                todo &= todo - 1u;
                float4* sr = s_r[wave];
                float* fr = reinterpret_cast<float*>(sr);
                wave_lds_fence();
                if (v == vv) {
#pragma unroll
                    for (int k = 0; k < 8; ++k)
                        sr[8 * g + k] = make_float4(r[4 * k], r[4 * k + 1], r[4 * k + 2], r[4 * k + 3]);
                }
                wave_lds_fence();
                const float rv = __shfl(rx, vv);
                const float h0_ = tq::div_rn(fr[lane], rv), h1_ = tq::div_rn(fr[lane + 64], rv);
                wave_lds_fence();
                fr[lane] = h0_;
                fr[lane + 64] = h1_;
                wave_lds_fence();
#pragma unroll
                for (int half = 0; half < 2; ++half) {
                    const uint32_t w0 = (uint32_t)__builtin_amdgcn_readlane((int)amb, vv + 32 * half);
                    const uint32_t w1 = (uint32_t)__builtin_amdgcn_readlane((int)amb, vv + 32 * half + 16);
                    if ((w0 | w1) == 0u) continue;
                    const bool need = ((lane < 32 ? w0 : w1) >> (lane & 31)) & 1u;
                    bool pos = false;
                    if (need) {
                        const float4* si = reinterpret_cast<const float4*>(a.S) + (64 * half + lane) * (D / 4);
                        float p = 0.0f;
#pragma unroll 8
                        for (int k = 0; k < D / 4; ++k) {
                            const float4 e = sr[k], c = si[k];
                            p = __builtin_fmaf(e.x, c.x, p);
                            p = __builtin_fmaf(e.y, c.y, p);
                            p = __builtin_fmaf(e.z, c.z, p);
                            p = __builtin_fmaf(e.w, c.w, p);
                        }
                        pos = p >= 0.0f;
                    }
                    const uint64_t bits = __builtin_amdgcn_ballot_w64(pos);
                    if (v == vv && (g >> 1) == half)
                        sb = (sb & ~amb) | ((uint32_t)(bits >> (32 * (g & 1))) & amb);
                }
            }
        }
        if (live) {
            if (g == 0) a.rnorms[slot] = (uint16_t)rho16;
            if constexpr (!GROUP) {
                reinterpret_cast<uint32_t*>(a.signs + slot * (D / 8))[g] = sb;
            } else {
                sb &= valid;
                uint8_t* dst = a.signs + slot * sign_bytes + 4 * g;
                const int left = sign_bytes - 4 * g;
                if (left >= 4) {
                    __builtin_memcpy(dst, &sb, 4);
                } else {
#pragma unroll
                    for (int e = 0; e < 3; ++e)
                        if (e < left) dst[e] = (uint8_t)(sb >> (8 * e));
                }
            }
        }
    }
}

// ------------------------------------------------------------------ calls of few vectors
// The chains themselves, on the fp32 matrix cores: a workgroup of eight waves encodes a tile of 16
// vectors, wave w the outputs [16 w, 16 w + 16) of each product (32 v_mfma_f32_16x16x4_f32, the fma
// chain over d = 4 s + k), and the vectors meet in LDS between the products.  Lane 16 g + v feeds
// element 4 s + g of vector v and gets back outputs 16 w + 4 g + (0..3) of it.  The matrices are staged
// in LDS once per workgroup, rows MS floats apart (reads of one column block by 16 rows and four
// columns hit 64 banks).  The norms are chains of 128 fma that every wave runs for all 16 vectors, one
// lane each (four alike), while its SIMD's other wave does the same.
//
// Latency-bound while a CU has one tile (up to 4096 vectors): the matrices' arrival and six barriers'
// worth of chains; beyond, about 8 us a tile with the sketch and 4 without, of which the products'
// issue is a quarter.  3-bit keys with the sketch / 4-bit values, us: one thread per output (the kernel
// below 1024 vectors) 24.5 / 9.2 at 2408 vectors and 31.8 / 11.4 at 4096, this one 11.1 / 6.4 and
// 11.5 / 6.7.
//
// The lines: up to 1024 vectors the one-thread-per-output kernels have at most a workgroup of four
// vectors per CU and are ahead (7.5 / 4.1 against 10.1 / 5.8 at 8, 9.8 / 5.3 against 10.7 / 6.3 at 1024);
// their callers keep those.  From TILE_MAX_* vectors the kernels above are: with the sketch 33.8 here
// against 46.5 there at 16384, 49.4 against 48.7 at 24576; without, 17.8 against 21.0 at 16384 and 25.3 against
// 18.9 at 24576 (channel groups the same within 10%).  Between, a plain call of one tile per wave is ahead
// of both in one pass (tq_quantize.hip).
constexpr int64_t TILE_MAX_PROD = 24576, TILE_MAX_MSE = 20480;
constexpr int MS = D + 4;
constexpr int BS = 36;  // floats between lanes' 32 elements in the exchange buffers

__device__ __forceinline__ int lane_slot(int v, int g) { return (4 * v + g) * BS; }

template <int BITS, bool GROUP, bool PROD>
__global__ __launch_bounds__(MQ_THREADS) void tile_kernel(EncodeArgs a) {
    constexpr int NB = (1 << BITS) - 1;
    __shared__ float s_r[D * MS];
    __shared__ float s_s[PROD ? D * MS : 1];
    __shared__ float4 s_a[64 * BS / 4];  // x as rows of MS floats; then C[code], then rhat, by lane
    __shared__ float4 s_b[64 * BS / 4];  // u by lane; then the residual as rows
    __shared__ uint8_t s_code[16][D];
    __shared__ float s_bound[NB];
    __shared__ float s_cent[PROD ? NB + 1 : 1];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int v = lane & 15, g = lane >> 4;
    const int sub_dim = GROUP ? a.sub_dim : D;
    const int row_bytes = GROUP ? (sub_dim * BITS + 7) >> 3 : D * BITS / 8;
    const int sign_bytes = (sub_dim + 7) >> 3;
    float* const fa = reinterpret_cast<float*>(s_a);
    float* const fb = reinterpret_cast<float*>(s_b);
    const uint32_t mw = a.mask[wave >> 1] >> (16 * (wave & 1) + 4 * g);  // this lane's four channels

    // channels 16 wave + 4 g + (0..3) of vector tile * 16 + v
    auto fetch = [&](int64_t tile, int64_t* slot) -> uint2 {
        const int64_t vi = tile * 16 + v;
        uint2 w = make_uint2(0u, 0u);
        *slot = -1;
        if (vi < a.n_vec) {
            w = reinterpret_cast<const uint2*>(row_of(a, (uint32_t)vi, slot))[4 * wave + g];
            if constexpr (GROUP) w.x &= pair_mask(mw, 0), w.y &= pair_mask(mw, 1);
        }
        return w;
    };
    const int64_t n_tiles = (a.n_vec + 15) / 16;
    int64_t next_slot;
    uint2 next = fetch(blockIdx.x, &next_slot);

    {
        constexpr int N = D * D / 4 / MQ_THREADS;
        f32x4 m[N], p[PROD ? N : 1];
#pragma unroll
        for (int i = 0; i < N; ++i) {
            m[i] = reinterpret_cast<const f32x4*>(a.R)[threadIdx.x + i * MQ_THREADS];
            if constexpr (PROD) p[i] = reinterpret_cast<const f32x4*>(a.S)[threadIdx.x + i * MQ_THREADS];
        }
        for (int i = threadIdx.x; i < NB; i += MQ_THREADS) s_bound[i] = a.boundaries[i];
        if constexpr (PROD)
            for (int i = threadIdx.x; i <= NB; i += MQ_THREADS) s_cent[i] = a.centers[i];
#pragma unroll
        for (int i = 0; i < N; ++i) {
            const int at = threadIdx.x + i * MQ_THREADS, dst = (at >> 5) * MS + 4 * (at & 31);
            *reinterpret_cast<f32x4*>(s_r + dst) = m[i];
            if constexpr (PROD) *reinterpret_cast<f32x4*>(s_s + dst) = p[i];
        }
    }
    // product of 16 rows (row m at `rows` + m * step_m, element 4 s + k at 4 s * step_k + k * step_k) with the 16
    // vectors whose elements lane 16 g + v finds at src
    auto product = [&](const float* rows, int step_m, int step_k, const float* src) {
        f32x4 b[8];
#pragma unroll
        for (int c = 0; c < 8; ++c) b[c] = *reinterpret_cast<const f32x4*>(src + lane_slot(v, g) + 4 * c);
        const float* am = rows + v * step_m + g * step_k;
        f32x4 acc = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
        for (int s = 0; s < 32; ++s) acc = mfma_f32(am[4 * s * step_k], b[s >> 2][s & 3], acc);
        return acc;
    };
    // sum of squares of row v as a chain, then its root (0 -> 1)
    auto norm_of = [&](const float* rows) {
        float ss = 0.0f;
#pragma unroll
        for (int c = 0; c < D / 4; ++c) {
            const f32x4 e = *reinterpret_cast<const f32x4*>(rows + v * MS + 4 * c);
#pragma unroll
            for (int k = 0; k < 4; ++k) ss = __builtin_fmaf(e[k], e[k], ss);
        }
        const float n = tq::sqrt_rn(ss);
        return n > 0.0f ? n : 1.0f;
    };
    // element i of this lane's four goes to the lane that feeds it: dim 16 wave + 4 g + i = 4 (4 wave + g) + i
    auto deal = [&](float* dst, int i, float e) { dst[lane_slot(v, i) + 4 * wave + g] = e; };

    for (int64_t tile = blockIdx.x; tile < n_tiles; tile += gridDim.x) {
        const int64_t slot = next_slot;
        const float x[4] = {lo_half(next.x), hi_half(next.x), lo_half(next.y), hi_half(next.y)};
        next = fetch(tile + gridDim.x, &next_slot);
        *reinterpret_cast<f32x4*>(fa + v * MS + 16 * wave + 4 * g) = f32x4{x[0], x[1], x[2], x[3]};
        __syncthreads();
        const float n = norm_of(fa);
        const uint32_t n16 = tq::f32_to_f16(n);
        if (wave == 0 && g == 0 && slot >= 0) a.norms[slot] = (uint16_t)n16;
#pragma unroll
        for (int i = 0; i < 4; ++i) deal(fb, i, tq::div_rn(x[i], n));
        __syncthreads();

        // ---- z_j, codes
        const f32x4 z = product(s_r + 16 * wave * MS, MS, 1, fb);
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const int j = 16 * wave + 4 * g + i;
            const uint32_t code = !GROUP || j < sub_dim ? bucket_lds(z[i], s_bound, BITS) : 0u;
            s_code[v][j] = (uint8_t)code;
            if constexpr (PROD) deal(fa, i, !GROUP || j < sub_dim ? s_cent[code] : 0.0f);
        }
        __syncthreads();
        // ---- the code rows: stream bits [32 k, 32 k + 32) of vector t / 32 by thread t = 32 vector + k
        {
            const int t = threadIdx.x >> 5, k = threadIdx.x & 31;
            // the tile's slots live in the lanes of vector t
            const int64_t row_slot = __shfl(slot, (t & 15));
            if (k < 4 * BITS && 4 * k < row_bytes && row_slot >= 0) {
                const int b0 = 32 * k, last = std::min((b0 + 31) / BITS, sub_dim - 1);
                uint64_t acc = 0;
                for (int j = b0 / BITS; j <= last; ++j)
                    acc |= (uint64_t)s_code[t][j] << (j * BITS - b0 + 32);  // shift in [33 - BITS, 63]
                const uint32_t word = (uint32_t)(acc >> 32);
                uint8_t* dst = a.codes + row_slot * row_bytes + 4 * k;
                const int left = row_bytes - 4 * k;
                if (!GROUP) {
                    *reinterpret_cast<uint32_t*>(dst) = word;
                } else if (left >= 4) {
                    __builtin_memcpy(dst, &word, 4);
                } else {
#pragma unroll
                    for (int e = 0; e < 3; ++e)
                        if (e < left) dst[e] = (uint8_t)(word >> (8 * e));
                }
            }
        }
        if constexpr (PROD) {
            // ---- residual: khat_d = bf16((chain j of C[code_j] R[j][d]) * f32(f16(n))), d = 16 wave + 4 g + i
            const f32x4 kh = product(s_r + 16 * wave, 1, MS, fa);
            const float nf = tq::f16_to_f32(n16);
            f32x4 r;
#pragma unroll
            for (int i = 0; i < 4; ++i) r[i] = x[i] - tq::bf16_to_f32(tq::f32_to_bf16(kh[i] * nf));
            *reinterpret_cast<f32x4*>(fb + v * MS + 16 * wave + 4 * g) = r;  // u was read before the barrier above
            __syncthreads();
            const float rho = norm_of(fb);
            if (wave == 0 && g == 0 && slot >= 0) a.rnorms[slot] = (uint16_t)tq::f32_to_f16(rho);
#pragma unroll
            for (int i = 0; i < 4; ++i) deal(fa, i, tq::div_rn(r[i], rho));
            __syncthreads();
            // ---- signs
            const f32x4 p = product(s_s + 16 * wave * MS, MS, 1, fa);
            uint32_t bits = 0u;
#pragma unroll
            for (int i = 0; i < 4; ++i)
                if (!GROUP || 16 * wave + 4 * g + i < sub_dim) bits |= (p[i] >= 0.0f ? 1u : 0u) << (4 * g + i);
            bits |= (uint32_t)__shfl_xor((int)bits, 16);
            bits |= (uint32_t)__shfl_xor((int)bits, 32);
            if (g == 0 && slot >= 0) {
                uint8_t* dst = a.signs + slot * sign_bytes + 2 * wave;
                if (!GROUP) {
                    *reinterpret_cast<uint16_t*>(dst) = (uint16_t)bits;
                } else {
                    if (2 * wave < sign_bytes) dst[0] = (uint8_t)bits;
                    if (2 * wave + 1 < sign_bytes) dst[1] = (uint8_t)(bits >> 8);
                }
            }
        }
        __syncthreads();  // every wave is done with the tile
    }
}

// Workgroups of a kernel that fit on the device at once (each loops over tiles, so more would only
// repeat the LDS set-up).
template <auto KERNEL>
int64_t resident(int threads) {
    static std::atomic<int64_t> cached[tq::MAX_DEVICES];
    return tq::once_per_device(cached, 256, [threads](int dev) {
        int cus = 0, per_cu = 0;
        if (hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess) cus = 256;
        if (hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, KERNEL, threads, 0) != hipSuccess || per_cu < 1)
            per_cu = 1;
        return (int64_t)cus * per_cu;
    });
}

template <auto KERNEL>
int launch(const EncodeArgs& a, int64_t groups, int threads, hipStream_t s) {
    hipLaunchKernelGGL(KERNEL, dim3((unsigned)std::min(groups, resident<KERNEL>(threads))), dim3(threads), 0, s, a);
    TQ_CHECK_LAUNCH();
    return TQ_OK;
}

template <int BITS, bool GROUP>
int encode(const EncodeArgs& a, hipStream_t s) {
    const int64_t tiles = (a.n_vec + 15) / 16;
    if (a.n_vec < (a.S ? TILE_MAX_PROD : TILE_MAX_MSE)) {
        if (!a.S) return launch<tile_kernel<BITS, GROUP, false>>(a, tiles, MQ_THREADS, s);
        if constexpr (GROUP || BITS <= 3) return launch<tile_kernel<BITS, GROUP, true>>(a, tiles, MQ_THREADS, s);
    }
    // two tiles per wave share each matrix fragment read from LDS; a call with fewer tiles than the
    // device has waves spreads them instead
    const int64_t waves = resident<codes_kernel<BITS, GROUP, 2>>(CT) * CW;
    const int st = tiles > waves ? launch<codes_kernel<BITS, GROUP, 2>>(a, (tiles + 1) / 2, CT, s)
                                 : launch<codes_kernel<BITS, GROUP, 1>>(a, tiles, CT, s);
    if (st != TQ_OK || !a.S) return st;
    if constexpr (GROUP || BITS <= 3)
        return launch<residual_kernel<BITS, GROUP>>(a, (tiles + MQ_WAVES - 1) / MQ_WAVES, MQ_THREADS, s);
    return TQ_ERR_INVALID_ARGUMENT;
}

}  // namespace

namespace tqenc {

int launch_encode(EncodeArgs a, int bits, bool group, hipStream_t s) {
    a.tok_div = make_fastdiv((uint32_t)a.tokens);
    a.head_div = make_fastdiv((uint32_t)a.heads);
    if (!group) {
        switch (bits) {
            case 1: return encode<1, false>(a, s);
            case 2: return encode<2, false>(a, s);
            case 3: return encode<3, false>(a, s);
            case 4: return encode<4, false>(a, s);
            default: return TQ_ERR_INVALID_ARGUMENT;
        }
    }
    switch (bits) {
        case 1: return encode<1, true>(a, s);
        case 2: return encode<2, true>(a, s);
        case 3: return encode<3, true>(a, s);
        case 4: return encode<4, true>(a, s);
        case 5: return encode<5, true>(a, s);
        case 6: return encode<6, true>(a, s);
        case 7: return encode<7, true>(a, s);
        case 8: return encode<8, true>(a, s);
        default: return TQ_ERR_INVALID_ARGUMENT;
    }
}

}  // namespace tqenc
