// tq_mfma.h -- fp32 matrix-core chains shared by the encoders and decoders (gfx950).
//
// v_mfma_f32_16x16x4_f32 adds the four products of its k = 0..3 to the accumulator one after
// another, each with one rounding (an fma chain in k order), so a chain of 32 of them over
// k-steps s = 0..31 covering d = 4s + k is the fma chain d = 0..127, bit for bit, denormals
// and signed zeros included.
//
// A wave works on a tile of 16 vectors.  Lane l = 16 g + v (v = l % 16, g = l / 16) holds
// element 4s + g of vector v for s = 0..31: the B operand (k = g, column v) of every product;
// a product's accumulator comes back to the lanes of its column v.  The matrix is the A
// operand, read from an LDS image laid out per (16-row tile t, k-step block sb): 64 lanes x 4
// consecutive k-steps, one 16-byte read per lane per block, lane slots xor-swizzled
// (slot = l ^ (l >> 4)).  In the CONTIG row order, row m = 4q + i of tile t is output index
// 32q + 4t + i, so lane g ends up holding outputs [32g, 32g + 32) of its vector.

#pragma once

#include <cstdint>
#include <utility>

#include "tq_common.h"

namespace tqmx {

constexpr int MXD = TQ_DIM;

typedef float f32x4 __attribute__((ext_vector_type(4)));
constexpr int MQ_WAVES = 8;                 // waves per workgroup, each on its own tiles
constexpr int MQ_THREADS = 64 * MQ_WAVES;

__device__ __forceinline__ f32x4 mfma_f32(float a, float b, f32x4 c) {
    return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0);
}

// floor(n / d) = (n * m) >> s for 0 <= n < 2^31 and 1 <= d < 2^31, with l = ceil(log2 d),
// s = 31 + l and m = ceil(2^s / d) < 2^32: then 2^s <= m d <= 2^s + 2^l (Granlund and
// Montgomery, "Division by invariant integers using multiplication", 1994, Theorem 4.2).
struct FastDiv {
    uint32_t m, s;
};
inline FastDiv make_fastdiv(uint32_t d) {
    uint32_t l = 0;
    while ((1ull << l) < d) ++l;
    return {(uint32_t)(((1ull << (31 + l)) + d - 1) / d), 31 + l};
}
__device__ __forceinline__ uint32_t fdiv(uint32_t n, FastDiv f) {
    return (uint32_t)(((uint64_t)n * f.m) >> f.s);
}

// fp32 -> bf16, nearest even, two at a time (v_cvt_pk_bf16_f32: the bits of tq::f32_to_bf16 for all
// 2^32 inputs), and back.
__device__ __forceinline__ uint32_t bf16_pair(float a, float b) {
    typedef float f32x2 __attribute__((ext_vector_type(2)));
    typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
    const f32x2 p = {a, b};
    return __builtin_bit_cast(uint32_t, __builtin_convertvector(p, bf16x2));
}
__device__ __forceinline__ float lo_half(uint32_t p) { return __uint_as_float(p << 16); }
__device__ __forceinline__ float hi_half(uint32_t p) { return __uint_as_float(p & 0xFFFF0000u); }

// cv[s] = cent[code of index 4 s + g], s = 0..31, from a vector's code row w (BITS words per 32 codes,
// one zero word past the row's end).  The row is shifted down by g codes once; index 4 s + g then sits
// at the fixed bit 4 s BITS, and the words, indexed by constants, stay in registers.
template <int BITS, int... I>
__device__ __forceinline__ void take_centers(const uint32_t* w, const float* cent, float* cv,
                                             std::integer_sequence<int, I...>) {
    ((cv[I] = cent[tq::extract_bits<BITS>(w, 4 * I * BITS)]), ...);
}
template <int BITS>
__device__ __forceinline__ void centers_of(uint32_t* w, int g, const float* cent, float* cv) {
#pragma unroll
    for (int c = 0; c < 4 * BITS; ++c) w[c] = __builtin_amdgcn_alignbit(w[c + 1], w[c], g * BITS);
    take_centers<BITS>(w, cent, cv, std::make_integer_sequence<int, 32>{});
}

// Rotation / QJL products of one tile: acc[t][i] = chain over d of b[d] * M[row(t, 4g + i)][d],
// with b held as described above (b[s] = element 4s + g) and `a` this lane's slot of image M.
// NT < 8 computes the row tiles t = 0..NT-1 of an image pointer advanced by t0 * 8 * 64.
template <int NT = 8>
__device__ __forceinline__ void image_products(const float4* __restrict__ a, const float* b, f32x4* acc) {
#pragma unroll
    for (int t = 0; t < NT; ++t) acc[t] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
    // two register sets of A values: block sb + 1 is read while block sb's products run; the
    // scheduling barriers keep the compiler from hoisting every block's reads to the top
    float4 cur[NT], nxt[NT];
#pragma unroll
    for (int t = 0; t < NT; ++t) cur[t] = a[t * 8 * 64];
#pragma unroll
    for (int sb = 0; sb < 8; ++sb) {
        if (sb + 1 < 8) {
#pragma unroll
            for (int t = 0; t < NT; ++t) nxt[t] = a[(t * 8 + sb + 1) * 64];
        }
#pragma unroll
        for (int e = 0; e < 4; ++e) {
#pragma unroll
            for (int t = 0; t < NT; ++t) {
                const float ae = e == 0 ? cur[t].x : e == 1 ? cur[t].y : e == 2 ? cur[t].z : cur[t].w;
                acc[t] = mfma_f32(ae, b[4 * sb + e], acc[t]);
            }
        }
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int t = 0; t < NT; ++t) cur[t] = nxt[t];
    }
}

// CONTIG image of M^T for a matrix M of `rows` <= MXD rows of MXD floats: row r of the image
// is column r of M, and its k-index d is row d - (MXD - rows) of M, the first MXD - rows
// k-indices zero.  A chain over the image then starts with that many zero products, which
// leave its +0 start unchanged (+0 plus a zero of either sign is +0), so it is the fma chain
// over M's rows, bit for bit.
// A float4 of the image holds one column's rows d, d + 4, d + 8, d + 12, so a thread reads four columns of
// those four rows and writes four float4: a quarter of the LDS writes of one row at a time, whose words
// met in 8 of the banks.  Lanes go round over (k, q) first, the low bits of a float4's place, then over t,
// neighbours in memory.  All reads are in flight ahead of the first write, in the decoder those of both
// matrices.  The image is most of a small call: 8192 keys with QJL 15.3 -> 11.3 us and values
// 8.5 -> 7.1 us, 65536 48.9 -> 45.1 and 27.5 -> 26.1 us; 2M rows as before.
struct TransposedImage {
    static constexpr int N = MXD * MXD / 16 / MQ_THREADS;
    float4 v[N][4];
    __device__ __forceinline__ void load(const float* __restrict__ M, int rows = MXD) {
        const int pad = MXD - rows;
#pragma unroll
        for (int i = 0; i < N; ++i) {
            const int u = threadIdx.x + i * MQ_THREADS;  // k = u % 4, q = u / 4 % 4, t = u / 16 % 8, block u / 128
            const int col = 32 * ((u >> 2) & 3) + 4 * ((u >> 4) & 7), d0 = 16 * (u >> 7) + (u & 3);
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                const int d = d0 + 4 * e;
                v[i][e] = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
                if (d >= pad)  // M may start at any float
                    __builtin_memcpy(&v[i][e], M + (size_t)(d - pad) * MXD + col, sizeof(float4));
            }
        }
    }
    __device__ __forceinline__ void store(float4* img) const {
#pragma unroll
        for (int i = 0; i < N; ++i) {
            const int u = threadIdx.x + i * MQ_THREADS, k = u & 3, q = (u >> 2) & 3, t = (u >> 4) & 7;
            float4* blk = img + (t * 8 + (u >> 7)) * 64;  // columns 32 q + 4 t + j are rows 4 q + j of tile t
            blk[(16 * k + 4 * q + 0) ^ k] = make_float4(v[i][0].x, v[i][1].x, v[i][2].x, v[i][3].x);
            blk[(16 * k + 4 * q + 1) ^ k] = make_float4(v[i][0].y, v[i][1].y, v[i][2].y, v[i][3].y);
            blk[(16 * k + 4 * q + 2) ^ k] = make_float4(v[i][0].z, v[i][1].z, v[i][2].z, v[i][3].z);
            blk[(16 * k + 4 * q + 3) ^ k] = make_float4(v[i][0].w, v[i][1].w, v[i][2].w, v[i][3].w);
        }
    }
};
__device__ __forceinline__ void build_image_transposed(float* img, const float* __restrict__ M, int rows = MXD) {
    TransposedImage m;
    m.load(M, rows);
    m.store(reinterpret_cast<float4*>(img));
}

}  // namespace tqmx
