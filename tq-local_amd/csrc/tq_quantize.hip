// tq_quantize.hip -- TurboQuant encoder kernels for gfx950 (prefill and decode-append).
//
// Every kernel evaluates the encoder in one fixed fp32 order (the CPU oracle restates the
// reference in the same order), so their outputs are bit-identical to it and to each other:
//
//   norm^2 = fma chain d=0..127 of x_d*x_d;  n = sqrt_rn;  n==0 -> 1
//   u_d    = x_d /_rn n
//   z_j    = fma chain d=0..127 of u_d*R[j][d]          (z = u @ R^T)
//   code_j = #{i : boundaries_i < z_j}                   (torch.bucketize right=False)
//   Q_prod residual:  khat_d = bf16((fma chain j=0..127 of C[code_j]*R[j][d]) * f32(f16(n)))
//                     r = x - khat;  rho = sqrt_rn(fma chain r_d^2) (0 -> 1);  rhat = r /_rn rho
//                     sign_i = (fma chain d of rhat_d*S[i][d]) >= 0
//
// Two encoders: those of tq_encode.hip for calls of at least MQ_MIN_VECTORS vectors (prefill; the
// figures at the line stand there) and a small-batch kernel with one thread per output index of each
// vector (decode-append).
//
// Reference: runtime/packed_qmse_cache.py:376-402 (_encode_group), :285-310
// (_encode_keys_qjl_group), :404-435 (_decode_group), :13-43 (_pack_indices),
// :148-154 (_pack_qjl_signs).

#include <algorithm>
#include <type_traits>
#include <utility>

#include "tq_encode.h"

namespace {

using namespace tqmx;
constexpr int D = TQ_DIM;

// #{i : b[i] < z} (torch.bucketize right=False): one compare and one add-with-carry per
// boundary; the empty asm keeps the count a plain running sum (no bitmask reassociation).
template <int NB>
__device__ __forceinline__ uint32_t bucket_count(float z, const float* __restrict__ b) {
    uint32_t c = 0;
#pragma unroll
    for (int i = 0; i < NB; ++i) {
        c += (b[i] < z) ? 1u : 0u;
        __asm__("" : "+v"(c));
    }
    return c;
}

// ------------------------------------------------------------------ small-batch encoder
// Below MQ_MIN_VECTORS vectors (decode-append encodes B * Hkv of them per step) a workgroup
// encodes AV vectors with D threads each: thread (v, j) owns output index j of vector v in
// every matrix-vector product and runs that output's fma chain alone, in the fixed order
// above, so the result is bit for bit the chain of the oracle and of the prefill encoder.
// The matrices are staged in LDS with a row stride of MS = 132 floats: thread j reading row j
// 16 bytes at a time (the rotation and the QJL projection) touches 4 j + 4 k mod 64, distinct
// banks for the 16 lanes of an LDS pass, and thread d reading column d (the residual decode)
// touches consecutive banks.  The norms are fma chains over the vector held in LDS, run by
// every thread of the vector (the same operands in the same order: one value in all of them).
//
// A call of few vectors is bound by one workgroup's LDS reads along five chains of 128 (when the
// matrices are staged, beside or before the norm, makes no difference).  So the vectors spread over
// the CUs: one per workgroup while there are that many, the other waves only staging.  3-bit keys with
// the sketch / 4-bit values at 8 vectors, us: 8.7 / 4.6 with four per workgroup, 8.3 / 4.5 with two,
// 7.5 / 4.1 with one.
constexpr int AT = 4 * D;      // threads per workgroup
constexpr int MS = D + 4;      // LDS row stride of a staged matrix, floats

template <int BITS, bool PROD, int AV>
__global__ __launch_bounds__(AT) void append_kernel(
    const uint16_t* __restrict__ x, int heads, int64_t tokens, int64_t n_vec, int64_t x_sb, int64_t x_sh,
    int64_t x_st, const float* __restrict__ R, const float* __restrict__ centers,
    const float* __restrict__ boundaries, const float* __restrict__ S, uint8_t* __restrict__ codes,
    uint16_t* __restrict__ norms, uint8_t* __restrict__ signs, uint16_t* __restrict__ rnorms, int64_t out_cap,
    int64_t out_offset, FastDiv tok_div, FastDiv head_div) {
    __shared__ float4 sR[D * MS / 4];
    __shared__ float4 sS[PROD ? D * MS / 4 : 1];
    __shared__ float4 sx[AV][D / 4];    // the vector in fp32, later rhat
    __shared__ float4 su[AV][D / 4];    // u = x / n, later the residual
    __shared__ float4 sc[AV][D / 4];    // C[code_j]
    __shared__ uint8_t scode[AV][D];
    __shared__ float scent[1 << BITS];

    const int tid = threadIdx.x;
    const int vi = tid / D, j = tid % D;  // vector of the workgroup (two whole waves), output index
    const bool works = vi < AV;           // the waves of further vectors only stage and wait
    const int64_t v = (int64_t)blockIdx.x * AV + vi;
    const bool active = works && v < n_vec;  // threads of missing vectors compute on unused LDS, store nothing
    float* const fx = reinterpret_cast<float*>(sx[works ? vi : 0]);
    float* const fu = reinterpret_cast<float*>(su[works ? vi : 0]);
    float* const fc = reinterpret_cast<float*>(sc[works ? vi : 0]);

    // ---- the matrices, the codebook and the vector into LDS (row r of a matrix at r * MS)
    constexpr int N = D * D / 4 / AT;
    f32x4 mR[N], mS[PROD ? N : 1];
#pragma unroll
    for (int i = 0; i < N; ++i) mR[i] = reinterpret_cast<const f32x4*>(R)[tid + i * AT];
    if constexpr (PROD) {
#pragma unroll
        for (int i = 0; i < N; ++i) mS[i] = reinterpret_cast<const f32x4*>(S)[tid + i * AT];
    }
    int64_t slot = 0;
    if (active) {
        int64_t gh, b;
        if (n_vec < ((int64_t)1 << 31)) {
            const uint32_t q = fdiv((uint32_t)v, tok_div);
            gh = q;
            b = fdiv(q, head_div);
        } else {
            gh = v / tokens;
            b = gh / heads;
        }
        const int64_t t = v - gh * tokens, h = gh - b * heads;
        fx[j] = tq::bf16_to_f32(x[b * x_sb + h * x_sh + t * x_st + j]);
        slot = gh * out_cap + out_offset + t;
    }
    if (PROD && tid < (1 << BITS)) scent[tid] = centers[tid];
#pragma unroll
    for (int i = 0; i < N; ++i) {
        const int k = tid + i * AT, at = k / (D / 4) * (MS / 4) + k % (D / 4);
        reinterpret_cast<f32x4*>(sR)[at] = mR[i];
        if constexpr (PROD) reinterpret_cast<f32x4*>(sS)[at] = mS[i];
    }
    __syncthreads();

    // ---- norm, u = x / n
    auto norm_of = [](const float4* row) {
        float ss = 0.0f;
#pragma unroll
        for (int d4 = 0; d4 < D / 4; ++d4) {
            const float4 e = row[d4];
            ss = __builtin_fmaf(e.x, e.x, ss);
            ss = __builtin_fmaf(e.y, e.y, ss);
            ss = __builtin_fmaf(e.z, e.z, ss);
            ss = __builtin_fmaf(e.w, e.w, ss);
        }
        const float n = tq::sqrt_rn(ss);
        return n > 0.0f ? n : 1.0f;
    };
    auto chain = [](const float4* a, const float4* b) {
        float z = 0.0f;
#pragma unroll
        for (int d4 = 0; d4 < D / 4; ++d4) {
            const float4 uu = a[d4], rr = b[d4];
            z = __builtin_fmaf(uu.x, rr.x, z);
            z = __builtin_fmaf(uu.y, rr.y, z);
            z = __builtin_fmaf(uu.z, rr.z, z);
            z = __builtin_fmaf(uu.w, rr.w, z);
        }
        return z;
    };
    float xj = 0.0f, r = 0.0f;
    uint32_t n16 = 0u;
    if (works) {
        const float n = norm_of(sx[vi]);
        xj = fx[j];
        fu[j] = tq::div_rn(xj, n);
        n16 = tq::f32_to_f16(n);
        if (active && j == 0) norms[slot] = (uint16_t)n16;
    }
    __syncthreads();

    // ---- z_j = fma chain d of u_d R[j][d]; code_j
    if (works) {
        const uint32_t code = bucket_count<(1 << BITS) - 1>(chain(su[vi], sR + j * (MS / 4)), boundaries);
        scode[vi][j] = (uint8_t)code;
        if constexpr (PROD) fc[j] = scent[code];
    }
    __syncthreads();

    // ---- the code row: thread j < ROW / 4 assembles dword j (stream bits [32 j, 32 j + 32))
    constexpr int ROW = D * BITS / 8;
    if (active && j < ROW / 4) {
        const int b0 = 32 * j;
        uint64_t acc = 0;
        for (int k = b0 / BITS; k <= (b0 + 31) / BITS; ++k)
            acc |= (uint64_t)scode[vi][k] << (k * BITS - b0 + 32);  // shift in [33 - BITS, 63]
        reinterpret_cast<uint32_t*>(codes + slot * ROW)[j] = (uint32_t)(acc >> 32);
    }

    if constexpr (PROD) {
        // ---- residual: khat_d = bf16((fma chain jj of C[code_jj] R[jj][d]) * f32(f16(n))), d = j
        if (works) {
            const float* fR = reinterpret_cast<const float*>(sR);
            float acc = 0.0f;
#pragma unroll
            for (int k4 = 0; k4 < D / 4; ++k4) {
                const float4 cc = sc[vi][k4];
                acc = __builtin_fmaf(cc.x, fR[(4 * k4 + 0) * MS + j], acc);
                acc = __builtin_fmaf(cc.y, fR[(4 * k4 + 1) * MS + j], acc);
                acc = __builtin_fmaf(cc.z, fR[(4 * k4 + 2) * MS + j], acc);
                acc = __builtin_fmaf(cc.w, fR[(4 * k4 + 3) * MS + j], acc);
            }
            r = xj - tq::bf16_to_f32(tq::f32_to_bf16(acc * tq::f16_to_f32(n16)));
            fu[j] = r;  // u was last read by the rotation, before the barrier above
        }
        __syncthreads();
        if (works) {
            const float rho = norm_of(su[vi]);
            fx[j] = tq::div_rn(r, rho);  // x was last read before the second barrier
            if (active && j == 0) rnorms[slot] = (uint16_t)tq::f32_to_f16(rho);
        }
        __syncthreads();
        // ---- sign_i = (fma chain d of rhat_d S[i][d]) >= 0, i = j; a wave holds 64 of them
        if (works) {
            const float p = chain(sx[vi], sS + j * (MS / 4));
            const uint64_t sb = __builtin_amdgcn_ballot_w64(p >= 0.0f);  // bit l: index 64 (j / 64) + l
            if (active && (j & 63) == 0)
                reinterpret_cast<uint2*>(signs + slot * (D / 8))[j >> 6] = make_uint2((uint32_t)sb, (uint32_t)(sb >> 32));
        }
    }
}

// At least this many vectors take the prefill encoder (tq_encode.hip).
constexpr int64_t MQ_MIN_VECTORS = 1025;

// ------------------------------------------------------------------- decoders
// out = bf16((C[code] @ R) * f32(norm)); with QJL (keys of Q_prod) the reference's
// correction is added in bf16: corr = bf16(((s @ S) * rnorm) * sqrt(pi/2)/D),
// out = bf16(f32(khat) + f32(corr))   (runtime/packed_qmse_cache.py:312-330, 404-435).
// Output dim d is the fma chain j = 0..127 of C[code_j] * R[j][d] (of sign_j * S[j][d] for
// the correction), the residual decode's order.  On the matrix cores these are the image
// products above with A = R^T (S^T): a CONTIG image of the transposed matrix leaves dims
// [32g, 32g + 32) of vector v in lane 16 g + v, which stores them as 64 contiguous bytes.
// The B operand is C[code] of index 4s + g; each of a vector's four lanes loads the whole
// code row and takes its own indices from it.

template <int BITS, bool QJL, int PARTS>
__global__ __launch_bounds__(MQ_THREADS) void dequantize_kernel(
    const uint8_t* __restrict__ codes, const uint16_t* __restrict__ norms, const uint8_t* __restrict__ signs,
    const uint16_t* __restrict__ rnorms, int64_t tokens, int64_t cap, int64_t n_vec, const float* __restrict__ R,
    const float* __restrict__ centers, const float* __restrict__ S, uint16_t* __restrict__ out, FastDiv tok_div) {
    __shared__ float4 s_img[(QJL ? 2 : 1) * D * D / 4];  // R^T image (+ S^T image)
    __shared__ float s_cent[1 << BITS];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int v = lane & 15, g = lane >> 4;
    constexpr int NT = 8 / PARTS;  // row tiles (16 output dims each) per work item
    constexpr int ROW = D * BITS / 8;  // code bytes per vector
    constexpr int RW = ROW / 4;
    const int64_t n_items = (n_vec + 15) / 16 * PARTS;

    // work item = (tile of 16 vectors, part): part p computes row tiles [p NT, p NT + NT), the
    // dims 32g + [4 p NT, 4 p NT + 4 NT) of each of lane 16 g + v's vector
    uint4 raw[BITS], raw_sign;
    uint32_t raw_norm = 0u, raw_rnorm = 0u;
    auto fetch = [&](int64_t item) {
        const uint32_t vi = (uint32_t)(item / PARTS) * 16u + (uint32_t)v;  // n_vec < 2^31
        // a lane past the end reads slot 0's row, which exists, and stores nothing
        int64_t slot = 0;
        if (item < n_items && vi < (uint64_t)n_vec) {
            const uint32_t gh = fdiv(vi, tok_div);
            slot = (int64_t)gh * cap + (vi - gh * (uint32_t)tokens);
        }
        const uint4* c4 = reinterpret_cast<const uint4*>(codes + slot * ROW);
#pragma unroll
        for (int c = 0; c < BITS; ++c) raw[c] = c4[c];
        raw_norm = norms[slot];
        if constexpr (QJL) {
            raw_sign = reinterpret_cast<const uint4*>(signs + slot * (D / 8))[0];
            raw_rnorm = rnorms[slot];
        }
    };
    // the first item's rows are on their way while the images are built
    int64_t item = (int64_t)blockIdx.x * MQ_WAVES + wave;
    fetch(item);
    float* img = reinterpret_cast<float*>(s_img);
    build_image_transposed(img, R);
    if constexpr (QJL) build_image_transposed(img + D * D, S);
    if (threadIdx.x < (1 << BITS)) s_cent[threadIdx.x] = centers[threadIdx.x];
    __syncthreads();  // the only barrier: each wave then works on its own tiles

    for (; item < n_items; item += (int64_t)gridDim.x * MQ_WAVES) {
        const int64_t tile = item / PARTS;
        const int t0 = (int)(item % PARTS) * NT;
        const float4* a_img = s_img + t0 * 8 * 64 + (lane ^ g);
        const uint32_t vi = (uint32_t)tile * 16u + (uint32_t)v;  // n_vec < 2^31
        const bool live = vi < (uint64_t)n_vec;
        uint32_t w[RW + 1];  // the code row, one zero word past its end
#pragma unroll
        for (int c = 0; c < BITS; ++c)
            w[4 * c] = raw[c].x, w[4 * c + 1] = raw[c].y, w[4 * c + 2] = raw[c].z, w[4 * c + 3] = raw[c].w;
        w[RW] = 0u;
        const float nf = tq::f16_to_f32(raw_norm);
        const uint4 sw = raw_sign;
        const float rn = tq::f16_to_f32(raw_rnorm);
        float cv[32];
        centers_of<BITS>(w, g, s_cent, cv);
        // the next item's rows beside this one's products (Q_mse kernels, four waves on a SIMD, would
        // lose one to the registers)
        if (QJL) fetch(item + (int64_t)gridDim.x * MQ_WAVES);
        f32x4 acc[NT];
        image_products<NT>(a_img, cv, acc);
        uint32_t kh[2 * NT];  // bf16 pairs of dims 32g + 4 t0 + 2p, + 2p + 1
#pragma unroll
        for (int p = 0; p < 2 * NT; ++p)
            kh[p] = bf16_pair(acc[p >> 1][2 * (p & 1)] * nf, acc[p >> 1][2 * (p & 1) + 1] * nf);
        if constexpr (QJL) {
            // sign of index 4s + g: word s / 8, bit 4 (s % 8) + g of the 16-byte sign row
            // +-1: the inverted bit as the sign
            const uint32_t sws[4] = {~sw.x >> g, ~sw.y >> g, ~sw.z >> g, ~sw.w >> g};
            float sv[32];
#pragma unroll
            for (int s = 0; s < 32; ++s)
                sv[s] = __uint_as_float(((sws[s >> 3] << (31 - 4 * (s & 7))) & 0x80000000u) | 0x3F800000u);
            f32x4 pacc[NT];
            image_products<NT>(a_img + D * D / 4, sv, pacc);
            const float qs = 1.2533141373155003f / D;  // sqrt(pi/2)/D rounded to fp32
#pragma unroll
            for (int p = 0; p < 2 * NT; ++p) {
                const uint32_t c = bf16_pair((pacc[p >> 1][2 * (p & 1)] * rn) * qs, (pacc[p >> 1][2 * (p & 1) + 1] * rn) * qs);
                kh[p] = bf16_pair(lo_half(kh[p]) + lo_half(c), hi_half(kh[p]) + hi_half(c));
            }
        }
        if (live) {
            uint4* o4 = reinterpret_cast<uint4*>(out + (int64_t)vi * D + 32 * g + 4 * t0);
#pragma unroll
            for (int i = 0; i < NT / 2; ++i) o4[i] = make_uint4(kh[4 * i], kh[4 * i + 1], kh[4 * i + 2], kh[4 * i + 3]);
        }
        if (!QJL) fetch(item + (int64_t)gridDim.x * MQ_WAVES);
    }
}

bool aligned16(const void* p) { return (reinterpret_cast<uintptr_t>(p) & 15u) == 0; }

int check_common(const uint16_t* x, int batch, int heads, int64_t tokens, int dim, int64_t x_sb, int64_t x_sh,
                 int64_t x_st, int64_t out_cap, int64_t out_offset) {
    if (!x || batch < 0 || heads < 0 || tokens < 0 || out_offset < 0) return TQ_ERR_INVALID_ARGUMENT;
    if (out_offset + tokens > out_cap) return TQ_ERR_INVALID_ARGUMENT;
    if (dim != TQ_DIM) return TQ_ERR_UNSUPPORTED;
    if (!aligned16(x) || (x_sb % 8) || (x_sh % 8) || (x_st % 8)) return TQ_ERR_UNSUPPORTED;
    return TQ_OK;
}

bool prefill_size(int64_t n_vec) { return n_vec >= MQ_MIN_VECTORS && n_vec < ((int64_t)1 << 31); }

tqenc::EncodeArgs plain_args(const uint16_t* x, int batch, int heads, int64_t tokens, int64_t x_sb, int64_t x_sh,
                             int64_t x_st, const float* R, const float* centers, const float* boundaries,
                             const float* S, uint8_t* codes, uint16_t* norms, uint8_t* signs, uint16_t* rnorms,
                             int64_t out_cap, int64_t out_offset) {
    return {x, heads, tokens, (int64_t)batch * heads * tokens, x_sb, x_sh, x_st, R, centers, boundaries, S, codes, norms,
            signs, rnorms, out_cap, out_offset, {~0u, ~0u, ~0u, ~0u}, TQ_DIM, {}, {}};
}

// Workgroups of a matrix-core kernel that fit on the device at once (each loops over tiles,
// so more would only repeat the LDS image set-up).
template <auto KERNEL>
int64_t resident_groups() {
    static std::atomic<int64_t> cached[tq::MAX_DEVICES];
    return tq::once_per_device(cached, 256, [](int dev) {
        int cus = 0, per_cu = 0;
        if (hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess) cus = 256;
        if (hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, KERNEL, MQ_THREADS, 0) != hipSuccess || per_cu < 1)
            per_cu = 1;
        return (int64_t)cus * per_cu;
    });
}

template <int BITS, bool PROD, int AV>
int launch_append_by(const tqenc::EncodeArgs& a, hipStream_t s) {
    hipLaunchKernelGGL((append_kernel<BITS, PROD, AV>), dim3((unsigned)((a.n_vec + AV - 1) / AV)), dim3(AT), 0, s, a.x,
                       a.heads, a.tokens, a.n_vec, a.x_sb, a.x_sh, a.x_st, a.R, a.centers, a.boundaries, a.S, a.codes,
                       a.norms, a.signs, a.rnorms, a.out_cap, a.out_offset, make_fastdiv((uint32_t)a.tokens),
                       make_fastdiv((uint32_t)a.heads));
    TQ_CHECK_LAUNCH();
    return TQ_OK;
}

// Vectors per workgroup: as few as leave one workgroup (137 KB of LDS) per CU.  Keys / values, us: 256
// vectors 8.1 / 4.4 at one, 8.7 / 4.7 at two; 384 14.1 / 5.0 at one, 8.8 / 4.9 at two; 512 8.9 / 4.9 at
// two, 9.3 / 5.0 at four; 768 16.0 / 5.5 at two, 9.5 / 5.0 at four.
constexpr int64_t APPEND_ONE = 256, APPEND_TWO = 512;

template <int BITS, bool PROD>
int launch_append(const tqenc::EncodeArgs& a, hipStream_t s) {
    if (a.n_vec == 0) return TQ_OK;
    if (a.n_vec <= APPEND_ONE) return launch_append_by<BITS, PROD, 1>(a, s);
    if (a.n_vec <= APPEND_TWO) return launch_append_by<BITS, PROD, 2>(a, s);
    return launch_append_by<BITS, PROD, 4>(a, s);
}

}  // namespace

extern "C" int tq_quantize_mse(const uint16_t* x, int batch, int heads, int64_t tokens, int dim, int64_t x_sb,
                               int64_t x_sh, int64_t x_st, int bits, const float* rotation,
                               const float* boundaries, uint8_t* codes, uint16_t* norms, int64_t out_cap,
                               int64_t out_offset, void* stream) {
    int st = check_common(x, batch, heads, tokens, dim, x_sb, x_sh, x_st, out_cap, out_offset);
    if (st != TQ_OK) return st;
    if (!rotation || !boundaries || !codes || !norms) return TQ_ERR_INVALID_ARGUMENT;
    if (!aligned16(codes) || !aligned16(rotation)) return TQ_ERR_UNSUPPORTED;
    const tqenc::EncodeArgs a = plain_args(x, batch, heads, tokens, x_sb, x_sh, x_st, rotation, nullptr, boundaries,
                                           nullptr, codes, norms, nullptr, nullptr, out_cap, out_offset);
    hipStream_t s = static_cast<hipStream_t>(stream);
    if (bits >= 1 && bits <= 4 && prefill_size(a.n_vec)) return tqenc::launch_encode(a, bits, false, s);
    switch (bits) {
        case 1: return launch_append<1, false>(a, s);
        case 2: return launch_append<2, false>(a, s);
        case 3: return launch_append<3, false>(a, s);
        case 4: return launch_append<4, false>(a, s);
        default: return TQ_ERR_INVALID_ARGUMENT;
    }
}

extern "C" int tq_quantize_prod(const uint16_t* x, int batch, int heads, int64_t tokens, int dim, int64_t x_sb,
                                int64_t x_sh, int64_t x_st, int mse_bits, const float* rotation,
                                const float* centers, const float* boundaries, const float* qjl, uint8_t* codes,
                                uint16_t* norms, uint8_t* signs, uint16_t* rnorms, int64_t out_cap,
                                int64_t out_offset, void* stream) {
    int st = check_common(x, batch, heads, tokens, dim, x_sb, x_sh, x_st, out_cap, out_offset);
    if (st != TQ_OK) return st;
    if (!rotation || !centers || !boundaries || !qjl || !codes || !norms || !signs || !rnorms)
        return TQ_ERR_INVALID_ARGUMENT;
    if (!aligned16(codes) || !aligned16(signs) || !aligned16(rotation) || !aligned16(qjl)) return TQ_ERR_UNSUPPORTED;
    const tqenc::EncodeArgs a = plain_args(x, batch, heads, tokens, x_sb, x_sh, x_st, rotation, centers, boundaries, qjl,
                                           codes, norms, signs, rnorms, out_cap, out_offset);
    hipStream_t s = static_cast<hipStream_t>(stream);
    if (mse_bits >= 1 && mse_bits <= 3 && prefill_size(a.n_vec)) return tqenc::launch_encode(a, mse_bits, false, s);
    switch (mse_bits) {
        case 1: return launch_append<1, true>(a, s);
        case 2: return launch_append<2, true>(a, s);
        case 3: return launch_append<3, true>(a, s);
        default: return TQ_ERR_INVALID_ARGUMENT;
    }
}

namespace {

template <int BITS, bool QJL, int PARTS>
int launch_dequantize_parts(const uint8_t* codes, const uint16_t* norms, const uint8_t* signs,
                            const uint16_t* rnorms, int64_t tokens, int64_t cap, int64_t n_vec,
                            const float* rotation, const float* centers, const float* qjl, uint16_t* out,
                            hipStream_t s) {
    const int64_t items = (n_vec + 15) / 16 * PARTS;
    const int64_t wgs = std::min<int64_t>((items + MQ_WAVES - 1) / MQ_WAVES,
                                          resident_groups<dequantize_kernel<BITS, QJL, PARTS>>());
    hipLaunchKernelGGL((dequantize_kernel<BITS, QJL, PARTS>), dim3((unsigned)wgs), dim3(MQ_THREADS), 0, s, codes,
                       norms, signs, rnorms, tokens, cap, n_vec, rotation, centers, qjl, out,
                       make_fastdiv((uint32_t)tokens));
    TQ_CHECK_LAUNCH();
    return TQ_OK;
}

// A call with fewer tiles than the device holds waves splits each tile's row tiles over 2 or 4
// waves: the same chains, each wave running a half or a quarter of a tile's MFMAs.
template <int BITS, bool QJL>
int run_dequantize(const uint8_t* codes, const uint16_t* norms, const uint8_t* signs, const uint16_t* rnorms,
                   int64_t tokens, int64_t cap, int64_t n_vec, const float* rotation, const float* centers,
                   const float* qjl, uint16_t* out, hipStream_t s) {
    const int64_t tiles = (n_vec + 15) / 16;
    const int64_t waves = resident_groups<dequantize_kernel<BITS, QJL, 1>>() * MQ_WAVES;
    if (4 * tiles <= waves)
        return launch_dequantize_parts<BITS, QJL, 4>(codes, norms, signs, rnorms, tokens, cap, n_vec, rotation,
                                                     centers, qjl, out, s);
    if (2 * tiles <= waves)
        return launch_dequantize_parts<BITS, QJL, 2>(codes, norms, signs, rnorms, tokens, cap, n_vec, rotation,
                                                     centers, qjl, out, s);
    return launch_dequantize_parts<BITS, QJL, 1>(codes, norms, signs, rnorms, tokens, cap, n_vec, rotation, centers,
                                                 qjl, out, s);
}

template <bool QJL>
int launch_dequantize(const uint8_t* codes, const uint16_t* norms, const uint8_t* signs, const uint16_t* rnorms,
                      int64_t groups, int64_t tokens, int64_t cap, int dim, int bits, const float* rotation,
                      const float* centers, const float* qjl, uint16_t* out, void* stream) {
    if (!codes || !norms || !rotation || !centers || !out || groups < 0 || tokens < 0 || tokens > cap)
        return TQ_ERR_INVALID_ARGUMENT;
    if (QJL && (!signs || !rnorms || !qjl)) return TQ_ERR_INVALID_ARGUMENT;
    if (dim != TQ_DIM) return TQ_ERR_UNSUPPORTED;
    if (!aligned16(codes) || !aligned16(out) || (QJL && !aligned16(signs))) return TQ_ERR_UNSUPPORTED;
    if (bits < 1 || bits > 4) return TQ_ERR_INVALID_ARGUMENT;
    const int64_t n_vec = groups * tokens;
    if (n_vec == 0) return TQ_OK;
    if (n_vec >= ((int64_t)1 << 31)) return TQ_ERR_UNSUPPORTED;
    auto run = [&](auto b) {
        return run_dequantize<decltype(b)::value, QJL>(codes, norms, signs, rnorms, tokens, cap, n_vec, rotation,
                                                        centers, qjl, out, static_cast<hipStream_t>(stream));
    };
    switch (bits) {
        case 1: return run(std::integral_constant<int, 1>{});
        case 2: return run(std::integral_constant<int, 2>{});
        case 3: return run(std::integral_constant<int, 3>{});
        default: return run(std::integral_constant<int, 4>{});
    }
}

}  // namespace

extern "C" int tq_dequantize_mse(const uint8_t* codes, const uint16_t* norms, int64_t groups, int64_t tokens,
                                 int64_t cap, int dim, int bits, const float* rotation, const float* centers,
                                 uint16_t* out, void* stream) {
    return launch_dequantize<false>(codes, norms, nullptr, nullptr, groups, tokens, cap, dim, bits, rotation,
                                    centers, nullptr, out, stream);
}

extern "C" int tq_dequantize_prod(const uint8_t* codes, const uint16_t* norms, const uint8_t* signs,
                                  const uint16_t* rnorms, int64_t groups, int64_t tokens, int64_t cap, int dim,
                                  int mse_bits, const float* rotation, const float* centers, const float* qjl,
                                  uint16_t* out, void* stream) {
    if (mse_bits > 3) return TQ_ERR_INVALID_ARGUMENT;
    return launch_dequantize<true>(codes, norms, signs, rnorms, groups, tokens, cap, dim, mse_bits, rotation,
                                   centers, qjl, out, stream);
}
