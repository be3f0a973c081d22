/*
 * quant_matmul.hip -- the projections beside the attention path on gfx950:
 * Q8_K quantization of activations and the Q4_K x Q8_K matrix-vector /
 * small-batch product (`wo` after attention, fused Q/K/V before it).
 *
 * Formats are the reference's packed GGUF blocks
 * (tools/lfm2_cpuid_quants.c:76-127):
 *   block_q4_K, 144 B: fp16 d, fp16 dmin, scales[12], qs[128].  Sub-block j
 *     (32 weights) has a 6-bit scale and min packed in scales[]; its weights
 *     are the low (even j) or high (odd j) nibbles of qs[32*(j/2) .. +32]:
 *     w = d*sc*q - dmin*m.
 *   block_q8_K, 292 B: float d, int8 qs[256], int16 bsums[16] (sums of 16
 *     consecutive qs): x = d*q.
 *
 * Arithmetic follows the reference exactly where it is exact, and in its
 * order where it rounds:
 *   quantize  d = max|x| / 127, iscale = 127 / max|x| (correctly rounded),
 *             q = round-half-even(x * iscale), bsums of the unsaturated q
 *             (lfm2_quantize_row_q8_K_avx2_cpuid, tools/lfm2_cpuid_quants.c:585-635);
 *   dot       per super-block the integer sums sum(sc*q4*q8) and
 *             sum(m*bsum) (exact), then sumf += (d*d8)*dot - (dmin*d8)*mins
 *             with every product and sum rounded separately, super-blocks in
 *             order (lfm2_vec_dot_q4_K_q8_K_avx2, include/lfm2_simd_avx2.h:364-412).
 * So results are bit-identical to that reference kernel.
 *
 * Up to four tokens (k_matmul_q): one wave per RPW consecutive rows; the 8
 * lanes of a lane group take the 8 16-byte parts of one super-block's qs
 * (part p holds 16 weights of sub-block 2*(p/2) in its low nibbles and 16 of
 * sub-block 2*(p/2)+1 in its high nibbles), so a wave covers 8 super-blocks
 * (2048 columns) per step, reading each weight byte once.  Integer dots use
 * v_dot4_i32_i8; the lane groups' sums meet by shuffles.  The product is
 * HBM-bound on the weights (4.5 bits per weight).  More tokens take the matrix
 * pipe (k_matmul_mfma), with the same arithmetic: 2048 columns, us per call
 * before -> after (where the earlier kernels ran dot4, or one 16 x 16 MFMA
 * tile per workgroup):
 *            64 tokens x 2048 rows   2000 tokens x 2048 rows
 *   Q4_K             8.2 -> 6.5            143.0 -> 32.1
 *   Q5_K             8.7 -> 7.3            156.3 -> 34.7
 *   Q6_K            35.6 -> 8.4            916.6 -> 39.8
 *   IQ4_XS          25.6 -> 7.2            611.7 -> 31.8
 *   Q4_0            31.8 -> 6.8            814.5 -> 44.3
 *   Q8_0            32.0 -> 7.3            816.3 -> 37.5
 */
#include <hip/hip_runtime.h>

#include <type_traits>

#include "kernels.h"
#include "lfm_attn.h"

namespace lfm {
namespace {

constexpr uint32_t kQ8K = 292u;
constexpr uint32_t kCus = 256u; /* compute units of an MI355X: sizes of a round of workgroups */

__device__ __forceinline__ uint32_t ld32(const uint8_t *p) { return *reinterpret_cast<const uint32_t *>(p); }

/* ---- Q8_K quantization: one wave per 256-value block ----------------------- */
__global__ __launch_bounds__(256) void k_quant_q8K(const float *__restrict__ x, uint8_t *__restrict__ y,
                                                   uint32_t n_blocks, uint32_t nb) {
    const uint32_t lane = threadIdx.x & 63u;
    const uint32_t blk  = blockIdx.x * 4u + (threadIdx.x >> 6);
    if (blk >= n_blocks) return;
    const uint32_t t = blk / nb, b = blk - t * nb;
    const float *xb = x + ((size_t)t * nb + b) * 256u + 4u * lane;
    const float v[4] = {xb[0], xb[1], xb[2], xb[3]};
    float amax = fmaxf(fmaxf(fabsf(v[0]), fabsf(v[1])), fmaxf(fabsf(v[2]), fabsf(v[3])));
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) amax = fmaxf(amax, __shfl_xor(amax, o));
    uint8_t *out = y + (size_t)blk * kQ8K;
    if (amax == 0.0f) {
        *reinterpret_cast<uint32_t *>(out + 4u + 4u * lane) = 0u;
        if (lane < 16u) *reinterpret_cast<int16_t *>(out + 260u + 2u * lane) = 0;
        if (lane == 0u) *reinterpret_cast<float *>(out) = 0.0f;
        return;
    }
    const float d      = amax / 127.0f;  /* correctly rounded (HIP default) */
    const float iscale = 127.0f / amax;
    int32_t q[4], part = 0;
    uint32_t packed = 0;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        q[i] = (int32_t)__builtin_rintf(v[i] * iscale); /* one rounding, then half-even */
        part += q[i];
        const int32_t s = q[i] > 127 ? 127 : (q[i] < -128 ? -128 : q[i]);
        packed |= (uint32_t)(uint8_t)(int8_t)s << (8 * i);
    }
    *reinterpret_cast<uint32_t *>(out + 4u + 4u * lane) = packed;
    part += __shfl_xor(part, 1);
    part += __shfl_xor(part, 2);
    if ((lane & 3u) == 0u) *reinterpret_cast<int16_t *>(out + 260u + (lane >> 1)) = (int16_t)part;
    if (lane == 0u) *reinterpret_cast<float *>(out) = d;
}

/* 6-bit scale and min of sub-block j (get_scale_min_k4,
 * tools/lfm2_cpuid_quants.c:180-189) from the 12 scale bytes held as the
 * words y (bytes 0-3), z (4-7) and w (8-11) of the block header.  Bytes are
 * picked by shifts, so a lane-dependent j needs no byte array in scratch. */
__device__ __forceinline__ void scale_min(uint32_t j, uint32_t y, uint32_t z, uint32_t w, int32_t *sc, int32_t *m) {
    const uint32_t sh = 8u * (j & 3u);
    const uint32_t b0 = (y >> sh) & 0xFFu, b4 = (z >> sh) & 0xFFu, b8 = (w >> sh) & 0xFFu;
    if (j < 4u) {
        *sc = (int32_t)(b0 & 63u);
        *m  = (int32_t)(b4 & 63u);
    } else {
        *sc = (int32_t)((b8 & 0x0Fu) | ((b0 >> 6) << 4));
        *m  = (int32_t)((b8 >> 4) | ((b4 >> 6) << 4));
    }
}

__device__ __forceinline__ float fp16_bits(uint32_t h) { return (float)__builtin_bit_cast(_Float16, (uint16_t)h); }

__device__ __forceinline__ float add_rounded(float a, float b) {
#pragma clang fp contract(off)
    return a + b;
}

__device__ __forceinline__ float mul_rounded(float a, float b) {
#pragma clang fp contract(off)
    return a * b;
}

__device__ __forceinline__ int32_t dot4(uint32_t a, uint32_t b, int32_t c) {
    return __builtin_amdgcn_sdot4((int)a, (int)b, c, false);
}

/* 4 bytes from a 2-byte aligned address */
__device__ __forceinline__ uint32_t ld16x2(const uint8_t *p) {
    const uint16_t *h = reinterpret_cast<const uint16_t *>(p);
    return (uint32_t)h[0] | ((uint32_t)h[1] << 16);
}

/* Per weight type: what lane p (0..7) of a super-block's lane group loads and
 * computes.  Both give two exact integer partials (a, b) that sum over the
 * 8 lanes, and the super-block's fp32 term in the reference's rounding order. */
template <int TYPE> struct QType;

/* Integer-partial types (Q4_K, Q5_K, Q6_K, IQ4_XS) combine their exact lane
 * sums in one fp32 term per super-block; the 32-weight block types (Q4_0,
 * Q8_0) give a float per lane (one block each) that the reference sums in
 * block order before scaling by d8 (kFloatParts). */
/* Q4_K: part p = qs bytes 16p..16p+15: 16 weights of sub-block 2*(p/2) (low
 * nibbles) and of sub-block 2*(p/2)+1 (high nibbles); a = sum(sc*q4*q8),
 * b = sum(m*bsum); term = (d*d8)*a - (dmin*d8)*b
 * (include/lfm2_simd_avx2.h:364-412). */
template <> struct QType<12> {
    static constexpr uint32_t kBytes = 144u;
    static constexpr bool kFloatParts = false;
    struct W { uint32_t q[4]; int32_t sc1, m1, sc2, m2; float d, dmin; };
    struct X { float d8; uint32_t lo[4], hi[4]; int32_t bl, bh; };
    static __device__ __forceinline__ void load_w(W &w, const uint8_t *blk, uint32_t p) {
        const uint4 hdr = *reinterpret_cast<const uint4 *>(blk);
        const uint4 qs  = *reinterpret_cast<const uint4 *>(blk + 16u + 16u * p);
        w.q[0] = qs.x;
        w.q[1] = qs.y;
        w.q[2] = qs.z;
        w.q[3] = qs.w;
        scale_min(2u * (p >> 1), hdr.y, hdr.z, hdr.w, &w.sc1, &w.m1);
        scale_min(2u * (p >> 1) + 1u, hdr.y, hdr.z, hdr.w, &w.sc2, &w.m2);
        w.d    = fp16_bits(hdr.x & 0xFFFFu);
        w.dmin = fp16_bits(hdr.x >> 16);
    }
    static __device__ __forceinline__ void load_x(X &x, const uint8_t *xb, uint32_t p) {
        const uint32_t jp = p >> 1, h = p & 1u;
        const uint32_t qlo = 4u + 64u * jp + 16u * h, qhi = qlo + 32u;
        x.d8 = *reinterpret_cast<const float *>(xb);
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            x.lo[i] = ld32(xb + qlo + 4u * i);
            x.hi[i] = ld32(xb + qhi + 4u * i);
        }
        x.bl = *reinterpret_cast<const int16_t *>(xb + 260u + 2u * (4u * jp + h));
        x.bh = *reinterpret_cast<const int16_t *>(xb + 260u + 2u * (4u * jp + 2u + h));
    }
    static __device__ __forceinline__ void partials(const W &w, const X &x, uint32_t, int32_t &a, int32_t &b) {
        int32_t lo = 0, hi = 0;
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            lo = dot4(w.q[i] & 0x0F0F0F0Fu, x.lo[i], lo);
            hi = dot4((w.q[i] >> 4) & 0x0F0F0F0Fu, x.hi[i], hi);
        }
        a = w.sc1 * lo + w.sc2 * hi;
        b = w.m1 * x.bl + w.m2 * x.bh;
    }
    static __device__ __forceinline__ float term(const W &w, float d8, int32_t a, int32_t b) {
#pragma clang fp contract(off)
        const float dd = w.d * d8, dm = w.dmin * d8;
        return dd * (float)a - dm * (float)b;
    }
};

/* Q6_K (ql[128], qh[64], int8 scales[16], fp16 d; 210 bytes, so blocks are
 * only 2-byte aligned): part p = half p/4, columns l in 8(p%4)..+8 of the
 * half's four 32-groups; a = sum(sc*u*q8), b = sc[2p]*bsum[2p] +
 * sc[2p+1]*bsum[2p+1]; term = (d*d8) * (float)(a - 32*b)
 * (include/lfm2_simd_avx2.h:551-634). */
template <> struct QType<14> {
    static constexpr uint32_t kBytes = 210u;
    static constexpr bool kFloatParts = false;
    struct W { uint32_t l0[2], l1[2], qh[2]; int32_t s[4], so0, so1; float d; };
    struct X { float d8; uint32_t x[4][2]; int32_t b0, b1; };
    static __device__ __forceinline__ void load_w(W &w, const uint8_t *blk, uint32_t p) {
        const uint32_t half = p >> 2, q = p & 3u;
        const uint8_t *ql = blk + 64u * half + 8u * q, *qh = blk + 128u + 32u * half + 8u * q;
#pragma unroll
        for (int i = 0; i < 2; ++i) {
            w.l0[i] = ld16x2(ql + 4u * i);
            w.l1[i] = ld16x2(ql + 32u + 4u * i);
            w.qh[i] = ld16x2(qh + 4u * i);
        }
        const int8_t *sc = reinterpret_cast<const int8_t *>(blk + 192u + 8u * half + (q >> 1));
        w.s[0] = sc[0];
        w.s[1] = sc[2];
        w.s[2] = sc[4];
        w.s[3] = sc[6];
        const int8_t *so = reinterpret_cast<const int8_t *>(blk + 192u + 2u * p);
        w.so0 = so[0];
        w.so1 = so[1];
        w.d   = fp16_bits(*reinterpret_cast<const uint16_t *>(blk + 208u));
    }
    static __device__ __forceinline__ void load_x(X &x, const uint8_t *xb, uint32_t p) {
        const uint32_t half = p >> 2, q = p & 3u;
        x.d8 = *reinterpret_cast<const float *>(xb);
#pragma unroll
        for (int k = 0; k < 4; ++k) {
            const uint8_t *g = xb + 4u + 128u * half + 32u * k + 8u * q;
            x.x[k][0] = ld32(g);
            x.x[k][1] = ld32(g + 4u);
        }
        const uint32_t bs = ld32(xb + 260u + 4u * p); /* bsums 2p, 2p+1 */
        x.b0 = (int16_t)(bs & 0xFFFFu);
        x.b1 = (int16_t)(bs >> 16);
    }
    static __device__ __forceinline__ void partials(const W &w, const X &x, uint32_t, int32_t &a, int32_t &b) {
        int32_t acc = 0;
#pragma unroll
        for (int i = 0; i < 2; ++i) {
            const uint32_t u1 = (w.l0[i] & 0x0F0F0F0Fu) | ((w.qh[i] & 0x03030303u) << 4);
            const uint32_t u2 = (w.l1[i] & 0x0F0F0F0Fu) | ((w.qh[i] & 0x0C0C0C0Cu) << 2);
            const uint32_t u3 = ((w.l0[i] >> 4) & 0x0F0F0F0Fu) | (w.qh[i] & 0x30303030u);
            const uint32_t u4 = ((w.l1[i] >> 4) & 0x0F0F0F0Fu) | ((w.qh[i] >> 2) & 0x30303030u);
            acc += w.s[0] * dot4(u1, x.x[0][i], 0) + w.s[1] * dot4(u2, x.x[1][i], 0) +
                   w.s[2] * dot4(u3, x.x[2][i], 0) + w.s[3] * dot4(u4, x.x[3][i], 0);
        }
        a = acc;
        b = w.so0 * x.b0 + w.so1 * x.b1;
    }
    static __device__ __forceinline__ float term(const W &w, float d8, int32_t a, int32_t b) {
#pragma clang fp contract(off)
        const float dd = w.d * d8;
        return dd * (float)(a - 32 * b);
    }
};

/* Q5_K (fp16 d, fp16 dmin, scales[12] as Q4_K, qh[32], qs[128]; 176 bytes):
 * part p = qs bytes 16p..16p+15 of 64-chunk c = p/2 with qh bytes
 * 16(p%2)..+15: low nibbles + 16 * qh bit 2c are sub-block 2c, high nibbles
 * + 16 * bit 2c+1 sub-block 2c+1; a, b and the term as Q4_K
 * (lfm2_vec_dot_q5_K_q8_K_avx2, tools/lfm2_cpuid_quants.c:690-740). */
template <> struct QType<13> {
    static constexpr uint32_t kBytes = 176u;
    static constexpr bool kFloatParts = false;
    using X = QType<12>::X;
    struct W { uint32_t lo[4], hi[4]; int32_t sc1, m1, sc2, m2; float d, dmin; };
    static __device__ __forceinline__ void load_w(W &w, const uint8_t *blk, uint32_t p) {
        const uint4 hdr = *reinterpret_cast<const uint4 *>(blk);
        const uint4 qs  = *reinterpret_cast<const uint4 *>(blk + 48u + 16u * p);
        const uint4 qh  = *reinterpret_cast<const uint4 *>(blk + 16u + 16u * (p & 1u));
        const uint32_t c = p >> 1;
        const uint32_t q[4] = {qs.x, qs.y, qs.z, qs.w}, h[4] = {qh.x, qh.y, qh.z, qh.w};
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            w.lo[i] = (q[i] & 0x0F0F0F0Fu) | (((h[i] >> (2u * c)) & 0x01010101u) << 4);
            w.hi[i] = ((q[i] >> 4) & 0x0F0F0F0Fu) | (((h[i] >> (2u * c + 1u)) & 0x01010101u) << 4);
        }
        scale_min(2u * c, hdr.y, hdr.z, hdr.w, &w.sc1, &w.m1);
        scale_min(2u * c + 1u, hdr.y, hdr.z, hdr.w, &w.sc2, &w.m2);
        w.d    = fp16_bits(hdr.x & 0xFFFFu);
        w.dmin = fp16_bits(hdr.x >> 16);
    }
    static __device__ __forceinline__ void load_x(X &x, const uint8_t *xb, uint32_t p) { QType<12>::load_x(x, xb, p); }
    static __device__ __forceinline__ void partials(const W &w, const X &x, uint32_t, int32_t &a, int32_t &b) {
        int32_t lo = 0, hi = 0;
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            lo = dot4(w.lo[i], x.lo[i], lo);
            hi = dot4(w.hi[i], x.hi[i], hi);
        }
        a = w.sc1 * lo + w.sc2 * hi;
        b = w.m1 * x.bl + w.m2 * x.bh;
    }
    static __device__ __forceinline__ float term(const W &w, float d8, int32_t a, int32_t b) {
#pragma clang fp contract(off)
        const float dd = w.d * d8, dm = w.dmin * d8;
        return dd * (float)a - dm * (float)b;
    }
};

/* IQ4_XS (fp16 d, scales_h, scales_l[4], qs[128]; 136 bytes): part p =
 * sub-block p, qs bytes 16p..16p+15 (low nibbles elements 0..15, high
 * 16..31) mapped through the IQ4_NL grid with v_perm_b32; a = ls * dot, b = 0;
 * term = (d*d8) * a (lfm2_vec_dot_iq4_xs_q8_K_avx2, tools/lfm2_cpuid_quants.c:832-880). */
template <> struct QType<23> {
    static constexpr uint32_t kBytes = 136u;
    static constexpr bool kFloatParts = false;
    struct W { uint32_t lo[4], hi[4]; int32_t ls; float d; };
    struct X { float d8; uint32_t lo[4], hi[4]; };
    /* the 16 grid values as int8 bytes, four per dword */
    static constexpr uint32_t kG0 = 0xBFAD9881u, kG1 = 0xF6EADDCFu, kG2 = 0x26190D01u, kG3 = 0x71594535u;
    static __device__ __forceinline__ uint32_t grid4(uint32_t nib) { /* 4 nibbles (one per byte) */
        const uint32_t sel = nib & 0x07070707u;
        const uint32_t lo  = __builtin_amdgcn_perm(kG1, kG0, sel);
        const uint32_t hi  = __builtin_amdgcn_perm(kG3, kG2, sel);
        const uint32_t m   = ((nib >> 3) & 0x01010101u) * 0xFFu;
        return (lo & ~m) | (hi & m);
    }
    static __device__ __forceinline__ void load_w(W &w, const uint8_t *blk, uint32_t p) {
        const uint2 hdr = *reinterpret_cast<const uint2 *>(blk);
        const uint2 q0  = *reinterpret_cast<const uint2 *>(blk + 8u + 16u * p);
        const uint2 q1  = *reinterpret_cast<const uint2 *>(blk + 16u + 16u * p);
        const uint32_t q[4] = {q0.x, q0.y, q1.x, q1.y};
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            w.lo[i] = grid4(q[i] & 0x0F0F0F0Fu);
            w.hi[i] = grid4((q[i] >> 4) & 0x0F0F0F0Fu);
        }
        const uint32_t sh = hdr.x >> 16, sl = hdr.y;
        w.ls = (int32_t)(((sl >> (8u * (p >> 1) + 4u * (p & 1u))) & 0x0Fu) | (((sh >> (2u * p)) & 3u) << 4)) - 32;
        w.d  = fp16_bits(hdr.x & 0xFFFFu);
    }
    static __device__ __forceinline__ void load_x(X &x, const uint8_t *xb, uint32_t p) {
        x.d8 = *reinterpret_cast<const float *>(xb);
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            x.lo[i] = ld32(xb + 4u + 32u * p + 4u * i);
            x.hi[i] = ld32(xb + 20u + 32u * p + 4u * i);
        }
    }
    static __device__ __forceinline__ void partials(const W &w, const X &x, uint32_t, int32_t &a, int32_t &b) {
        int32_t acc = 0;
#pragma unroll
        for (int i = 0; i < 4; ++i) acc = dot4(w.hi[i], x.hi[i], dot4(w.lo[i], x.lo[i], acc));
        a = w.ls * acc;
        b = 0;
    }
    static __device__ __forceinline__ float term(const W &w, float d8, int32_t a, int32_t) {
#pragma clang fp contract(off)
        const float dd = w.d * d8;
        return dd * (float)a;
    }
};

/* Q4_0 (fp16 d, qs[16]; 18 bytes per 32 weights, 2-byte aligned): part p =
 * block p of the super-block; its float d * (sum(u4*q8) - 8 * bsums) is
 * summed in block order (lfm2_vec_dot_q4_0_q8_K_avx2,
 * tools/lfm2_cpuid_quants.c:634-672). */
template <> struct QType<2> {
    static constexpr uint32_t kBytes = 144u; /* 8 blocks */
    static constexpr bool kFloatParts = true;
    struct W { uint32_t q[4]; float d; };
    struct X { float d8; uint32_t lo[4], hi[4]; int32_t s8; };
    static __device__ __forceinline__ void load_w(W &w, const uint8_t *blk, uint32_t p) {
        const uint8_t *b = blk + 18u * p;
        w.d = fp16_bits(*reinterpret_cast<const uint16_t *>(b));
#pragma unroll
        for (int i = 0; i < 4; ++i) w.q[i] = ld16x2(b + 2u + 4u * i);
    }
    static __device__ __forceinline__ void load_x(X &x, const uint8_t *xb, uint32_t p) {
        x.d8 = *reinterpret_cast<const float *>(xb);
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            x.lo[i] = ld32(xb + 4u + 32u * p + 4u * i);
            x.hi[i] = ld32(xb + 20u + 32u * p + 4u * i);
        }
        const uint32_t bs = ld32(xb + 260u + 4u * p);
        x.s8 = (int32_t)(int16_t)(bs & 0xFFFFu) + (int32_t)(int16_t)(bs >> 16);
    }
    static __device__ __forceinline__ float part_float(const W &w, const X &x) {
#pragma clang fp contract(off)
        int32_t acc = 0;
#pragma unroll
        for (int i = 0; i < 4; ++i) acc = dot4((w.q[i] >> 4) & 0x0F0F0F0Fu, x.hi[i], dot4(w.q[i] & 0x0F0F0F0Fu, x.lo[i], acc));
        return w.d * (float)(acc - 8 * x.s8);
    }
};

/* Q8_0 (fp16 d, int8 qs[32]; 34 bytes per 32 weights, 2-byte aligned): as
 * Q4_0 with d * sum(q*q8) (lfm2_vec_dot_q8_0_q8_K_avx2, include/lfm2_simd_avx2.h:639-674). */
template <> struct QType<8> {
    static constexpr uint32_t kBytes = 272u; /* 8 blocks */
    static constexpr bool kFloatParts = true;
    struct W { uint32_t q[8]; float d; };
    struct X { float d8; uint32_t v[8]; };
    static __device__ __forceinline__ void load_w(W &w, const uint8_t *blk, uint32_t p) {
        const uint8_t *b = blk + 34u * p;
        w.d = fp16_bits(*reinterpret_cast<const uint16_t *>(b));
#pragma unroll
        for (int i = 0; i < 8; ++i) w.q[i] = ld16x2(b + 2u + 4u * i);
    }
    static __device__ __forceinline__ void load_x(X &x, const uint8_t *xb, uint32_t p) {
        x.d8 = *reinterpret_cast<const float *>(xb);
#pragma unroll
        for (int i = 0; i < 8; ++i) x.v[i] = ld32(xb + 4u + 32u * p + 4u * i);
    }
    static __device__ __forceinline__ float part_float(const W &w, const X &x) {
#pragma clang fp contract(off)
        int32_t acc = 0;
#pragma unroll
        for (int i = 0; i < 8; ++i) acc = dot4(w.q[i], x.v[i], acc);
        return w.d * (float)acc;
    }
};

/* Up to four matrices over the same activations (Q, K, V, gate), each of its
 * own GGML type; waves [wave0[m], wave0[m+1]) cover matrix m, RPW rows each. */
struct MatSet {
    const uint8_t *w[4];
    float *out[4];
    uint32_t rows[4];
    uint32_t type[4];
    uint32_t wave0[5];
    uint32_t n;
};

/* ---- quantized weights x Q8_K: out[t][r] ----------------------------------------
 * RPW rows of one matrix and a chunk of TCH tokens per wave (grid y = token
 * chunks): per 8-super-block step a lane loads its part of the RPW rows'
 * weights and of the TCH tokens' activations in one batch, then forms the
 * RPW x TCH partials, sums them over its lane group, and adds the
 * super-blocks' terms to the row sums in order. */
template <int TYPE, int RPW, int TCH>
__device__ __forceinline__ void matmul_rows(const uint8_t *__restrict__ w, float *__restrict__ out, uint32_t n_rows,
                                            uint32_t r0, const uint8_t *__restrict__ xq, uint32_t nb,
                                            uint32_t n_tokens, uint32_t t0) {
    using Q = QType<TYPE>;
    const uint32_t lane = threadIdx.x & 63u;
    const uint32_t p = lane & 7u; /* part within the super-block    */
    const uint32_t g = lane >> 3; /* super-block slot of this step  */
    const size_t row_bytes = (size_t)nb * Q::kBytes;

    float sumf[TCH][RPW];
#pragma unroll
    for (int tt = 0; tt < TCH; ++tt)
#pragma unroll
        for (int r = 0; r < RPW; ++r) sumf[tt][r] = 0.0f;
    for (uint32_t b0 = 0; b0 < nb; b0 += 8u) {
        const uint32_t b = min(b0 + g, nb - 1u); /* slots past the end repeat a block, unused */
        typename Q::W wr[RPW];
#pragma unroll
        for (int r = 0; r < RPW; ++r) {
            const uint32_t row = min(r0 + (uint32_t)r, n_rows - 1u);
            Q::load_w(wr[r], w + row * row_bytes + (size_t)b * Q::kBytes, p);
        }
        typename Q::X xt[TCH];
#pragma unroll
        for (int tt = 0; tt < TCH; ++tt) {
            const uint32_t t = min(t0 + (uint32_t)tt, n_tokens - 1u);
            Q::load_x(xt[tt], xq + ((size_t)t * nb + b) * kQ8K, p);
        }
        float term[TCH][RPW];
#pragma unroll
        for (int r = 0; r < RPW; ++r)
#pragma unroll
            for (int tt = 0; tt < TCH; ++tt) {
                if constexpr (Q::kFloatParts) {
                    /* blocks of the super-block in order, then times d8 */
                    const float t  = Q::part_float(wr[r], xt[tt]);
                    const int base = (int)(lane & ~7u);
                    float bsum     = add_rounded(0.0f, __shfl(t, base));
#pragma unroll
                    for (int k = 1; k < 8; ++k) bsum = add_rounded(bsum, __shfl(t, base + k));
                    term[tt][r] = mul_rounded(xt[tt].d8, bsum);
                } else {
                    int32_t a, c;
                    Q::partials(wr[r], xt[tt], p, a, c);
#pragma unroll
                    for (int o = 1; o < 8; o <<= 1) {
                        a += __shfl_xor(a, o);
                        c += __shfl_xor(c, o);
                    }
                    term[tt][r] = Q::term(wr[r], xt[tt].d8, a, c);
                }
            }
        /* super-blocks b0 .. b0+7 in order; a block whose d8 is 0 adds nothing */
#pragma unroll
        for (uint32_t i = 0; i < 8u; ++i) {
            if (b0 + i >= nb) break;
#pragma unroll
            for (int tt = 0; tt < TCH; ++tt) {
                const float d8i = __shfl(xt[tt].d8, (int)(8u * i));
#pragma unroll
                for (int r = 0; r < RPW; ++r) {
                    const float ti = __shfl(term[tt][r], (int)(8u * i));
                    if (d8i != 0.0f) sumf[tt][r] = add_rounded(sumf[tt][r], ti);
                }
            }
        }
    }
    /* lane tt * RPW + r writes token t0 + tt, row r0 + r */
#pragma unroll
    for (int tt = 0; tt < TCH; ++tt)
#pragma unroll
        for (int r = 0; r < RPW; ++r)
            if (lane == (uint32_t)(tt * RPW + r) && t0 + tt < n_tokens && r0 + r < n_rows)
                out[(size_t)(t0 + tt) * n_rows + r0 + r] = sumf[tt][r];
}

/* one launch over every matrix of the set.  TYPE > 0: all matrices of that
 * type; TYPE == 0: each wave takes its matrix's type (a wave-uniform branch;
 * the kernel then needs the registers of the widest type, so sets of one
 * type take the specialised form) */
template <int TYPE, int RPW, int TCH>
__global__ __launch_bounds__(256) void k_matmul_q(const MatSet S, const uint8_t *__restrict__ xq, uint32_t nb,
                                                  uint32_t n_tokens) {
    const uint32_t wv = blockIdx.x * 4u + (threadIdx.x >> 6);
    if (wv >= S.wave0[S.n]) return;
    uint32_t m = 0;
    while (m + 1u < S.n && wv >= S.wave0[m + 1u]) ++m;
    const uint32_t r0 = (wv - S.wave0[m]) * RPW, t0 = blockIdx.y * TCH;
    if constexpr (TYPE != 0) {
        matmul_rows<TYPE, RPW, TCH>(S.w[m], S.out[m], S.rows[m], r0, xq, nb, n_tokens, t0);
        return;
    }
    switch (S.type[m]) {
    case 12u: matmul_rows<12, RPW, TCH>(S.w[m], S.out[m], S.rows[m], r0, xq, nb, n_tokens, t0); break;
    case 14u: matmul_rows<14, RPW, TCH>(S.w[m], S.out[m], S.rows[m], r0, xq, nb, n_tokens, t0); break;
    case 13u: matmul_rows<13, RPW, TCH>(S.w[m], S.out[m], S.rows[m], r0, xq, nb, n_tokens, t0); break;
    case 23u: matmul_rows<23, RPW, TCH>(S.w[m], S.out[m], S.rows[m], r0, xq, nb, n_tokens, t0); break;
    case 2u: matmul_rows<2, RPW, TCH>(S.w[m], S.out[m], S.rows[m], r0, xq, nb, n_tokens, t0); break;
    default: matmul_rows<8, RPW, TCH>(S.w[m], S.out[m], S.rows[m], r0, xq, nb, n_tokens, t0); break;
    }
}

template <int TYPE, int RPW, int TCH>
hipError_t launch_set(MatSet S, const void *x_q8, uint32_t nb, uint32_t n_tokens, hipStream_t stream) {
    S.wave0[0] = 0;
    for (uint32_t m = 0; m < S.n; ++m) S.wave0[m + 1] = S.wave0[m] + (S.rows[m] + RPW - 1u) / RPW;
    if (S.wave0[S.n] == 0u) return hipSuccess;
    hipLaunchKernelGGL((k_matmul_q<TYPE, RPW, TCH>), dim3((S.wave0[S.n] + 3u) / 4u, (n_tokens + TCH - 1u) / TCH),
                       dim3(256), 0, stream, S, static_cast<const uint8_t *>(x_q8), nb, n_tokens);
    return hipGetLastError();
}

/* one token: a row per wave (most waves in flight); two to four: two rows and
 * the tokens per wave share each weight and activation load */
template <int TYPE>
hipError_t launch_tokens(const MatSet &S, const void *x_q8, uint32_t nb, uint32_t n_tokens, hipStream_t stream) {
    if (n_tokens == 1u) return launch_set<TYPE, 1, 1>(S, x_q8, nb, n_tokens, stream);
    if (n_tokens == 2u) return launch_set<TYPE, 2, 2>(S, x_q8, nb, n_tokens, stream);
    return launch_set<TYPE, 2, 4>(S, x_q8, nb, n_tokens, stream);
}

/* ---- quantized weights x Q8_K on the matrix pipe -------------------------------
 * The integer sum of a super-block is one exact product of int8 matrices: its
 * scaled weights W = sc * q do not fit a byte, so they enter as two planes,
 * W = p0 + (p1 << kShift), each multiplied with the tokens' int8 activations by
 * v_mfma_i32_16x16x64_i8 (A = 16 tokens, B = 16 rows), and
 *   a[t][r] = acc0 + (acc1 << kShift)
 * is the reference's integer sum.  Sums over bsums (Q4_K and Q5_K mins, Q6_K
 * offsets) are one v_mfma_f32_16x16x32_f16 on each bsum's low byte and its
 * high byte times 256 (both exact in fp16): exact while the sum stays below
 * 2^24, which bsums of -2048..2047 keep (16 x 2048 x 128 = 2^22); no 16 int8
 * values sum to others, and a tile with such a bsum takes the dot4 kernel's
 * integer sums.  The 32-weight block types
 * (Q4_0, Q8_0) need their int sum per block, one v_mfma_i32_16x16x32_i8 each,
 * started from kMagic, whose bits read as a float are 1.5 * 2^23 + sum: then
 *   fma(d, that float, -d * 1.5 * 2^23) = d * sum, rounded once (d * 1.5 * 2^23
 * is exact), the conversion and product of the reference in one instruction.
 * The fp32 terms keep the reference's rounding order, so every element equals
 * the one-token dot4 kernel's bit for bit.
 *
 * K order ("pair" layout): lane slice g (lane >> 4) of a 64-weight chunk c
 * holds weights 8g..8g+7 of the chunk's first 32 and of its second 32, as one
 * 8-byte read of a nibble row gives them; activations are read in the same
 * order. */
typedef int32_t i32x4_t __attribute__((ext_vector_type(4)));
typedef float f32x4_t __attribute__((ext_vector_type(4)));
typedef _Float16 f16x8_t __attribute__((ext_vector_type(8)));
typedef uint16_t u16x2_t __attribute__((ext_vector_type(2)));
typedef uint32_t u32x4_t __attribute__((ext_vector_type(4)));
/* vector loads from addresses aligned to 2, 4 or 8 bytes only */
typedef uint32_t u32x4_a4 __attribute__((ext_vector_type(4), aligned(4)));
typedef uint32_t u32x4_a2 __attribute__((ext_vector_type(4), aligned(2)));

constexpr int32_t kMagic   = 0x4B400000; /* bits of 1.5 * 2^23 */
constexpr float kMagicF    = 12582912.0f;
constexpr uint32_t kLow4   = 0x0F0F0F0Fu;

__device__ __forceinline__ float sub_rounded(float a, float b) {
#pragma clang fp contract(off)
    return a - b;
}

__device__ __forceinline__ uint32_t pk_mul(uint32_t a, uint32_t b) {
    return __builtin_bit_cast(uint32_t, (u16x2_t)(__builtin_bit_cast(u16x2_t, a) * __builtin_bit_cast(u16x2_t, b)));
}
__device__ __forceinline__ uint32_t pk_add(uint32_t a, uint32_t b) {
    return __builtin_bit_cast(uint32_t, (u16x2_t)(__builtin_bit_cast(u16x2_t, a) + __builtin_bit_cast(u16x2_t, b)));
}
__device__ __forceinline__ uint32_t pk_mad(uint32_t a, uint32_t b, uint32_t c) {
    return __builtin_bit_cast(uint32_t, (u16x2_t)(__builtin_bit_cast(u16x2_t, a) * __builtin_bit_cast(u16x2_t, b) +
                                                  __builtin_bit_cast(u16x2_t, c)));
}
/* byte j of v in both 16-bit halves */
__device__ __forceinline__ uint32_t splat_byte(uint32_t v, uint32_t j) {
    return __builtin_amdgcn_perm(0u, v, 0x0C000C00u | j | (j << 16));
}
/* bytes 0 and 2 of even and odd, interleaved: weights 0, 1, 2, 3 */
__device__ __forceinline__ uint32_t weave(uint32_t even, uint32_t odd) {
    return __builtin_amdgcn_perm(odd, even, 0x06020400u);
}
__device__ __forceinline__ bool half_finite(uint32_t h) { return (h & 0x7C00u) != 0x7C00u; }

/* 6-bit scales and mins of the 8 sub-blocks (get_scale_min_k4), four per word */
struct ScaleMin {
    uint32_t sc03, sc47, m03, m47;
    __device__ __forceinline__ ScaleMin(uint32_t y, uint32_t z, uint32_t w)
        : sc03(y & 0x3F3F3F3Fu), sc47((w & kLow4) | ((y >> 2) & 0x30303030u)), m03(z & 0x3F3F3F3Fu),
          m47(((w >> 4) & kLow4) | ((z >> 2) & 0x30303030u)) {}
};
/* this lane's slice of the bsums product's B operand: slots 8g..8g+7 take the
 * mins of sub-blocks 4(g & 1)..+3, twice each */
__device__ __forceinline__ f16x8_t mins_half8(uint32_t m03, uint32_t m47, uint32_t g) {
    const uint32_t m = (g & 1u) ? m47 : m03;
    f16x8_t r;
#pragma unroll
    for (uint32_t j = 0; j < 4u; ++j) {
        const _Float16 v  = (_Float16)(uint16_t)((m >> (8u * j)) & 0xFFu);
        r[2u * j]         = v;
        r[2u * j + 1u]    = v;
    }
    return r;
}

/* ---- one super-block of ROWS weight rows and NTOK tokens through LDS -------------
 * The lanes of a fragment read 16 rows a row pitch apart, 8 bytes each: loaded
 * so from global memory, the address unit serves a cache line at a time and
 * bounds the product (Q8_0 2000 x 2048 tokens x rows: 93 us, its address unit
 * busy 72 % of the time).  So both operands move as runs of whole blocks, 16
 * consecutive bytes a lane, and are picked apart in LDS. */
template <int TYPE> struct WLayout; /* kPitch: LDS bytes per row, in an odd multiple of 8 or 16 bytes: no bank conflicts */
template <> struct WLayout<12> { static constexpr uint32_t kPitch = 144u, kPieces = 9u; };
template <> struct WLayout<13> { static constexpr uint32_t kPitch = 176u, kPieces = 11u; };
template <> struct WLayout<14> { static constexpr uint32_t kPitch = 208u, kPieces = 13u; }; /* d apart */
template <> struct WLayout<23> { static constexpr uint32_t kPitch = 136u, kPieces = 17u; }; /* 8-byte pieces */
template <> struct WLayout<2> { static constexpr uint32_t kPitch = 144u, kPieces = 8u; };   /* 16 quant bytes of a block; d apart */
template <> struct WLayout<8> { static constexpr uint32_t kPitch = 272u, kPieces = 8u; };   /* 32 */

template <int TYPE, uint32_t ROWS> struct WTile {
    static constexpr uint32_t kD = TYPE == 14 ? 1u : (TYPE == 2 || TYPE == 8) ? 8u : 0u; /* scales kept apart per row */
    uint8_t q[ROWS * WLayout<TYPE>::kPitch] __attribute__((aligned(16)));
    uint16_t d[kD ? ROWS * kD : 8u] __attribute__((aligned(16)));
};

/* ROWS rows from r0 (rows past the last repeat it) by THREADS threads: fetch
 * reads super-block b into registers, put writes the LDS image */
template <int TYPE, uint32_t ROWS, uint32_t THREADS> struct WStage {
    using L = WLayout<TYPE>;
    static constexpr uint32_t kTotal = ROWS * L::kPieces, N = (kTotal + THREADS - 1u) / THREADS;
    static constexpr uint32_t kBytes = QType<TYPE>::kBytes, kBlk = TYPE == 2 ? 18u : 34u;
    static constexpr bool kWhole = kTotal % THREADS == 0u;
    uint32_t off[N], at[N];
    u32x4_t v[N], v2[TYPE == 8 ? N : 1];
    uint32_t d[N], dq, dq_off;
    const uint8_t *base;
    uint32_t tid;

    __device__ __forceinline__ WStage(const uint8_t *w, uint32_t n_rows, uint32_t nb, uint32_t r0, uint32_t t)
        : dq(0u), dq_off(0u), base(w + (size_t)r0 * nb * kBytes), tid(t) {
        const uint32_t last = n_rows - 1u - r0, pitch = nb * kBytes;
#pragma unroll
        for (uint32_t i = 0; i < N; ++i) {
            const uint32_t e = kWhole ? t + THREADS * i : min(t + THREADS * i, kTotal - 1u);
            const uint32_t row = e / L::kPieces, p = e % L::kPieces;
            off[i] = min(row, last) * pitch + (TYPE == 23 ? 8u * p : TYPE == 2 || TYPE == 8 ? kBlk * p : 16u * p);
            at[i]  = row * L::kPitch + (TYPE == 23 ? 8u * p : TYPE == 8 ? 32u * p : 16u * p);
        }
        if constexpr (TYPE == 14) dq_off = min(t, last) * pitch + 208u;
    }
    __device__ __forceinline__ void fetch(uint32_t b) {
        const uint8_t *p = base + (size_t)b * kBytes;
#pragma unroll
        for (uint32_t i = 0; i < N; ++i) {
            if constexpr (TYPE == 12 || TYPE == 13) v[i] = *reinterpret_cast<const u32x4_t *>(p + off[i]);
            else if constexpr (TYPE == 23) {
                const uint2 x = *reinterpret_cast<const uint2 *>(p + off[i]);
                v[i][0] = x.x;
                v[i][1] = x.y;
            } else if constexpr (TYPE == 14) v[i] = *reinterpret_cast<const u32x4_a2 *>(p + off[i]);
            else {
                d[i] = *reinterpret_cast<const uint16_t *>(p + off[i]);
                v[i] = *reinterpret_cast<const u32x4_a2 *>(p + off[i] + 2u);
                if constexpr (TYPE == 8) v2[i] = *reinterpret_cast<const u32x4_a2 *>(p + off[i] + 18u);
            }
        }
        if constexpr (TYPE == 14)
            if (tid < ROWS) dq = *reinterpret_cast<const uint16_t *>(p + dq_off);
    }
    __device__ __forceinline__ void put(WTile<TYPE, ROWS> &W) const {
#pragma unroll
        for (uint32_t i = 0; i < N; ++i) {
            if (!kWhole && i == N - 1u && tid + THREADS * i >= kTotal) break;
            if constexpr (TYPE == 23) *reinterpret_cast<uint2 *>(W.q + at[i]) = make_uint2(v[i][0], v[i][1]);
            else *reinterpret_cast<u32x4_t *>(W.q + at[i]) = v[i];
            if constexpr (TYPE == 8) *reinterpret_cast<u32x4_t *>(W.q + at[i] + 16u) = v2[i];
            if constexpr (TYPE == 2 || TYPE == 8) W.d[tid + THREADS * i] = (uint16_t)d[i];
        }
        if constexpr (TYPE == 14)
            if (tid < ROWS) W.d[tid] = (uint16_t)dq;
    }
};

/* Per type: a lane's part (row, slice g) of the LDS image, and what it becomes.
 * p0, p1: the two planes of chunk c as MFMA operands. */
template <int TYPE> struct QPlane;

template <> struct QPlane<12> {
    static constexpr int kShift = 3; /* sc = 8 * s1 + s0, both <= 7: q * s <= 105 */
    struct Raw { u32x4_t hdr; uint2 q[4]; };
    struct Op { i32x4_t p0[4], p1[4]; f16x8_t mins; float d, dmin; bool finite; };
    static __device__ __forceinline__ void load(Raw &r, const uint8_t *blk, const uint16_t *, uint32_t g) {
        r.hdr = *reinterpret_cast<const u32x4_t *>(blk);
#pragma unroll
        for (uint32_t c = 0; c < 4u; ++c) r.q[c] = *reinterpret_cast<const uint2 *>(blk + 16u + 32u * c + 8u * g);
    }
    static __device__ __forceinline__ void prep(Op &o, const Raw &r, uint32_t g) {
        const ScaleMin s(r.hdr[1], r.hdr[2], r.hdr[3]);
        const uint32_t dig0[2] = {s.sc03 & 0x07070707u, s.sc47 & 0x07070707u};
        const uint32_t dig1[2] = {(s.sc03 >> 3) & 0x07070707u, (s.sc47 >> 3) & 0x07070707u};
#pragma unroll
        for (uint32_t c = 0; c < 4u; ++c) {
            const uint32_t b = 2u * (c & 1u);
            const uint32_t l0 = splat_byte(dig0[c >> 1], b), l1 = splat_byte(dig1[c >> 1], b);
            const uint32_t h0 = splat_byte(dig0[c >> 1], b + 1u), h1 = splat_byte(dig1[c >> 1], b + 1u);
            const uint32_t lx = r.q[c].x & kLow4, ly = r.q[c].y & kLow4;
            const uint32_t hx = (r.q[c].x >> 4) & kLow4, hy = (r.q[c].y >> 4) & kLow4;
            o.p0[c] = i32x4_t{(int)pk_mul(lx, l0), (int)pk_mul(ly, l0), (int)pk_mul(hx, h0), (int)pk_mul(hy, h0)};
            o.p1[c] = i32x4_t{(int)pk_mul(lx, l1), (int)pk_mul(ly, l1), (int)pk_mul(hx, h1), (int)pk_mul(hy, h1)};
        }
        o.mins   = mins_half8(s.m03, s.m47, g);
        o.d      = fp16_bits(r.hdr[0] & 0xFFFFu);
        o.dmin   = fp16_bits(r.hdr[0] >> 16);
        o.finite = half_finite(r.hdr[0]) && half_finite(r.hdr[0] >> 16);
    }
};

/* planes of 16-bit products We (weights 0, 2) and Wo (1, 3): W = p0 + 2^SH p1 */
template <int SH>
__device__ __forceinline__ void split_planes(uint32_t we, uint32_t wo, int32_t &p0, int32_t &p1) {
    constexpr uint32_t kMask = ((1u << SH) - 1u) * 0x01010101u;
    p0 = (int32_t)(weave(we, wo) & kMask);
    p1 = (int32_t)weave(we >> SH, wo >> SH);
}

template <> struct QPlane<13> {
    static constexpr int kShift = 4; /* sc * q <= 63 * 31 < 2^11 */
    struct Raw { u32x4_t hdr; uint2 qh; uint2 q[4]; };
    using Op = QPlane<12>::Op;
    static __device__ __forceinline__ void load(Raw &r, const uint8_t *blk, const uint16_t *, uint32_t g) {
        r.hdr = *reinterpret_cast<const u32x4_t *>(blk);
        r.qh  = *reinterpret_cast<const uint2 *>(blk + 16u + 8u * g);
#pragma unroll
        for (uint32_t c = 0; c < 4u; ++c) r.q[c] = *reinterpret_cast<const uint2 *>(blk + 48u + 32u * c + 8u * g);
    }
    static __device__ __forceinline__ void prep(Op &o, const Raw &r, uint32_t g) {
        const ScaleMin s(r.hdr[1], r.hdr[2], r.hdr[3]);
#pragma unroll
        for (uint32_t c = 0; c < 4u; ++c) {
            const uint32_t sc4 = c < 2u ? s.sc03 : s.sc47, b = 2u * (c & 1u);
            const uint32_t sc[2] = {splat_byte(sc4, b), splat_byte(sc4, b + 1u)};
            const uint32_t q[2] = {r.q[c].x, r.q[c].y}, h[2] = {r.qh.x, r.qh.y};
#pragma unroll
            for (uint32_t e = 0; e < 4u; ++e) { /* dwords lo.x, lo.y, hi.x, hi.y */
                const uint32_t hi = e >> 1;
                const uint32_t v = ((q[e & 1u] >> (4u * hi)) & kLow4) | (((h[e & 1u] >> (2u * c + hi)) & 0x01010101u) << 4);
                int32_t p0, p1;
                split_planes<kShift>(pk_mul(v & 0x00FF00FFu, sc[hi]), pk_mul((v >> 8) & 0x00FF00FFu, sc[hi]), p0, p1);
                o.p0[c][e] = p0;
                o.p1[c][e] = p1;
            }
        }
        o.mins   = mins_half8(s.m03, s.m47, g);
        o.d      = fp16_bits(r.hdr[0] & 0xFFFFu);
        o.dmin   = fp16_bits(r.hdr[0] >> 16);
        o.finite = half_finite(r.hdr[0]) && half_finite(r.hdr[0] >> 16);
    }
};

template <> struct QPlane<14> {
    static constexpr int kShift = 7; /* sc * u in [-128 * 63, 127 * 63]: 14 bits */
    struct Raw { uint2 ql[2][2], qh[2]; u32x4_t sc; uint32_t d; };
    struct Op { i32x4_t p0[4], p1[4]; f16x8_t mins; float d; bool finite; };
    static __device__ __forceinline__ void load(Raw &r, const uint8_t *blk, const uint16_t *d, uint32_t g) {
#pragma unroll
        for (uint32_t h = 0; h < 2u; ++h) {
            r.ql[h][0] = *reinterpret_cast<const uint2 *>(blk + 64u * h + 8u * g);
            r.ql[h][1] = *reinterpret_cast<const uint2 *>(blk + 64u * h + 32u + 8u * g);
            r.qh[h]    = *reinterpret_cast<const uint2 *>(blk + 128u + 32u * h + 8u * g);
        }
        r.sc = *reinterpret_cast<const u32x4_t *>(blk + 192u);
        r.d  = d[0];
    }
    static __device__ __forceinline__ void prep(Op &o, const Raw &r, uint32_t g) {
#pragma unroll
        for (uint32_t c = 0; c < 4u; ++c) { /* half h, 32-groups k = 2 kk and 2 kk + 1 */
            const uint32_t h = c >> 1, kk = c & 1u;
            const uint32_t s = r.sc[c] >> (8u * (g >> 1)); /* bytes 0 and 2: the lane's two 16-group scales */
            const int32_t sa = (int8_t)(s & 0xFFu), sb = (int8_t)((s >> 16) & 0xFFu);
            const uint32_t sc[2] = {((uint32_t)sa & 0xFFFFu) | ((uint32_t)sa << 16),
                                    ((uint32_t)sb & 0xFFFFu) | ((uint32_t)sb << 16)};
            const uint32_t qh[2] = {r.qh[h].x, r.qh[h].y};
#pragma unroll
            for (uint32_t e = 0; e < 4u; ++e) {
                const uint32_t odd = e >> 1, k = 2u * kk + odd;
                const uint32_t ql  = (e & 1u) ? r.ql[h][odd].y : r.ql[h][odd].x;
                const uint32_t u   = ((ql >> (4u * kk)) & kLow4) | (((qh[e & 1u] >> (2u * k)) & 0x03030303u) << 4);
                int32_t p0, p1;
                split_planes<kShift>(pk_mul(u & 0x00FF00FFu, sc[odd]), pk_mul((u >> 8) & 0x00FF00FFu, sc[odd]), p0, p1);
                o.p0[c][e] = p0;
                o.p1[c][e] = p1;
            }
        }
        /* minus the 16-group scales of bsums 8(g & 1)..+7 */
#pragma unroll
        for (uint32_t i = 0; i < 2u; ++i) {
            const uint32_t s = (g & 1u) ? r.sc[2u + i] : r.sc[i];
#pragma unroll
            for (uint32_t j = 0; j < 4u; ++j) o.mins[4u * i + j] = (_Float16)(int16_t)(-(int32_t)(int8_t)((s >> (8u * j)) & 0xFFu));
        }
        o.d      = fp16_bits(r.d);
        o.finite = half_finite(r.d);
    }
};

template <> struct QPlane<23> {
    static constexpr int kShift = 7; /* ls * grid in [-4064, 4064] */
    struct Raw { uint2 hdr; uint2 q[8]; };
    struct Op { i32x4_t p0[4], p1[4]; float d; bool finite; };
    /* the grid + 128 as unsigned bytes: ls * grid = ls * (grid + 128) - 128 ls */
    static __device__ __forceinline__ uint32_t grid4(uint32_t nib) {
        const uint32_t sel = nib & 0x07070707u;
        const uint32_t lo  = __builtin_amdgcn_perm(QType<23>::kG1 ^ 0x80808080u, QType<23>::kG0 ^ 0x80808080u, sel);
        const uint32_t hi  = __builtin_amdgcn_perm(QType<23>::kG3 ^ 0x80808080u, QType<23>::kG2 ^ 0x80808080u, sel);
        const uint32_t b   = (nib >> 3) & 0x01010101u;
        const uint32_t m   = (b << 8) - b;
        return (lo & ~m) | (hi & m);
    }
    static __device__ __forceinline__ void load(Raw &r, const uint8_t *blk, const uint16_t *, uint32_t g) {
        r.hdr = *reinterpret_cast<const uint2 *>(blk);
#pragma unroll
        for (uint32_t j = 0; j < 8u; ++j) r.q[j] = *reinterpret_cast<const uint2 *>(blk + 8u + 16u * j + 8u * (g & 1u));
    }
    static __device__ __forceinline__ void prep(Op &o, const Raw &r, uint32_t g) {
        const uint32_t sh = r.hdr.x >> 16, sl = r.hdr.y, nib = 4u * (g >> 1); /* elements 8g..: low nibbles for g < 2 */
#pragma unroll
        for (uint32_t j = 0; j < 8u; ++j) {
            const int32_t ls  = (int32_t)(((sl >> (4u * j)) & 0x0Fu) | (((sh >> (2u * j)) & 3u) << 4)) - 32;
            const uint32_t lp = ((uint32_t)ls & 0xFFFFu) | ((uint32_t)ls << 16);
            const int32_t off = -128 * ls;
            const uint32_t op = ((uint32_t)off & 0xFFFFu) | ((uint32_t)off << 16);
            const uint32_t q[2] = {r.q[j].x, r.q[j].y};
#pragma unroll
            for (uint32_t e = 0; e < 2u; ++e) {
                const uint32_t v = grid4((q[e] >> nib) & kLow4);
                int32_t p0, p1;
                split_planes<kShift>(pk_mad(v & 0x00FF00FFu, lp, op), pk_mad((v >> 8) & 0x00FF00FFu, lp, op), p0, p1);
                o.p0[j >> 1][2u * (j & 1u) + e] = p0;
                o.p1[j >> 1][2u * (j & 1u) + e] = p1;
            }
        }
        o.d      = fp16_bits(r.hdr.x & 0xFFFFu);
        o.finite = half_finite(r.hdr.x);
    }
};

/* Q4_0, Q8_0: p0[c] holds 8 weights of block 2c and 8 of block 2c + 1 */
struct BlockOp { i32x4_t p0[4]; float d[8]; bool finite; };
struct BlockRaw { uint2 q[8]; u32x4_t d; };
template <uint32_t BLK>
__device__ __forceinline__ void block_load(BlockRaw &r, const uint8_t *blk, const uint16_t *d, uint32_t at) {
    r.d = *reinterpret_cast<const u32x4_t *>(d);
#pragma unroll
    for (uint32_t j = 0; j < 8u; ++j) r.q[j] = *reinterpret_cast<const uint2 *>(blk + BLK * j + at);
}
template <int TYPE>
__device__ __forceinline__ void block_prep(BlockOp &o, const BlockRaw &r, uint32_t nib) {
    o.finite = true;
#pragma unroll
    for (uint32_t j = 0; j < 8u; ++j) {
        uint32_t x = r.q[j].x, y = r.q[j].y;
        if constexpr (TYPE == 2) {
            x = (x >> nib) & kLow4;
            y = (y >> nib) & kLow4;
        }
        o.p0[j >> 1][2u * (j & 1u)]      = (int)x;
        o.p0[j >> 1][2u * (j & 1u) + 1u] = (int)y;
        const uint32_t d = (r.d[j >> 1] >> (16u * (j & 1u))) & 0xFFFFu;
        o.d[j]   = fp16_bits(d);
        o.finite = o.finite && half_finite(d);
    }
}
template <> struct QPlane<2> {
    using Raw = BlockRaw;
    using Op  = BlockOp;
    static __device__ __forceinline__ void load(Raw &r, const uint8_t *blk, const uint16_t *d, uint32_t g) {
        block_load<16u>(r, blk, d, 8u * (g & 1u));
    }
    static __device__ __forceinline__ void prep(Op &o, const Raw &r, uint32_t g) { block_prep<2>(o, r, 4u * (g >> 1)); }
};
template <> struct QPlane<8> {
    using Raw = BlockRaw;
    using Op  = BlockOp;
    static __device__ __forceinline__ void load(Raw &r, const uint8_t *blk, const uint16_t *d, uint32_t g) {
        block_load<32u>(r, blk, d, 8u * g);
    }
    static __device__ __forceinline__ void prep(Op &o, const Raw &r, uint32_t) { block_prep<8>(o, r, 0u); }
};

template <int TYPE> constexpr bool kHasBsums = TYPE == 12 || TYPE == 13 || TYPE == 14;

/* A operands of one token (lane l16) and super-block: x[c] is slice g of chunk
 * c, bs slice g of the bsums product (slots 0..15 low bytes, 16..31 high bytes
 * times 256). */
struct XOp { i32x4_t x[4]; f16x8_t bs; };

/* NTOK tokens in LDS: 16-B slices (chunk c, slice g) of a token at 16 * ((4c +
 * g) ^ (token & 15)), so that a fragment read has no bank conflicts */
template <int TYPE, uint32_t NTOK> struct XTile {
    uint8_t x[NTOK * 256u] __attribute__((aligned(16)));
    f16x8_t bs[kHasBsums<TYPE> ? NTOK * 4u : 1u];
    float d8[NTOK] __attribute__((aligned(16)));
    int32_t cin[TYPE == 2 ? 8u * NTOK : 4u] __attribute__((aligned(16))); /* [block][token]: kMagic - 8 * bsums */

    __device__ __forceinline__ void read(XOp &o, uint32_t t0, uint32_t l16, uint32_t g) const {
        const uint8_t *p = x + (t0 + l16) * 256u + ((g ^ (l16 & 3u)) << 4);
#pragma unroll
        for (uint32_t c = 0; c < 4u; ++c) o.x[c] = *reinterpret_cast<const i32x4_t *>(p + 64u * (c ^ (l16 >> 2)));
        if constexpr (kHasBsums<TYPE>) o.bs = bs[(t0 + l16) * 4u + g];
    }
    __device__ __forceinline__ f32x4_t scales(uint32_t t0, uint32_t g) const {
        return *reinterpret_cast<const f32x4_t *>(&d8[t0 + 4u * g]);
    }
    __device__ __forceinline__ void inits(i32x4_t (&c)[8], uint32_t t0, uint32_t g) const {
        if constexpr (TYPE == 2)
#pragma unroll
            for (uint32_t k = 0; k < 8u; ++k) c[k] = *reinterpret_cast<const i32x4_t *>(&cin[k * NTOK + t0 + 4u * g]);
    }
};

/* tokens t0 .. t0 + NTOK - 1 (past the last they repeat it) by THREADS threads */
template <int TYPE, uint32_t NTOK, uint32_t THREADS> struct XStage {
    static constexpr uint32_t N = NTOK * 16u / THREADS, NB = kHasBsums<TYPE> ? (NTOK * 2u + THREADS - 1u) / THREADS : 0u;
    static constexpr uint32_t NC = TYPE == 2 ? NTOK * 8u / THREADS : 0u, kStep = THREADS / 16u;
    static_assert(NTOK <= THREADS && NTOK * 8u % THREADS == 0u && 16u % (kStep < 16u ? kStep : 16u) == 0u, "staging shape");
    u32x4_t v[N], bv[NB ? NB : 1];
    uint32_t cv[NC ? NC : 1], off[N], boff[NB ? NB : 1], coff[NC ? NC : 1], doff;
    float d;
    uint64_t wide = 0; /* lanes of this wave that staged a bsum outside -2048..2047 (in SGPRs: the registers are full) */
    const uint8_t *base;
    uint32_t tid;

    __device__ __forceinline__ XStage(const uint8_t *xq, uint32_t n_tokens, uint32_t nb, uint32_t t0, uint32_t t)
        : d(0.0f), base(xq + (size_t)t0 * nb * kQ8K), tid(t) {
        const uint32_t last = n_tokens - 1u - t0, pitch = nb * kQ8K;
#pragma unroll
        for (uint32_t i = 0; i < N; ++i) off[i] = min((t >> 4) + kStep * i, last) * pitch + 4u + 16u * (t & 15u);
#pragma unroll
        for (uint32_t i = 0; i < NB; ++i) boff[i] = min(min((t + THREADS * i) >> 1, NTOK - 1u), last) * pitch + 260u + 16u * (t & 1u);
#pragma unroll
        for (uint32_t i = 0; i < NC; ++i) coff[i] = min((t + THREADS * i) >> 3, last) * pitch + 260u + 4u * (t & 7u);
        doff = min(t, last) * pitch;
    }
    __device__ __forceinline__ void fetch(uint32_t b) {
        const uint8_t *p = base + (size_t)b * kQ8K;
#pragma unroll
        for (uint32_t i = 0; i < N; ++i) v[i] = *reinterpret_cast<const u32x4_a4 *>(p + off[i]);
#pragma unroll
        for (uint32_t i = 0; i < NB; ++i) bv[i] = *reinterpret_cast<const u32x4_a4 *>(p + boff[i]);
#pragma unroll
        for (uint32_t i = 0; i < NC; ++i) cv[i] = ld32(p + coff[i]);
        if (tid < NTOK) d = *reinterpret_cast<const float *>(p + doff);
    }
    __device__ __forceinline__ void put(XTile<TYPE, NTOK> &X) const {
        /* 16-B piece sp: slices 2(sp & 1) and +1 of chunk sp >> 2, half (sp >> 1) & 1 */
        const uint32_t sp = tid & 15u, c4 = 4u * (sp >> 2) + 2u * (sp & 1u), half = 8u * ((sp >> 1) & 1u);
#pragma unroll
        for (uint32_t i = 0; i < N; ++i) {
            const uint32_t tk = (tid >> 4) + kStep * i;
            uint8_t *row = X.x + tk * 256u + half;
            *reinterpret_cast<uint2 *>(row + ((c4 ^ (tk & 15u)) << 4))        = make_uint2(v[i][0], v[i][1]);
            *reinterpret_cast<uint2 *>(row + (((c4 + 1u) ^ (tk & 15u)) << 4)) = make_uint2(v[i][2], v[i][3]);
        }
#pragma unroll
        for (uint32_t i = 0; i < NB; ++i) {
            const uint32_t e = tid + THREADS * i;
            if (NTOK * 2u % THREADS == 0u || e < NTOK * 2u) {
                f16x8_t lo, hi; /* 8 bsums: low bytes, and high bytes times 256 */
#pragma unroll
                for (uint32_t j = 0; j < 8u; ++j) {
                    const int32_t s = (int16_t)((bv[i][j >> 1] >> (16u * (j & 1u))) & 0xFFFFu);
                    lo[j] = (_Float16)(int16_t)(s & 0xFF);
                    hi[j] = (_Float16)(int16_t)(s & ~0xFF);
                }
                X.bs[(e >> 1) * 4u + (e & 1u)]      = lo;
                X.bs[(e >> 1) * 4u + 2u + (e & 1u)] = hi;
            }
        }
#pragma unroll
        for (uint32_t i = 0; i < NC; ++i) {
            const uint32_t e = tid + THREADS * i;
            X.cin[(e & 7u) * NTOK + (e >> 3)] =
                kMagic - 8 * ((int32_t)(int16_t)(cv[i] & 0xFFFFu) + (int32_t)(int16_t)(cv[i] >> 16));
        }
        if (tid < NTOK) X.d8[tid] = d;
    }
    /* the bsums just staged (not between put and the barrier, where the other
     * waves would wait for it too) */
    __device__ __forceinline__ void check() {
#pragma unroll
        for (uint32_t i = 0; i < NB; ++i) {
            uint32_t m = 0; /* bits 12..15 of each half of bsum + 2048: outside the range */
#pragma unroll
            for (uint32_t j = 0; j < 4u; ++j) m |= pk_add(bv[i][j], 0x08000800u);
            wide |= __builtin_amdgcn_ballot_w64((m & 0xF000F000u) != 0u);
        }
    }
};

/* Integer sums of a 16 x 16 tile and super-block: lane (l16, g) holds tokens
 * 4g..4g+3 of row l16.  cin (Q4_0): kMagic - 8 * bsums of each block for the
 * four tokens. */
template <int TYPE> struct TileAcc { i32x4_t a0, a1; f32x4_t bm; };
template <> struct TileAcc<2> { i32x4_t v[8]; };
template <> struct TileAcc<8> { i32x4_t v[8]; };

template <int TYPE>
__device__ __forceinline__ void tile_sums(TileAcc<TYPE> &s, const typename QPlane<TYPE>::Op &o, const XOp &x,
                                          const i32x4_t *cin, i32x4_t magic) {
    if constexpr (QType<TYPE>::kFloatParts) {
#pragma unroll
        for (int k = 0; k < 8; ++k) {
            const int c = k >> 1, e = 2 * (k & 1);
            const long a = (long)(((uint64_t)(uint32_t)x.x[c][e + 1] << 32) | (uint32_t)x.x[c][e]);
            const long b = (long)(((uint64_t)(uint32_t)o.p0[c][e + 1] << 32) | (uint32_t)o.p0[c][e]);
            s.v[k] = __builtin_amdgcn_mfma_i32_16x16x32_i8(a, b, TYPE == 2 ? cin[k] : magic, 0, 0, 0);
        }
    } else {
        s.a0 = (i32x4_t)0;
        s.a1 = (i32x4_t)0;
#pragma unroll
        for (int c = 0; c < 4; ++c) {
            s.a0 = __builtin_amdgcn_mfma_i32_16x16x64_i8(x.x[c], o.p0[c], s.a0, 0, 0, 0);
            s.a1 = __builtin_amdgcn_mfma_i32_16x16x64_i8(x.x[c], o.p1[c], s.a1, 0, 0, 0);
        }
        if constexpr (kHasBsums<TYPE>) s.bm = __builtin_amdgcn_mfma_f32_16x16x32_f16(x.bs, o.mins, (f32x4_t)0.0f, 0, 0, 0);
    }
}

/* their fp32 terms; d8: the four tokens' scales */
template <int TYPE>
__device__ __forceinline__ f32x4_t tile_terms(const TileAcc<TYPE> &s, const typename QPlane<TYPE>::Op &o, f32x4_t d8) {
    f32x4_t term;
    if constexpr (QType<TYPE>::kFloatParts) {
        f32x4_t sum;
#pragma unroll
        for (int k = 0; k < 8; ++k) {
            const float off = -(o.d[k] * kMagicF);
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                const int32_t vi = s.v[k][i]; /* a bit cast of the element itself reads element 0 */
                const float t    = __builtin_fmaf(o.d[k], __builtin_bit_cast(float, vi), off);
                sum[i]           = k == 0 ? t : add_rounded(sum[i], t);
            }
        }
#pragma unroll
        for (int i = 0; i < 4; ++i) term[i] = mul_rounded(d8[i], sum[i]);
    } else {
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            int32_t a = s.a0[i] + (int32_t)((uint32_t)s.a1[i] << QPlane<TYPE>::kShift);
            if constexpr (TYPE == 14) a += 32 * (int32_t)s.bm[i]; /* - 32 * bsums (bm holds their negative) */
            term[i] = mul_rounded(mul_rounded(o.d, d8[i]), (float)a);
            if constexpr (TYPE == 12 || TYPE == 13)
                term[i] = sub_rounded(term[i], mul_rounded(mul_rounded(o.dmin, d8[i]), s.bm[i]));
        }
    }
    return term;
}

/* kMagic in four registers that the compiler keeps: as a known constant it
 * would set them anew before every product */
__device__ __forceinline__ i32x4_t magic_splat() {
    i32x4_t v = (i32x4_t)kMagic;
    asm volatile("" : "+v"(v));
    return v;
}

/* a row and token at a time: rows whose scales are not all finite, where a
 * super-block whose d8 is 0 must be left out (elsewhere its term is a zero,
 * which changes no sum), and tokens whose bsums are not sums of int8 values */
template <int TYPE>
__device__ __noinline__ void slow_rows(const uint8_t *w, float *out, uint32_t n_rows, uint32_t r0, uint32_t r1,
                                       const uint8_t *xq, uint32_t nb, uint32_t n_tokens, uint32_t t0, uint32_t t1) {
    for (uint32_t r = r0; r < min(r1, n_rows); ++r)
        for (uint32_t t = t0; t < min(t1, n_tokens); ++t) matmul_rows<TYPE, 1, 1>(w, out, n_rows, r, xq, nb, n_tokens, t);
}

/* ---- few tokens: the super-blocks of a tile over the four waves ------------------
 * A workgroup computes a 16-token x 16-row tile.  Its four waves compute the
 * terms of different super-blocks (a term depends on its super-block alone) into
 * LDS; then each thread adds its element's terms in super-block order.
 * Latency-bound: as many waves as the product has 16 x 16 x 256 pieces / 2,
 * and every load of a wave's two super-blocks is issued before the first is
 * used. */
constexpr uint32_t kMfmaChunk = 8u; /* super-blocks per round (two per wave) */

template <int TYPE> struct FewShared {
    struct { XTile<TYPE, 16u> x; WTile<TYPE, 16u> w; } t[4]; /* one per wave */
    float terms[kMfmaChunk][256]; /* [super-block of the round][token * 16 + row] */
};

template <int TYPE>
__device__ __forceinline__ void few_tile(const uint8_t *__restrict__ w, float *__restrict__ out, uint32_t n_rows,
                                         uint32_t r0, const uint8_t *__restrict__ xq, uint32_t nb, uint32_t n_tokens,
                                         uint32_t t0, FewShared<TYPE> &S) {
    using Q = QPlane<TYPE>;
    const uint32_t tid = threadIdx.x, lane = tid & 63u, l16 = lane & 15u, g = lane >> 4;
    const uint32_t wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    WStage<TYPE, 16u, 64u> ws[2] = {{w, n_rows, nb, r0, lane}, {w, n_rows, nb, r0, lane}};
    XStage<TYPE, 16u, 64u> xs[2] = {{xq, n_tokens, nb, t0, lane}, {xq, n_tokens, nb, t0, lane}};
    auto &mine = S.t[wave];
    const i32x4_t magic = magic_splat();
    int bad = 0;
    float sumf = 0.0f; /* element tid: token t0 + tid / 16, row r0 + tid % 16 */
    for (uint32_t c0 = 0; c0 < nb; c0 += kMfmaChunk) {
#pragma unroll
        for (uint32_t u = 0; u < 2u; ++u) {
            const uint32_t b = min(c0 + 2u * wave + u, nb - 1u); /* slots past the end repeat a block, unused */
            ws[u].fetch(b);
            xs[u].fetch(b);
        }
#pragma unroll
        for (uint32_t u = 0; u < 2u; ++u) {
            const uint32_t k = 2u * wave + u;
            if (c0 + k >= nb) break;
            ws[u].put(mine.w);
            xs[u].put(mine.x);
            xs[u].check();
            __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
            __builtin_amdgcn_wave_barrier(); /* the image is this wave's own */
            __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
            typename Q::Raw raw;
            typename Q::Op op;
            XOp x;
            i32x4_t cin[8];
            Q::load(raw, mine.w.q + l16 * WLayout<TYPE>::kPitch, mine.w.d + l16 * WTile<TYPE, 16u>::kD, g);
            mine.x.read(x, 0u, l16, g);
            mine.x.inits(cin, 0u, g);
            const f32x4_t d8 = mine.x.scales(0u, g);
            Q::prep(op, raw, g);
            bad |= !op.finite;
            TileAcc<TYPE> acc;
            tile_sums<TYPE>(acc, op, x, cin, magic);
            const f32x4_t term = tile_terms<TYPE>(acc, op, d8);
#pragma unroll
            for (int i = 0; i < 4; ++i) S.terms[k][(4u * g + (uint32_t)i) * 16u + l16] = term[i];
            __builtin_amdgcn_wave_barrier();
        }
        __syncthreads();
        const uint32_t n_k = min(kMfmaChunk, nb - c0);
        for (uint32_t k = 0; k < n_k; ++k) sumf = add_rounded(sumf, S.terms[k][tid]);
        __syncthreads();
    }
    if (__syncthreads_or(bad || (xs[0].wide | xs[1].wide) != 0u)) {
        slow_rows<TYPE>(w, out, n_rows, r0 + 4u * wave, r0 + 4u * wave + 4u, xq, nb, n_tokens, t0, t0 + 16u);
        return;
    }
    const uint32_t t = t0 + (tid >> 4), r = r0 + (tid & 15u);
    if (t < n_tokens && r < n_rows) out[(size_t)t * n_rows + r] = sumf;
}

/* ---- many tokens: a tile of 64 rows x 16 T tokens per workgroup --------------------
 * Both operands of a super-block are staged in LDS.  Each of the four waves
 * makes MFMA operands of its 16 rows once per super-block and meets T tiles of
 * 16 tokens with them; the next super-block's loads are in flight meanwhile.
 * Per 16 x 16 x 256 piece: 9 MFMAs (8 for the types without bsums) beside about
 * 8 VALU instructions per element for the term (18 for Q4_0 and Q8_0, a rounded
 * product and sum per 32 weights), which bound it. */
template <int TYPE, uint32_t T> struct ManyShared {
    XTile<TYPE, 16u * T> x;
    WTile<TYPE, 64u> w;
    uint32_t wide[4]; /* per wave: it staged a bsum that is no sum of int8 values */
};

template <int TYPE, uint32_t T>
__device__ __forceinline__ void many_tile(const uint8_t *__restrict__ w, float *__restrict__ out, uint32_t n_rows,
                                          uint32_t r0, const uint8_t *__restrict__ xq, uint32_t nb, uint32_t n_tokens,
                                          uint32_t t0, ManyShared<TYPE, T> &S) {
    using Q = QPlane<TYPE>;
    const uint32_t tid = threadIdx.x, lane = tid & 63u, l16 = lane & 15u, g = lane >> 4;
    const uint32_t wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    WStage<TYPE, 64u, 256u> ws(w, n_rows, nb, r0, tid);
    XStage<TYPE, 16u * T, 256u> xs(xq, n_tokens, nb, t0, tid);
    const i32x4_t magic = magic_splat();
    f32x4_t sum[T];
#pragma unroll
    for (uint32_t t = 0; t < T; ++t) sum[t] = (f32x4_t)0.0f;
    bool bad = false;
    ws.fetch(0u);
    xs.fetch(0u);
    for (uint32_t b = 0; b < nb; ++b) {
        if (b) __syncthreads(); /* the last super-block's reads are done */
        ws.put(S.w);
        xs.put(S.x);
        if (kHasBsums<TYPE> && b + 1u == nb) { /* every wave's finding, without a barrier of its own */
            xs.check();
            S.wide[wave] = xs.wide != 0u; /* the same from every lane */
        }
        __syncthreads();
        if (b + 1u < nb) {
            xs.check();
            ws.fetch(b + 1u);
            xs.fetch(b + 1u);
        }
        typename Q::Raw raw;
        typename Q::Op op;
        Q::load(raw, S.w.q + (16u * wave + l16) * WLayout<TYPE>::kPitch, S.w.d + (16u * wave + l16) * WTile<TYPE, 64u>::kD, g);
        Q::prep(op, raw, g);
        bad |= !op.finite;
        /* step t: fragments of tile t + 1 from LDS, the products of tile t,
         * the terms of tile t - 1: the matrix pipe works beside the VALU */
        XOp x[2];
        i32x4_t cin[2][8];
        TileAcc<TYPE> acc[2];
        S.x.read(x[0], 0u, l16, g);
        S.x.inits(cin[0], 0u, g);
#pragma unroll
        for (uint32_t t = 0; t <= T; ++t) {
            __builtin_amdgcn_sched_barrier(0);
            if (t + 1u < T) {
                S.x.read(x[(t + 1u) & 1u], 16u * (t + 1u), l16, g);
                S.x.inits(cin[(t + 1u) & 1u], 16u * (t + 1u), g);
            }
            f32x4_t d8;
            if (t > 0u) d8 = S.x.scales(16u * (t - 1u), g);
            if (t < T) tile_sums<TYPE>(acc[t & 1u], op, x[t & 1u], cin[t & 1u], magic);
            if (t > 0u) {
                const f32x4_t term = tile_terms<TYPE>(acc[(t - 1u) & 1u], op, d8);
#pragma unroll
                for (int i = 0; i < 4; ++i) sum[t - 1u][i] = add_rounded(sum[t - 1u][i], term[i]);
            }
        }
    }
    const uint32_t rw = r0 + 16u * wave, row = rw + l16;
    if constexpr (kHasBsums<TYPE>) bad |= (S.wide[0] | S.wide[1] | S.wide[2] | S.wide[3]) != 0u;
    if (__any(bad)) {
        slow_rows<TYPE>(w, out, n_rows, rw, rw + 16u, xq, nb, n_tokens, t0, t0 + 16u * T);
        return;
    }
#pragma unroll
    for (uint32_t t = 0; t < T; ++t)
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const uint32_t tok = t0 + 16u * t + 4u * g + (uint32_t)i;
            if (tok < n_tokens && row < n_rows) out[(size_t)tok * n_rows + row] = sum[t][i];
        }
}

/* Row tiles of every matrix of the set, in one launch: block x -> (matrix,
 * rows), block y -> tokens.  TYPE as in k_matmul_q; T 0: few_tile (16 rows),
 * else many_tile (64 rows). */
template <int TYPE, uint32_t T>
__device__ __forceinline__ void mfma_tile(const MatSet &S, uint32_t m, uint32_t bx, const uint8_t *xq, uint32_t nb,
                                          uint32_t n_tokens, uint8_t *sh) {
    if constexpr (T == 0u)
        few_tile<TYPE>(S.w[m], S.out[m], S.rows[m], bx * 16u, xq, nb, n_tokens, blockIdx.y * 16u,
                       *reinterpret_cast<FewShared<TYPE> *>(sh));
    else
        many_tile<TYPE, T>(S.w[m], S.out[m], S.rows[m], bx * 64u, xq, nb, n_tokens, blockIdx.y * (16u * T),
                           *reinterpret_cast<ManyShared<TYPE, T> *>(sh));
}

template <int TYPE, uint32_t T> constexpr size_t mfma_lds() {
    if constexpr (T == 0u) return sizeof(FewShared<TYPE>);
    else return sizeof(ManyShared<TYPE, T>);
}
constexpr size_t max_of(size_t a, size_t b) { return a > b ? a : b; }
template <uint32_t T>
constexpr size_t kMixedLds = max_of(max_of(max_of(mfma_lds<12, T>(), mfma_lds<13, T>()), max_of(mfma_lds<14, T>(), mfma_lds<23, T>())),
                                    max_of(mfma_lds<2, T>(), mfma_lds<8, T>()));

template <int TYPE, uint32_t T>
__global__ __launch_bounds__(256, 2) void k_matmul_mfma(const MatSet S, const uint8_t *__restrict__ xq, uint32_t nb,
                                                        uint32_t n_tokens) {
    __shared__ __attribute__((aligned(16))) uint8_t sh[TYPE != 0 ? mfma_lds<TYPE == 0 ? 12 : TYPE, T>() : kMixedLds<T>];
    uint32_t m = 0;
    while (m + 1u < S.n && blockIdx.x >= S.wave0[m + 1u]) ++m;
    const uint32_t bx = blockIdx.x - S.wave0[m];
    if constexpr (TYPE != 0) {
        mfma_tile<TYPE, T>(S, m, bx, xq, nb, n_tokens, sh);
        return;
    }
    switch (S.type[m]) {
    case 12u: mfma_tile<12, T>(S, m, bx, xq, nb, n_tokens, sh); break;
    case 14u: mfma_tile<14, T>(S, m, bx, xq, nb, n_tokens, sh); break;
    case 13u: mfma_tile<13, T>(S, m, bx, xq, nb, n_tokens, sh); break;
    case 23u: mfma_tile<23, T>(S, m, bx, xq, nb, n_tokens, sh); break;
    case 2u: /* launch_mfma takes T = 8 for sets without Q4_0 only */
        if constexpr (T <= 4u) mfma_tile<2, T>(S, m, bx, xq, nb, n_tokens, sh);
        break;
    default: mfma_tile<8, T>(S, m, bx, xq, nb, n_tokens, sh); break;
    }
}

template <int TYPE, uint32_t T>
hipError_t launch_tiles(MatSet S, const void *x_q8, uint32_t nb, uint32_t n_tokens, hipStream_t stream) {
    constexpr uint32_t kRows = T == 0u ? 16u : 64u, kTokens = T == 0u ? 16u : 16u * T;
    S.wave0[0] = 0;
    for (uint32_t m = 0; m < S.n; ++m) S.wave0[m + 1] = S.wave0[m] + (S.rows[m] + kRows - 1u) / kRows;
    hipLaunchKernelGGL((k_matmul_mfma<TYPE, T>), dim3(S.wave0[S.n], (n_tokens + kTokens - 1u) / kTokens), dim3(256), 0,
                       stream, S, static_cast<const uint8_t *>(x_q8), nb, n_tokens);
    return hipGetLastError();
}

/* Five or more tokens.  Measured on MI355X, us per call over 2048 columns:
 *  - few_tile up to 1024 of its 16 x 16 tiles, against T = 2.  A CU holds three
 *    such workgroups (133 to 166 registers; Q6_K, Q8_0 and mixed sets also by
 *    LDS), so 768 are a round and 1024 a round and a third: 128 tokens x 2048
 *    rows Q4_K 9.1 against 9.9, Q5_K 11.3 / 12.1, Q6_K 12.6 / 14.3, IQ4_XS 11.4
 *    / 12.7, Q4_0 9.9 / 11.5, Q8_0 10.3 / 11.7, a mixed set 12.4 / 14.6; two
 *    whole rounds, x 3072 rows, Q4_K 11.8 against 9.9;
 *  - T = 2 while a CU gets at most one such workgroup: 256 x 2048 10.1, T = 4
 *    13.4; 700 x 2048 (704 workgroups) Q6_K 27.1 against 26.9, IQ4_XS 25.3
 *    against 22.8;
 *  - T = 8, which prepares a row's weights half as often, where it needs no
 *    more than half the rounds of T = 4 (two workgroups a CU): 2000 x 2048
 *    Q4_K 32.1 against 35.9, Q6_K 39.8 against 49.5; 1500 x 3072, two rounds
 *    against three, 46.1 against 44.7.  Q4_0 keeps T = 4: eight accumulator
 *    starts per tile do not fit the registers (spilled: 55.7 against 44.3). */
template <int TYPE>
hipError_t launch_mfma(const MatSet &S, const void *x_q8, uint32_t nb, uint32_t n_tokens, hipStream_t stream) {
    uint64_t t16 = 0, t64 = 0;
    bool q4_0 = false;
    for (uint32_t m = 0; m < S.n; ++m) {
        t16 += (S.rows[m] + 15u) / 16u;
        t64 += (S.rows[m] + 63u) / 64u;
        q4_0 = q4_0 || S.type[m] == 2u;
    }
    auto tok = [&](uint32_t per) { return (uint64_t)((n_tokens + per - 1u) / per); };
    if (t16 * tok(16u) <= 4u * kCus) return launch_tiles<TYPE, 0u>(S, x_q8, nb, n_tokens, stream);
    if (t64 * tok(32u) <= kCus) return launch_tiles<TYPE, 2u>(S, x_q8, nb, n_tokens, stream);
    auto rounds = [&](uint64_t wgs) { return (wgs + 2u * kCus - 1u) / (2u * kCus); };
    if constexpr (TYPE != 2)
        if (!q4_0 && 2u * rounds(t64 * tok(128u)) <= rounds(t64 * tok(64u)))
            return launch_tiles<TYPE, 8u>(S, x_q8, nb, n_tokens, stream);
    return launch_tiles<TYPE, 4u>(S, x_q8, nb, n_tokens, stream);
}

} // namespace

int launch_quantize_q8_K(const float *x, void *y, uint32_t n_rows, uint32_t n_cols, hipStream_t stream) {
    const uint32_t nb       = n_cols / 256u;
    const uint64_t n_blocks = (uint64_t)n_rows * nb;
    if (n_blocks == 0u) return LFM_ATTN_OK;
    hipLaunchKernelGGL(k_quant_q8K, dim3((uint32_t)((n_blocks + 3u) / 4u)), dim3(256), 0, stream, x,
                       static_cast<uint8_t *>(y), (uint32_t)n_blocks, nb);
    return hip_status(hipGetLastError());
}

int launch_matmul_q(uint32_t n_mats, float *const *outs, const void *const *ws, const uint32_t *types,
                    const uint32_t *rows, uint32_t n_cols, const void *x_q8, uint32_t n_tokens, hipStream_t stream) {
    if (n_tokens == 0u) return LFM_ATTN_OK;
    const uint32_t nb = n_cols / 256u;
    /* one launch over all matrices, whatever their types */
    MatSet S{};
    for (uint32_t m = 0; m < n_mats && m < 4u; ++m) {
        if (rows[m] == 0u) continue;
        S.w[S.n]    = static_cast<const uint8_t *>(ws[m]);
        S.out[S.n]  = outs[m];
        S.rows[S.n] = rows[m];
        S.type[S.n] = types[m];
        ++S.n;
    }
    if (S.n == 0u) return LFM_ATTN_OK;
    bool one_type = true;
    for (uint32_t m = 1; m < S.n; ++m) one_type = one_type && S.type[m] == S.type[0];
    hipError_t e;
    /* five or more tokens go to the matrix pipe (Q6_K 2048 x 2048: 4 tokens 6.0 us
     * both ways, 6 tokens 8.6 -> 6.0; Q4_K 8.1 -> 4.7) */
    if (n_tokens >= 5u) {
        switch (one_type ? S.type[0] : 0u) {
        case 12u: e = launch_mfma<12>(S, x_q8, nb, n_tokens, stream); break;
        case 14u: e = launch_mfma<14>(S, x_q8, nb, n_tokens, stream); break;
        case 13u: e = launch_mfma<13>(S, x_q8, nb, n_tokens, stream); break;
        case 23u: e = launch_mfma<23>(S, x_q8, nb, n_tokens, stream); break;
        case 2u: e = launch_mfma<2>(S, x_q8, nb, n_tokens, stream); break;
        case 8u: e = launch_mfma<8>(S, x_q8, nb, n_tokens, stream); break;
        default: e = launch_mfma<0>(S, x_q8, nb, n_tokens, stream); break;
        }
        return hip_status(e);
    }
    switch (one_type ? S.type[0] : 0u) {
    case 12u: e = launch_tokens<12>(S, x_q8, nb, n_tokens, stream); break;
    case 14u: e = launch_tokens<14>(S, x_q8, nb, n_tokens, stream); break;
    case 13u: e = launch_tokens<13>(S, x_q8, nb, n_tokens, stream); break;
    case 23u: e = launch_tokens<23>(S, x_q8, nb, n_tokens, stream); break;
    case 2u: e = launch_tokens<2>(S, x_q8, nb, n_tokens, stream); break;
    case 8u: e = launch_tokens<8>(S, x_q8, nb, n_tokens, stream); break;
    default: e = launch_tokens<0>(S, x_q8, nb, n_tokens, stream); break;
    }
    return hip_status(e);
}

} // namespace lfm
