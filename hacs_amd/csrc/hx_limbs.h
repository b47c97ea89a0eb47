// hx_limbs.h -- the balanced signed 8-bit limb split of residues mod p and the exact recombination
// of limb-product anti-diagonals, shared by the limb GEMM (hx_gemm.hip) and the MFMA trailing update
// inside the batched elimination (hx_rref_batch.hip).
//
//  * A canonical residue x < p (p <= 4278124287) is replaced by its balanced representative
//    v = x or x - p, |v| <= (p-1)/2, written in L signed base-256 digits d_s in [-128, 127]:
//    v = sum_s d_s 256^s (L = 4 covers p <= 4278124287, 3 covers p <= 16711423, 2 p <= 65279, 1 p <= 255).
//  * A product of two such numbers is sum_d 256^d D_d with D_d = sum_{s+t=d} a_s b_t; summed over K
//    terms, |D_d| <= pairs(d) K 2^14 (< 2^31 for K <= limb_k_chunk(L)).  Recombination:
//    x = sum_{d<=3} D_d 2^(8d) + sum_{d>=4} D_d w_d with w_d = 2^(8d) mod p balanced into (-p/2, p/2]:
//    |x| < 6 * 2^60 + 2^56 < 2^63, then one Barrett reduction of x + p ceil(2^63 / p) in [0, 2^64).
#pragma once

#include "hx_common.h"

namespace hx {

// Balanced signed base-256 digits of a canonical residue x (x < p): L digits in [-128, 127].
__device__ __forceinline__ void limbs_of(uint32_t x, uint32_t p, uint32_t half, int L, int32_t* d) {
    int32_t v = x > half ? (int32_t)((int64_t)x - (int64_t)p) : (int32_t)x;
#pragma unroll
    for (int s = 0; s < 3; ++s) {
        if (s >= L - 1) break;
        const int32_t t = ((v + 128) & 255) - 128;
        d[s] = t;
        v = (v - t) >> 8;
    }
#pragma unroll
    for (int s = 0; s < 4; ++s)
        if (s == L - 1) d[s] = v;
}

// The same digits of four residues at once, byte b of w[s] = digit s of x[b]: the balanced value plus 0x80808080
// carries exactly where a digit wraps, so its bytes are the digits plus 128 (the top one, in [-128, 127] by the
// limb count, too); the four words' bytes are then transposed.  About six operations per residue.
template <int L>
__device__ __forceinline__ void limb_split4(const uint32_t (&x)[4], uint32_t p, uint32_t half, uint32_t (&w)[L]) {
    const uint32_t K = 0x80808080u, Kp = K - p;
    uint32_t u[4];
#pragma unroll
    for (int b = 0; b < 4; ++b) u[b] = x[b] + (x[b] > half ? Kp : K);
    const uint32_t t0 = __builtin_amdgcn_perm(u[1], u[0], 0x05010400u), t2 = __builtin_amdgcn_perm(u[3], u[2], 0x05010400u);
    w[0] = __builtin_amdgcn_perm(t2, t0, 0x05040100u) ^ K;
    if (L > 1) w[L > 1 ? 1 : 0] = __builtin_amdgcn_perm(t2, t0, 0x07060302u) ^ K;
    if (L > 2) {
        const uint32_t t1 = __builtin_amdgcn_perm(u[1], u[0], 0x07030602u), t3 = __builtin_amdgcn_perm(u[3], u[2], 0x07030602u);
        w[L > 2 ? 2 : 0] = __builtin_amdgcn_perm(t3, t1, 0x05040100u) ^ K;
        if (L > 3) w[L > 3 ? 3 : 0] = __builtin_amdgcn_perm(t3, t1, 0x07060302u) ^ K;
    }
}

// The recombination constants for modulus p.
struct LimbConsts {
    uint64_t off;     // p * ceil(2^63 / p)
    int32_t w[3];     // 2^(8d) mod p, balanced, d = 4, 5, 6
};

inline LimbConsts limb_consts(uint32_t p) {
    LimbConsts c;
    c.off = ((1ull << 63) / p + 1) * (uint64_t)p;
    uint64_t w = 1;
    for (int d = 1; d <= 6; ++d) {
        w = (w << 8) % p;
        if (d >= 4) c.w[d - 4] = (int32_t)(w <= p / 2 ? (int64_t)w : (int64_t)w - (int64_t)p);
    }
    return c;
}

// sum_d 256^d D_d mod p from the ND = 2L - 1 anti-diagonal sums of one output.
template <int ND>
__device__ __forceinline__ uint32_t limb_recombine(const int32_t (&D)[ND], const LimbConsts& c, const DevMod& M) {
    int64_t x = 0;
#pragma unroll
    for (int d = 0; d < ND; ++d) {
        if (d <= 3)
            x += (int64_t)D[d] * (int64_t)(1u << (8 * d));
        else
            x += (int64_t)D[d] * (int64_t)c.w[d - 4];
    }
    return red64((uint64_t)x + c.off, M);
}

typedef int limb_v4i __attribute__((ext_vector_type(4)));
typedef int limb_v16i __attribute__((ext_vector_type(16)));

// The residues mod p < 2^31 of a 32 x 32 block of a product of depth at most 64 (KS k-steps of 32) from the
// operands' limb fragments.  The anti-diagonals come in pairs from the top: P_j = 2^8 D_{2j} + D_{2j-1} (weight
// 2^{8(2j-1)}, j = L-1 .. 1), shifted inside the accumulator between the two, and D_0.  |D_d| <= 4 * 64 * 2^14 =
// 2^22, so the pairs stay below 2^31.  x = sum_j 2^{8(2j-1)} P_j + D_0 is kept twice: exactly mod 2^32, and in a
// double (|x| < 2^71: error below 2^71 * 2^-51).  q = rint(x / p) from the double is within 1/2 + 2^20 / p < 0.6 of
// x / p for four limbs (p > 2^23; far closer for fewer), so x - q p, exact mod 2^32, lies in (-p, p).
// About 20 operations per output, none of them 64-bit integer.
struct SmallConsts {
    uint32_t p;
    double inv;                  // 1 / p
};
template <int L, int KS>
__device__ __forceinline__ void limb_small_product(const limb_v4i (&a)[KS][L], const limb_v4i (&b)[KS][L],
                                                   const SmallConsts& c, uint32_t (&out)[16]) {
    double xf[16];
    uint32_t xl[16];
    auto diag = [&](int d, limb_v16i acc) {
#pragma unroll
        for (int s = 0; s < L; ++s)
#pragma unroll
            for (int ks = 0; ks < KS; ++ks)
                if (d - s >= 0 && d - s < L)
                    acc = __builtin_amdgcn_mfma_i32_32x32x32_i8(a[ks][s], b[ks][d - s], acc, 0, 0, 0);
        return acc;
    };
    limb_v16i zero;
#pragma unroll
    for (int e = 0; e < 16; ++e) zero[e] = 0;
#pragma unroll
    for (int j = L - 1; j >= 1; --j) {
        limb_v16i acc = diag(2 * j, zero);
#pragma unroll
        for (int e = 0; e < 16; ++e) acc[e] = (int)((uint32_t)acc[e] << 8);
        acc = diag(2 * j - 1, acc);
        const double w = (double)(1ull << (8 * (2 * j - 1)));
#pragma unroll
        for (int e = 0; e < 16; ++e) {
            xf[e] = j == L - 1 ? (double)acc[e] * w : __builtin_fma((double)acc[e], w, xf[e]);
            const uint32_t low = 2 * j - 1 < 4 ? (uint32_t)acc[e] << (8 * (2 * j - 1)) : 0u;
            xl[e] = j == L - 1 ? low : xl[e] + low;
        }
    }
    const limb_v16i acc = diag(0, zero);
#pragma unroll
    for (int e = 0; e < 16; ++e) {
        const double x = L == 1 ? (double)acc[e] : xf[e] + (double)acc[e];
        const uint32_t l = L == 1 ? (uint32_t)acc[e] : xl[e] + (uint32_t)acc[e];
        // rint by the 1.5 * 2^52 shift: the low word of the sum is q mod 2^32 (|q| < 2^48)
        const uint32_t q = (uint32_t)__double_as_longlong(__builtin_fma(x, c.inv, 6755399441055744.0));
        const int32_t r = (int32_t)(l - q * c.p);
        out[e] = (uint32_t)(r + ((r >> 31) & (int32_t)c.p));
    }
}

}  // namespace hx
