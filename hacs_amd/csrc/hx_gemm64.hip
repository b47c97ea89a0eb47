// hx_gemm64.hip -- C op= A B mod p for 64-bit residues, every modulus 2 <= p < 2^64 (the device
// u64 GEMM of Cuda/cuda_kernels.cu:104-164; the CPU path of record is kernels::gemm<uint64_t>,
// ModArithmetic/Kernels.h:184).  Two routes with the same bytes:
//
//  * The residue route (gemm64_residue; k >= 96, or k >= 40 with small planes; outside a stream capture): the operands modulo up to 19
//    pairwise coprime bytes, one int8 MFMA product per modulus (res_gemm_kernel, hx_gemm.hip), and the CRT
//    back to 64 bits.  2048^3 mod 2^61 - 1: 17 products, 0.256 ms = 3.4e13 multiply-adds/s for the whole
//    call, against 4.19 ms (2.05e12) on the plain kernel; 512^3 0.049 against 0.364 ms.  Bound by the int8
//    products and the HBM passes over the residue planes (17 bytes per operand entry and per output).
//
//  * The plain kernel (gemm64_kernel; everything else): each 64 x 64 -> 128-bit product is formed from four
//    32 x 32 -> 64 partial products and added into a 160-bit accumulator (w0 + w1 2^64 + w2 2^128, exact for
//    K < 2^32), and the sum is reduced once: T = w0 + w1 2^64 + w2 2^128 mod p.  For odd p by Montgomery
//    (R = 2^64): REDC(w1 mod p, w0) = (w1 2^64 + w0) R^-1, multiplied by R^2 mod p and reduced again;
//    the w2 term is w2 (2^128 mod p).  For even p (no Montgomery inverse) by binary long division of
//    the 128-bit words.  Tiling: 64 x 64 outputs per 256-thread workgroup, 4 x 4 per thread (rows ty + 16 i,
//    columns tx + 16 j), K staged by 16 through a double-buffered LDS tile (A transposed, padded rows), the
//    next stage's global loads issued before the current stage's products.  VALU-bound: ~14 integer
//    operations per mod-p multiply-add.
//
// The bytes of both equal the oracle's exact integer arithmetic.
#include <algorithm>
#include <cmath>
#include <cstring>

#include "hx_common.h"
#include "hx_residue.h"

namespace hx {
namespace {

constexpr int G64_TILE = 64, G64_BK = 16, G64_T = 256;

struct Mod64 {
    uint64_t p, ninv, r2, two64;    // ninv = -p^-1 mod 2^64 (odd p); r2 = 2^128 mod p; two64 = 2^64 mod p
    int odd;
};

struct Gemm64Args {
    uint32_t m, n, k;
    const uint64_t* A;
    int64_t ars, acs;
    const uint64_t* B;
    int64_t brs, bcs;
    uint64_t* C;
    int64_t crs, ccs;
    int op;
};

__device__ __forceinline__ uint64_t add64m(uint64_t a, uint64_t b, uint64_t p) {
    const uint64_t r = a + b;
    return (r < a || r >= p) ? r - p : r;
}
__device__ __forceinline__ uint64_t sub64m(uint64_t a, uint64_t b, uint64_t p) { return a >= b ? a - b : a + (p - b); }

// (hi 2^64 + lo) R^-1 mod p for hi < p, odd p (Montgomery, R = 2^64).
__device__ __forceinline__ uint64_t redc128(uint64_t hi, uint64_t lo, const Mod64& M) {
    const uint64_t m = lo * M.ninv;
    const uint64_t mlo = m * M.p, mhi = __umul64hi(m, M.p);
    const uint64_t s = lo + mlo;                       // == 0 mod 2^64 by construction
    const uint64_t carry = s < lo ? 1u : 0u;
    // hi + mhi + carry < 2p; it may pass 2^64 when p > 2^63: then subtract p in 128-bit terms
    const uint64_t t1 = hi + mhi;
    const uint64_t c1 = t1 < hi ? 1u : 0u;
    const uint64_t t = t1 + carry;
    const uint64_t c2 = t < t1 ? 1u : 0u;
    return (c1 | c2 || t >= M.p) ? t - M.p : t;
}
__device__ __forceinline__ uint64_t mont_mul64(uint64_t a, uint64_t b, const Mod64& M) {
    return redc128(__umul64hi(a, b), a * b, M);
}
// (hi 2^64 + lo) mod p for any p >= 2 by binary long division (the even-modulus path).
__device__ uint64_t mod128_div(uint64_t hi, uint64_t lo, uint64_t p) {
    uint64_t r = hi % p;
    for (int b = 63; b >= 0; --b) {
        const uint64_t top = r >> 63;
        r = (r << 1) | ((lo >> b) & 1u);
        if (top || r >= p) r -= p;
    }
    return r;
}
__device__ __forceinline__ uint64_t reduce160(uint64_t w0, uint64_t w1, uint32_t w2, const Mod64& M) {
    uint64_t r;
    if (M.odd) {
        const uint64_t h = w1 >= M.p ? w1 % M.p : w1;
        r = mont_mul64(redc128(h, w0, M), M.r2, M);          // (h 2^64 + w0) mod p
        if (w2) r = add64m(r, mont_mul64(mont_mul64((uint64_t)w2, M.r2, M), M.r2, M), M.p);   // w2 2^128
    } else {
        r = mod128_div(w1, w0, M.p);
        if (w2) {
            // w2 2^128 mod p = ((w2 2^64 mod p) 2^64) mod p
            const uint64_t t = mod128_div((uint64_t)w2, 0, M.p);
            r = add64m(r, mod128_div(t, 0, M.p), M.p);
        }
    }
    return r;
}

// acc += a b exactly (a, b < 2^64; 160-bit accumulator w0, w1, w2)
__device__ __forceinline__ void mac128(uint64_t& w0, uint64_t& w1, uint32_t& w2, uint64_t a, uint64_t b) {
    const uint64_t lo = a * b, hi = __umul64hi(a, b);
    w0 += lo;
    const uint64_t c0 = w0 < lo ? 1u : 0u;
    const uint64_t h = hi + c0;                           // hi <= 2^64 - 2, so no wrap
    w1 += h;
    w2 += w1 < h ? 1u : 0u;
}

__global__ __launch_bounds__(G64_T) void gemm64_kernel(Gemm64Args g, Mod64 M) {
    __shared__ uint64_t As[2][G64_BK][G64_TILE + 1];
    __shared__ uint64_t Bs[2][G64_BK][G64_TILE];
    const uint32_t ntn = (g.n + G64_TILE - 1) / G64_TILE;
    const uint32_t i0 = (blockIdx.x / ntn) * G64_TILE, j0 = (blockIdx.x % ntn) * G64_TILE;
    const uint32_t tid = threadIdx.x, tx = tid % 16, ty = tid / 16;
    uint64_t w0[4][4], w1[4][4];
    uint32_t w2[4][4];
#pragma unroll
    for (int a = 0; a < 4; ++a)
#pragma unroll
        for (int b = 0; b < 4; ++b) {
            w0[a][b] = 0;
            w1[a][b] = 0;
            w2[a][b] = 0;
        }
    // loader roles: A tile 64 rows x 16 k (thread: k = tid % 16, rows tid / 16 + 16 e), B tile 16 k x 64
    // columns (thread: column tid % 64, k = tid / 64 + 4 e) -- unit-stride directions first
    uint64_t ra[4], rb[4];
    auto load = [&](uint32_t k0) {
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            const uint32_t row = i0 + tid / 16 + 16 * e, kk = k0 + tid % 16;
            ra[e] = (row < g.m && kk < g.k) ? g.A[(int64_t)row * g.ars + (int64_t)kk * g.acs] : 0u;
            const uint32_t col = j0 + tid % 64, kb = k0 + tid / 64 + 4 * e;
            rb[e] = (col < g.n && kb < g.k) ? g.B[(int64_t)kb * g.brs + (int64_t)col * g.bcs] : 0u;
        }
    };
    auto store = [&](int buf) {
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            As[buf][tid % 16][tid / 16 + 16 * e] = ra[e];
            Bs[buf][tid / 64 + 4 * e][tid % 64] = rb[e];
        }
    };
    load(0);
    store(0);
    __syncthreads();
    int buf = 0;
    for (uint32_t k0 = 0; k0 < g.k; k0 += G64_BK) {
        const bool more = k0 + G64_BK < g.k;
        if (more) load(k0 + G64_BK);                       // in flight during the products below
#pragma unroll 4
        for (int kk = 0; kk < G64_BK; ++kk) {
            uint64_t av[4], bv[4];
#pragma unroll
            for (int a = 0; a < 4; ++a) av[a] = As[buf][kk][ty + 16 * a];
#pragma unroll
            for (int b = 0; b < 4; ++b) bv[b] = Bs[buf][kk][tx + 16 * b];
#pragma unroll
            for (int a = 0; a < 4; ++a)
#pragma unroll
                for (int b = 0; b < 4; ++b) mac128(w0[a][b], w1[a][b], w2[a][b], av[a], bv[b]);
        }
        if (more) {
            store(buf ^ 1);
            __syncthreads();
            buf ^= 1;
        }
    }
#pragma unroll
    for (int a = 0; a < 4; ++a) {
        const uint32_t i = i0 + ty + 16 * a;
        if (i >= g.m) continue;
#pragma unroll
        for (int b = 0; b < 4; ++b) {
            const uint32_t j = j0 + tx + 16 * b;
            if (j >= g.n) continue;
            const uint64_t r = reduce160(w0[a][b], w1[a][b], w2[a][b], M);
            uint64_t* c = g.C + (int64_t)i * g.crs + (int64_t)j * g.ccs;
            *c = g.op == HX_OP_SET ? r : g.op == HX_OP_ADD ? add64m(*c, r, M.p) : sub64m(*c, r, M.p);
        }
    }
}

Mod64 mod64_of(const hx_modctx64& c) { return Mod64{c.p, c.ninv, c.r2, c.two64, (int)(c.p & 1u)}; }

// ---- the residue route ------------------------------------------------------------------------
// The product of balanced operands (|a_b| <= p / 2) modulo N pairwise coprime moduli q_i <= 255, one int8
// MFMA product each, and the CRT back to the residue mod p: hx_gemm.hip's route with the operands and the
// recombination on 64-bit words.  N is the least count with prod q_i > 2.05 k (p/2)^2 (at most 19).

struct Split64 {
    uint32_t nmod;
    uint32_t q[RES_MAXQ], tlo[RES_MAXQ], thi[RES_MAXQ];   // bytes 2^(8j) mod q, j = 0 .. 3 and 4 .. 7
    uint32_t kq[RES_MAXQ];                                // q - (2^63 mod q)
    float iq[RES_MAXQ];
};

struct Prep64 {
    const uint64_t* src;         // entry (row r, k c) at src[r s_r + c s_c]
    int64_t s_r, s_c;
    uint32_t R, K;               // rows and k of the operand (past them: zero)
    uint32_t Kp;                 // bytes per output row
    int8_t* out;
    size_t plane;
    uint64_t p;
};

// Residue planes of one 32-row x 128-k tile.  The entries a_b + 2^63 go through LDS as T[k][row] (row XOR 4 times
// the 16-k chunk: the strided reads below spread over the banks), loaded along whichever index is contiguous
// in memory; each thread then turns 16 k of one row into 16 bytes per plane (res_chunk: 128 contiguous bytes per eight rows).
// With w = a_b + 2^63 (a word of 8 bytes w_j), t = sum_j w_j (2^(8j) mod q) + q - (2^63 mod q) is congruent to
// a_b and below 8 * 255 * 254 + 255 < 2^19, so fp32 holds it and t fl(1/q) + 1/2 is within 2^19 / 173 * 2^-22
// < 8e-4 of t / q + 1/2, whose fractional part is at least 1 / (2q) > 0.0019 from an integer for odd q:
// the truncation is round(t / q).  (q = 254: a tie may go either way, +-127 are the same residue.)
__global__ __launch_bounds__(256) void prep64_kernel(Prep64 a, Split64 c) {
    __shared__ uint64_t T[128][33];
    const uint32_t r0 = blockIdx.x * 32, c0 = blockIdx.y * 128;
    const int tid = threadIdx.x;
    const uint64_t p = a.p, half = p / 2;
    auto put = [&](uint32_t r, uint32_t cc) {
        const uint32_t row = r0 + r, k = c0 + cc;
        const uint64_t v = (row < a.R && k < a.K) ? a.src[(int64_t)row * a.s_r + (int64_t)k * a.s_c] : 0u;
        T[cc][r ^ (((cc >> 4) & 7) << 2)] = (v > half ? v - p : v) + 0x8000000000000000ull;
    };
    if (a.s_c == 1) {
#pragma unroll 8
        for (int t = 0; t < 16; ++t) put((tid >> 7) + 2 * t, tid & 127);
    } else {
#pragma unroll 8
        for (int t = 0; t < 16; ++t) put(tid & 31, (tid >> 5) + 8 * t);
    }
    __syncthreads();
    const uint32_t r = tid >> 3, qd = tid & 7;
    if (c0 + 16 * qd >= a.Kp) return;
    uint64_t w[16];
#pragma unroll
    for (int j = 0; j < 16; ++j) w[j] = T[16 * qd + j][r ^ (qd << 2)];
    int8_t* out = a.out + res_chunk(r0 + r, c0 / 16 + qd, a.Kp);
    for (uint32_t i = 0; i < c.nmod; ++i) {
        const uint32_t Q = c.q[i], TL = c.tlo[i], TH = c.thi[i], KQ = c.kq[i];
        const float IQ = c.iq[i];
        uint32_t o[4] = {0, 0, 0, 0};
#pragma unroll
        for (int j = 0; j < 16; ++j) {
            const uint32_t t = __builtin_amdgcn_udot4((uint32_t)(w[j] >> 32), TH,
                                                      __builtin_amdgcn_udot4((uint32_t)w[j], TL, KQ, false), false);
            const uint32_t qt = (uint32_t)fmaf((float)t, IQ, 0.5f);
            o[j / 4] |= ((t - __umul24(qt, Q)) & 0xffu) << (8 * (j % 4));
        }
        *(uint4*)(out + (size_t)i * a.plane) = make_uint4(o[0], o[1], o[2], o[3]);
    }
}

// x mod p from the N product residues s_i = x (M / q_i)^-1 mod q_i (M = prod q_i): sum_i s_i M / q_i = x + T M with
// T = round(sum_i s_i / q_i), so x = sum_i s_i (M / q_i mod p) - T (M mod p).  The 64-bit constants are split
// in 16-bit digits (24-bit products, digit sums below 19 * 254 * 2^16 < 2^29), the fraction sum is in fixed
// point with f_i = round(2^20 / q_i) (error <= 19 * 254 / 2 units of 2^-20 < 0.0024, inside the 0.5 - 0.488
// margin), and the total, below 2^78, is reduced once.
struct Crt64 {
    const uint8_t* R;
    size_t r_plane;
    ResBlocks g;
    uint32_t nmod;
    uint16_t c[RES_MAXQ][4];     // (M / q_i) mod p, digits of 16 bits
    uint32_t f[RES_MAXQ];
    uint64_t pmm;                // p - (M mod p)
    uint32_t m, n;
    uint64_t* C;
    int64_t crs, ccs;
    int op;
};

// One 32 x 32 block per two waves: eight outputs per thread, planes read 8 bytes per lane.
__global__ __launch_bounds__(256) void crt64_kernel(Crt64 a, Mod64 M) {
    const uint32_t blk = blockIdx.x * 2 + (threadIdx.x >> 7), lane = threadIdx.x & 63, h = (threadIdx.x >> 6) & 1;
    uint32_t row0, col;
    res_block(a.g, blk, row0, col);
    if (row0 >= a.m || col >= a.n) return;
    row0 += 16 * h + 4 * (lane >> 5);
    col += lane & 31;
    uint32_t d[8][4] = {}, fr[8] = {};
    const uint8_t* src = a.R + (size_t)blk * 1024 + lane * 16 + 8 * h;
#pragma unroll 2
    for (uint32_t i = 0; i < a.nmod; ++i) {
        const uint2 v = *(const uint2*)(src + (size_t)i * a.r_plane);
        const uint32_t w[2] = {v.x, v.y};
#pragma unroll
        for (int r = 0; r < 8; ++r) {
            const uint32_t sb = (w[r / 4] >> (8 * (r % 4))) & 0xffu;
#pragma unroll
            for (int e = 0; e < 4; ++e) d[r][e] += __umul24(sb, a.c[i][e]);
            fr[r] += __umul24(sb, a.f[i]);
        }
    }
    if (col >= a.n) return;
#pragma unroll
    for (int r = 0; r < 8; ++r) {
        const uint32_t row = row0 + (r / 4) * 8 + r % 4;
        if (row >= a.m) continue;
        const uint32_t T = (fr[r] + (1u << 19)) >> 20;
        unsigned __int128 x = (unsigned __int128)T * a.pmm;
#pragma unroll
        for (int e = 0; e < 4; ++e) x += (unsigned __int128)d[r][e] << (16 * e);
        const uint64_t res = reduce160((uint64_t)x, (uint64_t)(x >> 64), 0, M);
        uint64_t* c = a.C + (int64_t)row * a.crs + (int64_t)col * a.ccs;
        *c = a.op == HX_OP_SET ? res : a.op == HX_OP_ADD ? add64m(*c, res, M.p) : sub64m(*c, res, M.p);
    }
}

// The least N with prod_{i<N} q_i > 2.05 k (p/2)^2 for 1 <= k <= RES_KMAX (the logarithms' rounding errors are
// far below the 1e-9 kept in hand; 19 moduli reach 2^147.6, the bound stays below 2^145.1).
uint32_t moduli64(uint64_t p, uint32_t k) {
    const double need = std::log2(2.05) + std::log2((double)k) + 2.0 * std::log2((double)(p / 2)) + 1e-9;
    double have = 0.0;
    for (int i = 0; i < RES_MAXQ; ++i) {
        have += std::log2((double)res_modulus(i));
        if (have > need) return (uint32_t)i + 1;
    }
    return 0;
}

// Shallower products stay on the plain kernel: the splits and the CRT cost the same at any k, the plain kernel's
// time grows with k (mod 2^61 - 1, us plain / residue: 2048 x 2048 x 16 59 / 109, x 64 180 / 122; 32^3 27 / 33,
// 64^3 56 / 32; 512^3 364 / 49, 2048^3 4190 / 256).
constexpr uint32_t RES64_MIN_K = 40, RES64_ANY_K = 96;
// Between them only where the planes are small beside the plain kernel's rounds of 256 tiles (bytes <= 350000 k a
// round; mod 2^61 - 1, us plain / residue, k = 40 and 64: 34 x 4096 39 / 40 and 51 / 41 at 13 MB; 1000 x 1000 45 / 50 and
// 54 / 50 at 20 MB; 1 x 8192 37 / 51 and 47 / 52 at 25 MB; 10 x 20000 56 / 91 and 72 / 91 at 66 MB, x 128 141 / 100).
constexpr size_t RES64_WS = (size_t)4 << 30;      // bytes of planes held at a time; C runs in blocks that fit

// C op= A B by the residue route; false, with nothing launched, where it does not apply.
bool gemm64_residue(const hx_modctx64& ctx, const Gemm64Args& g, hipStream_t s) {
    if (g.k == 0 || !stream_scratch_safe(s)) return false;
    auto up = [](uint64_t x, uint64_t a) { return (x + a - 1) / a * a; };
    const uint64_t p = ctx.p;
    const uint32_t kc = std::min<uint32_t>(g.k, RES_KMAX / 64 * 64), N = moduli64(p, kc);
    if (N == 0) return false;
    const uint32_t side = residue_side(g.m, g.n, N);
    const uint64_t Kp0 = up(kc, 64);
    uint64_t mb = up(g.m, side), nb = up(g.n, side);
    auto bytes = [&] { return N * (mb * Kp0 + nb * Kp0 + mb * nb); };
    const uint64_t tiles = (uint64_t)((g.m + G64_TILE - 1) / G64_TILE) * ((g.n + G64_TILE - 1) / G64_TILE);
    if (g.k < RES64_ANY_K && (double)bytes() > 350e3 * g.k * std::max(1.0, (double)tiles / 256)) return false;
    while (bytes() > RES64_WS && (mb > side || nb > side)) (mb >= nb ? mb : nb) = up((mb >= nb ? mb : nb) / 2, side);
    ScratchLease planes;                         // held until every block is launched
    try {
        planes = stream_scratch(s, SCRATCH_U64, bytes());
    } catch (const Error& e) {
        if (e.code != HX_E_NOMEM) throw;
        return false;
    }
    char* const ws = (char*)planes.ptr;
    if (ws == nullptr) return false;

    Split64 sp{};
    ResArgs ra{};
    Crt64 ca{};
    sp.nmod = ca.nmod = N;
    // M / q_i mod p from prefix and suffix products (also M / q_i mod q_i, inverted by Euclid)
    uint64_t suf[RES_MAXQ + 1], pre = 1 % p;
    suf[N] = 1 % p;
    for (uint32_t i = N; i-- > 0;) suf[i] = (uint64_t)((unsigned __int128)suf[i + 1] * res_modulus((int)i) % p);
    for (uint32_t i = 0; i < N; ++i) {
        const uint32_t q = res_modulus((int)i);
        const uint64_t ci = (uint64_t)((unsigned __int128)pre * suf[i + 1] % p);
        pre = (uint64_t)((unsigned __int128)pre * q % p);
        uint32_t mq = 1;
        for (uint32_t j = 0; j < N; ++j)
            if (j != i) mq = mq * res_modulus((int)j) % q;
        int32_t r0 = (int32_t)q, r1 = (int32_t)mq, t0 = 0, t1 = 1;
        while (r1 != 0) {
            const int32_t d = r0 / r1, r2 = r0 - d * r1, t2 = t0 - d * t1;
            r0 = r1, r1 = r2, t0 = t1, t1 = t2;
        }
        HX_CHECK(r0 == 1, "residue route: moduli not coprime");
        const uint32_t y = (uint32_t)(t0 < 0 ? t0 + (int32_t)q : t0);
        sp.q[i] = q;
        res_modulus_consts(ra, i, q, y);
        uint32_t w8 = 1, wt[8];
        for (int j = 0; j < 8; ++j) {
            wt[j] = w8;
            w8 = w8 * 256 % q;
        }
        sp.tlo[i] = wt[0] | wt[1] << 8 | wt[2] << 16 | wt[3] << 24;
        sp.thi[i] = wt[4] | wt[5] << 8 | wt[6] << 16 | wt[7] << 24;
        sp.kq[i] = q - (uint32_t)(0x8000000000000000ull % q);
        sp.iq[i] = 1.0f / (float)q;
        for (int e = 0; e < 4; ++e) ca.c[i][e] = (uint16_t)(ci >> (16 * e));
        ca.f[i] = ((1u << 20) + q / 2) / q;
    }
    ca.pmm = p - pre;
    const Mod64 M = mod64_of(ctx);

    auto split = [&](const uint64_t* src, int64_t s_r, int64_t s_c, uint32_t R, uint32_t rows, uint32_t K, uint32_t Kp,
                     int8_t* out, const char* what) {
        const Prep64 a{src, s_r, s_c, R, K, Kp, out, (size_t)rows * Kp, p};
        prep64_kernel<<<dim3(rows / 32, (Kp + 127) / 128), 256, 0, s>>>(a, sp);
        after_launch(what);
    };
    for (uint64_t k0 = 0; k0 < g.k; k0 += kc) {
        const uint32_t K = (uint32_t)std::min<uint64_t>(kc, g.k - k0), Kp = (uint32_t)up(K, 64);
        for (uint64_t j0 = 0; j0 < g.n; j0 += nb) {
            const uint32_t n = (uint32_t)std::min<uint64_t>(nb, g.n - j0), Np = (uint32_t)up(n, side);
            int8_t* B8 = (int8_t*)ws;
            split(g.B + (int64_t)j0 * g.bcs + (int64_t)k0 * g.brs, g.bcs, g.brs, n, Np, K, Kp, B8, "prep64(B)");
            for (uint64_t i0 = 0; i0 < g.m; i0 += mb) {
                const uint32_t m = (uint32_t)std::min<uint64_t>(mb, g.m - i0), Mp = (uint32_t)up(m, side);
                int8_t* A8 = B8 + (size_t)N * Np * Kp;
                split(g.A + (int64_t)i0 * g.ars + (int64_t)k0 * g.acs, g.ars, g.acs, m, Mp, K, Kp, A8, "prep64(A)");
                ra.A8 = A8;
                ra.B8 = B8;
                ra.a_plane = (size_t)Mp * Kp;
                ra.b_plane = (size_t)Np * Kp;
                ra.Kp = Kp;
                ra.ntm = Mp / side;
                ra.ntn = Np / side;
                ra.R = (uint8_t*)(A8 + (size_t)N * Mp * Kp);
                ra.r_plane = (size_t)Mp * Np;
                residue_product(ra, N, side, s);
                ca.R = ra.R;
                ca.r_plane = ra.r_plane;
                ca.g = ResBlocks{side, ra.ntn};
                ca.m = m;
                ca.n = n;
                ca.C = g.C + (int64_t)i0 * g.crs + (int64_t)j0 * g.ccs;
                ca.crs = g.crs;
                ca.ccs = g.ccs;
                ca.op = k0 == 0 ? g.op : g.op == HX_OP_SUB ? HX_OP_SUB : HX_OP_ADD;
                crt64_kernel<<<(uint32_t)(ra.r_plane / 2048), 256, 0, s>>>(ca, M);
                after_launch("crt64_kernel");
            }
        }
    }
    return true;
}

}  // namespace
}  // namespace hx

using namespace hx;

extern "C" {

HX_API int hx_modctx64_init(uint64_t p, hx_modctx64* out) {
    return guard("hx_modctx64_init", [&] {
        HX_CHECK(out != nullptr, "out is NULL");
        HX_CHECK(p >= 2, "modulus must be >= 2");
        std::memset(out, 0, sizeof(*out));
        out->p = p;
        out->two64 = (uint64_t)(((unsigned __int128)1 << 64) % p);
        const unsigned __int128 t = (unsigned __int128)out->two64 * out->two64;
        out->r2 = (uint64_t)(t % p);
        if (p & 1u) {
            uint64_t inv = p;                       // p^-1 mod 2^64 by Newton (p odd: right to 3 bits)
            for (int i = 0; i < 6; ++i) inv *= 2u - p * inv;
            out->ninv = 0u - inv;
        }
    });
}

HX_API int hx_gemm_u64(const hx_modctx64* ctx, hx_view A, hx_view B, hx_view C, int op, hx_stream s) {
    return guard("hx_gemm_u64", [&] {
        HX_CHECK(ctx != nullptr && ctx->p >= 2, "bad modulus context");
        HX_CHECK(A.cols == B.rows && C.rows == A.rows && C.cols == B.cols, "gemm: shape mismatch");
        HX_CHECK(op == HX_OP_SET || op == HX_OP_ADD || op == HX_OP_SUB, "gemm: bad op");
        HX_CHECK(!views_overlap(C, A, 8, 8) && !views_overlap(C, B, 8, 8), "gemm: C aliases an operand");
        HX_CHECK(C.rows == 0 || C.cols == 0 || C.base != nullptr, "gemm: C is NULL");
        HX_CHECK((uint64_t)A.cols < (1ull << 32), "gemm: k must be below 2^32");
        if (C.rows == 0 || C.cols == 0) return;
        Gemm64Args g{C.rows, C.cols, A.cols, (const uint64_t*)A.base, A.rs, A.cs, (const uint64_t*)B.base, B.rs, B.cs,
                     (uint64_t*)C.base, C.rs, C.cs, op};
        if (g.k >= RES64_MIN_K && gemm64_residue(*ctx, g, (hipStream_t)s)) {
            stat_add(ST_GEMMS, 1);
            return;
        }
        const uint32_t tiles = ((g.m + G64_TILE - 1) / G64_TILE) * ((g.n + G64_TILE - 1) / G64_TILE);
        gemm64_kernel<<<tiles, G64_T, 0, (hipStream_t)s>>>(g, mod64_of(*ctx));
        after_launch("gemm64_kernel");
        stat_add(ST_GEMMS, 1);
    });
}

}  // extern "C"
