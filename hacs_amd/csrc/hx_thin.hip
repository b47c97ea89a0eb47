// hx_thin.hip -- C op= A B mod p for products too shallow or too small for the limb kernels: the limbs are split
// on the fly (no planes in memory, no separate passes) and each 32 x 32 block is one short burst of int8 MFMAs.
//
// One wave owns 32 columns; a workgroup of four waves 128.  Each wave splits its B fragment (up to 64 k) once and
// keeps it in registers; the workgroup walks down `nb` blocks of 32 rows of A, which its 256 threads split
// together into LDS in fragment order (double-buffered: one barrier per block), and every wave multiplies the
// block by its B fragment, reduces (limb_small_product) and applies the op.  Deeper products of few rows take K
// in steps of 64, one block of rows per workgroup, adding the residues.
//
// What bounds it: at k <= 64 the read and write of C and the reduction's ~20 operations per output (the 16
// MFMAs of a four-limb block take less than either).  4095 x 4033 x 32 mod 2^31 - 1: 34 us for C = A B,
// 47 us for C -= A B (132 MB of C: 2.8 TB/s), against 100 and 118 us on the plain kernel; 96 x 80 x 64 about 6 us
// on the device against 18.
#include "hx_gemm.h"
#include "hx_limbs.h"

#include <algorithm>

namespace hx {
namespace {

constexpr int TH_N = 128;                // columns per workgroup
// Where the automatic choice comes here (us, plain / limb kernel 4 / here, mod 2147483629): every depth up to 64
// (4095 x 4033 x 4 91 / 69 / 31, x 32 100 / 71 / 34, x 64 162 / 72 / 45; 64^3 18 / 18 / 12; 1000^2 x 4 13 / 20 / 12),
// (16^3 12 / 18 / 12: smaller ones stay on the plain kernel), and to 256 for products below 4e6 multiply-adds (128^3 30 / 21 / 12, 100 x 100 x 256 52 / 25 / 20; 80 x 80 x 512
// 98 / 30 / 36).
constexpr uint32_t TH_KMAX = 256;

struct ThinArgs {
    GemmArgs g;
    uint32_t half;
    SmallConsts c;
    uint32_t ntn;                        // workgroups across
    uint32_t nb;                         // blocks of 32 rows per workgroup
};

// KS k-steps of 32 at a time.  DEEP: K runs in steps of 64 (KS = 2, nb = 1).  RMW: the op reads C.
template <int L, int KS, bool DEEP, bool RMW>
__global__ __launch_bounds__(256) void thin_kernel(ThinArgs t) {
    __shared__ __attribute__((aligned(16))) uint32_t As[2][KS][L][256];
    const GemmArgs& g = t.g;
    const uint32_t tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, lr = lane & 31, lg = lane >> 5;
    const uint32_t col = (blockIdx.x % t.ntn) * TH_N + wave * 32 + lr;
    const uint32_t row0 = (blockIdx.x / t.ntn) * 32 * t.nb;
    const uint32_t nb = min(t.nb, (g.m - row0 + 31) / 32);
    const bool cok = col < g.n;

    // this thread's part of an A block: row tid % 32, k = 4 (tid / 32) .. + 3 of each k-step
    const uint32_t ar = tid & 31, ak = (tid >> 5) * 4;
    uint32_t av[KS][4];
    auto load_a = [&](uint32_t rb, uint32_t k0) {
        const uint32_t row = row0 + 32 * rb + ar;
        const uint32_t* src = g.A + (int64_t)row * g.ars;
#pragma unroll
        for (int ks = 0; ks < KS; ++ks)
#pragma unroll
            for (int b = 0; b < 4; ++b) {
                const uint32_t k = k0 + 32 * ks + ak + b;
                av[ks][b] = row < g.m && k < g.k ? src[(int64_t)k * g.acs] : 0u;
            }
    };
    auto store_a = [&](int buf) {
#pragma unroll
        for (int ks = 0; ks < KS; ++ks) {
            uint32_t w[L];
            limb_split4<L>(av[ks], t.c.p, t.half, w);
            // fragment order: lane ar + 32 (k / 16), 16 bytes per lane
#pragma unroll
            for (int s = 0; s < L; ++s) As[buf][ks][s][(ar + 32 * (ak >> 4)) * 4 + ((ak >> 2) & 3)] = w[s];
        }
    };
    limb_v4i fb[KS][L];
    uint32_t bv[KS][16];
    auto load_b = [&](uint32_t k0) {
#pragma unroll
        for (int ks = 0; ks < KS; ++ks)
#pragma unroll
            for (int i = 0; i < 16; ++i) {
                const uint32_t k = k0 + 32 * ks + 16 * lg + i;
                bv[ks][i] = cok && k < g.k ? g.B[(int64_t)k * g.brs + (int64_t)col * g.bcs] : 0u;
            }
    };
    auto split_b = [&] {
#pragma unroll
        for (int ks = 0; ks < KS; ++ks)
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                const uint32_t v[4] = {bv[ks][4 * j], bv[ks][4 * j + 1], bv[ks][4 * j + 2], bv[ks][4 * j + 3]};
                uint32_t w[L];
                limb_split4<L>(v, t.c.p, t.half, w);
#pragma unroll
                for (int s = 0; s < L; ++s) fb[ks][s][j] = (int)w[s];
            }
    };
    auto read_a = [&](int buf, limb_v4i (&fa)[KS][L]) {
#pragma unroll
        for (int ks = 0; ks < KS; ++ks)
#pragma unroll
            for (int s = 0; s < L; ++s) fa[ks][s] = *(const limb_v4i*)&As[buf][ks][s][lane * 4];
    };

    uint32_t cn[16];
    auto load_c = [&](uint32_t rb) {
        const uint32_t r0 = row0 + 32 * rb + 4 * lg;
#pragma unroll
        for (int e = 0; e < 16; ++e) {
            const uint32_t row = r0 + (e / 4) * 8 + e % 4;
            cn[e] = cok && row < g.m ? g.Cin[(int64_t)row * g.cirs + (int64_t)col * g.cics] : 0u;
        }
    };

    load_a(0, 0);
    load_b(0);
    if (RMW) load_c(0);
    store_a(0);
    split_b();
    for (uint32_t rb = 0; rb < nb; ++rb) {
        __syncthreads();                         // block rb is in LDS, every wave done with the other buffer
        const uint32_t r0 = row0 + 32 * rb + 4 * lg;
        if (!DEEP && rb + 1 < nb) load_a(rb + 1, 0);
        limb_v4i fa[KS][L];
        read_a(rb & 1, fa);
        uint32_t cv[16];                         // this block's C; the next one's on its way
        if (RMW) {
#pragma unroll
            for (int e = 0; e < 16; ++e) cv[e] = cn[e];
            if (!DEEP && rb + 1 < nb) load_c(rb + 1);
        }
        uint32_t r[16];
        if (DEEP) {
            // the next step's entries are on their way while this one is multiplied
            for (uint32_t k0 = 64, it = 1;; k0 += 64, ++it) {
                const bool more = k0 < g.k;
                if (more) {
                    load_a(0, k0);
                    load_b(k0);
                }
                uint32_t r2[16];
                limb_small_product<L, KS>(fa, fb, t.c, r2);
#pragma unroll
                for (int e = 0; e < 16; ++e) r[e] = it == 1 ? r2[e] : addm(r[e], r2[e], t.c.p);
                if (!more) break;
                store_a(it & 1);
                split_b();
                __syncthreads();
                read_a(it & 1, fa);
            }
        } else {
            limb_small_product<L, KS>(fa, fb, t.c, r);
        }
        if (!DEEP && rb + 1 < nb) store_a((rb + 1) & 1);
        if (cok) {
#pragma unroll
            for (int e = 0; e < 16; ++e) {
                const uint32_t row = r0 + (e / 4) * 8 + e % 4;
                if (row < g.m)
                    g.Cout[(int64_t)row * g.cors + (int64_t)col * g.cocs] =
                        RMW ? apply_op(cv[e], r[e], g.op, t.c.p) : r[e];
            }
        }
    }
}

template <int L, bool RMW>
void launch_thin(const ThinArgs& t, uint32_t blocks, hipStream_t s) {
    if (t.g.k <= 32) thin_kernel<L, 1, false, RMW><<<blocks, 256, 0, s>>>(t);
    else if (t.g.k <= 64) thin_kernel<L, 2, false, RMW><<<blocks, 256, 0, s>>>(t);
    else thin_kernel<L, 2, true, RMW><<<blocks, 256, 0, s>>>(t);
    after_launch("thin_kernel");
}
template <int L>
void launch_thin(const ThinArgs& t, uint32_t blocks, hipStream_t s) {
    if (t.g.op == HX_OP_SET) launch_thin<L, false>(t, blocks, s);
    else launch_thin<L, true>(t, blocks, s);
}

}  // namespace

bool thin_applies(const hx_modctx& ctx, uint32_t m, uint32_t n, uint32_t k) {
    if (ctx.limbs == 0 || ctx.p >= 0x80000000u || k == 0 || (uint64_t)m * n < 256) return false;
    return k <= 64 || (k <= TH_KMAX && (double)m * n * k < 4.0e6);
}

void gemm_thin(const hx_modctx& ctx, const GemmArgs& g, hipStream_t s) {
    HX_CHECK(g.m_dev == nullptr && g.k_dev == nullptr && g.a_rows == nullptr && g.a_cols == nullptr &&
                 g.c_rows == nullptr && ctx.limbs >= 1 && ctx.p < 0x80000000u && g.k >= 1,
             "thin product: no plan for this product");
    if (g.m == 0 || g.n == 0) return;
    ThinArgs t{};
    t.g = g;
    t.half = (ctx.p - 1) / 2;
    t.c = SmallConsts{ctx.p, 1.0 / (double)ctx.p};
    t.ntn = (g.n + TH_N - 1) / TH_N;
    const uint32_t rblocks = (g.m + 31) / 32;
    // as many row blocks per workgroup (one split of B) as leave two workgroups per compute unit
    // (4095 x 4033 x 32: 8 blocks 34 us, 4 blocks 37, 2 blocks 43, 1 block 52; 7 blocks, 608 workgroups, 20 us more where C
    // is read).  Of one workgroup across, reading C at k <= 32 where the loads of C decide, only the waves with
    // columns count: 100000 x 16 x 32 40 us with one block, 49 with six (plain kernel 38); at k = 64 or without the
    // read the longer walk is at least as fast (mod 65521 18 us / 20).
    const uint64_t waves = t.ntn == 1 && g.op != HX_OP_SET && g.k <= 32 ? (g.n + 31) / 32 : 4 * (uint64_t)t.ntn;
    t.nb = g.k > 64 ? 1 : (uint32_t)std::clamp<uint64_t>(rblocks * waves / 2048, 1, 8);
    const uint32_t blocks = t.ntn * ((rblocks + t.nb - 1) / t.nb);
    switch (ctx.limbs) {
        case 1: launch_thin<1>(t, blocks, s); break;
        case 2: launch_thin<2>(t, blocks, s); break;
        case 3: launch_thin<3>(t, blocks, s); break;
        default: launch_thin<4>(t, blocks, s); break;
    }
}

}  // namespace hx
