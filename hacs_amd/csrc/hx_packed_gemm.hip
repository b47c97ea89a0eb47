// hx_packed_gemm.hip -- C = A B over F_2 / F_3 on bit-packed rows as a 4-bit matrix product on the MFMAs.
//
// The entries of F_2 ({0, 1}) and F_3 ({0, 1, -1}) are exact in the 4-bit format e2m1 (codes 0x0, 0x2 = +1,
// 0xA = -1), every product of two entries is 0 or +-1, and a sum of at most PG_KMAX = 2^23 of them is an
// integer below 2^24: exact in the float accumulators of v_mfma_f32_32x32x64_f8f6f4 in any order.  The
// result entry is that integer mod P, written back as bits.
//
//  * pg_prep_a_kernel / pg_prep_b_kernel expand the operands into nibble planes, k contiguous (A's rows; B's
//    columns, transposed 64 x 64 bits per wave in registers).  Both put bit 4 i + d of every 32-bit group
//    in nibble i of word d: the order of k inside a group is free as long as A and B share it, and this one
//    costs a shift and a mask per eight entries.
//  * pg_kernel: 256 x 256 (or 128 x 128) outputs per 512-thread workgroup, 128 k per stage copied straight
//    into a three-stage LDS ring, the next fragments read while the MFMAs of the current ones run.  The
//    epilogue reduces the sums mod P and packs 32 columns per ballot.
//
// What bounds it: the matrix cores and, about as much, the LDS reads that feed them (six 1 KB fragments per
// eight 32-cycle MFMAs and wave).  8192^3 over F_3: 0.263 ms for the call (the expansion of both operands
// included, 4.2 P multiply-adds/s) against 5.51 ms on subset-sum tables in LDS; 4096^3 51 us against 2.76 ms
// (F_2: 44 us against 0.98 ms); 64^3 15.5 us against 24 us, 4096 x 4096 x 128 over F_2 14 us against 33 us:
// it is the faster one at every size measured but long F_2 operands of one word of k, so the tables remain for those
// and for captures, where this route's planes (library scratch that a later call may move) must not be recorded
// in a graph.
#include "hx_packed_gemm.h"

#include <algorithm>

namespace hx {
namespace {

typedef int v4i __attribute__((ext_vector_type(4)));
typedef int v8i __attribute__((ext_vector_type(8)));
typedef float v16f __attribute__((ext_vector_type(16)));

constexpr uint32_t PG_KMAX = 1u << 23;       // terms of one exact float sum (multiple of 128)
constexpr size_t PG_WS = 512u << 20;         // bytes of operand planes held at a time; K runs in chunks that fit

__device__ __forceinline__ int pg_swz(int row) { return ((row >> 2) & 3) ^ (row & 2); }
constexpr int pg_wait(int vm, int lgkm) { return (vm & 15) | ((vm >> 4) << 14) | (7 << 4) | ((lgkm & 15) << 8); }

// Word d of the 16-byte nibble strip of 32 entries: nibble i holds entry 4 i + d (nz = non-zero, neg = -1).
__device__ __forceinline__ v4i pg_nibbles(uint32_t nz, uint32_t neg) {
    v4i v;
#pragma unroll
    for (int d = 0; d < 4; ++d)
        v[d] = (int)((((nz >> d) & 0x11111111u) << 1) | (((neg >> d) & 0x11111111u) << 3));
    return v;
}

// A's rows: one 32-entry group per thread (4 bytes per plane in, 16 bytes out).  Groups past `groups` (the
// chunk's words) and rows past m are zero.  g0: the chunk's first 32-entry group.
template <int P>
__global__ __launch_bounds__(256) void pg_prep_a_kernel(const uint64_t* A, uint32_t lda, uint32_t m, uint32_t g0,
                                                        uint32_t groups, uint32_t Kb, uint32_t Mp, uint8_t* out) {
    const uint32_t per = Kb / 16;
    const uint64_t idx = (uint64_t)blockIdx.x * 256 + threadIdx.x;
    if (idx >= (uint64_t)Mp * per) return;
    const uint32_t row = (uint32_t)(idx / per), g = (uint32_t)(idx % per);
    uint32_t one = 0, two = 0;
    if (row < m && g < groups) {
        const uint32_t* r = (const uint32_t*)(A + (size_t)row * lda * (P - 1)) + g0 + g;
        one = r[0];
        if (P == 3) two = r[2 * (size_t)lda];
    }
    *(v4i*)(out + (size_t)row * Kb + 16 * (size_t)g) = pg_nibbles(one | two, two);
}

// A 64 x 64 bit transpose over a wave: lane l holds row l on entry and column l on return.
__device__ __forceinline__ uint64_t pg_transpose(uint64_t x, int lane) {
    const uint64_t keep[6] = {0x00000000ffffffffull, 0x0000ffff0000ffffull, 0x00ff00ff00ff00ffull,
                              0x0f0f0f0f0f0f0f0full, 0x3333333333333333ull, 0x5555555555555555ull};
#pragma unroll
    for (int t = 0; t < 6; ++t) {
        const int sft = 32 >> t;
        const uint64_t y = (uint64_t)__shfl_xor((unsigned long long)x, sft), mk = keep[t];
        x = (lane & sft) ? ((x & ~mk) | ((y >> sft) & mk)) : ((x & mk) | ((y & mk) << sft));
    }
    return x;
}

// B's columns: wave w of a workgroup takes the 64 columns of word 4 blockIdx.y + w, 128 k (one stage) per
// blockIdx.x: two transposes per plane, 64 contiguous bytes out per column.  Rows at or past kend (the chunk's
// end, at most k) and words past nw read as zero.
template <int P>
__global__ __launch_bounds__(256) void pg_prep_b_kernel(const uint64_t* B, uint32_t ldb, uint32_t k0, uint32_t kend,
                                                        uint32_t nw, uint32_t Kb, uint32_t Np, uint8_t* out) {
    const int lane = threadIdx.x & 63;
    const uint32_t c = blockIdx.y * 4 + (threadIdx.x >> 6);
    if (64 * c >= Np) return;                    // (whole waves; Np is a multiple of 128)
    uint8_t* dst = out + (size_t)(64 * c + lane) * Kb + 64 * (size_t)blockIdx.x;
#pragma unroll
    for (int h = 0; h < 2; ++h) {
        const uint32_t t = k0 + 128 * blockIdx.x + 64 * h + lane;
        uint64_t one = 0, two = 0;
        if (t < kend && c < nw) {
            const uint64_t* r = B + (size_t)t * ldb * (P - 1) + c;
            one = r[0];
            if (P == 3) two = r[ldb];
        }
        one = pg_transpose(one, lane);
        if (P == 3) two = pg_transpose(two, lane);
        const uint64_t nz = one | two;
        *(v4i*)(dst + 32 * h) = pg_nibbles((uint32_t)nz, (uint32_t)two);
        *(v4i*)(dst + 32 * h + 16) = pg_nibbles((uint32_t)(nz >> 32), (uint32_t)(two >> 32));
    }
}

struct PgArgs {
    const uint8_t* A4;           // Mp rows of Kb bytes (two entries per byte)
    const uint8_t* B4;           // Np rows of Kb bytes
    uint32_t Kb;                 // multiple of 64
    uint32_t ntm, ntn;
    uint32_t m, nw;              // rows and words per plane of C
    uint64_t* C;
    uint32_t ldc;
    int accumulate;
};

// Consecutive workgroups go round-robin over the 8 XCDs: each XCD gets a contiguous run of tiles, in groups
// of 8 tile rows, so the planes' rows a run touches stay in its L2.
__device__ __forceinline__ void pg_tile_of(uint32_t b, uint32_t ntm, uint32_t ntn, uint32_t& tm, uint32_t& tn) {
    const uint32_t T = ntm * ntn, per = T / 8;
    const uint32_t t = b < per * 8 ? (b % 8) * per + b / 8 : b;
    const uint32_t width = 8 * ntn, group = t / width, gm = min(ntm - 8 * group, 8u), in = t % width;
    tm = 8 * group + in % gm;
    tn = in / gm;
}

// 64 LA x 128 LB outputs per workgroup of eight waves (two down, four across), LA x LB blocks of 32 x 32 per
// wave: rows 64 s + 32 wm, columns 128 t + 32 wn.
template <int LA, int LB>
struct PgTile {
    static constexpr int SA = LA * 64 * 64, STAGE = SA + LB * 128 * 64, NBLK = 4 * LA + 8 * LB, PER = NBLK / 8;
    static_assert(NBLK % 8 == 0, "every wave copies the same number of 1 KB blocks");

    // stage kt: NBLK blocks of 16 rows x 64 bytes, one 16-byte-per-lane direct-to-LDS copy each
    static __device__ __forceinline__ void issue(const PgArgs& a, const uint8_t* Ab, const uint8_t* Bb, int wave,
                                                 uint32_t kt, uint8_t* st) {
        const size_t k0 = (size_t)kt * 64;
#pragma unroll
        for (int i = 0; i < PER; ++i) {
            const int blk = wave + 8 * i;
            const uint8_t* src;
            uint8_t* dst;
            if (blk < 4 * LA) {
                const int b = blk >> 2, g = blk & 3;
                src = Ab + (size_t)(b * 64 + 16 * g) * a.Kb + k0;
                dst = st + b * 4096 + g * 1024;
            } else {
                const int b = (blk - 4 * LA) >> 3, g = (blk - 4 * LA) & 7;
                src = Bb + (size_t)(b * 128 + 16 * g) * a.Kb + k0;
                dst = st + SA + b * 8192 + g * 1024;
            }
            __builtin_amdgcn_global_load_lds((const void*)src, (__attribute__((address_space(3))) void*)dst, 16, 0, 0);
        }
    }
    struct Frag {
        v4i a[LA], b[LB];
    };
    static __device__ __forceinline__ void read(const uint8_t* st, int ks, int wm, int wn, int lane, Frag& f) {
        const int lr = lane & 31, q = ks * 2 + (lane >> 5), ra = wm * 32 + lr, rb = wn * 32 + lr;
#pragma unroll
        for (int s = 0; s < LA; ++s) f.a[s] = *(const v4i*)(st + s * 4096 + ra * 64 + 16 * (q ^ pg_swz(ra)));
#pragma unroll
        for (int t = 0; t < LB; ++t) f.b[t] = *(const v4i*)(st + SA + t * 8192 + rb * 64 + 16 * (q ^ pg_swz(rb)));
    }
    static __device__ __forceinline__ void mfma(const Frag& f, v16f (&acc)[LA][LB]) {
        const v4i z = {0, 0, 0, 0};
#pragma unroll
        for (int s = 0; s < LA; ++s)
#pragma unroll
            for (int t = 0; t < LB; ++t) {
                const v8i va = __builtin_shufflevector(f.a[s], z, 0, 1, 2, 3, 4, 5, 6, 7);
                const v8i vb = __builtin_shufflevector(f.b[t], z, 0, 1, 2, 3, 4, 5, 6, 7);
                // formats 4 / 4: e2m1 on both sides; zero scale operands: the unscaled instruction
                acc[s][t] = __builtin_amdgcn_mfma_scale_f32_32x32x64_f8f6f4(va, vb, acc[s][t], 4, 4, 0, 0, 0, 0);
            }
    }
};

template <int P, int LA, int LB>
__global__ __launch_bounds__(512, 1) void pg_kernel(PgArgs a) {
    using T = PgTile<LA, LB>;
    __shared__ __attribute__((aligned(1024))) uint8_t s0[T::STAGE];
    __shared__ __attribute__((aligned(1024))) uint8_t s1[T::STAGE];
    __shared__ __attribute__((aligned(1024))) uint8_t s2[T::STAGE];
    uint32_t tm, tn;
    pg_tile_of(blockIdx.x, a.ntm, a.ntn, tm, tn);
    const uint32_t m0 = tm * (64 * LA), n0 = tn * (128 * LB);
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int wm = wave & 1, wn = wave >> 1;
    v16f acc[LA][LB];
#pragma unroll
    for (int s = 0; s < LA; ++s)
#pragma unroll
        for (int t = 0; t < LB; ++t)
#pragma unroll
            for (int r = 0; r < 16; ++r) acc[s][t][r] = 0.0f;

    const int br = lane >> 2, bq = (lane & 3) ^ pg_swz(br);
    const uint8_t* Ab = a.A4 + (size_t)(m0 + br) * a.Kb + 16 * bq;
    const uint8_t* Bb = a.B4 + (size_t)(n0 + br) * a.Kb + 16 * bq;
    const uint32_t KT = a.Kb / 64;
    auto barrier = [&] {
        __atomic_signal_fence(__ATOMIC_SEQ_CST);
        __builtin_amdgcn_s_barrier();
        __atomic_signal_fence(__ATOMIC_SEQ_CST);
    };
    T::issue(a, Ab, Bb, wave, 0, s0);
    if (KT > 2) {
        T::issue(a, Ab, Bb, wave, 1, s1);
        T::issue(a, Ab, Bb, wave, 2, s2);
        __builtin_amdgcn_s_waitcnt(pg_wait(2 * T::PER, 15));
    } else {
        if (KT > 1) T::issue(a, Ab, Bb, wave, 1, s1);
        __builtin_amdgcn_s_waitcnt(pg_wait(0, 15));
    }
    barrier();
    typename T::Frag fa, fb;
    T::read(s0, 0, wm, wn, lane, fa);
    __builtin_amdgcn_s_waitcnt(pg_wait(63, 0));
    // stage kt: MFMAs of its first half while the second half is read; stage kt + 1 landed and every wave done
    // reading stage kt (barrier); stage kt + 3 copied into its slot; MFMAs of the second half while the next
    // stage's first half is read.  `more`: stage kt + 3 exists, so stage kt + 2 may stay in flight at the
    // barrier (the steady loop has no branch: the compiler's own wait tracking then adds no waits to it).
    auto body = [&](uint32_t kt, uint8_t* cur, const uint8_t* nxt, bool more) {
        T::read(cur, 1, wm, wn, lane, fb);
        __builtin_amdgcn_sched_barrier(0);
        T::mfma(fa, acc);
        __builtin_amdgcn_sched_barrier(0);
        __builtin_amdgcn_s_waitcnt(pg_wait(63, 0));
        if (more) __builtin_amdgcn_s_waitcnt(pg_wait(T::PER, 15));
        else __builtin_amdgcn_s_waitcnt(pg_wait(0, 15));
        barrier();
        if (more) T::issue(a, Ab, Bb, wave, kt + 3, cur);
        T::read(nxt, 0, wm, wn, lane, fa);
        __builtin_amdgcn_sched_barrier(0);
        T::mfma(fb, acc);
        __builtin_amdgcn_sched_barrier(0);
        __builtin_amdgcn_s_waitcnt(pg_wait(63, 0));
    };
    uint32_t kt = 0;
    for (; kt + 5 < KT; kt += 3) {
        body(kt, s0, s1, true);
        body(kt + 1, s1, s2, true);
        body(kt + 2, s2, s0, true);
    }
    uint8_t* const ring[3] = {s0, s1, s2};
#pragma unroll
    for (int j = 0; j < 5; ++j)                 // at most five stages left, the last one below
        if (kt + j + 1 < KT) body(kt + j, ring[j % 3], ring[(j + 1) % 3], kt + j + 3 < KT);
    const uint32_t ls = (KT - 1) % 3;
    T::read(ls == 0 ? s0 : ls == 1 ? s1 : s2, 1, wm, wn, lane, fb);
    T::mfma(fa, acc);
    T::mfma(fb, acc);

    // accumulator register r: rows (r / 4) 8 + r % 4 (lanes 0 .. 31) and + 4 (lanes 32 .. 63), column lane % 32.
    // Lane r + 16 h keeps the 32 column bits of register r's row of half h.
    const int keep = lane & 15, kh = (lane >> 4) & 1;
    const uint32_t krow = (uint32_t)((keep / 4) * 8 + kh * 4 + keep % 4);
#pragma unroll
    for (int s = 0; s < LA; ++s)
#pragma unroll
        for (int t = 0; t < LB; ++t) {
            uint32_t one = 0, two = 0;
#pragma unroll
            for (int r = 0; r < 16; ++r) {
                const int32_t v = (int32_t)acc[s][t][r];
                uint64_t b1, b2 = 0;
                if (P == 2) {
                    b1 = __ballot(v & 1);
                } else {
                    const uint32_t e = (uint32_t)(v + 3 * 5592406) % 3u;        // 3 * 5592406 > 2^24 > |v|
                    b1 = __ballot(e == 1);
                    b2 = __ballot(e == 2);
                }
                if (keep == r) {
                    one = kh ? (uint32_t)(b1 >> 32) : (uint32_t)b1;
                    two = kh ? (uint32_t)(b2 >> 32) : (uint32_t)b2;
                }
            }
            const uint32_t row = m0 + s * 64 + wm * 32 + krow, cw = (n0 + t * 128 + wn * 32) / 32;
            if (lane < 32 && row < a.m && cw < 2 * a.nw) {
                uint32_t* c = (uint32_t*)(a.C + (size_t)row * a.ldc * (P - 1)) + cw;
                if (P == 2) {
                    c[0] = a.accumulate ? c[0] ^ one : one;
                } else {
                    uint32_t* c2 = c + 2 * (size_t)a.ldc;
                    if (a.accumulate) {
                        const uint32_t x1 = c[0], x2 = c2[0], x0 = ~(x1 | x2), y0 = ~(one | two);
                        const uint32_t z1 = (x1 & y0) | (x0 & one) | (x2 & two), z2 = (x2 & y0) | (x0 & two) | (x1 & one);
                        one = z1;
                        two = z2;
                    }
                    c[0] = one;
                    c2[0] = two;
                }
            }
        }
}

inline uint64_t up(uint64_t x, uint64_t a) { return (x + a - 1) / a * a; }

}  // namespace

template <int P>
bool packed_gemm(uint32_t m, uint32_t n, uint32_t k, const uint64_t* A, uint32_t lda, const uint64_t* B, uint32_t ldb,
                 uint64_t* C, uint32_t ldc, bool accumulate, hipStream_t s) {
    if (m == 0 || n == 0 || k == 0 || !stream_scratch_safe(s)) return false;
    // the 128 x 128 tile where 256 x 256 tiles would leave compute units idle
    const bool small = up(m, 256) / 256 * (up(n, 256) / 256) < 256;
    const uint64_t tile = small ? 128 : 256, Mp = up(m, tile), Np = up(n, tile);
    if (Mp > 0xffffffffu || Np > 0xffffffffu) return false;
    // One word of A over F_2 and long operands: the tables take one pass, the planes pad k to 128 (us, tables / here:
    // 1000000 x 64 x 64 69 / 84, 1000 x 300000 x 64 93 / 105; 100000 x 64 x 64 18 / 17, 20000^2 x 64 128 / 121, 1000000 x 64 x 200
    // 257 / 107; over F_3 201 / 135 for the first).
    if (P == 2 && k <= 64 && Mp + Np > 200000) return false;
    // pg_kernel's grid: a launch holds fewer than 2^32 threads (C of 69 GB and more runs on the tables)
    if ((Mp / tile) * (Np / tile) * 512 >= (uint64_t)1 << 32) return false;
    const uint64_t fit = PG_WS / (Mp + Np) * 2 / 128 * 128;                     // k whose planes fit PG_WS
    if (fit == 0) return false;
    const uint32_t chunk = (uint32_t)std::min<uint64_t>({up(k, 128), fit, PG_KMAX});
    ScratchLease planes;                         // held until every chunk is launched
    try {
        planes = stream_scratch(s, SCRATCH_PACKED, (Mp + Np) * (chunk / 2));
    } catch (const Error& e) {
        if (e.code != HX_E_NOMEM) throw;
        return false;
    }
    uint8_t* const ws = (uint8_t*)planes.ptr;
    if (ws == nullptr) return false;
    const uint32_t nw = (n + 63) / 64;
    for (uint64_t k0 = 0; k0 < k; k0 += chunk) {
        const uint32_t kend = (uint32_t)std::min<uint64_t>(k, k0 + chunk);
        const uint32_t Kb = (uint32_t)(up(kend - k0, 128) / 2);
        PgArgs a{};
        a.A4 = ws;
        a.B4 = ws + Mp * Kb;
        a.Kb = Kb;
        a.ntm = (uint32_t)(Mp / tile);
        a.ntn = (uint32_t)(Np / tile);
        a.m = m;
        a.nw = nw;
        a.C = C;
        a.ldc = ldc;
        a.accumulate = accumulate || k0 != 0;
        const uint32_t groups = (uint32_t)(up(kend - k0, 64) / 32);
        pg_prep_a_kernel<P><<<(uint32_t)((Mp * (Kb / 16) + 255) / 256), 256, 0, s>>>(A, lda, m, (uint32_t)(k0 / 32), groups,
                                                                                     Kb, (uint32_t)Mp, ws);
        after_launch("pg_prep_a_kernel");
        pg_prep_b_kernel<P><<<dim3(Kb / 64, (uint32_t)((Np + 255) / 256)), 256, 0, s>>>(
            B, ldb, (uint32_t)k0, kend, nw, Kb, (uint32_t)Np, ws + Mp * Kb);
        after_launch("pg_prep_b_kernel");
        if (small) pg_kernel<P, 2, 1><<<a.ntm * a.ntn, 512, 0, s>>>(a);
        else pg_kernel<P, 4, 2><<<a.ntm * a.ntn, 512, 0, s>>>(a);
        after_launch("pg_kernel");
    }
    return true;
}

template bool packed_gemm<2>(uint32_t, uint32_t, uint32_t, const uint64_t*, uint32_t, const uint64_t*, uint32_t, uint64_t*,
                             uint32_t, bool, hipStream_t);
template bool packed_gemm<3>(uint32_t, uint32_t, uint32_t, const uint64_t*, uint32_t, const uint64_t*, uint32_t, uint64_t*,
                             uint32_t, bool, hipStream_t);

}  // namespace hx
