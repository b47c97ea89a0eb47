// hx_f2.hip -- linear algebra over F_2 on bit-packed rows (binary::BitMatrix, Binary/BitMatrix.h:49-140):
// the in-place reduced row echelon form with its rank and pivot columns (rref, BitMatrix.h:101-105),
// and the product C = A B (multiply_m4rm, BitMatrix.h:129).
//
// Layout (the reference's): row i of an m x n bit matrix is `ldw` 64-bit words, bit j of the row is
// bit j % 64 of word j / 64; padding bits (columns >= n) are zero and stay zero.
//
// Over F_2 an exact XOR elimination is exact arithmetic and the RREF, its pivot columns (the column
// rank profile) and hence the rank are unique functions of A, so any correct elimination order gives
// the reference's bytes (BitMatrix.h:24-28) -- this one is designed for the GPU:
//
//  * Column panels of 64 (one word).  Every row keeps a 64-bit mask over the panel's pivot slots t:
//    row_i = orig_i + sum_{t in mask_i} orig_{P_t} (orig = the rows at the panel's start), so the rest of each
//    row is one product away.  Any pivot row serves (the RREF does not depend on it), so the search is not
//    run over all rows: one wave eliminates the panel word of the first 128 rows that have one (f2_wave_eliminate:
//    a ballot per column, no barrier, Gauss-Jordan), and every other row then takes the pivots of its own
//    bits in one step, by byte tables of the pivots' words and masks.  What is left non-zero after two such
//    rounds (few independent rows among the first ones) goes through a column-by-column search over all rows.
//  * One launch per panel (f2_panel_update_kernel): block 0 runs panel w -- first bringing word w up to date with
//    panel w - 1 -- while the other blocks apply panel w - 1 to the words behind w: per group of 8 slots a
//    256-entry LDS table of all XOR combinations of those 8 pivot rows, one lookup per byte of a row's mask
//    (the words before the panel need nothing: a row that is not a pivot is zero there).  f2_copy_kernel then
//    sets the panel's pivot rows aside.
//    8192^2 of rank 6000: 3.7 ms, against 16.3 ms with one search over all rows per column (two barriers each,
//    104 us per panel) and a separate update.  Bound by block 0's chain: 32 us per panel, of it 9 us the 64
//    columns of the wave's elimination, 6 us the other rows' table look-ups, 4 us each the word's load and the
//    previous panel, the rest tables, candidates and the store; then 4 us f2_copy_kernel.
//  * f2_finish: the pivot rows in pivot order to the top, zero rows below (the non-pivot rows are
//    zero after the last panel: every row is reduced against every pivot).
//  * The product runs on the matrix cores (hx_packed_gemm.hip).  Where that route does not
//    apply (hx_packed_gemm.h): f2_gemm_kernel, the same tables over B's rows, 64 at a time, accumulating
//    the output words in registers (one lookup per byte of A's word).
#include <algorithm>
#include <cstring>
#include <vector>

#include "hx_common.h"
#include "hx_packed_gemm.h"

namespace hx {
namespace {

constexpr int F2_PT = 1024;              // threads of the panel kernel
constexpr int F2_RMAX = 16;              // rows per thread held in registers (m <= 16384)
constexpr int F2_UT = 256;               // threads of the table kernels
constexpr int F2_WS = 4;                 // words per table-kernel workgroup
constexpr int F2_ROWS = 1024;            // rows per table-kernel workgroup

// Device-side state of one elimination.
struct F2State {
    uint32_t rank;                       // pivots so far
    uint32_t k;                          // this panel's pivots
};

constexpr int F2_CAND = 128;             // rows of one wave's elimination (two per lane)
constexpr int F2_ROUNDS = 2;             // such rounds before the column-by-column search

// LDS of the panel block (aliased by the update blocks' tables).
struct F2PanelLds {
    uint64_t tab[8][256][2];             // per byte of a row's word: XOR of the pivots' words / masks
    uint64_t prev[8][256];               // the previous panel's pivot rows at this word, per byte of a mask
    uint64_t px[64], pc[64];             // by column: the pivot row's reduced word and its combination (0: none)
    uint64_t cx[F2_CAND], cc[F2_CAND];   // candidate rows: word, mask
    uint32_t crow[F2_CAND];
    uint64_t wor[F2_PT / 64];
    uint32_t wcnt[F2_PT / 64];
    uint32_t slot_row[64], slot_col[64]; // by slot (order of discovery)
    uint32_t col_slot[64];
    uint64_t newcols;                    // this round's pivot columns
    uint32_t k;
    uint64_t s_pw[2], s_pc[2];
    uint32_t s_min[2][F2_PT / 64];
    uint8_t pcol1[F2_PT * F2_RMAX];      // by row: 1 + its pivot column in this round (0: none)
};

// One wave's Gauss-Jordan elimination of the n <= 128 candidate rows (lane, lane + 64) over the columns `cols`:
// per column the first unused row with the bit.  Slots start at k0; fills px, pc, slot_row, slot_col, col_slot,
// pcol1, newcols and k.  Branch-free over the lanes, the pivot row through scalar registers, the slots' rows and
// columns collected in lane t of two registers: 64 columns are one serial chain, whose length is what a panel costs.
__device__ __forceinline__ void f2_wave_eliminate(F2PanelLds& L, uint32_t n, uint64_t cols, uint32_t k0, int lane) {
    uint32_t x0[2] = {}, x1[2] = {}, c0[2] = {}, c1[2] = {};       // words and masks in halves
    if (lane < (int)n) {
        x0[0] = (uint32_t)L.cx[lane];
        x0[1] = (uint32_t)(L.cx[lane] >> 32);
        c0[0] = (uint32_t)L.cc[lane];
        c0[1] = (uint32_t)(L.cc[lane] >> 32);
    }
    if (lane + 64 < (int)n) {
        x1[0] = (uint32_t)L.cx[lane + 64];
        x1[1] = (uint32_t)(L.cx[lane + 64] >> 32);
        c1[0] = (uint32_t)L.cc[lane + 64];
        c1[1] = (uint32_t)(L.cc[lane + 64] >> 32);
    }
    auto lane_of = [](uint32_t v, int l) { return (uint32_t)__builtin_amdgcn_readlane((int)v, l); };
    k0 = __builtin_amdgcn_readfirstlane((int)k0);         // (uniform: in scalar registers)
    const uint32_t half[2] = {(uint32_t)__builtin_amdgcn_readfirstlane((int)(uint32_t)cols),
                              (uint32_t)__builtin_amdgcn_readfirstlane((int)(uint32_t)(cols >> 32))};
    uint64_t used0 = 0, used1 = 0, found = 0;
    uint32_t k = k0;
    int vpos = 0, vcol = 0;                              // lane t: slot k0 + t's candidate and column
#pragma unroll
    for (int h = 0; h < 2; ++h) {
        uint32_t todo = half[h];
        while (todo) {
            const int q = __builtin_ctz(todo);
            todo &= todo - 1;
            int m0 = __builtin_amdgcn_sbfe((int)x0[h], q, 1), m1 = __builtin_amdgcn_sbfe((int)x1[h], q, 1);
            const uint64_t f0 = __ballot(m0 != 0) & ~used0, f1 = __ballot(m1 != 0) & ~used1;
            if ((f0 | f1) == 0) continue;
            uint32_t pl, ph, ql, qh;
            int p;
            if (f0) {
                p = __builtin_ctzll(f0);
                pl = lane_of(x0[0], p);
                ph = lane_of(x0[1], p);
                ql = lane_of(c0[0], p);
                qh = lane_of(c0[1], p);
                used0 |= 1ull << p;
                m0 = lane == p ? 0 : m0;
            } else {
                p = __builtin_ctzll(f1);
                pl = lane_of(x1[0], p);
                ph = lane_of(x1[1], p);
                ql = lane_of(c1[0], p);
                qh = lane_of(c1[1], p);
                used1 |= 1ull << p;
                m1 = lane == p ? 0 : m1;
                p += 64;
            }
            const uint64_t bit = 1ull << k;
            ql ^= (uint32_t)bit;
            qh ^= (uint32_t)(bit >> 32);
            const bool mine = lane == (int)(k - k0);
            vpos = mine ? p : vpos;
            vcol = mine ? q + 32 * h : vcol;
            x0[0] ^= m0 & pl;
            x0[1] ^= m0 & ph;
            c0[0] ^= m0 & ql;
            c0[1] ^= m0 & qh;
            x1[0] ^= m1 & pl;
            x1[1] ^= m1 & ph;
            c1[0] ^= m1 & ql;
            c1[1] ^= m1 & qh;
            found |= 1ull << (q + 32 * h);
            ++k;
        }
    }
    L.px[lane] = 0;
    L.pc[lane] = 0;
    L.cx[lane] = (uint64_t)x0[1] << 32 | x0[0];
    L.cx[lane + 64] = (uint64_t)x1[1] << 32 | x1[0];
    L.cc[lane] = (uint64_t)c0[1] << 32 | c0[0];
    L.cc[lane + 64] = (uint64_t)c1[1] << 32 | c1[0];
    __builtin_amdgcn_wave_barrier();
    if (lane < (int)(k - k0)) {
        const uint32_t t = k0 + lane, row = L.crow[vpos];
        L.px[vcol] = L.cx[vpos];
        L.pc[vcol] = L.cc[vpos] ^ (1ull << t);
        L.slot_row[t] = row;
        L.slot_col[t] = (uint32_t)vcol;
        L.col_slot[vcol] = t;
        L.pcol1[row] = (uint8_t)(vcol + 1);
    }
    if (lane == 0) {
        L.newcols = found;
        L.k = k;
    }
}

// All 256 XOR combinations of 8 words a (stride sa words apart): thread j of 16 writes the 16 entries with high
// nibble j in Gray-code order, entries `st` words apart.
__device__ __forceinline__ void f2_combine16(const uint64_t* a, int sa, uint32_t j, uint64_t* out, int st) {
    uint64_t v = 0;
#pragma unroll
    for (int b = 0; b < 4; ++b)
        if ((j >> b) & 1u) v ^= a[(4 + b) * sa];
    const uint64_t r[4] = {a[0], a[sa], a[2 * sa], a[3 * sa]};
    uint32_t s = 0;
    out[(16 * j) * st] = v;
#pragma unroll
    for (int i = 1; i < 16; ++i) {
        const int b = __builtin_ctz(i);
        s ^= 1u << b;
        v ^= r[b];
        out[(16 * j + s) * st] = v;
    }
}

struct F2Args {
    uint64_t* A;
    uint32_t ldw, m;
    uint8_t* done;                       // 1 once a row is a pivot row
    uint64_t* cmask[2];                  // by panel parity: every row's slot mask
    uint32_t* prow;
    uint32_t* pcol;
    F2State* st;                         // [2], by panel parity
    uint32_t* slots;                     // rows of the current panel's slots
    uint64_t* B;                         // the previous panel's pivot rows (words behind it), by slot
    uint64_t* in[2];                     // by word parity: a panel's word of every row, set aside by the update
    uint64_t* out[2];                    // by word parity: the reduced panel word, put in place a launch later
};

// Panel w (block 0): rows i = tid + F2_PT r in registers.
template <int R>
__device__ __forceinline__ void f2_panel(const F2Args& a, uint32_t w, uint64_t vmask, F2PanelLds& L) {
    const uint32_t tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, m = a.m;
    uint64_t* cm_out = a.cmask[w & 1];
    const uint64_t* cm_prev = a.cmask[(w & 1) ^ 1];
    const uint64_t* in = a.in[w & 1];
    uint64_t* out = a.out[w & 1];
    F2State prev{0, 0};
    if (w > 0) prev = a.st[(w & 1) ^ 1];
    uint64_t x[R], cm[R];
    uint32_t dn = 0;                                     // bit r: row tid + F2_PT r is a pivot row
#pragma unroll
    for (int r = 0; r < R; ++r) {
        const uint32_t i = tid + F2_PT * r;
        x[r] = i >= m ? 0u : w < 2 ? a.A[(size_t)i * a.ldw + w] : in[i];
        cm[r] = prev.k && i < m ? cm_prev[i] : 0u;
        if (i >= m || a.done[i]) dn |= 1u << r;
        L.pcol1[i] = 0;
    }
    if (prev.k) {                                        // (uniform) panel w - 1 on this word
        if (tid < 64) L.px[tid] = tid < prev.k ? a.B[(size_t)tid * a.ldw + w] : 0u;
        __syncthreads();
        if (tid < 128) f2_combine16(&L.px[8 * (tid >> 4)], 1, tid & 15, &L.prev[tid >> 4][0], 1);
        __syncthreads();
#pragma unroll
        for (int r = 0; r < R; ++r) {
            uint64_t v = 0;
#pragma unroll
            for (int g = 0; g < 8; ++g) v ^= L.prev[g][(cm[r] >> (8 * g)) & 255u];
            x[r] ^= v;
            if (r % 4 == 3) __builtin_amdgcn_sched_barrier(0);       // (at most four rows' lookups in flight)
        }
    }
#pragma unroll
    for (int r = 0; r < R; ++r) cm[r] = 0;
    const uint32_t rank0 = prev.rank;
    uint32_t k = 0;
    uint64_t cols = vmask;                               // columns without a pivot yet
    uint64_t left = 0;
    for (int round = 0; round <= F2_ROUNDS; ++round) {
        // which columns any row that is not a pivot still has
        uint64_t o = 0;
#pragma unroll
        for (int r = 0; r < R; ++r)
            if (!((dn >> r) & 1u)) o |= x[r];
#pragma unroll
        for (int off = 32; off >= 1; off >>= 1) o |= (uint64_t)__shfl_xor((unsigned long long)o, off);
        if (lane == 0) L.wor[wave] = o;
        __syncthreads();
        left = 0;
#pragma unroll
        for (int v = 0; v < F2_PT / 64; ++v) left |= L.wor[v];
        left &= cols;
        if (left == 0 || round == F2_ROUNDS) break;      // (uniform)
        // candidates: the first rows (r major) that are not pivots and have a bit
        uint32_t n = 0;
#pragma unroll
        for (int r = 0; r < R; ++r) {
            if (n >= F2_CAND) break;                     // (uniform)
            const bool has = !((dn >> r) & 1u) && x[r] != 0;
            const uint64_t bal = __ballot(has);
            if (lane == 0) L.wcnt[wave] = (uint32_t)__popcll(bal);
            __syncthreads();
            uint32_t base = n, total = 0;
#pragma unroll
            for (int v = 0; v < F2_PT / 64; ++v) {
                const uint32_t c = L.wcnt[v];
                if (v < (int)wave) base += c;
                total += c;
            }
            const uint32_t pos = base + __builtin_amdgcn_mbcnt_hi((uint32_t)(bal >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)bal, 0));
            if (has && pos < F2_CAND) {
                L.cx[pos] = x[r];
                L.cc[pos] = cm[r];
                L.crow[pos] = tid + F2_PT * r;
            }
            n = min(n + total, (uint32_t)F2_CAND);
            __syncthreads();
        }
        if (wave == 0) f2_wave_eliminate(L, n, left, k, (int)lane);
        __syncthreads();
        const uint64_t nc = L.newcols;
        k = L.k;
        if (tid < 256) {
            const uint32_t g = (tid >> 4) & 7, h = tid >> 7;
            f2_combine16(h ? &L.pc[8 * g] : &L.px[8 * g], 1, tid & 15, &L.tab[g][0][h], 2);
        }
        __syncthreads();
#pragma unroll
        for (int r = 0; r < R; ++r) {
            const uint32_t i = tid + F2_PT * r;
            const uint32_t pq = L.pcol1[i];
            if (pq) {                                    // a pivot of this round: its own reduced row
                x[r] = L.px[pq - 1];
                cm[r] = L.pc[pq - 1] ^ (1ull << L.col_slot[pq - 1]);     // (its own slot is the row itself)
                dn |= 1u << r;
                L.pcol1[i] = 0;
            } else {
                const uint64_t b = x[r] & nc;
                uint64_t dx = 0, dc = 0;
#pragma unroll
                for (int g = 0; g < 8; ++g) {
                    const ulonglong2 e = *(const ulonglong2*)&L.tab[g][(b >> (8 * g)) & 255u][0];
                    dx ^= e.x;
                    dc ^= e.y;
                }
                x[r] ^= dx;
                cm[r] ^= dc;
            }
            if (r % 2 == 1) __builtin_amdgcn_sched_barrier(0);
        }
        cols &= ~nc;
        __syncthreads();
    }
    // column by column over all rows: what two rounds left
    uint32_t par = 0;
    while (left) {
        const int q = __builtin_ctzll(left);
        left &= left - 1;
        const uint32_t slot = par & 1;
        ++par;
        uint32_t key = 0xffffffffu;
#pragma unroll
        for (int r = R - 1; r >= 0; --r)
            if (!((dn >> r) & 1u) && ((x[r] >> q) & 1u)) key = ((uint32_t)r << 10) | tid;
#pragma unroll
        for (int off = 32; off >= 1; off >>= 1) key = min(key, (uint32_t)__shfl_xor((int)key, off));
        if (lane == 0) L.s_min[slot][wave] = key;
        __syncthreads();
        uint32_t best = L.s_min[slot][0];
#pragma unroll
        for (int v = 1; v < F2_PT / 64; ++v) best = min(best, L.s_min[slot][v]);
        if (best == 0xffffffffu) continue;               // (uniform) no pivot in this column
        const uint32_t pr = best >> 10, pt = best & 1023u;
        if (tid == pt) {
            uint64_t pw = 0, pc = 0;
#pragma unroll
            for (int r = 0; r < R; ++r)
                if ((uint32_t)r == pr) {
                    pw = x[r];
                    pc = cm[r];
                }
            L.s_pw[slot] = pw;
            L.s_pc[slot] = pc;
            dn |= 1u << pr;
            L.slot_row[k] = pt + F2_PT * pr;
            L.slot_col[k] = (uint32_t)q;
        }
        __syncthreads();
        const uint64_t pw = L.s_pw[slot], pc = L.s_pc[slot] ^ (1ull << k);
#pragma unroll
        for (int r = 0; r < R; ++r) {
            const bool piv = tid == pt && (uint32_t)r == pr;
            if (!piv && ((x[r] >> q) & 1u)) {
                x[r] ^= pw;
                cm[r] ^= pc;
            }
        }
        ++k;
    }
    __syncthreads();
    uint32_t tid1 = tid;                                 // (row addresses computed again: not kept in registers)
    asm volatile("" : "+v"(tid1));
#pragma unroll
    for (int r = 0; r < R; ++r) {
        const uint32_t i = tid1 + F2_PT * r;
        if (i < m) {
            out[i] = x[r];
            cm_out[i] = cm[r];
            if ((dn >> r) & 1u) a.done[i] = 1;
        }
    }
    // the pivots in column order; the slots in the order of discovery
    if (tid < k) {
        uint32_t pos = 0;
        for (uint32_t t = 0; t < k; ++t) pos += L.slot_col[t] < L.slot_col[tid];
        a.prow[rank0 + pos] = L.slot_row[tid];
        a.pcol[rank0 + pos] = 64 * w + L.slot_col[tid];
        a.slots[tid] = L.slot_row[tid];
    }
    if (tid == 0) {
        a.st[w & 1].k = k;
        a.st[w & 1].rank = rank0 + k;
    }
}

// LDS of an update block: per group of 8 slots all XOR combinations of those pivot rows' four words.
struct F2UpdateLds {
    uint64_t tab[8][256][F2_WS];
    uint64_t rows[64][F2_WS];
};

// Panel u on words [c0, c0 + 4) of rows [r0, r0 + 1024), words at or below `skip` excepted.  Word skip + 1, the next
// panel's, is also set aside (also when panel u has no pivots).
__device__ __forceinline__ void f2_update(const F2Args& a, uint32_t u, uint32_t c0, uint32_t skip, uint32_t r0, F2UpdateLds& L) {
    const uint32_t k = a.st[u & 1].k, tid = threadIdx.x;
    if (k == 0 && (skip + 1 < c0 || skip + 1 >= c0 + F2_WS)) return;
    if (tid < 64 * F2_WS) {
        const uint32_t t = tid / F2_WS, c = c0 + tid % F2_WS;
        L.rows[t][tid % F2_WS] = t < k && c > skip && c < a.ldw ? a.B[(size_t)t * a.ldw + c] : 0u;
    }
    __syncthreads();
    if (tid < 512) {
        const uint32_t c = tid & 3, j = (tid >> 2) & 15, g = tid >> 6;
        f2_combine16(&L.rows[8 * g][c], F2_WS, j, &L.tab[g][0][c], F2_WS);
    }
    __syncthreads();
    const uint32_t h = 2 * (tid & 1), c = c0 + h;
    const bool v0 = c > skip && c < a.ldw, v1 = c + 1 > skip && c + 1 < a.ldw;
    if (!v0 && !v1) return;
    const uint64_t* cm = a.cmask[u & 1];
    uint64_t* next = a.in[(skip + 1) & 1];
#pragma unroll
    for (uint32_t e = 0; e < F2_ROWS; e += F2_PT / 2) {
        const uint32_t i = r0 + e + (tid >> 1);
        if (i >= a.m) break;
        const uint64_t msk = cm[i];
        uint64_t* p = a.A + (size_t)i * a.ldw + c;
        uint64_t a0 = v0 ? p[0] : 0, a1 = v1 ? p[1] : 0;
#pragma unroll
        for (int g = 0; g < 8; ++g) {
            const ulonglong2 t = *(const ulonglong2*)&L.tab[g][(msk >> (8 * g)) & 255u][h];
            a0 ^= t.x;
            a1 ^= t.y;
        }
        if (v0) p[0] = a0;
        if (v1) p[1] = a1;
        if (c == skip + 1) next[i] = a0;
        if (c + 1 == skip + 1) next[i] = a1;
    }
}

union F2Lds {
    F2PanelLds panel;
    F2UpdateLds update;
    __device__ F2Lds() {}
};

// Block 0: panel w (when `panel`).  Then rblocks blocks (w > 0) put word w - 1 in place.  The others: panel w - 1 on
// the words behind w (behind w - 1 without a panel w), slabs of four words, nslab slabs from word c_first.  (One
// block alone reads and writes a word of 8192 rows in 17 and 4 us while the others stream the matrix, its
// contiguous copy in 4 and 2.)
template <int R>
__global__ __launch_bounds__(F2_PT) void f2_panel_update_kernel(F2Args a, uint32_t w, uint64_t vmask, int panel,
                                                                uint32_t c_first, uint32_t nslab, uint32_t rblocks) {
    __shared__ __attribute__((aligned(16))) F2Lds lds;
    uint32_t b = blockIdx.x;
    if (panel) {
        if (b == 0) {
            f2_panel<R>(a, w, vmask, lds.panel);
            return;
        }
        --b;
    }
    if (b < rblocks) {
        const uint32_t i = b * F2_ROWS + threadIdx.x;
        if (i < a.m) a.A[(size_t)i * a.ldw + w - 1] = a.out[(w & 1) ^ 1][i];
        return;
    }
    b -= rblocks;
    f2_update(a, w - 1, c_first + F2_WS * (b % nslab), panel ? w : w - 1, F2_ROWS * (b / nslab), lds.update);
}

// The words behind w of the panel's pivot rows, as they are before the panel's own update.
__global__ void f2_copy_kernel(F2Args a, uint32_t w) {
    const uint32_t t = blockIdx.x;
    if (t >= a.st[w & 1].k) return;
    const uint64_t* src = a.A + (size_t)a.slots[t] * a.ldw;
    for (uint32_t c = w + 1 + threadIdx.x; c < a.ldw; c += blockDim.x) a.B[(size_t)t * a.ldw + c] = src[c];
}

// The LDS tables of one workgroup: for each group g of 8 rows of Bsrc (rows 8g .. 8g + 7, fewer than
// `kb` counting as zero) and each of the F2_WS words c0 .. c0 + 3: tab[g][s][c] = XOR of the rows
// whose bit is set in s.
__device__ __forceinline__ void f2_build_tables(uint64_t (*tab)[256][F2_WS], const uint64_t* Bsrc, uint32_t ldb,
                                                uint32_t kb, uint32_t c0, uint32_t nw) {
    __shared__ uint64_t rows[64][F2_WS];
    for (uint32_t idx = threadIdx.x; idx < 64 * F2_WS; idx += F2_UT) {
        const uint32_t t = idx / F2_WS, c = idx % F2_WS;
        rows[t][c] = (t < kb && c0 + c < nw) ? Bsrc[(size_t)t * ldb + c0 + c] : 0u;
    }
    __syncthreads();
    for (uint32_t idx = threadIdx.x; idx < 8 * 256 * F2_WS; idx += F2_UT) {
        const uint32_t c = idx % F2_WS, s = (idx / F2_WS) % 256, g = idx / (F2_WS * 256);
        uint64_t v = 0;
#pragma unroll
        for (int b = 0; b < 8; ++b)
            if ((s >> b) & 1u) v ^= rows[8 * g + b][c];
        tab[g][s][c] = v;
    }
    __syncthreads();
}

// The RREF's row order: row t = pivot row prow[t] (t < rank), then zero rows.  T holds the pivot rows.
__global__ void f2_gather_kernel(const uint64_t* A, uint32_t ldw, const uint32_t* prow, const F2State* st, uint64_t* T) {
    const uint32_t rank = st->rank;
    for (size_t idx = (size_t)blockIdx.x * blockDim.x + threadIdx.x; idx < (size_t)rank * ldw;
         idx += (size_t)gridDim.x * blockDim.x)
        T[idx] = A[(size_t)prow[idx / ldw] * ldw + idx % ldw];
}
__global__ void f2_place_kernel(uint64_t* A, uint32_t ldw, uint32_t m, const F2State* st, const uint64_t* T) {
    const uint32_t rank = st->rank;
    for (size_t idx = (size_t)blockIdx.x * blockDim.x + threadIdx.x; idx < (size_t)m * ldw;
         idx += (size_t)gridDim.x * blockDim.x)
        A[idx] = idx < (size_t)rank * ldw ? T[idx] : 0u;
}

// C[i][c] (op=) sum over the bits b of A's row i of B[b][c]: per 64 rows of B one set of tables.
__global__ __launch_bounds__(F2_UT) void f2_gemm_kernel(const uint64_t* A, uint32_t lda, const uint64_t* B, uint32_t ldb,
                                                        uint64_t* C, uint32_t ldc, uint32_t m, uint32_t kw, uint32_t kbits,
                                                        uint32_t nw, int accumulate) {
    __shared__ uint64_t tab[8][256][F2_WS];
    const uint32_t c0 = blockIdx.x * F2_WS, wi = threadIdx.x % F2_WS, c = c0 + wi;
    const uint32_t r0 = blockIdx.y * F2_ROWS;
    constexpr int PER = F2_ROWS / (F2_UT / F2_WS);      // rows per thread (16)
    uint64_t acc[PER];
#pragma unroll
    for (int e = 0; e < PER; ++e) acc[e] = 0;
    for (uint32_t kb = 0; kb < kw; ++kb) {
        const uint32_t rows_left = kbits - 64 * kb;
        f2_build_tables(tab, B + (size_t)64 * kb * ldb, ldb, min(64u, rows_left), c0, nw);
#pragma unroll
        for (int e = 0; e < PER; ++e) {
            const uint32_t i = r0 + threadIdx.x / F2_WS + (F2_UT / F2_WS) * e;
            const uint64_t a = i < m ? A[(size_t)i * lda + kb] : 0u;
            uint64_t v = 0;
#pragma unroll
            for (int g = 0; g < 8; ++g) v ^= tab[g][(a >> (8 * g)) & 255u][wi];
            acc[e] ^= v;
        }
        __syncthreads();                                // the tables are rebuilt for the next 64 rows
    }
    if (c >= nw) return;
#pragma unroll
    for (int e = 0; e < PER; ++e) {
        const uint32_t i = r0 + threadIdx.x / F2_WS + (F2_UT / F2_WS) * e;
        if (i < m) C[(size_t)i * ldc + c] = accumulate ? (C[(size_t)i * ldc + c] ^ acc[e]) : acc[e];
    }
}

__global__ void f2_init_kernel(uint8_t* done, uint32_t m, F2State* st) {
    const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < m) done[i] = 0;
    if (i < 2) st[i] = F2State{0, 0};
}

}  // namespace
}  // namespace hx

using namespace hx;

namespace {
size_t f2_ws_bytes(uint32_t m, uint32_t n, uint32_t ldw) {
    const size_t mn = std::min(m, n);
    auto up = [](size_t b) { return (b + 255) / 256 * 256; };
    return up(m) + 6 * up((size_t)m * 8) + up(mn * 4) * 2 + up(2 * sizeof(F2State)) + up(64 * 4) + up((size_t)64 * ldw * 8) +
           up(mn * ldw * 8);
}
}  // namespace

extern "C" {

HX_API size_t hx_f2_rref_workspace_bytes(uint32_t m, uint32_t n, uint32_t ldw) {
    return (m == 0 || n == 0) ? 0 : f2_ws_bytes(m, n, std::max<uint32_t>(ldw, (n + 63) / 64));
}

}  // extern "C"

namespace {
// One pass of the panel elimination over m <= F2_PT * F2_RMAX rows (the panel kernel holds every row's
// panel word in registers).
void f2_rref_one(uint32_t m, uint32_t n, uint64_t* A, uint32_t ldw, uint32_t* rank, uint32_t* pivots, hx_stream s) {
    const hipStream_t st_ = (hipStream_t)s;
    const uint32_t mn = std::min(m, n), nwords = (n + 63) / 64;
    auto up = [](size_t b) { return (b + 255) / 256 * 256; };
    const size_t bytes = f2_ws_bytes(m, n, ldw);
    char* ws = (char*)arena_alloc(bytes);
    try {
        char* p = ws;
        uint8_t* done = (uint8_t*)p;
        p += up(m);
        uint64_t *cmask[2], *word[4];
        for (uint64_t** c : {&cmask[0], &cmask[1], &word[0], &word[1], &word[2], &word[3]}) {
            *c = (uint64_t*)p;
            p += up((size_t)m * 8);
        }
        uint32_t* prow = (uint32_t*)p;
        p += up((size_t)mn * 4);
        uint32_t* pcol = (uint32_t*)p;
        p += up((size_t)mn * 4);
        F2State* state = (F2State*)p;
        p += up(2 * sizeof(F2State));
        uint32_t* slots = (uint32_t*)p;
        p += up(64 * 4);
        uint64_t* B = (uint64_t*)p;
        p += up((size_t)64 * ldw * 8);
        uint64_t* T = (uint64_t*)p;
        f2_init_kernel<<<(m + 255) / 256, 256, 0, st_>>>(done, m, state);
        after_launch("f2_init_kernel");
        const int R = m <= 1024 ? 1 : m <= 2048 ? 2 : m <= 4096 ? 4 : m <= 8192 ? 8 : 16;
        const F2Args fa{A, ldw, m, done, {cmask[0], cmask[1]}, prow, pcol, state, slots, B,
                        {word[0], word[1]}, {word[2], word[3]}};
        const uint32_t rblocks = (m + F2_ROWS - 1) / F2_ROWS;
        for (uint32_t w = 0; w <= nwords; ++w) {
            // panel w beside panel w - 1 on the words behind w; after the last panel, its words (if any) alone
            const int panel = w < nwords;
            const uint32_t bits = panel ? std::min<uint32_t>(64, n - 64 * w) : 0;
            const uint64_t vmask = bits == 64 ? ~0ull : ((1ull << bits) - 1);
            const uint32_t first = panel ? w + 1 : w, c_first = first / F2_WS * F2_WS;
            const uint32_t nslab = w > 0 && first < ldw ? (ldw - c_first + F2_WS - 1) / F2_WS : 0;
            const uint32_t place = w > 0 ? rblocks : 0, grid = (panel ? 1 : 0) + place + nslab * rblocks;
            switch (R) {
                case 1: f2_panel_update_kernel<1><<<grid, F2_PT, 0, st_>>>(fa, w, vmask, panel, c_first, nslab, place); break;
                case 2: f2_panel_update_kernel<2><<<grid, F2_PT, 0, st_>>>(fa, w, vmask, panel, c_first, nslab, place); break;
                case 4: f2_panel_update_kernel<4><<<grid, F2_PT, 0, st_>>>(fa, w, vmask, panel, c_first, nslab, place); break;
                case 8: f2_panel_update_kernel<8><<<grid, F2_PT, 0, st_>>>(fa, w, vmask, panel, c_first, nslab, place); break;
                default: f2_panel_update_kernel<16><<<grid, F2_PT, 0, st_>>>(fa, w, vmask, panel, c_first, nslab, place); break;
            }
            after_launch("f2_panel_update_kernel");
            if (panel && w + 1 < ldw) {
                f2_copy_kernel<<<64, 128, 0, st_>>>(fa, w);
                after_launch("f2_copy_kernel");
            }
        }
        F2State* last = state + ((nwords - 1) & 1);
        const uint32_t g = (uint32_t)std::min<size_t>(4096, ((size_t)m * ldw + 255) / 256);
        f2_gather_kernel<<<g, 256, 0, st_>>>(A, ldw, prow, last, T);
        after_launch("f2_gather_kernel");
        f2_place_kernel<<<g, 256, 0, st_>>>(A, ldw, m, last, T);
        after_launch("f2_place_kernel");
        F2State h{};
        host_status(hx_download(&h, last, sizeof(h), s));
        *rank = h.rank;
        if (pivots && h.rank) host_status(hx_download(pivots, pcol, (size_t)h.rank * 4, s));
    } catch (...) {
        (void)hipStreamSynchronize(st_);
        arena_free(ws);
        throw;
    }
    arena_free(ws);
}
}  // namespace

extern "C" {

HX_API int hx_f2_rref(uint32_t m, uint32_t n, uint64_t* A, uint32_t ldw, uint32_t* rank, uint32_t* pivots, hx_stream s) {
    return guard("hx_f2_rref", [&] {
        HX_CHECK(rank != nullptr, "rank is NULL");
        *rank = 0;
        if (m == 0 || n == 0) return;
        HX_CHECK(A != nullptr, "A is NULL");
        HX_CHECK(ldw >= (n + 63) / 64, "ldw < ceil(n / 64)");
        const uint32_t cap = F2_PT * F2_RMAX;
        if (m <= cap) {
            f2_rref_one(m, n, A, ldw, rank, pivots, s);
            return;
        }
        // taller: the RREF of 16384 rows at a time stacked with the next rows (rank < 16384 needed)
        rref_stacked(m, A, ldw, cap, rank, pivots, (hipStream_t)s,
                     [&](uint32_t rows, uint64_t* W, uint32_t* rk, uint32_t* pv) { f2_rref_one(rows, n, W, ldw, rk, pv, s); },
                     "F_2 RREF: the rank reached 16384 with rows left (more than 16384 rows need a rank below 16384)");
    });
}

HX_API int hx_f2_gemm(uint32_t m, uint32_t n, uint32_t k, const uint64_t* A, uint32_t lda, const uint64_t* B,
                      uint32_t ldb, uint64_t* C, uint32_t ldc, int accumulate, hx_stream s) {
    return guard("hx_f2_gemm", [&] {
        const uint32_t kw = (k + 63) / 64, nw = (n + 63) / 64;
        HX_CHECK(m == 0 || n == 0 || C != nullptr, "C is NULL");
        HX_CHECK(lda >= kw && ldb >= nw && ldc >= nw, "leading dimension below the row's words");
        HX_CHECK(k == 0 || (A != nullptr && B != nullptr), "A or B is NULL");
        if (m == 0 || n == 0) return;
        if (packed_gemm<2>(m, n, k, A, lda, B, ldb, C, ldc, accumulate != 0, (hipStream_t)s)) return;
        const dim3 grid((nw + F2_WS - 1) / F2_WS, (m + F2_ROWS - 1) / F2_ROWS);
        f2_gemm_kernel<<<grid, F2_UT, 0, (hipStream_t)s>>>(A, lda, B, ldb, C, ldc, m, kw, k, nw, accumulate);
        after_launch("f2_gemm_kernel");
    });
}

}  // extern "C"
