// hx_residue.h -- the residue route's moduli and its int8 product (res_gemm_kernel, hx_gemm.hip), shared by the
// 32-bit (hx_gemm.hip) and 64-bit (hx_gemm64.hip) residue products.
#pragma once

#include "hx_common.h"

namespace hx {

constexpr int RES_MAXQ = 19;                     // moduli below; 12 reach 2^94, 19 reach 2^147
constexpr uint32_t RES_KMAX = 133144;            // k * 127^2 <= 2^31 - 1
// pairwise coprime: 3*5*17, 2*127, 11*23, 251, 13*19, then primes
constexpr uint8_t RES_Q[RES_MAXQ] = {255, 254, 253, 251, 247, 241, 239, 233, 229, 227,
                                     223, 211, 199, 197, 193, 191, 181, 179, 173};
__host__ __device__ constexpr uint32_t res_modulus(int i) { return RES_Q[i]; }

struct ResArgs {
    const int8_t* A8;            // residue plane i of A at A8 + i * a_plane: Mp rows of Kp bytes (res_chunk's order)
    const int8_t* B8;            // residue plane i of B at B8 + i * b_plane: Np rows of Kp bytes (the same)
    size_t a_plane, b_plane;
    uint32_t Kp;
    uint32_t ntm, ntn;
    uint8_t* R;                  // product residues of modulus i at R + i * r_plane (res_block's order)
    size_t r_plane;              // ntm ntn side^2 bytes
    uint32_t q[RES_MAXQ];
    uint32_t tpack[RES_MAXQ];    // bytes (y 2^(8j)) mod q, j = 0 .. 3, y = (M / q_i)^-1 mod q_i (the CRT's factor)
    uint32_t kq[RES_MAXQ];       // q - (y 2^31 mod q)
    float iq[RES_MAXQ];
};

// An operand plane lies as the MFMA fragments do: 1 KB per 32 rows x 32 k, 16 bytes per lane (row lane % 32, k
// 16 (lane / 32) .. + 15), the k blocks of 32 rows one after the other.  The byte offset of a row's 16-byte
// chunk c (k = 16 c ..) in a plane of Kp bytes per row (Kp a multiple of 64):
__device__ __forceinline__ size_t res_chunk(uint32_t row, uint32_t c, uint32_t Kp) {
    return ((size_t)(row >> 5) * (Kp >> 5) + (c >> 1)) * 1024 + (c & 1) * 512 + (row & 31) * 16;
}

// The product residues of a plane lie as the MFMA accumulators do: 1 KB per 32 x 32 block, 16 bytes per lane
// (byte r: row (r / 4) 8 + 4 (lane / 32) + r % 4, column lane % 32), so the product kernel stores and the CRT
// kernels load 16 bytes per lane.  Blocks of a tile: 64-row strip, 128-column strip, then the upper / lower 32
// rows and the four 32-column blocks of the 64 x 128 piece; tiles row by row.
struct ResBlocks {
    uint32_t side, ntn;          // tile side (256 or 128), tiles per row
};
__device__ __forceinline__ void res_block(const ResBlocks& g, uint32_t b, uint32_t& row, uint32_t& col) {
    const uint32_t per = g.side * g.side / 1024, tile = b / per, in = b % per;
    const uint32_t lb = g.side / 128, s = in / 8 / lb, t = in / 8 % lb;
    row = tile / g.ntn * g.side + 64 * s + 32 * ((in >> 2) & 1);
    col = tile % g.ntn * g.side + 128 * t + 32 * (in & 3);
}

// Modulus i's constants of the product's epilogue (q, y < 256).
inline void res_modulus_consts(ResArgs& a, uint32_t i, uint32_t q, uint32_t y) {
    a.q[i] = q;
    a.tpack[i] = y % q | y * 256u % q << 8 | (uint32_t)(y * 65536ull % q) << 16 | (uint32_t)(y * 16777216ull % q) << 24;
    a.kq[i] = q - (uint32_t)(y * 0x80000000ull % q);
    a.iq[i] = 1.0f / (float)q;
}

// The side of the square output tiles of an N-moduli product: Mp and Np are multiples of it.
uint32_t residue_side(uint32_t m, uint32_t n, uint32_t N);
// One int8 product per modulus (grid.y): R_i = (A_i B_i) y_i mod q_i.  a.ntm, a.ntn: tiles of `side`.
void residue_product(const ResArgs& a, uint32_t N, uint32_t side, hipStream_t s);

}  // namespace hx
