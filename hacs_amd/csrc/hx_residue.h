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
    const int8_t* A8;            // residue plane i of A at A8 + i * a_plane: Mp rows of Kp bytes
    const int8_t* B8;            // residue plane i of B at B8 + i * b_plane: Np rows of Kp bytes
    size_t a_plane, b_plane;
    uint32_t Kp;
    uint32_t ntm, ntn;
    uint8_t* R;                  // product residues of modulus i at R + i * r_plane: Mp rows of ldr bytes
    size_t r_plane;
    uint32_t ldr;
    uint32_t q[RES_MAXQ];
    uint32_t y[RES_MAXQ];        // (M / q_i)^-1 mod q_i, the CRT factor of modulus i
    double invq[RES_MAXQ];
};

// The side of the square output tiles of an N-moduli product: Mp and Np are multiples of it.
uint32_t residue_side(uint32_t m, uint32_t n, uint32_t N);
// One int8 product per modulus (grid.y): R_i = (A_i B_i) y_i mod q_i.  a.ntm, a.ntn: tiles of `side`.
void residue_product(const ResArgs& a, uint32_t N, uint32_t side, hipStream_t s);

}  // namespace hx
