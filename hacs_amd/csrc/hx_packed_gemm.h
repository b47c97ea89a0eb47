// hx_packed_gemm.h -- products over F_2 and F_3 of bit-packed matrices on the matrix cores (hx_packed_gemm.hip).
#pragma once

#include "hx_common.h"

namespace hx {

// C = A B (or C += A B) over F_P, P = 2 (one plane of words per row) or 3 (planes `one` and `two`, plane two
// `ld` words after plane one).  ld*: words per plane.  Returns false, with nothing launched, where this route
// does not apply: inside a stream capture, when its operand planes do not fit the device, past one launch's threads,
// and where the table kernel is the faster one (one word of k over F_2, long operands).
template <int P>
bool packed_gemm(uint32_t m, uint32_t n, uint32_t k, const uint64_t* A, uint32_t lda, const uint64_t* B, uint32_t ldb,
                 uint64_t* C, uint32_t ldc, bool accumulate, hipStream_t s);

}  // namespace hx
