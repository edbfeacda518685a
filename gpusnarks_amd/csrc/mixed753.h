// The mixed-radix transforms' odd passes on the matrix cores (mixed753.hip).
#pragma once

#include "gsn_launch.h"

namespace gsn {

// DFT constants per radix: 3 at 0, 5 at 6, 7 at 16; C[e] at off + e, S[e] at
// off + q + e
__host__ __device__ constexpr uint32_t mix_cs_offset(uint32_t q) { return q == 3 ? 0u : (q == 5 ? 6u : 16u); }
constexpr uint32_t MIX_CS_ELEMS = 30;

// One pass of radix q over stride L: T and CS hold byte matrices (the powers
// w_{n1}^e and the DFT constants), lo and hi the records of w^e.
struct MixedPass {
    E753 *dst;
    const E753 *src;
    uint32_t n1, log_n2, L;
    const void *T, *CS;
    const TW753 *lo, *hi;
    uint32_t h;
};

// 2^log_n2 >= 64 columns
template <class F>
void launch_mixed_mat(const MixedPass &a, uint32_t q, bool last, hipStream_t stream);
// Instead of `last`: the product by w^(j2 k1) and the transpose, row j2 of n1
// positions.
template <class F>
void launch_mixed_twist(const MixedPass &a, hipStream_t stream);
// The matrices of the residues of `count` records in device memory or (null)
// of `one`.
template <class F>
void launch_build_mat753_records(uint4 *out, uint32_t count, const TW753 *records, const TW753 &one,
                                 hipStream_t stream);

}  // namespace gsn
