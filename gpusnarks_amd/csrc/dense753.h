// Dense matrix-core passes of small 753-bit transforms (dense753.hip).
#pragma once

#include "gsn_launch.h"

namespace gsn {

// the smallest radix compiled as a last pass (matrix_passes' schedules end in
// no smaller one)
constexpr int DENSE_LAST = 5;
// radices compiled, and columns of a block
constexpr bool dense_supported(const PassCfg &c)
{
    return c.log_e == 1 && ((c.log_w == 5 && c.log_r >= 4 && c.log_r <= 6) || (c.log_w == 6 && c.log_r == 5));
}

// A Stockham pass: tw_col holds the matrices of w_R^e (e < R), tw_pass the
// records that outputs take along to the next pass, of radix 2^log_np.  Of
// `count` transforms, one after the other in both buffers.
template <class F>
void launch_dense753(const PassJob<F> &job, bool last, uint32_t count, hipStream_t stream);
// The tables of a pass of radix 2^log_r (mat, or null) and, with 2^log_s
// points through it and the ones before and a next pass of 2^log_next, its
// records w_n^(j c n / 2^(log_s + log_next)) at (j << log_s) + c (rec, or
// null), times *scale.
template <class F>
void launch_build_dense753(uint4 *mat, uint32_t log_r, TW753 *rec, uint32_t log_s, uint32_t log_next, const E753 *hi,
                           const TW753 *lo, uint32_t h, uint32_t log_n, const TW753 *scale, hipStream_t stream);

}  // namespace gsn
