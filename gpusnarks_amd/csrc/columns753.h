// Radix-2 transforms of the columns of an array, 753-bit fields
// (columns753.hip).
#pragma once

#include "gsn_launch.h"

namespace gsn {

// 2^log_n points of each of `cols` columns, in two passes of 2^r1 and 2^r2:
// x[j][c] at in, X[k][c] at out, both at row cols + c; ws holds as much and
// is neither of them.  fold1 and fold2 are launch_build_mat753's folded
// matrices of the passes (log_y = 0 and r1) for a root of order 2^log_n.
// columns_split: whether there is such a pair, and which.
template <class F>
void launch_columns753(const E753 *in, E753 *out, E753 *ws, uint32_t log_n, uint32_t cols, const void *fold1,
                       const void *fold2, hipStream_t stream);
constexpr bool columns_split(uint32_t log_n, uint32_t &r1, uint32_t &r2)
{
    r1 = (log_n + 1) / 2;
    r2 = log_n / 2;
    return r2 >= 4 && r1 <= 6;
}

}  // namespace gsn
