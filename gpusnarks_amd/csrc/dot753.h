// Inner products of the 753-bit fields (dot753.hip).
#pragma once

#include <hip/hip_runtime.h>

#include "field_core.h"

namespace gsn {

constexpr int DOT753_THREADS = 256, DOT753_BLOCKS = 256;

// partial[block] = the block's share of sum_i a_i b_i r_inv, or (b null) of
// sum_i a_i; canonical.
template <class F>
void launch_dot753(E753 *partial, const E753 *a, const E753 *b, size_t n, unsigned blocks, const TW753 &r_inv,
                   hipStream_t stream);

}  // namespace gsn
