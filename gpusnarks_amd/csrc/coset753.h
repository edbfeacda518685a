// Products by g^i, 753-bit fields (coset753.hip).
#pragma once

#include "gsn_launch.h"

namespace gsn {

// g^i = lo[i mod 2^h] hi[i >> h]: lo as records, hi as byte matrices, which a
// wavefront's 64 consecutive i share if 2^h >= 64.
struct CosetArgs {
    const TW753 *lo;
    const void *hi;
    uint32_t h;
};
// out[i] = in[i] g^i, n a multiple of 64
template <class F>
void launch_coset753(E753 *out, const E753 *in, const CosetArgs &t, size_t n, hipStream_t stream);
// The steps of an extended domain around its half transforms (gsn_domain.hip),
// c the matrix of G or K.
template <class F>
void launch_ext753(E753 *out, const E753 *in, const CosetArgs &t, const void *c, size_t m, bool inverse,
                   hipStream_t stream);

}  // namespace gsn
