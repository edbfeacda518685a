// Inner products of the 753-bit fields.
//
// A thread adds up to 8 products without reducing them, in 53 columns of
// 28-bit digits (27 products of 56 bits, 8 times, stay below 2^64), and
// reduces the sum once: 729 multiply-adds a product and 1158 a sum, against
// 1458 a Montgomery product.  Sums over lanes are not reduced either
// (256 p < 2^768).
//
// One wavefront per SIMD holds the columns, the operands and the next ones,
// which are requested before the product: with two wavefronts that load, then
// multiply, all of the chip waits for memory together (2^18 products: 25 us
// against 22; one Montgomery product at a time 27).  What is left is the
// multiply-adds' issue, about 13 us of it.
//
// One product a thread is a Montgomery product: 1458 multiply-adds on the
// only path against 1887.
#include "dot753.h"

#include "device_field.h"

namespace gsn {

constexpr int DOT_TERMS = 8;

template <class F>
__global__ __launch_bounds__(DOT753_THREADS) __attribute__((amdgpu_waves_per_eu(1))) void dot753_kernel(
    E753 *partial, const E753 *a, const E753 *b, size_t n, TW753 r_inv)
{
    constexpr uint32_t M28 = (1u << 28) - 1;
    const auto digits = [](uint32_t (&d)[27], const E753 &x) {
#pragma unroll
        for (int i = 0; i < 27; ++i) {
            const int w = 28 * i >> 5, sh = 28 * i & 31;
            d[i] = (sh > 4 && w + 1 < 24 ? __builtin_amdgcn_alignbit(x.v[w + 1], x.v[w], sh) : x.v[w] >> sh) & M28;
        }
    };
    __shared__ E753 sm[DOT753_THREADS / 64];
    const int t = threadIdx.x;
    const size_t stride = (size_t)gridDim.x * DOT753_THREADS;
    size_t i = (size_t)blockIdx.x * DOT753_THREADS + t;
    E753 acc{};
    if (!b) {
        for (; i < n; i += stride)
            acc = F::add_mod(acc, F::load(a, i));
    } else if (n <= stride) {
        if (i < n)
            acc = F::mont_mul(F::load(a, i), F::load(b, i));
    } else {
        E753 u = F::load(a, i), v = F::load(b, i);
        while (i < n) {
            uint64_t col[54] = {};
            for (int e = 0; e < DOT_TERMS && i < n; ++e) {
                uint32_t x[27], y[27];
                digits(x, u);
                digits(y, v);
                i += stride;
                if (i < n) {
                    u = F::load(a, i);
                    v = F::load(b, i);
                }
#pragma unroll
                for (int k = 0; k < 27; ++k)
#pragma unroll
                    for (int l = 0; l < 27; ++l)
                        col[k + l] += (uint64_t)x[k] * y[l];
            }
            uint64_t s = 0;
            E753 lo{}, hi{};
#pragma unroll
            for (int c = 0; c < 54; ++c) {
                s += col[c];
                const uint32_t d = (uint32_t)s & M28;
                s >>= 28;
                const int w = 28 * c >> 5, sh = 28 * c & 31;
                (w < 24 ? lo.v[w] : hi.v[w - 24]) |= d << sh;
                if (sh > 4 && w + 1 < 48)
                    (w + 1 < 24 ? lo.v[w + 1] : hi.v[w - 23]) |= d >> (32 - sh);
            }
            // (lo + 2^768 hi) 2^-768, hi < 2^742
            acc = F::add_mod(acc, F::canon(F::add(F::mul(lo, r_inv), hi)));
        }
    }
    const auto add_lanes = [&](int d) {
        E753 o;
#pragma unroll
        for (int l = 0; l < 24; ++l)
            o.v[l] = (uint32_t)__shfl_xor((int)acc.v[l], d);
        acc = F::add(acc, o);
    };
#pragma unroll
    for (int d = 1; d < 64; d *= 2)
        add_lanes(d);
    if ((t & 63) == 0)
        sm[t >> 6] = acc;
    __syncthreads();
    if (t < 64) {
        acc = sm[t & 3];
        add_lanes(1);
        add_lanes(2);
        if (t == 0)
            F::store(partial, blockIdx.x, F::canon(acc));
    }
}

template <class F>
void launch_dot753(E753 *partial, const E753 *a, const E753 *b, size_t n, unsigned blocks, const TW753 &r_inv,
                   hipStream_t st)
{
    hipLaunchKernelGGL(dot753_kernel<F>, dim3(blocks), dim3(DOT753_THREADS), 0, st, partial, a, b, n, r_inv);
}
template void launch_dot753<FMnt4>(E753 *, const E753 *, const E753 *, size_t, unsigned, const TW753 &, hipStream_t);
template void launch_dot753<FMnt6>(E753 *, const E753 *, const E753 *, size_t, unsigned, const TW753 &, hipStream_t);

}  // namespace gsn
