// Products by the powers of a coset's generator, 753-bit fields.
//
// g^i = lo[i mod 2^h] hi[i >> h], and 64 consecutive i share hi and, in an
// extended domain, the constant: these products are byte matrices times the
// wavefront's digits (matrix753_kernels.h), about 2000 clocks deep, and only
// lo's is a vector product of 6200.  A coset shift of 2^16 points 12.0 -> 9.5
// us, of 2^20 117 -> 95 (both products as vector ones before); an extended
// domain's step at 2^16 17 -> 13.  What is left is that product and the
// launch, at 2^20 (2.1 TB/s) two wavefronts per SIMD of it.
#include "coset753.h"

#include "matrix753_kernels.h"

namespace gsn {

template <class F>
struct Shared {  // products by constants that the whole wavefront shares
    using P = typename F::params;
    using M = Mat753<P>;
    typedef const gcv4i *Matrix;
    v16i bias;
    __device__ __forceinline__ Shared()
    {
#pragma unroll
        for (int i = 0; i < 16; ++i)
            bias[i] = M::BIAS;
        asm volatile("" : "+v"(bias));
    }
    static __device__ __forceinline__ Matrix matrix(const void *tab, uint32_t e)
    {
        return (Matrix)((const char *)uniform(tab) + (size_t)uniform(e) * MAT_BYTES);
    }
    // canonical v m for |v| < 2^766
    __device__ __forceinline__ E753 times(const E753 &v, Matrix mat) const
    {
        v4i b0[3], b1[3];
        M::digits(b0, b1, M::to_offset(v));
        E753 none, y;
        const Matrix m[1] = {mat};
        mat753_mul<P, 1, false>(b0, b1, m, bias, none, y);
        return F::canon(M::from_offset(M::to_offset(y)));
    }
};

template <class F>
__device__ __forceinline__ E753 coset_times(const Shared<F> &s, const E753 &v, const CosetArgs &t, size_t i)
{
    return s.times(F::mul(v, F::load_tw(t.lo, i & (((size_t)1 << t.h) - 1))), s.matrix(t.hi, (uint32_t)(i >> t.h)));
}

template <class F>
__global__ __launch_bounds__(256) void coset753_kernel(E753 *out, const E753 *in, CosetArgs t, size_t n)
{
    const size_t i = (size_t)blockIdx.x * 256 + threadIdx.x;
    if (i < n)  // whole wavefronts
        F::store(out, i, coset_times<F>(Shared<F>(), F::load(in, i), t, i));
}

template <class F, bool INVERSE>
__global__ __launch_bounds__(256) void ext753_kernel(E753 *out, const E753 *in, CosetArgs t, const void *c, size_t m)
{
    const size_t i = (size_t)blockIdx.x * 256 + threadIdx.x;
    if (i >= m)  // whole wavefronts
        return;
    const Shared<F> s;
    const E753 u = F::load(in, i), w = F::load(in, i + m);
    if constexpr (INVERSE) {  // c_(i+m) = (u - g^-i w) K, c_i = u - c_(i+m)
        const E753 v = coset_times<F>(s, w, t, i);
        const E753 hi = s.times(F::sub_mod(u, v), s.matrix(c, 0));
        F::store(out, i, F::sub_mod(u, hi));
        F::store(out, i + m, hi);
    } else {  // u + w and g^i (u + G w)
        const E753 v = F::add(u, s.times(w, s.matrix(c, 0)));
        F::store(out, i, F::add_mod(u, w));
        F::store(out, i + m, coset_times<F>(s, v, t, i));
    }
}

template <class F>
void launch_coset753(E753 *out, const E753 *in, const CosetArgs &t, size_t n, hipStream_t st)
{
    hipLaunchKernelGGL(coset753_kernel<F>, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, st, out, in, t, n);
}
template <class F>
void launch_ext753(E753 *out, const E753 *in, const CosetArgs &t, const void *c, size_t m, bool inverse,
                   hipStream_t st)
{
    const dim3 grid((unsigned)((m + 255) / 256)), block(256);
    if (inverse)
        hipLaunchKernelGGL((ext753_kernel<F, true>), grid, block, 0, st, out, in, t, c, m);
    else
        hipLaunchKernelGGL((ext753_kernel<F, false>), grid, block, 0, st, out, in, t, c, m);
}

#define GSN_COSET_FIELD(F)                                                                            \
    template void launch_coset753<F>(E753 *, const E753 *, const CosetArgs &, size_t, hipStream_t);   \
    template void launch_ext753<F>(E753 *, const E753 *, const CosetArgs &, const void *, size_t, bool, hipStream_t);
GSN_COSET_FIELD(FMnt4)
GSN_COSET_FIELD(FMnt6)

}  // namespace gsn
