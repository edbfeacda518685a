// Transforms of the 753-bit fields too small to fill the chip, on the matrix
// cores: Stockham passes whose R-point DFTs are dense sums of products,
//   Y_k = sum_j x_j w_R^(j k),
// so a pass has the depth of one accumulation and one product by a twiddle
// record instead of log R products (a vector product is 6200 clocks of one
// wavefront however empty the chip is, and 2^10 points are 8 wavefronts).
//
// Lanes are columns, so w_R^(j k) is the same for all of them and a term is a
// byte matrix times the lanes' digits (matrix753_kernels.h); terms add up in
// the accumulators, and one carry chain ends them.  Two radix-2 levels are
// free: for the parity of k, terms j and j + R/2 share a factor up to its
// sign (z_j = x_j +- x_(j+R/2), j < R/2), and outputs k and k + R/2 share all
// factors up to the sign of odd terms:
//   Y_k, Y_(k+R/2) = S_even +- S_odd,  S = sum z_j w_R^(j k).
//
// KS wavefronts share the terms of outputs k and k + R/2 of 32 columns, an
// even and an odd term at a time in their two halves; a block is four of
// them: KS = 4 spreads the least work over the most wavefronts, KS = 2 leaves
// fewer carry chains and sums between them where there are columns enough
// (2^15: 36 against 40 us; KS = 1: 48).  KS wavefronts read R/2 matrices
// (9216 B) and 32 R elements once: 123, 245, 490 KB for R = 16, 32, 64, which
// at the CU's 64 bytes a clock is 0.8, 1.6, 3.2 us and bounds the pass
// together with the final product (2.6 us) and the launch (3.5 us); 18 MFMAs
// per two terms take a quarter of it.  2^10 points, two passes: 16 us, on the
// vector kernels 35.  The reads grow as n R, so larger transforms go other
// ways (matrix_passes).
#include "dense753.h"
#include "matrix753_kernels.h"

namespace gsn {

// Accumulator start of the wave's even terms: column sums of up to 32
// terms (32 * 96 * 2^14 < 2^26) stay positive.  Over the 96 rows it adds
// 2^18 (2^768 - 1).
constexpr int DENSE_BIAS = 255 << 18;
constexpr uint32_t DENSE_BIAS_ROW0 = 1u << 18;

template <class F, int LOG_R, int KS>
struct DenseWave {
    using P = typename F::params;
    using M = Mat753<P>;
    static constexpr int R = 1 << LOG_R, ROUNDS = R / (4 * KS);

    struct Terms {  // an even and an odd term: matrices and each lane's x_j, x_(j + R/2)
        v4i m[2][9];
        E753 x0, x1;
    };
    __device__ __forceinline__ static void load(Terms &t, const PassArgs<F> &a, uint32_t k, size_t col, uint32_t j)
    {
        const int lane = (int)__lane_id();
        const uint32_t log_c = a.log_n - LOG_R;
        t.x0 = F::load(a.in, ((size_t)(j + (lane >> 5)) << log_c) + col);
        t.x1 = F::load(a.in, ((size_t)(j + R / 2 + (lane >> 5)) << log_c) + col);
#pragma unroll
        for (int h = 0; h < 2; ++h) {
            const gcv4i *m =
                (const gcv4i *)((const char *)uniform(a.tw_col) + (size_t)(((j + h) * k) & (R - 1)) * MAT_BYTES);
#pragma unroll
            for (int b = 0; b < 9; ++b)
                t.m[h][b] = m[64 * b + lane];
        }
    }
    // x0 + x1 or, for odd k, x0 - x1, as digits
    __device__ __forceinline__ static void operands(v4i (&b0)[3], v4i (&b1)[3], const Terms &t, uint32_t odd)
    {
        const uint32_t mask = 0u - odd;
        E753 z;
        unsigned c = odd;
#pragma unroll
        for (int i = 0; i < 24; ++i)
            z.v[i] = __builtin_addc(t.x0.v[i], t.x1.v[i] ^ mask, c, &c);
        M::digits(b0, b1, M::to_offset(z));
    }
    __device__ __forceinline__ static void add(v16i (&se)[3], v16i (&so)[3], const Terms &t, uint32_t odd)
    {
        v4i b0[3], b1[3];
        operands(b0, b1, t, odd);
#pragma unroll
        for (int I = 0; I < 3; ++I)
#pragma unroll
            for (int J = 0; J < 3; ++J) {
                se[I] = __builtin_amdgcn_mfma_i32_32x32x32_i8(t.m[0][3 * I + J], b0[J], se[I], 0, 0, 0);
                so[I] = __builtin_amdgcn_mfma_i32_32x32x32_i8(t.m[1][3 * I + J], b1[J], so[I], 0, 0, 0);
            }
    }
    // The limbs of S_even + S_odd in the low half of the wave and of
    // S_even - S_odd in the high one (rows as in mat753_mul), reduced to
    // |x| <= 0.51 p, two's complement modulo 2^768.
    __device__ __forceinline__ static E753 finish(const v16i (&se)[3], const v16i (&so)[3])
    {
        E753 y;
        uint32_t prev = DENSE_BIAS_ROW0;
        unsigned carry = 0;
#pragma unroll
        for (int I = 0; I < 3; ++I)
#pragma unroll
            for (int q = 0; q < 4; ++q) {
                uint64_t t[2];
#pragma unroll
                for (int h = 0; h < 2; ++h) {
                    uint32_t d[4];
#pragma unroll
                    for (int b = 0; b < 4; ++b)
                        d[b] = (uint32_t)(h ? se[I][4 * q + b] - so[I][4 * q + b] : se[I][4 * q + b] + so[I][4 * q + b]);
                    t[h] = (uint64_t)d[3] * (1u << 24) + ((uint64_t)d[2] * (1u << 16) + ((uint64_t)d[1] * 256u + d[0]));
                }
                const auto lo = __builtin_amdgcn_permlane32_swap((uint32_t)t[0], (uint32_t)t[1], false, false);
                const auto hi =
                    __builtin_amdgcn_permlane32_swap((uint32_t)(t[0] >> 32), (uint32_t)(t[1] >> 32), false, false);
                const int l = 8 * I + 2 * q;
                y.v[l] = __builtin_addc(lo[0], prev, carry, &carry);
                y.v[l + 1] = __builtin_addc(lo[1], hi[0], carry, &carry);
                prev = hi[1];
            }
        // |y| < 32 * 6144 p: the quotient from limbs 23 and 24
        const int32_t top = (int32_t)(prev + carry - DENSE_BIAS_ROW0);
        constexpr double TOP = (double)P::MOD[23] + (double)P::MOD[22] / 4294967296.0;
        const float f = ((float)top * 4294967296.0f + (float)y.v[23]) * (float)(1.0 / TOP);
        const int32_t nq = -(int32_t)__builtin_rintf(f);
        unsigned c = 0;
        int64_t s = 0;
#pragma unroll
        for (int i = 0; i < 24; ++i) {
            s += (int64_t)nq * (int32_t)M::SMOD.v[i];
            y.v[i] = __builtin_addc(y.v[i], (uint32_t)s, c, &c);
            s >>= 32;
        }
        return y;
    }
};

// 3 p: added to a sum of four reduced parts, |x| <= 2.04 p
template <class P>
struct ThreeP {
    static constexpr W24 make()
    {
        W24 o{};
        uint64_t c = 0;
        for (int i = 0; i < 24; ++i) {
            c += 3ull * P::MOD[i];
            o.v[i] = (uint32_t)c;
            c >>= 32;
        }
        return o;
    }
    static constexpr W24 V = make();
};

// A round's operands are requested while the one before is multiplied.  The
// record is loaded late: requested before the last round it cost the second
// wavefront per SIMD (2^15, KS = 4: 51 us).
template <class F, int LOG_R, int KS, bool LAST>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(2))) void dense753_kernel(PassArgs<F> a)
{
    using D = DenseWave<F, LOG_R, KS>;
    constexpr uint32_t R = D::R;
    constexpr int G = 4 / KS;
    a.in += (size_t)blockIdx.y << a.log_n;
    a.out += (size_t)blockIdx.y << a.log_n;
    static_assert(R / 2 / KS <= 32, "terms within DENSE_BIAS");
    __shared__ uint4 part[G * (KS - 1) * 6 * 64];
    const uint32_t tile = xcd_tile(blockIdx.x, gridDim.x);
    const uint32_t k = tile & (R / 2 - 1);
    const int lane = (int)__lane_id(), wave = (int)uniform(threadIdx.x >> 6), g = wave / KS, me = wave % KS;
    const size_t col = ((size_t)(tile >> (LOG_R - 1)) * G + g) * 32 + (lane & 31);

    v16i se[3], so[3];
#pragma unroll
    for (int I = 0; I < 3; ++I)
#pragma unroll
        for (int i = 0; i < 16; ++i) {
            se[I][i] = DENSE_BIAS;
            so[I][i] = 0;
        }
    typename D::Terms t;
    D::load(t, a, k, col, 2 * me);
#pragma unroll
    for (int r = 0; r + 1 < D::ROUNDS; ++r) {
        typename D::Terms next;
        D::load(next, a, k, col, 2 * (KS * (r + 1) + me));
        D::add(se, so, t, k & 1);
        __builtin_amdgcn_sched_barrier(0);
        t = next;
    }
    D::add(se, so, t, k & 1);
    E753 y = D::finish(se, so);
    uint4 *const p = part + g * (KS - 1) * 6 * 64 + lane;
    if (me) {
#pragma unroll
        for (int q = 0; q < 6; ++q)
            p[((me - 1) * 6 + q) * 64] = make_uint4(y.v[4 * q], y.v[4 * q + 1], y.v[4 * q + 2], y.v[4 * q + 3]);
    }
    __syncthreads();
    if (me)
        return;
#pragma unroll
    for (int i = 0; i + 1 < KS; ++i) {
        unsigned c = 0;
#pragma unroll
        for (int q = 0; q < 6; ++q) {
            const uint4 v = p[(i * 6 + q) * 64];
            y.v[4 * q] = __builtin_addc(y.v[4 * q], v.x, c, &c);
            y.v[4 * q + 1] = __builtin_addc(y.v[4 * q + 1], v.y, c, &c);
            y.v[4 * q + 2] = __builtin_addc(y.v[4 * q + 2], v.z, c, &c);
            y.v[4 * q + 3] = __builtin_addc(y.v[4 * q + 3], v.w, c, &c);
        }
    }
    // where this lane's output goes, and its twiddle in the next pass
    const uint32_t kk = k + (lane >> 5) * (R / 2);
    const size_t ns = (size_t)1 << a.log_ns;
    const size_t at = ((col >> a.log_ns) << (a.log_ns + LOG_R)) + ((size_t)kk << a.log_ns) + (col & (ns - 1));
    unsigned c = 0;
#pragma unroll
    for (int i = 0; i < 24; ++i)
        y.v[i] = __builtin_addc(y.v[i], ThreeP<typename F::params>::V.v[i], c, &c);
    if constexpr (LAST) {
        F::store(a.out, at, F::canon(y));
    } else {
        const uint32_t log_c = a.log_n - a.log_np, log_s = a.log_ns + LOG_R;
        const size_t j = at >> log_c, x = at & (((size_t)1 << log_c) - 1) & (((size_t)1 << log_s) - 1);
        F::store(a.out, at, F::mul(y, F::load_tw(a.tw_pass, (j << log_s) + x)));
    }
}

// matrices of w_n^(i mul), i < entries
template <class F>
__global__ __launch_bounds__(64) void build_dense753_kernel(uint4 *out, uint32_t entries, const E753 *hi,
                                                           const TW753 *lo, uint32_t h, uint32_t log_n, uint64_t mul)
{
    write_matrices<F>(out, entries, [&](uint32_t i) { return root_power<F>(hi, lo, h, log_n, i * mul); });
}
// records of w_n^(j c mul) at (j << log_c) + c, times scale if use_scale
template <class F>
__global__ __launch_bounds__(64) void build_dense753_records_kernel(TW753 *out, uint32_t count, const E753 *hi,
                                                                    const TW753 *lo, uint32_t h, uint32_t log_n,
                                                                    uint32_t log_c, uint64_t mul, TW753 scale, int use_scale)
{
    const uint32_t i = blockIdx.x * 64 + threadIdx.x;
    if (i >= count)
        return;
    const size_t j = i >> log_c, c = i & ((1u << log_c) - 1u);
    E753 v = root_power<F>(hi, lo, h, log_n, j * c * mul);
    if (use_scale)
        v = F::canon(F::mul(v, scale));
    out[i] = F::make_tw(v);
}

template <class F, int LOG_R, int KS>
static void launch_r(const PassJob<F> &job, bool last, uint32_t count, hipStream_t st)
{
    const dim3 grid((1u << (job.a.log_n - 8)) * KS, count), block(256);
    if constexpr (LOG_R >= DENSE_LAST) {
        if (last) {
            hipLaunchKernelGGL((dense753_kernel<F, LOG_R, KS, true>), grid, block, 0, st, job.a);
            return;
        }
    }
    hipLaunchKernelGGL((dense753_kernel<F, LOG_R, KS, false>), grid, block, 0, st, job.a);
}
template <class F>
void launch_dense753(const PassJob<F> &job, bool last, uint32_t count, hipStream_t st)
{
    if (job.log_w == 6) {
        launch_r<F, 5, 2>(job, last, count, st);
        return;
    }
    switch (job.log_r) {
    case 4: launch_r<F, 4, 4>(job, last, count, st); break;
    case 5: launch_r<F, 5, 4>(job, last, count, st); break;
    case 6: launch_r<F, 6, 4>(job, last, count, st); break;
    default: break;
    }
}
template <class F>
void launch_build_dense753(uint4 *mat, uint32_t log_r, TW753 *rec, uint32_t log_s, uint32_t log_next, const E753 *hi,
                           const TW753 *lo, uint32_t h, uint32_t log_n, const TW753 *scale, hipStream_t st)
{
    const TW753 one{};
    if (mat)
        hipLaunchKernelGGL(build_dense753_kernel<F>, dim3(mat_blocks(1u << log_r)), dim3(64), 0, st, mat, 1u << log_r,
                           hi, lo, h, log_n, (uint64_t)1 << (log_n - log_r));
    if (rec) {
        const uint32_t count = 1u << (log_s + log_next);
        hipLaunchKernelGGL(build_dense753_records_kernel<F>, dim3((count + 63) / 64), dim3(64), 0, st, rec, count, hi,
                           lo, h, log_n, log_s, (uint64_t)1 << (log_n - log_s - log_next), scale ? *scale : one,
                           (int)(scale != nullptr));
    }
}

#define GSN_DENSE_FIELD(F)                                                                                        \
    template void launch_dense753<F>(const PassJob<F> &, bool, uint32_t, hipStream_t);                                    \
    template void launch_build_dense753<F>(uint4 *, uint32_t, TW753 *, uint32_t, uint32_t, const E753 *,          \
                                           const TW753 *, uint32_t, uint32_t, const TW753 *, hipStream_t);
GSN_DENSE_FIELD(FMnt4)
GSN_DENSE_FIELD(FMnt6)

}  // namespace gsn
