// Odd passes of the mixed-radix transforms of the 753-bit fields on the
// matrix cores.
//
// The q-point DFTs of every column j2 (gsn_domain.hip describes the passes):
// a wavefront takes 64 consecutive columns of one group, so every factor --
// the twiddles of a pass and the DFT's constants -- is the same for all its
// lanes and a product is a byte matrix times the lanes' digits
// (matrix753_kernels.h).  A sum of products by constants is one accumulation:
// each U_k, V_k below takes (q-1)/2 products and a single carry chain.
//
// A radix-7 group of 64 columns takes 24 products and 6 chains: 432 MFMAs
// (13.8k matrix-core cycles) and about 3.3k vector instructions, against 24
// products of about 1700 vector instructions in the vector kernel.  At
// 525 x 2^12 (2.15 million elements, 413 MB read and written a pass) the
// radix-7, 5, 5, 3 passes take 156, 167, 167 and 112 us (2.6 to 3.7 TB/s)
// against the vector kernel's 504, 413, 413 and 401, of which about 150 are
// the two products by w^(j2 k1).  No two lanes share these, so they stay
// vector ones: in the last pass (317 us) or, where a transpose follows, in
// mixed_twist_kernel.  The others wait on memory with one or two wavefronts
// per SIMD.
//
// Values between the passes are small signed numbers, in two's complement
// modulo 2^768.  Bounds: inputs of the first pass are below p, every further
// pass adds at most 2 p; a product is below B = 6144 p, a sum of three below
// 3 B < 127/255 2^768, and both are reduced to about p/2 before they are
// added to anything.
#include "matrix753_kernels.h"
#include "mixed753.h"

namespace gsn {

// Accumulators start higher than in Mat753: up to three products' columns.
constexpr int MIX_BIAS = (1 << 23) - (1 << 15);
constexpr uint32_t MIX_BIAS_ROW0 = 1u << 15;

// x reduced to |x| <= 0.51 p, two's complement
template <class P>
__device__ __forceinline__ E753 reduce_signed(const E753 &x)
{
    constexpr double TOP = (double)P::MOD[23] + (double)P::MOD[22] / 4294967296.0;
    const int32_t nq = -(int32_t)__builtin_rintf((float)(int32_t)x.v[23] * (float)(1.0 / TOP));
    E753 o;
    unsigned c = 0;
    int64_t s = 0;
#pragma unroll
    for (int i = 0; i < 24; ++i) {
        s += (int64_t)nq * (int32_t)Mat753<P>::SMOD.v[i];
        o.v[i] = __builtin_addc(x.v[i], (uint32_t)s, c, &c);
        s >>= 32;
    }
    return o;
}
// x + K p for a small constant K: positive where |x| < K p
template <class P, uint32_t K>
struct MultipleOfP {
    static constexpr W24 make()
    {
        W24 o{};
        uint64_t c = 0;
        for (int i = 0; i < 24; ++i) {
            c += (uint64_t)K * P::MOD[i];
            o.v[i] = (uint32_t)c;
            c >>= 32;
        }
        return o;
    }
    static constexpr W24 V = make();
};
__device__ __forceinline__ E753 sub768(const E753 &a, const E753 &b)
{
    E753 r;
    unsigned c = 0;
#pragma unroll
    for (int i = 0; i < 24; ++i)
        r.v[i] = __builtin_subc(a.v[i], b.v[i], c, &c);
    return r;
}

// A wavefront's share of row block I of H matrices.
template <int H>
struct MatBlocks {
    v4i b[H][3];
    __device__ __forceinline__ void load(const gcv4i *const (&m)[H], int I)
    {
        const int lane = (int)__lane_id();
#pragma unroll
        for (int h = 0; h < H; ++h)
#pragma unroll
            for (int J = 0; J < 3; ++J)
                b[h][J] = m[h][64 * (3 * I + J) + lane];
    }
};

// sum over h < H of the products of digits (b0[h], b1[h]) and the matrices
// m[h], one per wavefront; two's complement.  AHEAD: blk holds m's row block
// 0 and takes that of `next`, every block being requested one block ahead of
// its use (radix 7 at 525 x 2^12: 156 us against 295 with the loads left to
// the scheduler; radix 3 has no registers for it at its two wavefronts).
template <class P, int H, bool AHEAD>
__device__ __forceinline__ E753 mat753_sum(const v4i (*b0)[3], const v4i (*b1)[3], MatBlocks<H> &blk,
                                           const gcv4i *const (&m)[H], const gcv4i *const (&next)[H],
                                           const v16i &bias)
{
    E753 y;
    uint32_t prev = 0;
    unsigned carry = 0;
#pragma unroll
    for (int I = 0; I < 3; ++I) {
        MatBlocks<H> ahead;
        if (!AHEAD)
            blk.load(m, I);
        else if (I < 2)
            ahead.load(m, I + 1);
        else
            ahead.load(next, 0);
        v16i d0 = bias, d1 = bias;
#pragma unroll
        for (int h = 0; h < H; ++h)
#pragma unroll
            for (int J = 0; J < 3; ++J) {
                d0 = __builtin_amdgcn_mfma_i32_32x32x32_i8(blk.b[h][J], b0[h][J], d0, 0, 0, 0);
                d1 = __builtin_amdgcn_mfma_i32_32x32x32_i8(blk.b[h][J], b1[h][J], d1, 0, 0, 0);
            }
        if (AHEAD)
            blk = ahead;
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            const uint32_t u0 = (uint32_t)d0[4 * q] + ((uint32_t)d0[4 * q + 1] << 8);
            const uint32_t u1 = (uint32_t)d0[4 * q + 2] + ((uint32_t)d0[4 * q + 3] << 8);
            const uint32_t v0 = (uint32_t)d1[4 * q] + ((uint32_t)d1[4 * q + 1] << 8);
            const uint32_t v1 = (uint32_t)d1[4 * q + 2] + ((uint32_t)d1[4 * q + 3] << 8);
            const auto s0 = __builtin_amdgcn_permlane32_swap(u0, v0, false, false);
            const auto s1 = __builtin_amdgcn_permlane32_swap(u1, v1, false, false);
            const int l = 8 * I + 2 * q;
            const uint32_t n0 = l == 0 ? s0[0] + MIX_BIAS_ROW0 : s0[0];
            y.v[l] = __builtin_addc(n0, __builtin_amdgcn_alignbit(s1[0], prev, 16), carry, &carry);
            y.v[l + 1] = __builtin_addc(s0[1], __builtin_amdgcn_alignbit(s1[1], s1[0], 16), carry, &carry);
            prev = s1[1];
        }
        if (AHEAD)
            __builtin_amdgcn_sched_barrier(0);
    }
    return y;
}

// v w^e, canonical
template <class F>
__device__ __forceinline__ E753 twist(const E753 &v, const MixedPass &a, uint64_t e)
{
    E753 t;
    unsigned c = 0;
#pragma unroll
    for (int l = 0; l < 24; ++l)
        t.v[l] = __builtin_addc(v.v[l], MultipleOfP<typename F::params, 32>::V.v[l], c, &c);
    t = F::mul(t, F::load_tw(a.lo, (size_t)(e & ((1ull << a.h) - 1))));
    return F::canon(F::mul(t, F::load_tw(a.hi, (size_t)(e >> a.h))));
}

// One pass.  START: the first one (no twiddles, canonical inputs); LAST: also
// times w^(j2 k1), canonical outputs.
template <class F, int Q, bool START, bool LAST>
__device__ __forceinline__ void mixed_mat_body(const MixedPass &a)
{
    using P = typename F::params;
    using M = Mat753<P>;
    constexpr int H = (Q - 1) / 2;
    constexpr bool AHEAD = Q > 3;
    const uint32_t nq = a.n1 / Q, span = a.n1 / (a.L * Q);
    const int lane = (int)__lane_id();
    const uint32_t log_c = a.log_n2 - 6;
    const uint32_t wave =
        uniform(xcd_tile(blockIdx.x, gridDim.x) * (uint32_t)(blockDim.x >> 6) + (uint32_t)(threadIdx.x >> 6));
    const uint32_t j = wave >> log_c;
    if (j >= nq)
        return;
    const size_t j2 = ((size_t)(wave & ((1u << log_c) - 1u)) << 6) + lane;
    const uint32_t k = j % a.L, jb = j / a.L;
    const auto matrix = [&](const void *tab, uint32_t e) {
        return (const gcv4i *)((const char *)tab + (size_t)e * MAT_BYTES);
    };
    v16i bias;
#pragma unroll
    for (int i = 0; i < 16; ++i)
        bias[i] = MIX_BIAS;
    asm volatile("" : "+v"(bias));

    E753 x[Q];
#pragma unroll
    for (int r = 0; r < Q; ++r)
        x[r] = F::load(a.src, ((size_t)(j + r * nq) << a.log_n2) + j2);
    if (!START && k != 0) {  // r k span < n1: w_{Lq}^(r k) = T[r k span]
        MatBlocks<1> blk;
        const gcv4i *m[1] = {matrix(a.T, k * span)};
        if (AHEAD)
            blk.load(m, 0);
#pragma unroll
        for (int r = 1; r < Q; ++r) {
            v4i d[2][1][3];
            M::digits(d[0][0], d[1][0], M::to_offset(x[r]));
            const gcv4i *const next[1] = {r + 1 < Q ? matrix(a.T, (uint32_t)(r + 1) * k * span) : m[0]};
            x[r] = mat753_sum<P, 1, AHEAD>(d[0], d[1], blk, m, next, bias);
            m[0] = next[0];
        }
    }
    const uint32_t pos0 = jb * a.L * Q + k;
    const auto put = [&](uint32_t s, const E753 &v) {
        const uint32_t pos = pos0 + s * a.L;
        const size_t i = ((size_t)pos << a.log_n2) + j2;
        if constexpr (LAST) {
            F::store(a.dst, i, twist<F>(v, a, (uint64_t)j2 * pos));
        } else {
            F::store(a.dst, i, v);
        }
    };
    // a_m = x_m + x_(q-m), b_m = x_m - x_(q-m), as digits
    v4i da[2][H][3], db[2][H][3];
    E753 s0 = x[0];
#pragma unroll
    for (int m = 1; m <= H; ++m) {
        E753 am = F::add(x[m], x[Q - m]);
        const E753 bm = sub768(x[m], x[Q - m]);
        if (!START)
            am = reduce_signed<P>(am);
        s0 = F::add(s0, am);
        M::digits(da[0][m - 1], da[1][m - 1], M::to_offset(am));
        M::digits(db[0][m - 1], db[1][m - 1], M::to_offset(bm));
    }
    // X_k, X_(q-k) = x_0 + U_k +- V_k, U_k = sum a_m C[m k], V_k = sum b_m S[m k]
    const gcv4i *mc[H + 1][H], *ms[H][H];
#pragma unroll
    for (int kk = 1; kk <= H; ++kk)
#pragma unroll
        for (int m = 1; m <= H; ++m) {
            mc[kk - 1][m - 1] = matrix(a.CS, mix_cs_offset(Q) + (uint32_t)(m * kk) % Q);
            ms[kk - 1][m - 1] = matrix(a.CS, mix_cs_offset(Q) + Q + (uint32_t)(m * kk) % Q);
        }
#pragma unroll
    for (int m = 0; m < H; ++m)
        mc[H][m] = mc[0][m];
    MatBlocks<H> blk;
    if (AHEAD)
        blk.load(mc[0], 0);
    put(0, s0);
#pragma unroll
    for (int kk = 1; kk <= H; ++kk) {
        const E753 base =
            F::add(x[0], reduce_signed<P>(mat753_sum<P, H, AHEAD>(da[0], da[1], blk, mc[kk - 1], ms[kk - 1], bias)));
        const E753 V = reduce_signed<P>(mat753_sum<P, H, AHEAD>(db[0], db[1], blk, ms[kk - 1], mc[kk], bias));
        put((uint32_t)kk, F::add(base, V));
        put((uint32_t)(Q - kk), sub768(base, V));
    }
}

// Radix 7 holds more than two wavefronts' registers, and radix 5 would spill
// its matrices' blocks (169 against 160 us).  Radix 3 fits, and its LAST's
// vector products want both (317 against 428 us with one).
template <class F, int Q, bool START, bool LAST>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(Q > 3 ? 1 : 2))) void mixed_mat_kernel(MixedPass a)
{
    mixed_mat_body<F, Q, START, LAST>(a);
}

// dst[j2 n1 + pos] = src[pos n2 + j2] w^(j2 pos).  A block takes 64 rows j2 of
// four neighbouring pos, so that their stores meet in the cache.  The products
// by records bound it, with the transpose under them: 258 us at 525 x 2^12,
// where a transpose alone takes 107 and the products cost the last odd pass
// 205.
template <class F>
__global__ __launch_bounds__(256) void mixed_twist_kernel(MixedPass a)
{
    const uint32_t groups = (a.n1 + 3) / 4, g = blockIdx.x / groups;
    const uint32_t pos = 4 * (blockIdx.x - g * groups) + (threadIdx.x >> 6);
    const size_t j2 = (size_t)g * 64 + (threadIdx.x & 63);
    if (pos < a.n1)
        F::store(a.dst, j2 * a.n1 + pos,
                 twist<F>(F::load(a.src, ((size_t)pos << a.log_n2) + j2), a, (uint64_t)j2 * pos));
}

// matrices of the residues of records, or (null) of one
template <class F>
__global__ __launch_bounds__(64) void build_mat753_records_kernel(uint4 *out, uint32_t entries, const TW753 *records,
                                                                 TW753 one)
{
    write_matrices<F>(out, entries, [&](uint32_t i) {
        const TW753 r = records ? F::load_tw(records, i) : one;
        uint32_t d[27];
#pragma unroll
        for (int l = 0; l < 27; ++l)
            d[l] = l < 26 ? r.w[l] : 0u;
        E753 v;
        F::from29(v.v, d);
        return v;
    });
}

template <class F, int Q>
static void launch_q(const MixedPass &a, bool last, hipStream_t st)
{
    const size_t waves = (size_t)(a.n1 / Q) << (a.log_n2 - 6);
    const dim3 grid((unsigned)((waves + 3) / 4)), block(256);
    if (a.L == 1 && last)
        hipLaunchKernelGGL((mixed_mat_kernel<F, Q, true, true>), grid, block, 0, st, a);
    else if (a.L == 1)
        hipLaunchKernelGGL((mixed_mat_kernel<F, Q, true, false>), grid, block, 0, st, a);
    else if (last)
        hipLaunchKernelGGL((mixed_mat_kernel<F, Q, false, true>), grid, block, 0, st, a);
    else
        hipLaunchKernelGGL((mixed_mat_kernel<F, Q, false, false>), grid, block, 0, st, a);
}

template <class F>
void launch_mixed_mat(const MixedPass &a, uint32_t q, bool last, hipStream_t st)
{
    switch (q) {
    case 3: launch_q<F, 3>(a, last, st); break;
    case 5: launch_q<F, 5>(a, last, st); break;
    default: launch_q<F, 7>(a, last, st); break;
    }
}
template <class F>
void launch_mixed_twist(const MixedPass &a, hipStream_t st)
{
    hipLaunchKernelGGL(mixed_twist_kernel<F>, dim3(((a.n1 + 3) / 4) << (a.log_n2 - 6)), dim3(256), 0, st, a);
}
template <class F>
void launch_build_mat753_records(uint4 *out, uint32_t count, const TW753 *records, const TW753 &one, hipStream_t st)
{
    hipLaunchKernelGGL(build_mat753_records_kernel<F>, dim3(mat_blocks(count)), dim3(64), 0, st, out, count, records,
                       one);
}

template void launch_mixed_mat<FMnt4>(const MixedPass &, uint32_t, bool, hipStream_t);
template void launch_mixed_mat<FMnt6>(const MixedPass &, uint32_t, bool, hipStream_t);
template void launch_mixed_twist<FMnt4>(const MixedPass &, hipStream_t);
template void launch_mixed_twist<FMnt6>(const MixedPass &, hipStream_t);
template void launch_build_mat753_records<FMnt4>(uint4 *, uint32_t, const TW753 *, const TW753 &, hipStream_t);
template void launch_build_mat753_records<FMnt6>(uint4 *, uint32_t, const TW753 *, const TW753 &, hipStream_t);

}  // namespace gsn
