// 753-bit passes on the matrix cores.
//
// A product by a twiddle that 32 lanes share is a matrix product: with the
// bytes y_k of y as signed digits,
//   y w = sum_k y_k (256^k w)  ==  sum_k y_k c_k  (mod p),  c_k = 256^k w mod p,
// so the 96 byte columns of the result are the 96 x 96 byte matrix of the
// c_k (fixed per twiddle, built with the plan) times the 96 digits of each
// lane's y: nine 32x32x32 int8 MFMAs per 32 lanes.  The reduction modulo p
// is inside the constants, so no quotient is formed: the result is below
// 96 * 128 * p / 2 in magnitude and one carry chain over the column sums
// gives its limbs.  Per 64 products and their butterflies this issues 18
// MFMAs (576 matrix-core cycles) and about 230 vector instructions, against
// about 1540 vector instructions for the quotient-estimate product
// (F753::mul), whose 1158 multiply-adds bound the vector kernel.
//
// What bounds it: no single unit.  Of a 1024-element tile of a full launch
// (2^20: 53 / 92 / 87 / 62 us for the four passes, 200 MB of elements each,
// so 3.8 / 2.2 / 2.3 / 3.2 TB/s) the vector instructions are a third of the
// time, the MFMAs an eighth, the loads of matrices and elements through the
// CU's 64 bytes a clock about a quarter; with two wavefronts per SIMD (the
// registers) they overlap only in part.
//
// Values inside these passes are signed and kept in offset form,
//   x^ = x + 0x8080..80  mod 2^768,
// so that the bytes of x^, each with its top bit flipped, are exactly the
// signed digits of x; sums and differences x0 +- t keep the offset.
//
// Bounds.  A product is below B = 6144 (1 + 2^-15) p.  x0 is reduced to about
// p/2 at every second step, so values stay below 2 B + 6 p, but for two places
// where a third product comes before the next reduction: step 1 of MAT_MID2
// (both halves of whose step 0 are products) and step 0 of COL_LAST (which
// reads what COL_FIRST left, up to 2 B + p).  VALUE_MAX p = 3 B + p is inside
// the digits' range, 127/255 2^768, by 0.1%.
#pragma once

#include <type_traits>

#include "ntt_kernels.h"

namespace gsn {

typedef int v4i __attribute__((ext_vector_type(4)));
typedef int v16i __attribute__((ext_vector_type(16)));

struct W24 {
    uint32_t v[24];
};

// Constants of the offset form.
template <class P>
struct Mat753 {
    using F = F753<P>;
    static constexpr uint32_t K80 = 0x80808080u;
    // Accumulators start at BIAS in every byte row, so that column sums are
    // positive; over the 96 rows BIAS 256^m sums to 2^782 - 2^14 = -2^14 mod
    // 2^768, which row 0 makes up for.
    static constexpr int BIAS = (1 << 22) - (1 << 14);
    static constexpr uint32_t BIAS_ROW0 = 1u << 14;
    static constexpr uint32_t VALUE_MAX = 18434u;
    static_assert((uint64_t)VALUE_MAX * (P::MOD[23] + 1ull) <= 0x7F7F7F7Full, "values are sums of signed byte digits");
    // a multiple of p above what a last pass or a single product leaves, 2 B + p
    // at most: x + LIFT p is positive and below 2^768
    static constexpr uint32_t LIFTED_MAX = 12290u, LIFT = 12400u;
    static_assert(LIFT > LIFTED_MAX && (uint64_t)(LIFT + LIFTED_MAX) * (P::MOD[23] + 1ull) < 1ull << 32,
                  "lifted values are positive and below 2^768");

    static constexpr W24 lift_offset()  // LIFT p - 0x8080..80 mod 2^768
    {
        W24 o{};
        uint64_t c = 0, b = 0;
        for (int i = 0; i < 24; ++i) {
            c += (uint64_t)LIFT * P::MOD[i];
            const uint64_t d = (uint64_t)(uint32_t)c - K80 - b;
            o.v[i] = (uint32_t)d;
            b = (d >> 32) & 1;
            c >>= 32;
        }
        return o;
    }
    // p in signed 32-bit digits
    static constexpr W24 signed_mod()
    {
        W24 o{};
        uint64_t c = 0;
        for (int i = 0; i < 24; ++i) {
            c += P::MOD[i];
            o.v[i] = (uint32_t)c;
            c = (c >> 32) + ((c >> 31) & 1);
        }
        return o;
    }
    static constexpr W24 LIFT_OFF = lift_offset();
    static constexpr W24 SMOD = signed_mod();

    // x + 0x8080..80 mod 2^768
    __device__ __forceinline__ static E753 to_offset(const E753 &x)
    {
        E753 o;
        unsigned c = 0;
#pragma unroll
        for (int i = 0; i < 24; ++i)
            o.v[i] = __builtin_addc(x.v[i], K80, c, &c);
        return o;
    }
    // a positive representative below 2^768 of the value with offset form x
    __device__ __forceinline__ static E753 from_offset(const E753 &x)
    {
        E753 o;
        unsigned c = 0;
#pragma unroll
        for (int i = 0; i < 24; ++i)
            o.v[i] = __builtin_addc(x.v[i], LIFT_OFF.v[i], c, &c);
        return o;
    }
    // x reduced to |x| <= 0.51 p, both in offset form: the quotient comes
    // from the top limb alone (p is above 2^16 units of it)
    __device__ __forceinline__ static E753 reduce(const E753 &x)
    {
        constexpr double TOP = (double)P::MOD[23] + (double)P::MOD[22] / 4294967296.0;
        const int32_t xt = (int32_t)(x.v[23] - K80);
        const int32_t nq = -(int32_t)__builtin_rintf((float)xt * (float)(1.0 / TOP));
        E753 o;
        unsigned c = 0;
        int64_t s = 0;
#pragma unroll
        for (int i = 0; i < 24; ++i) {
            s += (int64_t)nq * (int32_t)SMOD.v[i];
            o.v[i] = __builtin_addc(x.v[i], (uint32_t)s, c, &c);
            s >>= 32;
        }
        return o;
    }
    // (x0 + t, x0 - t), x0 in offset form
    __device__ __forceinline__ static void butterfly(E753 &x0, E753 &t)
    {
        unsigned c = 0, b = 0;
#pragma unroll
        for (int i = 0; i < 24; ++i) {
            const uint32_t a = x0.v[i], d = t.v[i];
            x0.v[i] = __builtin_addc(a, d, c, &c);
            t.v[i] = __builtin_subc(a, d, b, &b);
        }
    }

    // The digits of each lane's x as MFMA right operands: b0 holds lanes
    // 0..31 as columns, b1 lanes 32..63.  K block J holds bytes 32 J ..
    // 32 J + 31, the first 16 in the low half of the wave and the rest in
    // the high half, so one swap of half waves per word pair makes both.
    __device__ __forceinline__ static void digits(v4i (&b0)[3], v4i (&b1)[3], const E753 &x)
    {
#pragma unroll
        for (int J = 0; J < 3; ++J)
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                const auto s = __builtin_amdgcn_permlane32_swap(x.v[8 * J + i] ^ K80, x.v[8 * J + 4 + i] ^ K80, false,
                                                                false);
                b0[J][i] = (int)s[0];
                b1[J][i] = (int)s[1];
            }
    }
};

typedef __attribute__((address_space(1))) const v4i gcv4i;

// y w for the wave's 64 lanes: b0, b1 are the digits of y, m the matrices of
// w: one for the whole wave, or (GROUPS = 2) one per half, or (GROUPS = 4)
// one per 16 lanes, each half then taking two products of which the other's
// digits are masked out.  The result is signed, modulo 2^768 (no offset).
//
// The 32 x 32 result block I of a half wave leaves rows 8 q + 4 h + (0..3)
// of its columns in registers 4 q .. 4 q + 3 of half h: four byte columns of
// limb 8 I + 2 q + h.  They combine into two words there (bytes 0, 1 and
// bytes 2, 3), and one swap of half waves per word brings both halves'
// limbs to their own lanes.
// With BUTTERFLY the product t goes straight into x0 + t (in x0) and x0 - t
// (in y), x0 in offset form: three carry chains interleaved limb by limb, so
// that no carry waits on the instruction right before it.  Else y = t.
template <class P, int GROUPS, bool BUTTERFLY>
__device__ __forceinline__ void mat753_mul(const v4i (&b0)[3], const v4i (&b1)[3], const gcv4i *const (&m)[GROUPS],
                                           v16i bias, E753 &x0, E753 &y)
{
    uint32_t prev = 0;
    unsigned carry = 0, carry_x = 0, borrow_y = 0;
    const auto limb = [&](int l, uint32_t n0, uint32_t n1) {
        const uint32_t v = __builtin_addc(n0, n1, carry, &carry);
        if constexpr (BUTTERFLY) {
            const uint32_t a = x0.v[l];
            x0.v[l] = __builtin_addc(a, v, carry_x, &carry_x);
            y.v[l] = __builtin_subc(a, v, borrow_y, &borrow_y);
        } else {
            y.v[l] = v;
        }
    };
    const int lane = (int)__lane_id();
    v4i lo0[3], lo1[3], hi0[3], hi1[3];
    if constexpr (GROUPS == 4) {
        const int mask = (lane & 16) ? -1 : 0;
#pragma unroll
        for (int J = 0; J < 3; ++J) {
            hi0[J] = b0[J] & mask;
            hi1[J] = b1[J] & mask;
            lo0[J] = b0[J] & ~mask;
            lo1[J] = b1[J] & ~mask;
        }
    }
    v4i blk[GROUPS][3];
#pragma unroll
    for (int g = 0; g < GROUPS; ++g)
#pragma unroll
        for (int J = 0; J < 3; ++J)
            blk[g][J] = m[g][64 * J + lane];
#pragma unroll
    for (int I = 0; I < 3; ++I) {
        v16i d0 = bias, d1 = bias;
        v4i next[GROUPS][3];
        if (I < 2)
#pragma unroll
            for (int g = 0; g < GROUPS; ++g)
#pragma unroll
                for (int J = 0; J < 3; ++J)
                    next[g][J] = m[g][64 * (3 * I + 3 + J) + lane];
#pragma unroll
        for (int J = 0; J < 3; ++J) {
            if constexpr (GROUPS == 4) {
                d0 = __builtin_amdgcn_mfma_i32_32x32x32_i8(blk[0][J], lo0[J], d0, 0, 0, 0);
                d1 = __builtin_amdgcn_mfma_i32_32x32x32_i8(blk[2][J], lo1[J], d1, 0, 0, 0);
                d0 = __builtin_amdgcn_mfma_i32_32x32x32_i8(blk[1][J], hi0[J], d0, 0, 0, 0);
                d1 = __builtin_amdgcn_mfma_i32_32x32x32_i8(blk[3][J], hi1[J], d1, 0, 0, 0);
            } else {
                d0 = __builtin_amdgcn_mfma_i32_32x32x32_i8(blk[0][J], b0[J], d0, 0, 0, 0);
                d1 = __builtin_amdgcn_mfma_i32_32x32x32_i8(blk[GROUPS - 1][J], b1[J], d1, 0, 0, 0);
            }
        }
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            const uint32_t u0 = (uint32_t)d0[4 * q] + ((uint32_t)d0[4 * q + 1] << 8);
            const uint32_t u1 = (uint32_t)d0[4 * q + 2] + ((uint32_t)d0[4 * q + 3] << 8);
            const uint32_t v0 = (uint32_t)d1[4 * q] + ((uint32_t)d1[4 * q + 1] << 8);
            const uint32_t v1 = (uint32_t)d1[4 * q + 2] + ((uint32_t)d1[4 * q + 3] << 8);
            const auto s0 = __builtin_amdgcn_permlane32_swap(u0, v0, false, false);
            const auto s1 = __builtin_amdgcn_permlane32_swap(u1, v1, false, false);
            const int l = 8 * I + 2 * q;
            const uint32_t n0 = l == 0 ? s0[0] + Mat753<P>::BIAS_ROW0 : s0[0];
            limb(l, n0, __builtin_amdgcn_alignbit(s1[0], prev, 16));
            limb(l + 1, s0[1], __builtin_amdgcn_alignbit(s1[1], s1[0], 16));
            prev = s1[1];
        }
        if constexpr (GROUPS >= 2)
            __builtin_amdgcn_sched_barrier(0);  // one block's accumulators at a time: the registers are short
        if (I < 2) {
#pragma unroll
            for (int g = 0; g < GROUPS; ++g)
#pragma unroll
                for (int J = 0; J < 3; ++J)
                    blk[g][J] = next[g][J];
        }
    }
}

// One tile of R = 2^LOG_R rows by W = 2^LOG_W columns, four elements per
// thread: a radix-2 decimation in time over positions 0 .. R - 1 of each
// column, two steps between exchanges.  Thread t = u W + c holds column c;
// its elements e = 0..3 start as positions 0 and 1 (bits 0 and 1 of e), i.e.
// rows u + R/2 (e & 1) + R/4 (e >> 1), and bit j of u is position
// LOG_R - 1 - j.  Steps 2p and 2p + 1 pair positions 2p and 2p + 1; then
// these trade places with positions 2p + 2 and 2p + 3, bits LOG_R - 3 - 2p
// and the next lower one of u.  So position q < 2p sits at bit LOG_R - 3 - q
// of u, and kk, the positions below a step, is the low part of brev(u): the
// lanes of a half wave share it, and with it the step's twiddle, except
// where the last bits of u fall inside the 16 or 32 lanes (GROUPS below).
//
// A transform of n = N1 N2 .. NP: the input index is j1 .. jP, most
// significant digit first, and pass i replaces ji by ki in place, so every
// pass reads and writes the same address but the first's source and the
// last's destination, where the output index is k1 + N1 k2 + ...  The
// twiddle of a pair of digits a < b is w_n^(jb N(b+1)..NP  ka N1..N(a-1)),
// to be applied between passes a and b, in a pass whose tiles let many
// elements share it:
//   (i - 1, i)   pass i holds k(i-1) fixed in a tile; the factor goes into
//                the steps' twiddles ("folded": step s multiplies by
//                w_{G 2^(s+1)}^(k(i-1) + G kk), G = N(i-1));
//   (i - 1, P)   the columns of a pass between the first and the last
//                (MAT_MID) are W consecutive jP, so it is one factor per
//                column: a product after the steps, with the rows of one
//                column across the lanes;
//   (1, 3)       of four passes: fixed in a tile of the second pass (j3 is),
//                so one product more on half of the elements at its step 0.
// The columns of the last pass are W consecutive k1.  n^-1 rides on the
// column factors of the first MAT_MID pass.

// Transforms of the columns of an array, lanes on adjacent ones
// (columns753.hip): COL_FIRST is MAT_FIRST with the columns after the digits
// j2 .., COL_LAST the second and last pass, k1 fixed and folded.  Their tiles
// may end early.
enum : int { COL_FIRST = 16, COL_LAST = 17 };

// What a pass needs, held in scalar registers: jobs come through a table
// whose loads the compiler takes for lane-varying.
struct MatArgs {
    const void *in;
    void *out;
    const void *fold, *col, *fix;  // matrices: folded, per column, and the pair (1, 3) (null: none)
    uint32_t log_n, log_s, log_g, log_np, log_n1, flags, blk;
    uint32_t cols;  // COL_FIRST, COL_LAST
};
__device__ __forceinline__ uint32_t uniform(uint32_t v) { return (uint32_t)__builtin_amdgcn_readfirstlane((int)v); }
template <class T>
__device__ __forceinline__ T *uniform(T *p)
{
    const uint64_t v = (uint64_t)p;
    return (T *)(((uint64_t)uniform((uint32_t)(v >> 32)) << 32) | uniform((uint32_t)v));
}
template <class F>
__device__ __forceinline__ MatArgs mat_args(const PassJob<F> &j, uint32_t tile)
{
    return MatArgs{uniform((const void *)j.a.in),        uniform((void *)j.a.out),
                   uniform((const void *)j.a.tw_col),    uniform((const void *)j.a.tw_pass),
                   uniform((const void *)j.a.tw_pass_a), uniform(j.a.log_n),
                   uniform(j.a.log_s),                   uniform(j.a.log_g),
                   uniform(j.a.log_np),                  uniform(j.a.log_n1),
                   uniform(j.a.flags),                   uniform(tile - j.first_tile),
                   0u};
}

// LDS of a tile.  Exchanges pass three of a thread's four elements.  Where rows
// and columns trade roles (linear global accesses, the column factors) half
// of the rows, or a block of 2^LOG_CB columns, is staged in rows of one
// column more and six planes 3 mod 16 quads apart, which spreads accesses
// along rows, along columns and along an element's quads over the banks.
constexpr int mat_log_cb(int log_r) { return 9 - log_r; }
constexpr int mat_plane(int quads) { return (quads + 12) / 16 * 16 + 3; }
constexpr int mat_lds_quads(int kind, int log_r, int log_w)
{
    const int exchange = 18 << (log_r + log_w - 2);
    const int columns = 6 * mat_plane(((1 << mat_log_cb(log_r)) + 1) << log_r);
    const int rows = 6 * mat_plane(((1 << log_w) + 1) << (log_r - 1));
    const int stage = kind == MAT_MID || kind == MAT_MID2 ? columns : rows;
    return exchange > stage ? exchange : stage;
}

template <class F, int KIND, int LOG_R, int LOG_W>
struct MatTile {
    using P = typename F::params;
    using M = Mat753<P>;
    static constexpr int R = 1 << LOG_R, W = 1 << LOG_W, T = R * W / 4, UB = LOG_R - 2;
    static constexpr int LOG_CB = mat_log_cb(LOG_R), CB = 1 << LOG_CB, RS = CB + 1, PL = mat_plane(R * RS),
                         PH = mat_plane(R / 2 * (W + 1));
    static constexpr bool FIRST = KIND == MAT_FIRST || KIND == COL_FIRST, MID = KIND == MAT_MID || KIND == MAT_MID2,
                          LAST = KIND == MAT_LAST, ENDS = LAST || KIND == COL_LAST,
                          COL = KIND == COL_FIRST || KIND == COL_LAST;
    typedef __attribute__((address_space(1))) const u32x4 gcq4;
    typedef __attribute__((address_space(1))) u32x4 gq4;

    const MatArgs &a;
    uint4 *lds;
    const int t, c, u;
    uint32_t jj;
    uint32_t valid = W;     // columns of the tile
    uint32_t kap;           // the folded digit, k(i-1)
    uint32_t top = 0;       // MAT_MID: jP of column 0
    uint32_t next = 0;      // MAT_MID: the digits between ji and jP
    size_t in0, in_stride;  // row r, column c of the tile: in0 + r in_stride + c (MAT_LAST: + c in_stride + r)
    size_t out0, out_stride;
    v16i bias;
    E753 x[4];

    __device__ __forceinline__ MatTile(const MatArgs &args, uint4 *mem)
        : a(args), lds(mem), t((int)threadIdx.x), c(t & (W - 1)), u(t >> LOG_W)
    {
        jj = UB ? __builtin_bitreverse32((uint32_t)u) >> ((32 - UB) & 31) : 0u;
        if constexpr (FIRST) {
            kap = 0;
            in0 = out0 = (size_t)a.blk * W;
            in_stride = out_stride = (size_t)(KIND == COL_FIRST ? a.cols : 1u) << (a.log_n - LOG_R);
            if constexpr (KIND == COL_FIRST)
                valid = (uint32_t)(in_stride - in0 < (size_t)W ? in_stride - in0 : (size_t)W);
        } else if constexpr (KIND == COL_LAST) {
            const uint32_t tiles = (a.cols + W - 1) / W;
            kap = a.blk / tiles;
            const uint32_t c0 = (a.blk - kap * tiles) * W;
            valid = a.cols - c0 < (uint32_t)W ? a.cols - c0 : (uint32_t)W;
            in0 = ((size_t)kap << LOG_R) * a.cols + c0;
            in_stride = a.cols;
            out0 = (size_t)kap * a.cols + c0;
            out_stride = (size_t)a.cols << a.log_g;
        } else if constexpr (MID) {
            // tiles with the same k(i-1), which read the same matrices, are
            // neighbours
            const uint32_t log_hi = a.log_n - LOG_R - a.log_s - a.log_g;  // digits before k(i-1)
            const uint32_t p = a.blk >> (a.log_s - LOG_W), lo = (a.blk << LOG_W) & ((1u << a.log_s) - 1u);
            kap = p >> log_hi;
            const uint32_t pre = ((p & ((1u << log_hi) - 1u)) << a.log_g) | kap;
            top = lo & ((1u << a.log_np) - 1u);
            next = lo >> a.log_np;
            in0 = out0 = ((size_t)pre << (a.log_s + LOG_R)) + lo;
            in_stride = out_stride = (size_t)1 << a.log_s;
        } else {
            // the digits k2 .. between k1 and jP: k(P-1), whose tiles read the
            // same matrices, slowest
            const uint32_t rev = a.blk >> (a.log_n1 - LOG_W), k1 = (a.blk << LOG_W) & ((1u << a.log_n1) - 1u);
            const uint32_t log_k = a.log_n - a.log_n1 - LOG_R - a.log_g;
            kap = rev >> log_k;  // rev = k2 or, of four passes, k2 + N2 k3
            const uint32_t mid = log_k ? ((rev & ((1u << log_k) - 1u)) << a.log_g) | kap : rev;
            in_stride = (size_t)1 << (a.log_n - a.log_n1);
            in0 = k1 * in_stride + ((size_t)mid << LOG_R);
            out0 = ((size_t)rev << a.log_n1) + k1;
            out_stride = (size_t)1 << (a.log_n - LOG_R);
        }
    }

    __device__ __forceinline__ E753 gload(size_t i) const
    {
        const gcq4 *p = (const gcq4 *)a.in + 6 * i;
        E753 r;
#pragma unroll
        for (int q = 0; q < 6; ++q) {
            const u32x4 v = p[q];
            r.v[4 * q] = v.x;
            r.v[4 * q + 1] = v.y;
            r.v[4 * q + 2] = v.z;
            r.v[4 * q + 3] = v.w;
        }
        return r;
    }
    // element at quad i of each plane
    __device__ __forceinline__ void lds_put(int i, int plane, const E753 &v)
    {
#pragma unroll
        for (int q = 0; q < 6; ++q)
            lds[q * plane + i] = make_uint4(v.v[4 * q], v.v[4 * q + 1], v.v[4 * q + 2], v.v[4 * q + 3]);
    }
    __device__ __forceinline__ E753 lds_get(int i, int plane) const
    {
        E753 r;
#pragma unroll
        for (int q = 0; q < 6; ++q) {
            const uint4 v = lds[q * plane + i];
            r.v[4 * q] = v.x;
            r.v[4 * q + 1] = v.y;
            r.v[4 * q + 2] = v.z;
            r.v[4 * q + 3] = v.w;
        }
        return r;
    }
    __device__ __forceinline__ void set_bias()
    {
#pragma unroll
        for (int i = 0; i < 16; ++i)
            bias[i] = M::BIAS;
        asm volatile("" : "+v"(bias));  // one set of registers for every product
    }

    // v times the matrix `entry` of tab: into (x0, v) := (x0 + t, x0 - t), or
    // v := t
    template <int GROUPS, bool BUTTERFLY>
    __device__ __forceinline__ void times(E753 &x0, E753 &v, const void *tab, uint32_t entry) const
    {
        v4i b0[3], b1[3];
        M::digits(b0, b1, v);
        const gcv4i *m[GROUPS];
#pragma unroll
        for (int i = 0; i < GROUPS; ++i)
            m[i] = (const gcv4i *)((const char *)tab + (size_t)(uint32_t)__builtin_amdgcn_readlane(
                                                           (int)entry, i * (64 / GROUPS)) * MAT_BYTES);
        mat753_mul<P, GROUPS, BUTTERFLY>(b0, b1, m, bias, x0, v);
    }
    // the steps that reduce x0 first: inputs are below 2 B + 6 p in MAT_MID,
    // below B in MAT_LAST, below 2 B + p in COL_LAST and below 6 p after the two
    // plain steps of MAT_FIRST
    static constexpr bool reduces(int s) { return MID ? s % 2 == 0 : ENDS ? s % 2 == 1 : s % 2 == 1 && s >= 3; }

    // step s on elements lo (bit clear) and up; kk = low K bits of jj plus
    // `more`: matrix entry ((2^s - 1) << log_g) + (kap << s) + kk
    template <int S, int K>
    __device__ __forceinline__ void step(E753 &lo, E753 &up, uint32_t more)
    {
        // lane bits 5 and 4 are bits 5 - LOG_W and 4 - LOG_W of u, positions
        // LOG_R - 3 less these
        constexpr bool D5 = LOG_W <= 5 && LOG_R - 3 - (5 - LOG_W) < K;
        constexpr bool D4 = LOG_W <= 4 && LOG_R - 3 - (4 - LOG_W) < K;
        if (reduces(S))
            lo = M::reduce(lo);
        times<D4 ? 4 : D5 ? 2 : 1, true>(
            lo, up, a.fold, (((1u << S) - 1u) << a.log_g) + (kap << S) + (jj & ((1u << K) - 1u)) + more);
    }

    // lanes with bit L set give p for the partner's q
    template <int L>
    __device__ __forceinline__ static void swap_lanes(E753 &p, E753 &q)
    {
#pragma unroll
        for (int i = 0; i < 24; ++i) {
            const auto s = L == 5 ? __builtin_amdgcn_permlane32_swap(p.v[i], q.v[i], false, false)
                                  : __builtin_amdgcn_permlane16_swap(p.v[i], q.v[i], false, false);
            p.v[i] = s[0];
            q.v[i] = s[1];
        }
    }
    // Through LDS with other wavefronts: of elements E0, E0 + 1 (and with a
    // second thread bit, B1, all four), the thread whose bits B0 and B1 are
    // `own` gives element e != own to the thread with bits e and takes that
    // thread's element `own` in its place.  `own` is the same for a whole
    // wavefront; the comments keep the branches from becoming selects.
    template <int B0, int B1, int E0>
    __device__ __forceinline__ void exchange_waves()
    {
        constexpr int N = B1 < 0 ? 2 : 4, S1 = B1 < 0 ? 0 : B1, AT = E0 / 2 * T;
        const int own =
            __builtin_amdgcn_readfirstlane(((t >> B0) & 1) | (B1 < 0 ? 0 : ((t >> S1) & 1) << 1));
        const int t0 = t & ~((1 << B0) | (B1 < 0 ? 0 : 1 << S1));
        const auto give = [&](int e) {
            lds_put(AT + ((e ^ own) - 1) * T + t0 + ((e & 1) << B0) + (B1 < 0 ? 0 : (e >> 1) << S1), 3 * T, x[E0 + e]);
        };
        const auto take = [&](int e) { x[E0 + e] = lds_get(AT + ((e ^ own) - 1) * T + t, 3 * T); };
        if constexpr (N == 2) {
            if (own) {
                asm volatile("; give 0");
                give(0);
                asm volatile("; end give 0");
            } else {
                asm volatile("; give 1");
                give(1);
                asm volatile("; end give 1");
            }
            __syncthreads();
            if (own) {
                asm volatile("; take 0");
                take(0);
                asm volatile("; end take 0");
            } else {
                asm volatile("; take 1");
                take(1);
                asm volatile("; end take 1");
            }
        } else {
#pragma unroll
            for (int e = 0; e < N; ++e)
                if (e != own) {
                    asm volatile("; give %0" ::"n"(e));
                    give(e);
                }
            __syncthreads();
#pragma unroll
            for (int e = 0; e < N; ++e)
                if (e != own) {
                    asm volatile("; take %0" ::"n"(e));
                    take(e);
                }
        }
    }
    // Bit 0 of e trades places with thread bit B0 and, if B1 >= 0, bit 1 of
    // e with thread bit B1 = B0 - 1.
    template <int B0, int B1>
    __device__ __forceinline__ void exchange()
    {
        if constexpr (B1 >= 6) {
            __syncthreads();
            exchange_waves<B0, B1, 0>();
        } else {
            if constexpr (B0 >= 6) {
                __syncthreads();
                exchange_waves<B0, -1, 0>();
                exchange_waves<B0, -1, 2>();
            } else {
                swap_lanes<B0>(x[0], x[1]);
                swap_lanes<B0>(x[2], x[3]);
            }
            if constexpr (B1 >= 0) {
                swap_lanes<B1>(x[0], x[2]);
                swap_lanes<B1>(x[1], x[3]);
            }
        }
    }

    // steps 2 p and 2 p + 1, and the exchange before them
    template <int PP>
    __device__ __forceinline__ void pairs()
    {
        if constexpr (2 * PP + 1 < LOG_R) {
            exchange<LOG_W + LOG_R - 1 - 2 * PP, LOG_W + LOG_R - 2 - 2 * PP>();
            step<2 * PP, 2 * PP>(x[0], x[1], 0u);
            step<2 * PP, 2 * PP>(x[2], x[3], 0u);
            step<2 * PP + 1, 2 * PP>(x[0], x[2], 0u);
            step<2 * PP + 1, 2 * PP>(x[1], x[3], 1u << (2 * PP));
            pairs<PP + 1>();
        } else if constexpr (2 * PP < LOG_R) {
            // the last position alone, in bit 0 of e; the one below stays in
            // bit 1
            exchange<LOG_W, -1>();
            step<2 * PP, 2 * PP - 1>(x[0], x[1], 0u);
            step<2 * PP, 2 * PP - 1>(x[2], x[3], 1u << (2 * PP - 1));
        }
    }
    // output row of element e
    __device__ __forceinline__ int row(int e) const
    {
        constexpr int B0 = LOG_R % 2 ? LOG_R - 1 : LOG_R - 2, B1 = LOG_R % 2 ? LOG_R - 2 : LOG_R - 1;
        return (int)jj + ((e & 1) << B0) + ((e >> 1) << B1);
    }

    // Staged rounds.  MAT_MID: columns h CB .. h CB + CB - 1 of all rows.
    __device__ __forceinline__ void stage_columns(int h)
    {
        __syncthreads();
        if (LOG_CB == LOG_W || (c >> LOG_CB) == h)
#pragma unroll
            for (int e = 0; e < 4; ++e)
                lds_put(row(e) * RS + (c & (CB - 1)), PL, x[e]);
        __syncthreads();
    }
    // The others: rows h R/2 .. of all columns, two elements per thread,
    // element (r, c) at quad r (W + 1) + c.
    __device__ __forceinline__ void stage_rows(int h)
    {
        __syncthreads();
#pragma unroll
        for (int e = 0; e < 4; ++e)
            if ((LOG_R % 2 ? e & 1 : e >> 1) == h)  // the top bit of row(e)
                lds_put((row(e) & (R / 2 - 1)) * (W + 1) + c, PH, x[e]);
        __syncthreads();
    }
    // ROWS rows of COLS columns from LDS to global rows r0 .., columns c0 ..:
    // consecutive lanes store consecutive quads.  3 T quads are whole rows,
    // so three places per thread and their multiples cover the block.
    template <int ROWS, int COLS, int STEP, int PLANE>
    __device__ __forceinline__ void stage_store(int r0, int c0) const
    {
        constexpr int N = ROWS * COLS * 6 / T / 3, DR = T / (2 * COLS);
        static_assert(N * DR == ROWS, "three places a thread cover the rows");
        gq4 *o = (gq4 *)a.out + 6 * (out0 + r0 * out_stride + c0);
        uint4 v[3 * N];
        int r[3], z[3];
#pragma unroll
        for (int k = 0; k < 3; ++k) {
            const int m = k * T + t;
            r[k] = m / (6 * COLS);
            z[k] = m % (6 * COLS);
            const uint4 *p = lds + (z[k] % 6) * PLANE + r[k] * STEP + z[k] / 6;
#pragma unroll
            for (int i = 0; i < N; ++i)
                v[k * N + i] = p[i * DR * STEP];
        }
#pragma unroll
        for (int k = 0; k < 3; ++k) {
            if (COL && z[k] >= 6 * (int)valid)
                continue;
            gq4 *p = o + (6 * out_stride * r[k] + z[k]);
#pragma unroll
            for (int i = 0; i < N; ++i) {
                u32x4 w;
                w.x = v[k * N + i].x;
                w.y = v[k * N + i].y;
                w.z = v[k * N + i].z;
                w.w = v[k * N + i].w;
                p[6 * out_stride * (i * DR)] = w;
            }
        }
    }
    // MAT_LAST: the input rows h R/2 .. of every column, each a contiguous run
    __device__ __forceinline__ void stage_load(int h)
    {
        constexpr int N = 2 * (R / 2) * W / T, DC = T / R;  // three places, N columns DC apart each
        const gcq4 *g = (const gcq4 *)a.in + 6 * (in0 + h * (R / 2));
        u32x4 v[3 * N];
        int col[3], z[3];
#pragma unroll
        for (int k = 0; k < 3; ++k) {
            const int m = k * T + t;
            col[k] = m / (3 * R);
            z[k] = m % (3 * R);
            const gcq4 *p = g + (6 * in_stride * col[k] + z[k]);
#pragma unroll
            for (int i = 0; i < N; ++i)
                v[k * N + i] = p[6 * in_stride * (i * DC)];
        }
        __syncthreads();
#pragma unroll
        for (int k = 0; k < 3; ++k) {
            uint4 *p = lds + (z[k] % 6) * PH + (z[k] / 6) * (W + 1) + col[k];
#pragma unroll
            for (int i = 0; i < N; ++i)
                p[i * DC] = make_uint4(v[k * N + i].x, v[k * N + i].y, v[k * N + i].z, v[k * N + i].w);
        }
        __syncthreads();
    }
    // input row of element e
    __device__ __forceinline__ int in_row(int e) const { return u + (e & 1) * (R / 2) + (e >> 1) * (R / 4); }

    // the column factors of a staged round: the lanes take the rows of one
    // column (two of 32 rows, four of 16)
    __device__ __forceinline__ void column_factors(int h)
    {
        constexpr int GROUPS = 64 >> LOG_R;
        const int lane = t & 63, r = lane & (R - 1);
#pragma unroll 1
        for (int k = 0; k < R * CB / T; ++k) {
            const int col = (k * (T / 64) + (t >> 6)) * GROUPS + (lane >> LOG_R);
            const uint32_t entry = (kap << a.log_np) + top + h * CB + col;
            E753 v = lds_get(r * RS + col, PL), none;
            times<GROUPS, false>(none, v, a.col, entry);
            lds_put(r * RS + col, PL, M::to_offset(v));
        }
        __syncthreads();
    }

    __device__ __forceinline__ void run()
    {
        if constexpr (LAST) {
#pragma unroll
            for (int h = 0; h < 2; ++h) {
                stage_load(h);
#pragma unroll
                for (int e = h; e < 4; e += 2)
                    x[e] = lds_get((in_row(e) & (R / 2 - 1)) * (W + 1) + c, PH);
            }
        } else {
#pragma unroll
            for (int e = 0; e < 4; ++e)
                x[e] = gload(in0 + in_row(e) * in_stride + (COL ? min(c, (int)valid - 1) : c));
        }
        set_bias();
        if constexpr (FIRST) {
            // canonical inputs, without an offset; steps 0 and 1 have the
            // twiddles 1 and, for x[3], w_4
            x[0] = M::to_offset(x[0]);
            M::butterfly(x[0], x[1]);
            M::butterfly(x[2], x[3]);  // without an offset
            M::butterfly(x[0], x[2]);
            x[3] = M::to_offset(x[3]);
            step<1, 0>(x[1], x[3], 1u);
        } else {
            if constexpr (KIND == MAT_MID2) {
                // entry 2 (k1 N3 + j3): the factor, and its product with
                // step 0's twiddle
                const uint32_t entry = 2 * ((kap << (a.log_s - a.log_np)) + next);
                E753 none;
#pragma unroll
                for (int e = 0; e < 4; e += 2) {
                    times<1, false>(none, x[e], a.fix, entry);
                    x[e] = M::to_offset(x[e]);
                    times<1, true>(x[e], x[e + 1], a.fix, entry + 1);
                }
            } else {
                step<0, 0>(x[0], x[1], 0u);
                step<0, 0>(x[2], x[3], 0u);
            }
            step<1, 0>(x[0], x[2], 0u);
            step<1, 0>(x[1], x[3], 1u);
        }
        pairs<1>();
        if constexpr (ENDS) {
#pragma unroll
            for (int e = 0; e < 4; ++e)
                x[e] = F::canon(M::from_offset(x[e]));
        }
#pragma unroll
        for (int h = 0; h < (MID ? W / CB : 2); ++h) {
            if constexpr (MID) {
                stage_columns(h);
                column_factors(h);
                stage_store<R, CB, RS, PL>(0, h * CB);
            } else {
                stage_rows(h);
                stage_store<R / 2, W, W + 1, PH>(h * (R / 2), 0);
            }
        }
    }
};

// Two waves per SIMD is the register budget.
template <class F, int KIND, int LOG_R, int LOG_W>
__global__ __launch_bounds__(1 << (LOG_R + LOG_W - 2)) __attribute__((amdgpu_waves_per_eu(2))) void mat753_kernel(
    PassJob<F> single, const PassJob<F> *__restrict__ jobs, const uint32_t *__restrict__ tile_job)
{
    __shared__ uint4 lds[mat_lds_quads(KIND, LOG_R, LOG_W)];
    const uint32_t tile = xcd_tile(blockIdx.x, gridDim.x);
    const MatArgs args = jobs ? mat_args(jobs[tile_job[tile]], tile) : mat_args(single, tile);
    MatTile<F, KIND, LOG_R, LOG_W>(args, lds).run();
}

// w_n^e for e < n = 2^log_n, canonical: hi[e >> h] lo[e mod 2^h] for e < n/2,
// and its negative past that
template <class F>
__device__ __forceinline__ E753 root_power(const E753 *hi, const TW753 *lo, uint32_t h, uint32_t log_n, size_t e)
{
    const size_t half = (size_t)1 << (log_n - 1), x = e & (half - 1);
    E753 v = F::canon(F::mul(hi[x >> h], F::load_tw(lo, x & (((size_t)1 << h) - 1u))));
    if (e >= half) {
        unsigned b = 0;
#pragma unroll
        for (int l = 0; l < 24; ++l)
            v.v[l] = __builtin_subc(F::params::MOD[l], v.v[l], b, &b);
    }
    return v;
}

// Byte matrices of the residues value(i), i < entries: a wavefront forms five,
// 12 lanes each, a lane the columns 8 t .. 8 t + 7: the first as a product,
// each next one as 256 times the one before it, centred and written as signed
// digits.  A plan's thousands of matrices would otherwise be thousands of
// products (a column each: 250 us for 4096, with the residues' own products,
// the same for a whole block, on the scalar unit).
constexpr uint32_t MATS_PER_WAVE = 5;
template <class F, class V>
__device__ __forceinline__ void write_matrices(uint4 *out, uint32_t entries, V value)
{
    using P = typename F::params;
    __shared__ __align__(16) uint8_t img[MATS_PER_WAVE * MAT_BYTES];
    const uint32_t first = blockIdx.x * MATS_PER_WAVE, group = threadIdx.x / 12;
    const uint32_t t = threadIdx.x - 12 * group, m = min(group, MATS_PER_WAVE - 1);  // (four lanes repeat the last's)
    const TW753 w = F::make_tw(value(min(first + m, entries - 1)));
    E753 v;
#pragma unroll
    for (int l = 0; l < 24; ++l)
        v.v[l] = (uint32_t)l == 2 * t ? 1u : 0u;
    v = F::canon(F::mul(v, w));
#pragma unroll 1
    for (uint32_t k = 8 * t;;) {
        // centre: v - p when v > p/2 (compare the top limbs; either choice is
        // right to within 2^-16 p)
        unsigned b = 0;
        E753 d;
#pragma unroll
        for (int l = 0; l < 24; ++l)
            d.v[l] = __builtin_subc(v.v[l], P::MOD[l], b, &b);
        const bool neg = v.v[23] > P::MOD[23] / 2;
        unsigned c = 0;
#pragma unroll
        for (int l = 0; l < 24; ++l) {
            const uint32_t x = __builtin_addc(neg ? d.v[l] : v.v[l], Mat753<P>::K80, c, &c) ^ Mat753<P>::K80;
#pragma unroll
            for (int byte = 0; byte < 4; ++byte) {
                const uint32_t r = 4 * l + byte;
                img[m * MAT_BYTES + ((r >> 5) * 3 + (k >> 5)) * 1024 + ((r & 31) + 32 * ((k & 31) >> 4)) * 16 +
                    (k & 15)] = (uint8_t)(x >> (8 * byte));
            }
        }
        if ((++k & 7) == 0)
            break;
#pragma unroll
        for (int l = 23; l > 0; --l)
            v.v[l] = __builtin_amdgcn_alignbit(v.v[l], v.v[l - 1], 24);
        v.v[0] <<= 8;
        v = F::canon(v);
    }
    __syncthreads();
    const uint32_t quads = min(MATS_PER_WAVE, entries - first) * (MAT_BYTES / 16);
    for (uint32_t q = threadIdx.x; q < quads; q += 64)
        out[(size_t)first * (MAT_BYTES / 16) + q] = reinterpret_cast<const uint4 *>(img)[q];
}

// Matrices of entries i.  FOLD: the twiddles of a pass's steps, entry
// ((2^s - 1) << log_y) + (g << s) + kk being w_{G 2^(s+1)}^(g + G kk),
// G = 2^log_y.  Else entry x 2^log_y + y is w_n^(x y mul), times *scale if
// use_scale; with pair, entries 2 (x 2^log_y + y) and the one after it are
// that and its product with w_n^(x add).
template <class F, bool FOLD>
__global__ __launch_bounds__(64) void build_mat753_kernel(uint4 *out, uint32_t entries, const E753 *hi,
                                                         const TW753 *lo, uint32_t h, uint32_t log_n, uint32_t log_y,
                                                         uint64_t mul, uint64_t add, int pair, TW753 scale,
                                                         int use_scale)
{
    write_matrices<F>(out, entries, [&](uint32_t i) {
        size_t e;
        if (FOLD) {
            const uint32_t s = 31u - (uint32_t)__builtin_clz((i >> log_y) + 1u);
            const uint32_t rest = i - (((1u << s) - 1u) << log_y);
            const uint32_t g = rest >> s, kk = rest & ((1u << s) - 1u);
            e = ((size_t)g + ((size_t)kk << log_y)) << (log_n - log_y - s - 1u);
        } else {
            const uint32_t z = pair ? i >> 1 : i;
            const size_t x = z >> log_y, y = z & ((1u << log_y) - 1u);
            e = x * y * mul + (pair && (i & 1) ? x * add : 0);
        }
        const E753 v = root_power<F>(hi, lo, h, log_n, e);
        return use_scale ? F::canon(F::mul(v, scale)) : v;
    });
}
constexpr uint32_t mat_blocks(uint32_t entries) { return (entries + MATS_PER_WAVE - 1) / MATS_PER_WAVE; }

// tiles of 32 columns; 2^4 rows only in MAT_MID (matrix_passes uses no others)
#define GSN_MAT753_CASE(F, K, R)                                                                                   \
    case R:                                                                                                        \
        hipLaunchKernelGGL((mat753_kernel<F, K, R, 5>), dim3(grid), dim3(1 << (R + 3)), 0, st, single, jobs,       \
                           tile_job);                                                                              \
        break;
#define GSN_MAT753_KIND(F, K)                                                                                      \
    switch (c.log_r) {                                                                                             \
        GSN_MAT753_CASE(F, K, 5)                                                                                   \
        GSN_MAT753_CASE(F, K, 6)                                                                                   \
    default: break;                                                                                                \
    }
#define GSN_MAT753_LAUNCHES(F)                                                                                        \
    template <>                                                                                                       \
    void launch_mat<F>(const PassJob<F> &single, const PassJob<F> *jobs, const uint32_t *tile_job, uint32_t grid,     \
                       const PassCfg &c, hipStream_t st)                                                              \
    {                                                                                                                 \
        switch (c.kind) {                                                                                             \
        case MAT_FIRST: GSN_MAT753_KIND(F, MAT_FIRST) break;                                                          \
        case MAT_MID:                                                                                                 \
            switch (c.log_r) {                                                                                        \
                GSN_MAT753_CASE(F, MAT_MID, 4)                                                                        \
                GSN_MAT753_CASE(F, MAT_MID, 5)                                                                        \
                GSN_MAT753_CASE(F, MAT_MID, 6)                                                                        \
            default: break;                                                                                           \
            }                                                                                                         \
            break;                                                                                                    \
        case MAT_MID2: GSN_MAT753_KIND(F, MAT_MID2) break;                                                              \
        default: GSN_MAT753_KIND(F, MAT_LAST)                                                                         \
        }                                                                                                             \
    }                                                                                                                 \
    template <>                                                                                                       \
    void launch_build_mat753<F>(uint4 *out, uint32_t entries, bool fold, const E753 *hi, const TW753 *lo, uint32_t h, \
                                uint32_t log_n, uint32_t log_y, uint64_t mul, uint64_t add, bool pair,                \
                                const TW753 *scale, hipStream_t st)                                                   \
    {                                                                                                                 \
        const TW753 one{};                                                                                            \
        if (fold)                                                                                                     \
            hipLaunchKernelGGL((build_mat753_kernel<F, true>), dim3(mat_blocks(entries)), dim3(64), 0, st, out,       \
                               entries, hi, lo, h, log_n, log_y, mul, add, 0, one, 0);                                \
        else                                                                                                          \
            hipLaunchKernelGGL((build_mat753_kernel<F, false>), dim3(mat_blocks(entries)), dim3(64), 0, st, out,      \
                               entries, hi, lo, h, log_n, log_y, mul, add, (int)pair, scale ? *scale : one,           \
                               (int)(scale != nullptr));                                                              \
    }

}  // namespace gsn
