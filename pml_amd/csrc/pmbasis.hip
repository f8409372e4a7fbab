// Approximant bases on the device: M-Basis (iterative, one order per step)
// and PM-Basis (divide and conquer on the order, with the device middle
// product and product), following
//   flint-extras/src/nmod_mat_poly_extra/nmod_mat_poly_mbasis.c:116-378
//   flint-extras/src/nmod_poly_mat_extra/approximant_basis.c:18-69
//   flint-extras/src/nmod_mat_extra/left_nullspace.c:42-102
//
// One M-Basis step at order `ord`:
//  1. residual = coefficient ord of appbas * F.  It is kept as a truncated
//     series R = appbas * F mod x^order, updated by the same row operations
//     as appbas (the value is unique, so this equals the reference's
//     nmod_mat_poly_mul_coeff);
//  2. perm = stable sort of (shift[i], i); residual rows permuted by it;
//  3. left nullspace of the permuted residual in compact form: from the
//     reduced row echelon form R of its transpose (computed fraction-free,
//     then each pivot row divided by its pivot), X[t][r] = -R[r][nonpivot_t],
//     permutation = (pivot columns) ++ (non-pivot columns);
//  4. nullity 0: appbas <- x^(order-ord) appbas, shift += order-ord, stop;
//     nullity m: nothing; otherwise with piv[i] = perm[permutation[i]]:
//     shift[piv[r]] += 1 (r < rank), row piv[rank+t] += sum_r X[t][r] row piv[r],
//     rows piv[r] multiplied by x (length grows when one of them reaches the top).
//
// Kernel 1 (one workgroup) does 2-4 for a window of consecutive orders: it
// holds the window's residual coefficients in LDS, updates them itself after
// each order, and writes every order's description; kernel 2 (a grid) then
// applies the window's row operations, one after the other, to tiles of
// appbas and of the rest of R held in LDS, reading one buffer and writing the
// other (a thread per coefficient where windows do not pay: mbasis_window).
// All control (nullity cases, basis length) stays on the device: a leaf is a
// fixed sequence of launches.  The steps
// skip the division by the pivots in 3: with D the product of the pivots,
// they apply D X and multiply the updated rows by D, so each basis row is the
// reference's row times a known nonzero scale, and the leaf divides the
// scales out at its end.  The step's decisions only read which entries are
// zero, which row scaling keeps, and the normalised kernel of the scaled
// residual, applied to the scaled rows, gives the scaled normalised update.
#include <algorithm>
#include <chrono>
#include <cstring>
#include <type_traits>

#include <climits>

#include "ctx.hpp"
#include "host_arith.hpp"
#include "rules.hpp"

namespace pmlg {

namespace {

constexpr int kStepThreads = 1024;
constexpr int kMaxM = 256;    // rows of F (basis dimension) in the device M-Basis step
constexpr int kMaxN = 128;    // columns of F: at most two rows of the transposed residual per lane
constexpr int kPanel = 4;     // widest Gauss-Jordan panel (LDS is sized for it)
constexpr int kWindow = 4;    // most orders one launch of the step kernel takes
constexpr int kTile = 16;     // coefficients of a tile of the update kernel, its w leading ones a halo
// Shapes accepted: the transposed residual and the panel buffers within what
// the 128 x 128 shape needs with 64-bit words
constexpr size_t kStepLdsMax = 147968;
constexpr size_t kLds = 159 * 1024;  // dynamic LDS of one workgroup (its static LDS is below 1 KiB)

// LDS bytes that decide whether an m x n residual with words of wbytes is
// accepted: shifts (m 64-bit words), At (n rows of odd stride m | 1), the
// pivot cofactors (kMaxN), two coefficient buffers (kMaxN x (kPanel + 1) each),
// then the int arrays (4 of m, 3 of kMaxN)
__host__ __device__ inline size_t step_lds_bytes(int m, int n, size_t wbytes)
{
    return (size_t)m * 8 +
           ((size_t)n * (m | 1) + kMaxN + 2 * (size_t)kMaxN * (kPanel + 1)) * wbytes +
           (4 * (size_t)m + 3 * (size_t)kMaxN) * sizeof(int);
}
// Residual coefficients that the step kernel holds in LDS for a window of w
// orders: all of them, which the windows' choice makes fit, but for a single
// order's too large for it (read from memory when the rows' places are known)
__host__ __device__ inline int window_slots(int m, int n, int w, size_t wbytes)
{
    const size_t base = step_lds_bytes(m, n, wbytes) + (size_t)m * (wbytes + sizeof(int));
    return w > 1 || base + (size_t)m * n * wbytes <= kLds ? w : 0;
}
// LDS bytes of the step kernel with a window of w orders: those of
// step_lds_bytes, the row scales and delays, and the coefficients
__host__ __device__ inline size_t window_lds_bytes(int m, int n, int w, size_t wbytes)
{
    return step_lds_bytes(m, n, wbytes) + (size_t)m * (wbytes + sizeof(int)) +
           (size_t)m * n * window_slots(m, n, w, wbytes) * wbytes;
}
// LDS bytes of the update kernel but the staged vectors: the tile, the
// window's row lists, the delays and a word per wave
__host__ __device__ inline size_t update_lds_bytes(int m, size_t wbytes)
{
    return ((size_t)m * kTile * wbytes + ((size_t)m * (kWindow + 1) + 8) * sizeof(int) + 15) & ~(size_t)15;
}
__host__ __device__ inline int pad16(int r)
{
    return (r + 15) & ~15;
}
// most words of one order's kernel vectors, rows padded to a multiple of 16
inline size_t staged_words(int m, int n)
{
    size_t most = 0;
    for (int r = 1; r <= std::min(m, n); ++r)
        most = std::max(most, (size_t)(m - r) * pad16(r));
    return most;
}
// Orders per window that LDS allows: the step kernel's coefficients, and the
// update kernel's vectors in half of it, so that two workgroups share a compute
// unit (32-bit words, 192 x 24 at order 1500: 161 us an order in windows of 4, 114 in
// windows of 2)
inline int window_orders(int m, int n, size_t wbytes)
{
    int w = kWindow;
    while (w > 1 && (window_lds_bytes(m, n, w, wbytes) > kLds ||
                     update_lds_bytes(m, wbytes) + staged_words(m, n) * w * wbytes > kLds / 2))
        --w;
    return w;
}
constexpr int kXPad = 32;     // words after X read (and discarded) by mbasis_update1_kernel's last group

// control words of one leaf
enum Ctl {
    C_CUR = 0,    // index (0/1) of the buffers holding the current appbas and R
    C_STEPS = 1,  // orders of this window that kernel 2 applies
    C_LEN = 2,    // length of appbas at the window's start
    C_DONE = 4,   // full-rank residual met: the leaf is finished
    C_SHIFT = 5,  // then: power of x that appbas is still to be multiplied by
    C_FLIP = 6,   // kernel 2 wrote the other buffers: swap before the next window
    C_RANK = 8,   // rank of the residual at each order of the window (0: nothing to do)
    C_WORDS = 16
};
static_assert(C_RANK + kWindow <= C_WORDS, "a rank per order of the window");

struct LeafArgs {
    int m, n;
    int ordL;     // order of the leaf
    int cap;      // coefficient capacity of appbas (ordL + 1)
    int window;   // orders per launch of the step kernel
    uint64_t *app[2];  // m x m x cap, entry-major
    uint64_t *R[2];    // m x n x ordL, entry-major
    uint64_t *Rn;      // the coming window's residual coefficients: m x n each, one after the other
    // Row scales.  The steps use unnormalised kernel vectors (own coefficient
    // D, the product of the step's pivots, instead of 1), so basis row i is
    // scale[i] times the normalised one; the leaf divides them out at its
    // end.  scale[m + s] holds D of the window's order s (in the step
    // kernel's arithmetic, as X).
    uint64_t *scale;   // m + kWindow words
    uint64_t *X;       // per order of the window: nullity x rank, row stride m, words of the arithmetic
    int *piv;          // per order of the window: m
    int64_t *shift;    // m
    int *ctl;          // C_WORDS
    // lengths that kernel 2's workgroups have seen appbas reach, two words per
    // column (tiles of even and odd number): one word that all of them raised
    // by atomics took 3 us of a window's update
    int *lens;
    ModConst mc;
};

__device__ __forceinline__ uint64_t mulmod_g(uint64_t a, uint64_t b, const ModConst &mc)
{
    if (mc.p < ((uint64_t)1 << 32))
        return barrett(a * b, mc.bm, mc.p);
    if (mc.bits > 62)
        return mulmod_any(a, b, mc);
    uint64_t hi, lo;
    mul128(a, b, hi, lo);
    return reduce128(hi, lo, mc);
}

__device__ __forceinline__ uint64_t submod_g(uint64_t a, uint64_t b, uint64_t p)
{
    return a >= b ? a - b : a + (p - b);
}

__device__ uint64_t invmod_g(uint64_t a, const ModConst &mc)
{
    // Fermat: a^(p-2)
    uint64_t e = mc.p - 2, r = 1, b = a;
    while (e) {
        if (e & 1)
            r = mulmod_g(r, b, mc);
        b = mulmod_g(b, b, mc);
        e >>= 1;
    }
    return r;
}

// Inverse of a in [1, p) modulo a prime p < 2^62 by the extended Euclidean
// algorithm, r_i = s_i a (mod p), with the quotients estimated in double
// precision.  f = fl(r0) / fl(r1) has relative error below 2^-51, so for
// f < 2^49 trunc(f) is within one of the quotient and one correction step
// fixes it; larger quotients (r1 tiny) are refined once on the remainder,
// which is then below (2^11 + 1) r1 in magnitude.  The cofactors stay below p
// in magnitude.  About 0.84 ln p division steps on average against ~log2 p
// dependent squarings for Fermat's a^(p-2).
__device__ uint64_t inv_euclid(uint64_t a, uint64_t p)
{
    uint64_t r0 = p, r1 = a;
    int64_t s0 = 0, s1 = 1;
    double d0 = (double)r0, d1 = (double)r1;  // fl(r0), fl(r1), carried along
    while (r1 != 0) {
        const double f = d0 / d1;
        uint64_t q = (uint64_t)f;
        int64_t rem = (int64_t)(r0 - q * r1);
        if (f >= 0x1p49) {
            const int64_t q2 = (int64_t)((double)rem / (double)r1);
            q += (uint64_t)q2;
            rem -= q2 * (int64_t)r1;
        }
        if (rem < 0) {
            rem += (int64_t)r1;
            --q;
        } else if ((uint64_t)rem >= r1) {
            rem -= (int64_t)r1;
            ++q;
        }
        const int64_t s2 = s0 - (int64_t)q * s1;
        r0 = r1;
        d0 = d1;
        r1 = (uint64_t)rem;
        d1 = (double)r1;
        s0 = s1;
        s1 = s2;
    }
    return s0 < 0 ? (uint64_t)(s0 + (int64_t)p) : (uint64_t)s0;
}

// Arithmetic of the step kernel (p an odd prime below 2^62).  Values in LDS
// are Montgomery residues: x 2^32 mod p for p < 2^30 (Mont32: one 32x32 -> 64
// product, one low product and one multiply-add per reduction), x 2^64 mod p
// otherwise (Mont64: a 64x64 -> 128 product, one low and one high 64-bit
// product, against two Barrett steps and a Shoup step for a plain 128-bit
// reduction).  Zero maps to zero, so pivot tests read the representation
// directly.
struct Mont64Arith {
    using V = uint64_t;
    uint64_t p, pinv, r1, r2;  // pinv = -p^-1 mod 2^64, r1 = 2^64 mod p, r2 = 2^128 mod p
    __device__ explicit Mont64Arith(const ModConst &c)
        : p(c.p), pinv(c.pinvneg), r1(c.r64), r2(mulmod_g(c.r64, c.r64, c)) {}
    __device__ V redc(uint64_t hi, uint64_t lo) const
    {
        // (hi 2^64 + lo + mm p) / 2^64 with mm = lo pinv mod 2^64: the low
        // words sum to 0 when lo = 0 and to 2^64 otherwise; for inputs below
        // p^2 the quotient is below 2p < 2^63
        const uint64_t mm = lo * pinv;
        const uint64_t u = hi + mulhi64(mm, p) + (lo != 0 ? 1 : 0);
        return u >= p ? u - p : u;
    }
    __device__ V mul(V a, V b) const
    {
        uint64_t hi, lo;
        mul128(a, b, hi, lo);
        return redc(hi, lo);
    }
    // Sums of up to eight products, reduced once: t < 8 p^2 <= 2^127, and the
    // REDC quotient is below (8p / 2^64 + 1) p < 3p < 2^64.
    struct Acc {
        uint64_t hi, lo;
    };
    __device__ Acc prod(V a, V b) const
    {
        Acc t;
        mul128(a, b, t.hi, t.lo);
        return t;
    }
    __device__ Acc fma(Acc t, V a, V b) const
    {
        mac128(t.hi, t.lo, a, b);
        return t;
    }
    __device__ V reduce(Acc t) const
    {
        const uint64_t mm = t.lo * pinv;
        uint64_t u = t.hi + mulhi64(mm, p) + (t.lo != 0 ? 1 : 0);
        u = u >= p ? u - p : u;
        return u >= p ? u - p : u;
    }
    // pv x - fr q as pv x + fr (p - q) < 2 p^2: one reduction, quotient < 1.5 p
    __device__ V msub(V pv, V x, V fr, V q) const
    {
        const Acc t = fma(prod(pv, x), fr, p - q);
        return redc(t.hi, t.lo);
    }
    // K independent msubs sharing pv and fr, formed stage by stage so that
    // their dependent multiplies interleave
    template <int K>
    __device__ void msub_n(V pv, const V (&x)[K], V fr, const V (&q)[K], V (&out)[K]) const
    {
        Acc t[K];
#pragma unroll
        for (int i = 0; i < K; ++i)
            t[i] = fma(prod(pv, x[i]), fr, p - q[i]);
        uint64_t mm[K];
#pragma unroll
        for (int i = 0; i < K; ++i)
            mm[i] = t[i].lo * pinv;
#pragma unroll
        for (int i = 0; i < K; ++i) {
            const uint64_t u = t[i].hi + mulhi64(mm[i], p) + (t[i].lo != 0 ? 1 : 0);
            out[i] = u >= p ? u - p : u;
        }
    }
    __device__ V sub(V a, V b) const { return a >= b ? a - b : a + (p - b); }
    // a factor of a lazy sum: -a as p - a (p itself for a = 0)
    __device__ V neg(V a) const { return p - a; }
    __device__ V add(V a, V b) const
    {
        const uint64_t t = a + b;  // < 2p < 2^63
        return t >= p ? t - p : t;
    }
    __device__ V one() const { return r1; }
    __device__ V to(uint64_t x) const { return mul(x, r2); }
    __device__ uint64_t from(V x) const { return redc(0, x); }
    static __device__ V load(const uint64_t *w) { return *w; }
    // a = x R: the plain inverse of a is x^-1 R^-1, and x^-1 R = mul(mul(a^-1, R^2), R^2)
    __device__ V inv(V a) const { return mul(mul(inv_euclid(a, p), r2), r2); }
};

struct Mont32Arith {
    using V = uint32_t;
    uint32_t p, pinv, r1, r2;  // pinv = -p^-1 mod 2^32, r1 = 2^32 mod p, r2 = 2^64 mod p
    __device__ explicit Mont32Arith(const ModConst &c)
        : p((uint32_t)c.p), pinv((uint32_t)c.pinvneg), r1((uint32_t)c.c32), r2((uint32_t)c.c64) {}
    __device__ V redc(uint64_t t) const
    {
        // t < p^2 < 2^60: t + m p < 2^60 + 2^62, and the quotient u is below 2p;
        // min(u, u - p) picks u - p exactly when u >= p (u - p wraps otherwise)
        const uint32_t mm = (uint32_t)t * pinv;
        const uint32_t u = (uint32_t)((t + (uint64_t)mm * p) >> 32);
        const uint32_t v = u - p;
        return v < u ? v : u;
    }
    __device__ V mul(V a, V b) const { return redc((uint64_t)a * b); }
    // Sums of up to eight products, reduced once: t < 8 p^2 < 2^63, t + mm p
    // < 2^63 + 2^62 and the quotient is below (8p / 2^32 + 1) p < 3p < 2^32.
    using Acc = uint64_t;
    __device__ Acc prod(V a, V b) const { return (uint64_t)a * b; }
    __device__ Acc fma(Acc t, V a, V b) const { return t + (uint64_t)a * b; }
    __device__ V reduce(Acc t) const
    {
        const uint32_t mm = (uint32_t)t * pinv;
        uint32_t u = (uint32_t)((t + (uint64_t)mm * p) >> 32);
        uint32_t v = u - p;
        u = v < u ? v : u;
        v = u - p;
        return v < u ? v : u;
    }
    // pv x - fr q as pv x + fr (p - q) < 2 p^2: one reduction, quotient < 2p
    __device__ V msub(V pv, V x, V fr, V q) const
    {
        return redc((uint64_t)pv * x + (uint64_t)fr * (p - q));
    }
    // K independent msubs sharing pv and fr, formed stage by stage so that
    // their dependent multiplies interleave
    template <int K>
    __device__ void msub_n(V pv, const V (&x)[K], V fr, const V (&q)[K], V (&out)[K]) const
    {
        uint64_t t[K];
#pragma unroll
        for (int i = 0; i < K; ++i)
            t[i] = (uint64_t)pv * x[i] + (uint64_t)fr * (p - q[i]);
        uint32_t mm[K];
#pragma unroll
        for (int i = 0; i < K; ++i)
            mm[i] = (uint32_t)t[i] * pinv;
#pragma unroll
        for (int i = 0; i < K; ++i) {
            const uint32_t u = (uint32_t)((t[i] + (uint64_t)mm[i] * p) >> 32);
            const uint32_t v = u - p;
            out[i] = v < u ? v : u;
        }
    }
    // a factor of a lazy sum: -a as p - a (p itself for a = 0)
    __device__ V neg(V a) const { return p - a; }
    __device__ V sub(V a, V b) const
    {
        // a - b, plus p when it wraps: min(d, d + p) as unsigned words
        const uint32_t d = a - b, e = d + p;
        return e < d ? e : d;
    }
    __device__ V add(V a, V b) const
    {
        // a + b < 2p < 2^31: min(s, s - p) as unsigned words
        const uint32_t t = a + b, u = t - p;
        return u < t ? u : t;
    }
    __device__ V one() const { return r1; }
    __device__ V to(uint64_t x) const { return mul((V)x, r2); }
    // a residue below p < 2^30 is the low half of its 64-bit word
    static __device__ V load(const uint64_t *w) { return *reinterpret_cast<const uint32_t *>(w); }
    __device__ uint64_t from(V x) const { return redc(x); }
    __device__ V inv(V a) const
    {
        // Fermat a^(p-2), in the Montgomery domain (r1 is 1 there)
        uint32_t e = p - 2;
        V r = r1, b = a;
        while (e) {
            if (e & 1)
                r = mul(r, b);
            b = mul(b, b);
            e >>= 1;
        }
        return r;
    }
};

// Moduli from 2^62 to 2^64, and p = 2: plain residues, every product
// reduced at once by the division of mod128_any (Moller-Granlund); sums of
// residues may carry out of 64 bits, so additions go through addmod_any.
// Slower than the Montgomery forms, which need p < 2^62 for their lazy sums.
struct BigArith {
    using V = uint64_t;
    ModConst mc;
    __device__ explicit BigArith(const ModConst &c) : mc(c) {}
    __device__ V mul(V a, V b) const { return mulmod_any(a, b, mc); }
    using Acc = uint64_t;  // a reduced running sum
    __device__ Acc prod(V a, V b) const { return mul(a, b); }
    __device__ Acc fma(Acc t, V a, V b) const { return addmod_any(t, mul(a, b), mc.p); }
    __device__ V reduce(Acc t) const { return t; }
    // pv x - fr q
    __device__ V msub(V pv, V x, V fr, V q) const
    {
        return addmod_any(mul(pv, x), mul(fr, q ? mc.p - q : 0), mc.p);
    }
    template <int K>
    __device__ void msub_n(V pv, const V (&x)[K], V fr, const V (&q)[K], V (&out)[K]) const
    {
#pragma unroll
        for (int i = 0; i < K; ++i)
            out[i] = msub(pv, x[i], fr, q[i]);
    }
    __device__ V sub(V a, V b) const { return a >= b ? a - b : a + (mc.p - b); }
    __device__ V neg(V a) const { return sub(0, a); }
    __device__ V add(V a, V b) const { return addmod_any(a, b, mc.p); }
    __device__ V one() const { return 1; }
    __device__ V to(uint64_t x) const { return x; }
    __device__ uint64_t from(V x) const { return x; }
    static __device__ V load(const uint64_t *w) { return *w; }
    __device__ V inv(V a) const
    {
        // Fermat a^(p-2)
        uint64_t e = mc.p - 2;
        V r = 1, b = a;
        while (e) {
            if (e & 1)
                r = mul(r, b);
            b = mul(b, b);
            e >>= 1;
        }
        return r;
    }
};

// workgroup barrier ordering LDS only: global loads in flight stay in flight
__device__ __forceinline__ void lds_barrier()
{
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup", "local");
    __builtin_amdgcn_s_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");
}

// value of v in lane l (l uniform across the wave)
__device__ __forceinline__ uint32_t lane_value(uint32_t v, int l)
{
    return (uint32_t)__builtin_amdgcn_readlane((int)v, l);
}
__device__ __forceinline__ uint64_t lane_value(uint64_t v, int l)
{
    return ((uint64_t)lane_value((uint32_t)(v >> 32), l) << 32) | lane_value((uint32_t)v, l);
}

// ---------------------------------------------------------------------------
// kernel 1: permutation, left nullspace, step description
// ---------------------------------------------------------------------------
// Fraction-free Gauss-Jordan on At = (permuted residual)^T (n x m): pivot rows
// stay where they are (prow[k] is the row of the k-th pivot); for a pivot at
// (pr, c) every other row r becomes
// pv * row_r - At[r][c] * row_pr with pv = At[pr][c].  The k-th row of the
// reduced row echelon form is row prow[k] divided by its pivot; the step
// multiplies by the other pivots' product (the pivot's cofactor) instead, so
// its kernel vectors are the normalised ones times the product of all pivots.
//
// The columns are taken P at a time (a panel).  One wave runs the pivot
// steps of the panel on the panel's columns only and composes them: every row
// ends as C[r][0] * (its own row at the panel's start) + sum_j C[r][j+1] *
// (the pivot row of panel column j at the panel's start), the same exact
// residues as the one-column-at-a-time sequence.  The waves then apply that
// combination to their own columns while the next panel is composed: one
// barrier per panel instead of one per column.
//
// One launch takes the w orders ord0 .. ord0 + w - 1.  The residual's
// coefficients of the window sit in LDS (Rw, slot d of row i its coefficient
// ord0 + d + delay[i]: multiplying a row by x only raises its delay), and after
// each order the kernel rows' coefficients of the orders still to come are
// combined here, so that a window costs one launch of each kernel.
//
// One workgroup and a chain of n pivots: latency bounds it, not throughput.  Of
// the 16.5 us that an order takes (64 x 32, 32-bit words, clock stamps) the
// elimination has 9.0, 8 panels of 0.57 (composition) + 0.42 (apply) + 0.06
// (barrier) each, the window's update 0 to 6.7 with the orders still to come
// (3.5 on average), the sort 0.8, the rest 2.2.  Step plus update kernel per
// order, with one order per launch and panels composed pivot by pivot / as it
// is: 17.7 + 9.5 / 16.1 + 3.5 us (64 x 32, 32-bit), 13.5 + 6.8 / 11.0 + 3.6 us
// (32 x 17, 64-bit).
template <typename Arith, int H>
__global__ void __launch_bounds__(kStepThreads) mbasis_step_kernel(LeafArgs a, int ord0, int w)
{
    extern __shared__ __attribute__((aligned(16))) unsigned char smem[];
    using V = typename Arith::V;
    // panel width: 4 columns for 32-bit words, 2 for 64-bit ones in the
    // one-row kernels, whose dearer products make a shorter composition pay
    // for the extra barriers; the two-row kernels (more than 64 residual
    // columns) are bound by the apply, which wider panels make shorter
    constexpr int P = sizeof(V) == 8 && H == 1 ? 2 : kPanel;
    static_assert(P <= kPanel, "LDS is sized for kPanel");
    // the split composition needs one row per lane and the Montgomery forms;
    // the composition by pairs does not fit the registers with two rows of
    // 64-bit words per lane
    constexpr bool kMont = !std::is_same<Arith, BigArith>::value;
    constexpr bool kFast = kMont && (H == 1 || sizeof(V) == 4);
    constexpr bool kHalf = H == 1 && kMont;
    const int m = a.m, n = a.n;
    const Arith ar(a.mc);
    const int ms = m | 1;                   // odd row stride of At
    const int mn = m * n;
    const int slots = window_slots(m, n, w, sizeof(V));
    // the composed panels' rows (16-byte aligned), 64-bit words (sh), then the
    // V arrays, then the int arrays (sizes as in window_lds_bytes, whose
    // coefficient buffers are sized for kPanel)
    struct alignas(16) Row {
        V v[P];
    };
    Row *Ck = reinterpret_cast<Row *>(smem);                         // 2 x kMaxN: slots 1 .. P
    V *C0 = reinterpret_cast<V *>(Ck + 2 * kMaxN);                   // 2 x kMaxN: slot 0
    int64_t *sh = reinterpret_cast<int64_t *>(C0 + 2 * kMaxN);       // m
    V *At = reinterpret_cast<V *>(sh + m);                           // n x ms
    V *cof = At + n * ms;                                            // kMaxN: pivot cofactors
    V *scl = cof + kMaxN;                                            // m: row scales
    V *Rw = scl + m;                                                 // slots x m x n
    int *perm = reinterpret_cast<int *>(Rw + slots * mn);            // m
    int *plist = perm + m;                                           // m
    int *colpiv = plist + m;                                         // m (columns of At)
    int *pos = colpiv + m;                                           // m (then: pivot row by column)
    int *delay = pos + m;                                            // m
    int *prow = delay + m;                                           // kMaxN (by rank)
    int *ispiv = prow + kMaxN;                                       // kMaxN (rows of At)
    // a composed panel: which columns took a pivot (and kFastPanel), the pivots'
    // rows, the panel's own coefficient K0 and what its pivots' cofactors are made
    // of (by pairs: 1 for the first two, D1 for the others; else the pivots)
    constexpr int kFastPanel = 1 << P;
    __shared__ int s_tk[2], s_prs[2][kPanel];
    __shared__ V s_K0[2], s_pre[2][kPanel];
    __shared__ V s_D;  // the step's D
    const int tid = threadIdx.x;
    const int lane = tid & 63;
    const int wave = tid >> 6;

    // Shifts, row scales, control words and the window's residual
    // coefficients (contiguous in the fixed buffer Rn, written by the previous
    // update or the leaf's initialisation: their loads wait for no control
    // word).  Thread 0 writes the control words back at the end.
    int *c = a.ctl;
    const int flip = c[C_FLIP], cur0 = c[C_CUR], done = c[C_DONE];
    if (wave == kStepThreads / 64 - 1) {
        int len = 1;
        for (int i = lane; i < 2 * m; i += 64)
            len = max(len, a.lens[i]);
        for (int d = 32; d > 0; d >>= 1)
            len = max(len, __shfl_xor(len, d));
        if (lane == 0)
            c[C_LEN] = len;
    }
    if (tid < m) {  // m <= kMaxM <= kStepThreads
        sh[tid] = a.shift[tid];
        scl[tid] = ord0 == 0 ? ar.one() : (V)a.scale[tid];
        delay[tid] = 0;
    }
    const int cur = flip ? cur0 ^ 1 : cur0;
    if (done) {
        if (tid == 0) {
            c[C_CUR] = cur;
            c[C_FLIP] = 0;
            c[C_STEPS] = 0;
        }
        return;
    }
    for (int q = tid; q < slots * mn; q += kStepThreads)
        Rw[q] = ar.to(Arith::load(a.Rn + q));
    // threads per row of the shift sort
    const int sortLog = m <= 64 ? 4 : m <= 128 ? 3 : 2;
    bool full = false;  // full-rank residual met (uniform)
    int steps = 0, rank = 0;
    for (int s = 0; s < w && !full; ++s) {
        if (tid < m)
            colpiv[tid] = 0;
        if (tid < kMaxN)
            ispiv[tid] = 0;
        lds_barrier();

        // stable permutation sorting (shift, index): pos[i] = #{j : (sh_j, j) < (sh_i, i)},
        // counted by 2^sortLog neighbouring threads per row
        {
            const int i = tid >> sortLog, g = tid & ((1 << sortLog) - 1);
            if (i < m) {
                const int64_t si = sh[i];
                int cnt = 0;
                for (int j = g; j < m; j += 1 << sortLog) {
                    const int64_t sj = sh[j];
                    cnt += (sj < si) || (sj == si && j < i) ? 1 : 0;
                }
                for (int d = 1; d < 1 << sortLog; d <<= 1)
                    cnt += __shfl_xor(cnt, d);
                if (g == 0) {
                    pos[i] = cnt;
                    perm[cnt] = i;
                }
            }
        }
        lds_barrier();
        // the residual coefficient of this order, transposed and permuted: one
        // row of the residual per wave, two where they have at most 32 columns
        for (int i = n <= 32 ? tid >> 5 : wave; i < m; i += kStepThreads / (n <= 32 ? 32 : 64)) {
            const int pi = pos[i];
            const size_t slot = slots > 0 ? (size_t)(s - delay[i]) * mn : 0;
            for (int j = n <= 32 ? tid & 31 : lane; j < n; j += 64)
                At[j * ms + pi] = slots > 0 ? Rw[slot + i * n + j] : ar.to(Arith::load(a.Rn + i * n + j));
        }
        lds_barrier();

        // Gauss-Jordan by panels of P columns.  Wave w owns the columns
        // [w cw, (w + 1) cw) of At and applies every panel's combination to them;
        // the owner of the next panel then composes it from its own updated
        // columns (the LDS operations of one wave take effect in program order)
        // while the other waves are still applying: one barrier per panel, with
        // the coefficients double-buffered.
        rank = 0;
        // columns per wave: P times a power of two (so that cw divides the
        // wave's 64 lanes), 16 waves covering m
        int cw = P;
        while (16 * cw < m)
            cw *= 2;
        // compose the panel of columns c0 .. c0 + P - 1 into buffer buf (the
        // lambdas are forced inline: called from two places, compose was left as
        // a call in the two-row kernels, its captures and arrays on the stack)
        auto compose = [&](const int c0, const int buf) __attribute__((always_inline)) {
            __builtin_amdgcn_s_setprio(2);
            {
                // rows lane + 64 h (h < H) of the panel, their pivot flags and the
                // coefficients C[.][0..P] of the composition
                V pn[H][P], cc[H][P + 1];
                bool isp[H], ok[H];
                int prs[P] = {0};
                V pvs[P];
                int tk = 0;  // panel columns that took a pivot
#pragma unroll
                for (int h = 0; h < H; ++h) {
                    const int r = lane + 64 * h;
                    ok[h] = r < n;
                    isp[h] = ok[h] && ispiv[r];
#pragma unroll
                    for (int j = 0; j < P; ++j)
                        pn[h][j] = ok[h] && c0 + j < m ? At[r * ms + c0 + j] : (V)0;
                    cc[h][0] = ar.one();
#pragma unroll
                    for (int s2 = 1; s2 <= P; ++s2)
                        cc[h][s2] = 0;
                }
                int nb = 0;
                // one pivot step on panel column j (a compile-time index: the
                // convergent ballots and lane reads keep the compiler from unrolling
                // a loop around them, and the arrays must stay in registers)
                auto step = [&](auto jc) __attribute__((always_inline)) {
                    constexpr int j = decltype(jc)::value;
                    // columns past m, or a full rank already reached, take no pivot
                    const bool open = c0 + j < m && rank + nb < n;
                    const unsigned long long b0 = __ballot(open && ok[0] && !isp[0] && pn[0][j] != 0);
                    const unsigned long long b1 =
                        H == 2 ? __ballot(open && ok[H - 1] && !isp[H - 1] && pn[H - 1][j] != 0) : 0ull;
                    if (!b0 && !b1)
                        return;  // no pivot in this column
                    const int pr = b0 ? __ffsll(b0) - 1 : 63 + __ffsll(b1);
                    const int pl = pr & 63, ph = pr >> 6;
                    // broadcast the pivot row (panel values and coefficients): the
                    // pivot lane is uniform, so its registers are read into
                    // scalar registers; its self coefficient cc[0] moves to slot
                    // j + 1
                    V qp[P], qc[P + 1];
#pragma unroll
                    for (int jj = j; jj < P; ++jj)
                        qp[jj] = lane_value(H == 2 && ph ? pn[H - 1][jj] : pn[0][jj], pl);
#pragma unroll
                    for (int s2 = 1; s2 <= j; ++s2)
                        qc[s2] = lane_value(H == 2 && ph ? cc[H - 1][s2] : cc[0][s2], pl);
                    qc[j + 1] = lane_value(H == 2 && ph ? cc[H - 1][0] : cc[0][0], pl);
                    const V pv = qp[j];
                    // Only the nonzero terms are formed: column j of every other
                    // row becomes pv * fr - fr * pv = 0, and slots past j are zero
                    // in every row until this step, so slot j + 1 is -fr * qc.
                    // Every lane computes and the pivot lane keeps its own values
                    // (selects, not branches, so the step stays one basic block);
                    // rows past n hold zeros and are never published.
#pragma unroll
                    for (int h = 0; h < H; ++h) {
                        const bool me = lane + 64 * h == pr;
                        const V fr = pn[h][j];
                        // the P products of this step: panel columns j + 1 .. P - 1,
                        // slots 1 .. j, and slot j + 1 (from zero)
                        V xs[P], qs[P], ts[P];
#pragma unroll
                        for (int jj = j + 1; jj < P; ++jj) {
                            xs[jj - j - 1] = pn[h][jj];
                            qs[jj - j - 1] = qp[jj];
                        }
#pragma unroll
                        for (int s2 = 1; s2 <= j; ++s2) {
                            xs[P - j - 2 + s2] = cc[h][s2];
                            qs[P - j - 2 + s2] = qc[s2];
                        }
                        xs[P - 1] = 0;
                        qs[P - 1] = qc[j + 1];
                        ar.msub_n(pv, xs, fr, qs, ts);
#pragma unroll
                        for (int jj = j + 1; jj < P; ++jj)
                            pn[h][jj] = me ? pn[h][jj] : ts[jj - j - 1];
                        pn[h][j] = me ? fr : (V)0;
#pragma unroll
                        for (int s2 = 1; s2 <= j; ++s2)
                            cc[h][s2] = me ? cc[h][s2] : ts[P - j - 2 + s2];
                        cc[h][j + 1] = me ? qc[j + 1] : ts[P - 1];
                        const V t0 = ar.mul(pv, cc[h][0]);
                        cc[h][0] = me ? (V)0 : t0;
                        isp[h] = isp[h] || me;
                    }
                    prs[j] = pr;
                    pvs[j] = pv;
                    tk |= 1 << j;
                    ++nb;
                };
                static_assert(P >= 1 && P <= 4, "the panel steps below are written out for up to 4 columns");
                step(std::integral_constant<int, 0>{});
                if constexpr (P > 1)
                    step(std::integral_constant<int, 1>{});
                if constexpr (P > 2)
                    step(std::integral_constant<int, 2>{});
                if constexpr (P > 3)
                    step(std::integral_constant<int, 3>{});
                // publish: coefficients, pivot flags, pivot rows
#pragma unroll
                for (int h = 0; h < H; ++h) {
                    const int r = lane + 64 * h;
                    if (ok[h]) {
                        C0[buf * kMaxN + r] = cc[h][0];
#pragma unroll
                        for (int s2 = 1; s2 <= P; ++s2)
                            Ck[buf * kMaxN + r].v[s2 - 1] = cc[h][s2];
                        ispiv[r] = isp[h] ? 1 : 0;
                    }
                }
                if (lane == 0) {
                    s_tk[buf] = tk;
#pragma unroll
                    for (int k = 0; k < P; ++k) {
                        s_prs[buf][k] = prs[k];
                        if (tk >> k & 1)
                            s_pre[buf][k] = pvs[k];
                    }
                }
            }
            __builtin_amdgcn_s_setprio(0);
        };
        // Residuals of at most 32 columns (n <= 32 rows of At) leave the upper
        // half of the composing wave idle in compose().  compose_half() puts the
        // coefficient slots there: upper lane 32 + r holds slots 0, 1, 2 of row r
        // (slots 0, 1 for P = 2) and lower lane r the row's panel values and the
        // last slots, in registers whose lower halves pass from a panel column to
        // a slot once that column is eliminated.  Each instruction then advances
        // a panel value and a coefficient at once: three multiply-subtracts per
        // pivot step instead of five (two instead of three for P = 2).
        //   P = 4, registers Z A B C: lower lane r holds row r in panel columns
        //   0..3, A becomes slot 3 before step 2 and B slot 4 before step 3;
        //   upper lane 32 + r holds slots 0, 1, 2 in A, B, C.
        //   P = 2, registers Z A B: lower lane r holds columns 0, 1 in Z, A and
        //   slot 2 in B; upper lane 32 + r holds slots 0, 1 in A, B.
        // Slot 0 takes pv * c0 as the multiply-subtract with q = 0 (pv c0 + fr p,
        // the same residue); a register that starts a slot holds zero, so the
        // slot's first value is -fr * q as in compose().
        auto compose_half = [&](const int c0, const int buf) __attribute__((always_inline)) {
            __builtin_amdgcn_s_setprio(2);
            {
                static_assert(P == 2 || P == 4, "compose_half is written out for panels of 2 and 4");
                const bool hi = lane >= 32;
                const int r = lane & 31;
                const bool ok = r < n;
                auto col = [&](const int j) -> V {
                    return !hi && ok && c0 + j < m ? At[r * ms + c0 + j] : (V)0;
                };
                V Z = col(0);
                V A = hi ? ar.one() : col(1);
                V B = P == 4 ? col(2) : (V)0;
                V C = P == 4 ? col(3) : (V)0;
                bool isp = !hi && ok && ispiv[r];
                int prs[P] = {0};
                V pvs[P];
                int tk = 0, nb = 0;
                // every lane gets the value of x in lane (lane & 31)
                auto low = [](const V x) -> V {
                    if constexpr (sizeof(V) == 4) {
                        return __builtin_amdgcn_permlane32_swap(x, x, false, false)[0];
                    } else {
                        const uint32_t l = (uint32_t)x, h = (uint32_t)(x >> 32);
                        const uint32_t l2 = __builtin_amdgcn_permlane32_swap(l, l, false, false)[0];
                        const uint32_t h2 = __builtin_amdgcn_permlane32_swap(h, h, false, false)[0];
                        return ((uint64_t)h2 << 32) | l2;
                    }
                };
                auto step = [&](auto jc) __attribute__((always_inline)) {
                    constexpr int j = decltype(jc)::value;
                    if constexpr (P == 4 && j == 2)
                        A = hi ? A : (V)0;  // column 1 is done: lower A is slot 3
                    if constexpr (P == 4 && j == 3)
                        B = hi ? B : (V)0;  // column 2 is done: lower B is slot 4
                    const V xj = j == 0 ? Z : j == 1 ? A : j == 2 ? B : C;
                    const bool open = c0 + j < m && rank + nb < n;
                    const unsigned long long b = __ballot(open && !hi && ok && !isp && xj != 0);
                    if (!b)
                        return;  // no pivot in this column
                    const int pr = __ffsll(b) - 1;  // a lower lane
                    const bool me = r == pr;
                    const V pv = lane_value(xj, pr);
                    const V fr = low(xj);
                    const V Q = lane_value(A, 32 + pr);  // the pivot row's slot 0
                    constexpr int G = P == 4 ? 3 : 2;
                    V xs[G], qs[G], ts[G], kp[G];  // operands, and what the pivot row keeps
                    const V zero = 0;
                    if constexpr (P == 4) {
                        xs[0] = A;
                        xs[1] = B;
                        xs[2] = C;
                        if constexpr (j == 0) {
                            const V p1 = lane_value(A, pr), p2 = lane_value(B, pr), p3 = lane_value(C, pr);
                            qs[0] = hi ? zero : p1;
                            qs[1] = hi ? Q : p2;
                            qs[2] = hi ? zero : p3;
                            kp[0] = hi ? zero : A;
                            kp[1] = hi ? Q : B;
                            kp[2] = C;
                        } else if constexpr (j == 1) {
                            const V p2 = lane_value(B, pr), p3 = lane_value(C, pr), q1 = lane_value(B, 32 + pr);
                            qs[0] = zero;
                            qs[1] = hi ? q1 : p2;
                            qs[2] = hi ? Q : p3;
                            kp[0] = hi ? zero : A;
                            kp[1] = B;
                            kp[2] = hi ? Q : C;
                        } else if constexpr (j == 2) {
                            const V p3 = lane_value(C, pr), q1 = lane_value(B, 32 + pr), q2 = lane_value(C, 32 + pr);
                            qs[0] = hi ? zero : Q;
                            qs[1] = hi ? q1 : zero;
                            qs[2] = hi ? q2 : p3;
                            kp[0] = hi ? zero : Q;
                            kp[1] = B;
                            kp[2] = C;
                        } else {
                            const V q3 = lane_value(A, pr), q1 = lane_value(B, 32 + pr), q2 = lane_value(C, 32 + pr);
                            qs[0] = hi ? zero : q3;
                            qs[1] = hi ? q1 : Q;
                            qs[2] = hi ? q2 : zero;
                            kp[0] = hi ? zero : A;
                            kp[1] = hi ? B : Q;
                            kp[2] = C;
                        }
                    } else {
                        xs[0] = A;
                        xs[1] = B;
                        if constexpr (j == 0) {
                            const V p1 = lane_value(A, pr);
                            qs[0] = hi ? zero : p1;
                            qs[1] = hi ? Q : zero;
                            kp[0] = hi ? zero : A;
                            kp[1] = hi ? Q : B;
                        } else {
                            const V q1 = lane_value(B, 32 + pr);
                            qs[0] = zero;
                            qs[1] = hi ? q1 : Q;
                            kp[0] = hi ? zero : A;
                            kp[1] = hi ? B : Q;
                        }
                    }
                    ar.msub_n(pv, xs, fr, qs, ts);
                    A = me ? kp[0] : ts[0];
                    B = me ? kp[1] : ts[1];
                    if constexpr (P == 4)
                        C = me ? kp[2] : ts[2];
                    isp = isp || me;  // read in the lower half only
                    prs[j] = pr;
                    pvs[j] = pv;
                    tk |= 1 << j;
                    ++nb;
                };
                step(std::integral_constant<int, 0>{});
                step(std::integral_constant<int, 1>{});
                if constexpr (P == 4) {
                    step(std::integral_constant<int, 2>{});
                    step(std::integral_constant<int, 3>{});
                }
                // publish: coefficients, pivot flags, pivot rows
                if (ok) {
                    V *ck = Ck[buf * kMaxN + r].v;
                    if (hi) {
                        C0[buf * kMaxN + r] = A;
                        ck[0] = B;
                        if constexpr (P == 4)
                            ck[1] = C;
                    } else {
                        if constexpr (P == 4) {
                            ck[2] = A;
                            ck[3] = B;
                        } else {
                            ck[1] = B;
                        }
                        ispiv[r] = isp ? 1 : 0;
                    }
                }
                if (lane == 0) {
                    s_tk[buf] = tk;
#pragma unroll
                    for (int k = 0; k < P; ++k) {
                        s_prs[buf][k] = prs[k];
                        if (tk >> k & 1)
                            s_pre[buf][k] = pvs[k];
                    }
                }
            }
            __builtin_amdgcn_s_setprio(0);
        };
        // While every panel so far went this way, the pivot rows are simply the
        // rows in order, rank, rank + 1, ..., taken two at a time: for rows s1,
        // s2 with the block [a b; c d] in columns 1, 2 and D1 = ad - bc, every
        // row becomes D1 row - C1 row_s1 - C2 row_s2, C1 = v1 d - v2 c, C2 = v2 a - v1 b
        // (v1, v2 its own values there), and rows s1, s2 their adjugate combinations
        // d row_s1 - b row_s2 and a row_s2 - c row_s1, as the same expression with
        // C1 = D1 - d, C2 = b and C1 = c, C2 = D1 - a.  Two such steps make a panel
        // of four.  Nothing is searched for, so no ballot, bit search and lane read
        // stands between one pivot and the next, and a panel is 6 dependent
        // reductions instead of 4 times 2; the two blocks' determinants must be
        // nonzero, else (false) this panel and the step's later ones are composed
        // pivot by pivot.  The pivots
        // come out as another nonzero multiple than there, which their cofactors
        // take up: a row outside the panel is multiplied by K0, the product of its
        // determinants (or of its pivots), and with D the product of all K0, the
        // cofactor D / pivot of a step's pivots is the product of the earlier steps'
        // determinants (pivots).
        // With n <= 32 (HALF) the lanes 32 + r repeat row r and form the second of
        // every pair of values while the lanes r form the first.
        auto compose_fast = [&](const int c0, const int buf, auto halfc) __attribute__((always_inline)) -> bool {
            constexpr bool HALF = decltype(halfc)::value;
            if (c0 + P > m || rank + P > n)
                return false;
            const bool hi = HALF && lane >= 32;
            // (loads without branches; lanes past row n - 1 repeat it and publish nothing)
            V pn[H][P];
            bool ok[H];
#pragma unroll
            for (int h = 0; h < H; ++h) {
                const int r = HALF ? lane & 31 : lane + 64 * h;
                ok[h] = r < n;
                const V *x = At + (ok[h] ? r : n - 1) * ms + c0;
#pragma unroll
                for (int j = 0; j < P; ++j)
                    pn[h][j] = x[j];
            }
            int sr[P];
#pragma unroll
            for (int k = 0; k < P; ++k)
                sr[k] = rank + k;
            // value of x in row r (uniform), and of panel column j
            auto at = [&](const V (&x)[H], const int r) -> V {
                return lane_value(H == 2 && r >= 64 ? x[H - 1] : x[0], r & 63);
            };
            auto col = [&](const int j, const int r) -> V {
                return lane_value(H == 2 && r >= 64 ? pn[H - 1][j] : pn[0][j], r & 63);
            };
            auto row_of = [&](const int h) { return HALF ? lane & 31 : lane + 64 * h; };
            // the other half's value
            auto other = [&](const V x) -> V {
                if constexpr (!HALF) {
                    return x;
                } else if constexpr (sizeof(V) == 4) {
                    const auto v = __builtin_amdgcn_permlane32_swap(x, x, false, false);
                    return hi ? v[0] : v[1];
                } else {
                    const uint32_t l = (uint32_t)x, u = (uint32_t)(x >> 32);
                    const auto vl = __builtin_amdgcn_permlane32_swap(l, l, false, false);
                    const auto vu = __builtin_amdgcn_permlane32_swap(u, u, false, false);
                    return hi ? ((uint64_t)vu[0] << 32) | vl[0] : ((uint64_t)vu[1] << 32) | vl[1];
                }
            };
            // C1, C2 (with HALF: its own one and the other half's) of a 2 x 2 step on
            // rows r1, r2 and the values x1, x2 (with HALF: own and other) of every row
            auto pair = [&](const V (&x1)[H], const V (&x2)[H], const V a, const V b, const V cc, const V d,
                            const V det, const int r1, const int r2, V (&C1)[H], V (&C2)[H]) {
                const V na = ar.sub(det, a), nd = ar.sub(det, d);
#pragma unroll
                for (int h = 0; h < H; ++h) {
                    const bool me1 = row_of(h) == r1, me2 = row_of(h) == r2;
                    const V t = ar.msub(x1[h], hi ? a : d, x2[h], hi ? b : cc);
                    C1[h] = me1 ? (hi ? b : nd) : me2 ? (hi ? na : cc) : t;
                    if constexpr (HALF) {
                        C2[h] = other(C1[h]);
                    } else {
                        const V u = ar.msub(x2[h], a, x1[h], b);
                        C2[h] = me1 ? b : me2 ? na : u;
                    }
                }
            };
            const V a1 = col(0, sr[0]), b1 = col(1, sr[0]);
            const V c1 = col(0, sr[1]), d1 = col(1, sr[1]);
            const V D1 = ar.msub(a1, d1, b1, c1);
            V x1[H], x2[H], C1[H], C2[H];
#pragma unroll
            for (int h = 0; h < H; ++h) {
                x1[h] = hi ? pn[h][1] : pn[h][0];
                x2[h] = hi ? pn[h][0] : pn[h][1];
            }
            pair(x1, x2, a1, b1, c1, d1, D1, sr[0], sr[1], C1, C2);
            V K0 = D1, k1[H], k2[H], k3[H], k4[H];  // with HALF: k1 | k2 in k1, k3 | k4 in k3
            if constexpr (P == 2) {
#pragma unroll
                for (int h = 0; h < H; ++h) {
                    k1[h] = ar.sub(0, C1[h]);
                    k2[h] = ar.sub(0, C2[h]);
                }
            } else {
                // the other two columns after the first step
                const V q13 = ar.neg(col(2, sr[0])), q14 = ar.neg(col(3, sr[0]));
                const V q23 = ar.neg(col(2, sr[1])), q24 = ar.neg(col(3, sr[1]));
                V v3[H], v4[H];
#pragma unroll
                for (int h = 0; h < H; ++h) {
                    v3[h] = ar.reduce(ar.fma(ar.fma(ar.prod(D1, hi ? pn[h][3] : pn[h][2]), C1[h], hi ? q24 : q13),
                                             C2[h], hi ? q14 : q23));
                    v4[h] = HALF ? other(v3[h])
                                 : ar.reduce(ar.fma(ar.fma(ar.prod(D1, pn[h][3]), C1[h], q14), C2[h], q24));
                }
                // the second block; with HALF lane 32 + r holds the fourth column
                const V a2 = at(v3, sr[2]), c2 = at(v3, sr[3]);
                const V b2 = HALF ? lane_value(v3[0], 32 + sr[2]) : at(v4, sr[2]);
                const V d2 = HALF ? lane_value(v3[0], 32 + sr[3]) : at(v4, sr[3]);
                const V D2 = ar.msub(a2, d2, b2, c2);
                V C3[H], C4[H];
                pair(v3, v4, a2, b2, c2, d2, D2, sr[2], sr[3], C3, C4);
                // D2 (D1 row - C1 q1 - C2 q2) - C3 (D1 q3 - c31 q1 - c32 q2) - C4 (D1 q4 - c41 q1 - c42 q2)
                const V c31 = at(C1, sr[2]), c41 = at(C1, sr[3]);
                const V c32 = HALF ? lane_value(C1[0], 32 + sr[2]) : at(C2, sr[2]);
                const V c42 = HALF ? lane_value(C1[0], 32 + sr[3]) : at(C2, sr[3]);
                const V nD1 = ar.sub(0, D1), nD2 = ar.sub(0, D2);
                K0 = ar.mul(D1, D2);
#pragma unroll
                for (int h = 0; h < H; ++h) {
                    k1[h] = ar.reduce(ar.fma(ar.fma(ar.prod(nD2, C1[h]), C3[h], hi ? c42 : c31), C4[h], hi ? c32 : c41));
                    k3[h] = ar.mul(C3[h], nD1);
                    if constexpr (!HALF) {
                        k2[h] = ar.reduce(ar.fma(ar.fma(ar.prod(nD2, C2[h]), C3[h], c32), C4[h], c42));
                        k4[h] = ar.mul(C4[h], nD1);
                    }
                }
            }
            if (K0 == 0)
                return false;
            // publish the coefficients (what the pivot by pivot composition reads
            // beside them is brought up to date when it first runs)
#pragma unroll
            for (int h = 0; h < H; ++h) {
                V *ck = Ck[buf * kMaxN + row_of(h)].v;
                if (ok[h]) {
                    if constexpr (HALF) {
                        ck[hi ? 1 : 0] = k1[h];
                        if constexpr (P == 4)
                            ck[hi ? 3 : 2] = k3[h];
                    } else {
                        ck[0] = k1[h];
                        ck[1] = k2[h];
                        if constexpr (P == 4) {
                            ck[2] = k3[h];
                            ck[3] = k4[h];
                        }
                    }
                }
            }
            if (lane == 0) {
                s_tk[buf] = kFastPanel | (kFastPanel - 1);
                s_K0[buf] = K0;
                s_pre[buf][0] = D1;
            }
            return true;
        };
        const bool half = kHalf && n <= 32;
        bool inorder = kFast;  // every panel so far by compose_fast (uniform)
        auto compose_panel = [&](const int c0, const int buf) __attribute__((always_inline)) {
            if constexpr (kFast) {
                if (inorder) {
                    __builtin_amdgcn_s_setprio(2);
                    bool done = false;
                    if constexpr (kHalf) {
                        if (half)
                            done = compose_fast(c0, buf, std::true_type{});
                    }
                    if (!half)
                        done = compose_fast(c0, buf, std::false_type{});
                    __builtin_amdgcn_s_setprio(0);
                    if (done)
                        return;
                    // the first panel pivot by pivot: the rows used before
                    for (int r = lane; r < rank; r += 64)
                        ispiv[r] = 1;
                }
            }
            if constexpr (kHalf) {
                if (half) {
                    compose_half(c0, buf);
                    return;
                }
            }
            compose(c0, buf);
        };
        // apply the combination in buffer buf to this wave's columns: the pivot
        // rows' values are read before any row is written.  Every term is
        // formed: a panel column without a pivot has row 0 in s_prs and zero
        // coefficients in every row, so its term is zero, and issuing all loads
        // before the products (no branch between them) keeps the LDS round
        // trips of a panel to three instead of one per term.
        // A pivot column of an earlier panel (below cdone) is zero but in its
        // pivot row, and no later pivot row has a nonzero there: the combination
        // only multiplies that row's value by the row's own coefficient.
        const int acl = lane & (cw - 1), ag = lane / cw, aG = 64 / cw;  // cw: a power of two
        const int acg = wave * cw + acl;
        auto apply = [&](const int buf, const int cdone) __attribute__((always_inline)) {
            if (acg >= m)
                return;
            // (in order: the pivot of column c < cdone = rank is in row c, and the
            // panel's pivot rows follow, so nothing is looked up)
            if (acg < cdone && (inorder || colpiv[acg])) {
                const int r = inorder ? acg : pos[acg];
                if (ag == (r & (aG - 1))) {
                    V *x = At + r * ms + acg;
                    *x = ar.mul(inorder ? s_K0[buf] : C0[buf * kMaxN + r], *x);
                }
                return;
            }
            V pvr[P];
            if (inorder) {
#pragma unroll
                for (int q = 0; q < P; ++q)
                    pvr[q] = At[(cdone + q) * ms + acg];
            } else {
                int prq[P];
#pragma unroll
                for (int q = 0; q < P; ++q)
                    prq[q] = s_prs[buf][q];
#pragma unroll
                for (int q = 0; q < P; ++q)
                    pvr[q] = At[prq[q] * ms + acg];
            }
            // rows in pairs (32-bit words: two rows of 64-bit words exceed the
            // registers), their loads before the products
            constexpr int RP = sizeof(V) == 4 ? 2 : 1;
            const V K0 = kFast ? s_K0[buf] : (V)0;  // slot 0 of every row (in order)
            for (int r = ag; r < n; r += RP * aG) {
                V *x[RP];
                Row cv[RP];
                V c0[RP];
#pragma unroll
                for (int e = 0; e < RP; ++e) {
                    const int re = r + e * aG < n ? r + e * aG : r;  // (then the same value again)
                    x[e] = At + re * ms + acg;
                    cv[e] = Ck[buf * kMaxN + re];
                    c0[e] = inorder ? K0 : C0[buf * kMaxN + re];
                }
                typename Arith::Acc acc[RP];
#pragma unroll
                for (int e = 0; e < RP; ++e)
                    acc[e] = ar.prod(c0[e], *x[e]);
#pragma unroll
                for (int q = 0; q < P; ++q)
#pragma unroll
                    for (int e = 0; e < RP; ++e)
                        acc[e] = ar.fma(acc[e], cv[e].v[q], pvr[q]);
#pragma unroll
                for (int e = 0; e < RP; ++e)
                    *x[e] = ar.reduce(acc[e]);
            }
        };
        if (wave == 0)
            compose_panel(0, 0);
        lds_barrier();
        V dall = ar.one();  // in the last wave: product of the panels' own coefficients
        for (int k = 0;; ++k) {
            const int buf = k & 1;
            const int tk = s_tk[buf] & (kFastPanel - 1), nb = __popc(tk);
            inorder = inorder && (s_tk[buf] & kFastPanel);
            if (nb > 0)
                apply(buf, k * P);
            if (wave == kStepThreads / 64 - 1 && lane < P) {
                // pivot bookkeeping, off the composing wave's path: the pivots' rows
                // and cofactors, read after the elimination, and their columns, read
                // from the next panel's apply on
                // (q: the cofactor of this lane's pivot, dall the product past the panel;
                // by pivots: the products of the earlier ones, one after the other
                // here, where no pivot step waits for them)
                V q = dall;
                if (inorder) {
                    if (lane >= 2)
                        q = ar.mul(dall, s_pre[buf][0]);
                    dall = ar.mul(dall, s_K0[buf]);
                } else {
#pragma unroll
                    for (int c = 0; c < P; ++c)
                        if (tk >> c & 1) {
                            q = lane == c ? dall : q;
                            dall = ar.mul(dall, s_pre[buf][c]);
                        }
                }
                if (tk >> lane & 1) {
                    const int at = rank + __popc(tk & ((1 << lane) - 1));
                    const int pr = inorder ? rank + lane : s_prs[buf][lane];
                    prow[at] = pr;
                    cof[at] = q;
                    colpiv[k * P + lane] = 1;
                    pos[k * P + lane] = pr;
                }
            }
            rank += nb;
            const int c1 = (k + 1) * P;
            if (c1 >= m || rank >= n)
                break;
            if (wave == c1 / cw)
                compose_panel(c1, buf ^ 1);
            lds_barrier();
        }
        // With D the product of the panels' own coefficients and cof[k] the cofactor
        // of pivot k (D over the pivot), the kernel vectors are D times the
        // normalised ones, and no inverse is needed in the step.  Pivots are
        // nonzero, so is D.
        if (tid == kStepThreads - 64)
            s_D = dall;
        lds_barrier();
        const V D = s_D;
        // permutation list of left_nullspace_compact: pivot columns, then the
        // others; one wave counts the pivot columns before each column by ballots
        if (tid >= kStepThreads - 64) {
            const int l = tid - (kStepThreads - 64);
            int base = 0;
#pragma unroll
            for (int h = 0; h < kMaxM / 64; ++h) {
                const int i = l + 64 * h;
                const bool pc = i < m && colpiv[i];
                const unsigned long long b = __ballot(pc);
                const int before = base + __popcll(b & ((1ull << l) - 1));
                if (i < m) {
                    if (pc)
                        plist[before] = i;
                    else
                        plist[rank + i - before] = i;
                }
                base += __popcll(b);
            }
        }
        lds_barrier();
        const int nullity = m - rank;
        if (nullity == 0) {
            full = true;  // appbas <- x^(ordL - ord) appbas ends the leaf
            break;
        }
        if (rank > 0) {
            // kernel vectors: one per wave at a time, lane r (and r + 64) its entry r
            V *X = reinterpret_cast<V *>(a.X) + (size_t)s * m * m;
            constexpr int RH = kMaxN / 64;
            V cf[RH];
            int xrow[RH];
#pragma unroll
            for (int h = 0; h < RH; ++h) {
                const int r = lane + 64 * h;
                cf[h] = r < rank ? cof[r] : (V)0;
                xrow[h] = r < rank ? prow[r] * ms : 0;
            }
            // (up to 32 pivots: a vector per 2^lg lanes)
            const int lg = rank <= 32 ? 32 - __builtin_clz(2 * rank - 1) - 1 : 6;
            if (lg < 6) {
                const int r = tid & ((1 << lg) - 1);
                const V cr = r < rank ? cof[r] : (V)0;
                const int xr = r < rank ? prow[r] * ms : 0;
                for (int t = tid >> lg; t < nullity && r < rank; t += kStepThreads >> lg) {
                    const int col = plist[rank + t];
                    const V v = ar.sub(0, ar.mul(At[xr + col], cr));
                    At[xr + col] = v;
                    X[(size_t)t * m + r] = v;
                }
            }
            for (int t = wave; lg == 6 && t < nullity; t += kStepThreads / 64) {
                const int col = plist[rank + t];
#pragma unroll
                for (int h = 0; h < RH; ++h) {
                    const int r = lane + 64 * h;
                    if (r < rank) {
                        const V v = ar.sub(0, ar.mul(At[xrow[h] + col], cf[h]));
                        At[xrow[h] + col] = v;
                        X[(size_t)t * m + r] = v;
                    }
                }
            }
            if (tid < m) {
                const int row = perm[plist[tid]];
                a.piv[s * m + tid] = row;
                // rows updated by a kernel vector take the factor D
                if (tid >= rank)
                    scl[row] = ar.mul(scl[row], D);
            }
            if (tid == 0)
                a.scale[m + s] = D;
            // The window's remaining coefficients, orders s + 1 .. w - 1: two kernel
            // rows per wave at a time, a lane per (order, column).  The vectors and
            // the pivot rows' places sit in registers, lane r for pivot r, and are
            // read lane by lane into scalar registers: per pivot one LDS load for
            // two products.  With at most 32 (order, column) pairs the wave's halves,
            // quarters or eighths take a kernel row each and read their vectors'
            // entries from LDS.  The pivot rows' coefficients are read before they
            // move up by their delay; a kernel row's own are read and written by its
            // lanes alone.
            lds_barrier();
            if (s + 1 < w) {
                const int ncol = (w - 1 - s) * n;
                int rbase[RH];
#pragma unroll
                for (int h = 0; h < RH; ++h) {
                    const int r = lane + 64 * h;
                    const int pr = r < rank ? perm[plist[r]] : 0;
                    rbase[h] = r < rank ? (s + 1 - delay[pr]) * mn + pr * n : 0;
                }
                constexpr int NW = kStepThreads / 64;
                const int gl = ncol <= 8 ? 3 : ncol <= 16 ? 4 : 5;  // log2 of a group's lanes
                for (int t0 = wave << (6 - gl); ncol <= 32 && t0 < nullity; t0 += NW << (6 - gl)) {
                    const int tg = t0 + (lane >> gl), ql = lane & ((1 << gl) - 1);
                    const bool live = tg < nullity && ql < ncol;
                    const int col = plist[rank + (live ? tg : t0)], i = perm[col];
                    int d = 0, j = live ? ql : 0;
                    while (j >= n) {
                        j -= n;
                        ++d;
                    }
                    const int off = d * mn + j;
                    V *own = Rw + (s + 1 - delay[i]) * mn + i * n;
                    V sum = ar.mul(D, own[off]);
#pragma unroll
                    for (int h = 0; h < RH; ++h)
                        for (int r0 = 0; r0 < 64 && r0 + 64 * h < rank; r0 += 8) {
                            V y[8], x[8];
#pragma unroll
                            for (int u = 0; u < 8; ++u) {
                                y[u] = Rw[__builtin_amdgcn_readlane(rbase[h], r0 + u) + off];
                                x[u] = At[__builtin_amdgcn_readlane(xrow[h], r0 + u) + col];
                                x[u] = r0 + u + 64 * h < rank ? x[u] : (V)0;
                            }
                            typename Arith::Acc p1 = ar.prod(x[0], y[0]);
#pragma unroll
                            for (int u = 1; u < 8; ++u)
                                p1 = ar.fma(p1, x[u], y[u]);
                            sum = ar.add(sum, ar.reduce(p1));
                        }
                    if (live)
                        own[off] = sum;
                }
                for (int t = wave; ncol > 32 && t < nullity; t += 2 * NW) {
                    const int t2 = t + NW < nullity ? t + NW : t;
                    const int col1 = plist[rank + t], col2 = plist[rank + t2];
                    const int i1 = perm[col1], i2 = perm[col2];
                    V xa[RH], xb[RH];
#pragma unroll
                    for (int h = 0; h < RH; ++h) {
                        const int r = lane + 64 * h;
                        xa[h] = r < rank ? At[xrow[h] + col1] : (V)0;
                        xb[h] = r < rank ? At[xrow[h] + col2] : (V)0;
                    }
                    V *own1 = Rw + (s + 1 - delay[i1]) * mn + i1 * n, *own2 = Rw + (s + 1 - delay[i2]) * mn + i2 * n;
                    for (int q0 = 0; q0 < ncol; q0 += 64) {
                        const int q = q0 + lane < ncol ? q0 + lane : 0;
                        int d = 0, j = q;
                        while (j >= n) {
                            j -= n;
                            ++d;
                        }
                        const int off = d * mn + j;
                        V sum1 = ar.mul(D, own1[off]), sum2 = ar.mul(D, own2[off]);
#pragma unroll
                        for (int h = 0; h < RH; ++h)
                            for (int r0 = 0; r0 < 64 && r0 + 64 * h < rank; r0 += 8) {
                                // (pivots past the rank: zero vectors, place 0)
                                typename Arith::Acc p1, p2;
                                constexpr int G = sizeof(V) == 4 ? 8 : 4;  // loads together
#pragma unroll
                                for (int g0 = 0; g0 < 8; g0 += G) {
                                    V y[G];
#pragma unroll
                                    for (int u = 0; u < G; ++u)
                                        y[u] = Rw[__builtin_amdgcn_readlane(rbase[h], r0 + g0 + u) + off];
#pragma unroll
                                    for (int u = 0; u < G; ++u) {
                                        const V x1 = lane_value(xa[h], r0 + g0 + u);
                                        const V x2 = lane_value(xb[h], r0 + g0 + u);
                                        p1 = g0 + u == 0 ? ar.prod(x1, y[u]) : ar.fma(p1, x1, y[u]);
                                        p2 = g0 + u == 0 ? ar.prod(x2, y[u]) : ar.fma(p2, x2, y[u]);
                                    }
                                }
                                sum1 = ar.add(sum1, ar.reduce(p1));
                                sum2 = ar.add(sum2, ar.reduce(p2));
                            }
                        if (q0 + lane < ncol) {
                            own1[off] = sum1;
                            own2[off] = sum2;  // (t2 = t: the same value again)
                        }
                    }
                }
            }
            lds_barrier();
            if (tid < rank) {
                const int row = perm[plist[tid]];
                sh[row] += 1;
                delay[row] += 1;
            }
        }
        if (tid == 0)
            c[C_RANK + s] = rank;
        steps = s + 1;
        lds_barrier();
    }
    if (tid < m) {
        a.shift[tid] = sh[tid] + (full ? a.ordL - (ord0 + steps) : 0);
        a.scale[tid] = scl[tid];
    }
    if (tid == 0) {
        c[C_CUR] = cur;
        c[C_STEPS] = steps;
        // (single orders: nothing to apply to a zero residual)
        c[C_FLIP] = steps > 0 && (a.window > 1 || rank > 0) ? 1 : 0;
        if (full) {
            c[C_DONE] = 1;
            c[C_SHIFT] = a.ordL - (ord0 + steps);
        }
    }
}

// ---------------------------------------------------------------------------
// kernel 2: apply a window to appbas and to the residual series
// ---------------------------------------------------------------------------
// One workgroup takes kTile - w coefficients d0 .. of one column (of appbas,
// then of R) for all m rows, and the w before them, which rows multiplied by x
// bring in: row i of the tile Y holds coefficients d0 - w .., and its
// coefficient d is at Y[i][d - d0 + w - del[i]] after del[i] such
// multiplications.  The window's orders are applied one after the other in
// LDS, a thread per coefficient of the tile and kernel row, so that the tile is
// read and written once per window instead of once per order, and the launch,
// the control words' round trip and the tile's are paid once.  Order s leaves
// the first s coefficients of the halo undefined.
// The window's kernel vectors are brought to LDS at the start, beside the tile
// (rows padded with zeros to a multiple of kGroup), so that the orders wait for
// no global load.
// Latency bounds it: 14.0 us per window of 4 orders (64 x 32, 32-bit words; 4 x
// 7.4 to 9.5 with a launch per order), of which 2.3 are the loads, 1.5 each
// order and the rest the launch's start and end.
constexpr int kUpdateThreads = 512;
constexpr int kGroup = 16;  // pivots taken together
template <typename Arith>
__global__ void __launch_bounds__(kUpdateThreads)
mbasis_update_kernel(LeafArgs a, int ord0, int w, int wnext, int tilesB, int tilesR)
{
    extern __shared__ __attribute__((aligned(16))) unsigned char smem[];
    using V = typename Arith::V;
    static_assert(kMaxM <= kUpdateThreads, "one row-list entry per thread");
    const int m = a.m, n = a.n;
    const int tid = threadIdx.x, lane = tid & 63;
    V *Y = reinterpret_cast<V *>(smem);              // m x kTile
    int *pl = reinterpret_cast<int *>(Y + m * kTile);  // kWindow x m: row lists
    int *del = pl + kWindow * m;                     // m
    V *Xs = reinterpret_cast<V *>(smem + update_lds_bytes(m, sizeof(V)));  // vectors by order
    const int q = tid % kTile, tg = tid / kTile;
    constexpr int TG = kUpdateThreads / kTile;
    // 2 x 2 entries per thread of 2 TG rows x 2 kTile entries of every
    // order's vectors, all of them in flight at once; entry e of row t (in X's
    // bounds whatever the rank, which the first ones do not wait for)
    constexpr int XR = 2 * TG, XE = 2 * kTile;
    V xv[kWindow][2][2];
    auto fetch = [&](int tb, int eb) {
#pragma unroll
        for (int s = 0; s < kWindow; ++s)
#pragma unroll
            for (int u = 0; u < 4; ++u) {
                const int t = tb + tg + (u >> 1) * TG, e = eb + q + (u & 1) * kTile;
                const size_t x = (size_t)(s < w ? s : 0) * m * m + (t < m ? t : 0) * m + (e < m ? e : 0);
                xv[s][u >> 1][u & 1] = reinterpret_cast<const V *>(a.X)[x];
            }
    };
    fetch(0, 0);
    const int steps = a.ctl[C_STEPS], cur = a.ctl[C_CUR], len = a.ctl[C_LEN];
    int ranks[kWindow];
    V D[kWindow];
#pragma unroll
    for (int s = 0; s < kWindow; ++s) {
        ranks[s] = a.ctl[C_RANK + s];
        D[s] = (V)a.scale[m + s];
    }
    // row lists of the window (orders past `steps` are not used)
    if (tid < m) {
#pragma unroll
        for (int s = 0; s < kWindow; ++s)
            pl[s * m + tid] = a.piv[s * m + tid];
        del[tid] = 0;
    }
    if (steps == 0)
        return;
    const bool basis = (int)blockIdx.x < m * tilesB;
    const int b = basis ? blockIdx.x : blockIdx.x - m * tilesB;
    const int tiles = basis ? tilesB : tilesR;
    const int j = b / tiles, tile = b - j * tiles;
    const int cols = basis ? m : n;
    const int stride = basis ? a.cap : a.ordL;
    const int out = kTile - w;  // coefficients a tile writes
    const int d0 = (basis ? 0 : ord0 + w) + tile * out;
    // coefficients read, and written
    const int lin = basis ? len : a.ordL;
    const int lout = basis ? (len + steps < a.cap ? len + steps : a.cap) : a.ordL;
    if (d0 >= lout)
        return;
    const uint64_t *src = basis ? a.app[cur] : a.R[cur];
    uint64_t *dst = basis ? a.app[cur ^ 1] : a.R[cur ^ 1];
    const Arith ar(a.mc);
    {
        // (four rows' loads in flight, of an entry that exists in any case)
        const int d = d0 - w + q;
        const bool in = d >= 0 && d < lin;
        const uint64_t *from = src + (size_t)j * stride + (in ? d : 0);
        const size_t rows = (size_t)cols * stride;
        for (int i0 = tg; i0 < m; i0 += 4 * TG) {
            V y[4];
#pragma unroll
            for (int u = 0; u < 4; ++u)
                y[u] = Arith::load(from + (i0 + u * TG < m ? i0 + u * TG : 0) * rows);
#pragma unroll
            for (int u = 0; u < 4; ++u)
                if (i0 + u * TG < m)
                    Y[(i0 + u * TG) * kTile + q] = in ? y[u] : (V)0;
        }
    }
    {
        int most = 0;  // entries of the longest vectors
#pragma unroll
        for (int s = 0; s < kWindow; ++s) {
            ranks[s] = s < steps ? ranks[s] : 0;
            most = ranks[s] > most ? ranks[s] : most;
        }
        for (int tb = 0; tb < m; tb += XR)
            for (int eb = 0; eb < most; eb += XE) {
                if (tb + eb > 0)
                    fetch(tb, eb);
                V *xs = Xs;
#pragma unroll
                for (int s = 0; s < kWindow; ++s) {
                    const int rank = ranks[s], nullity = m - rank, r16 = pad16(rank);
                    if (rank == 0)
                        continue;
#pragma unroll
                    for (int u = 0; u < 4; ++u) {
                        const int t = tb + tg + (u >> 1) * TG, e = eb + q + (u & 1) * kTile;
                        if (t < nullity && e < r16)
                            xs[t * r16 + e] = e < rank ? xv[s][u >> 1][u & 1] : (V)0;
                    }
                    xs += nullity * r16;
                }
            }
    }
    __syncthreads();
    const int tw = __builtin_amdgcn_readfirstlane(tg);  // the wave's first
    struct alignas(16) Group {
        V v[kGroup];
    };
    constexpr int RH = kMaxN / 64;
    int top = 0;  // length that a row multiplied by x reaches
    const V *xstage = Xs;
    for (int s = 0; s < steps; ++s) {
        int rank = 0;
        V Ds = 0;
#pragma unroll
        for (int u = 0; u < kWindow; ++u) {
            rank = u == s ? ranks[u] : rank;
            Ds = u == s ? D[u] : Ds;
        }
        if (rank == 0)
            continue;  // zero residual: nothing to do at this order
        const int *ps = pl + s * m;
        const int nullity = m - rank;
        const int xstride = pad16(rank);
        // places of the pivot rows' coefficient q = 0, lane r for pivot r (past
        // the rank: the first row, with zero entries in the vectors)
        int ybase[RH];
#pragma unroll
        for (int h = 0; h < RH; ++h) {
            const int i = ps[lane + 64 * h < rank ? lane + 64 * h : 0];
            ybase[h] = i * kTile - del[i];
        }
        // (a wave takes every round as a whole, its lanes read each other's ybase)
        for (int t0 = tw; t0 < nullity; t0 += TG) {
            const int t = t0 + tg - tw < nullity ? t0 + tg - tw : t0;
            // (q below s: coefficients already undefined, read as q = s)
            const int qq = q < s ? s : q, i = ps[rank + t];
            V *own = Y + i * kTile + qq - del[i];
            const V *x = xstage + (size_t)t * xstride;
            V sum = ar.mul(Ds, *own);
#pragma unroll
            for (int h = 0; h < RH; ++h)
                for (int r0 = 0; r0 < 64 && r0 + 64 * h < rank; r0 += kGroup) {
                    V v[kGroup], c[kGroup];
                    *reinterpret_cast<Group *>(c) = *reinterpret_cast<const Group *>(x + r0 + 64 * h);
#pragma unroll
                    for (int u = 0; u < kGroup; ++u)
                        v[u] = Y[__builtin_amdgcn_readlane(ybase[h], r0 + u) + qq];
                    // two chains of eight products, the most one reduction takes
                    typename Arith::Acc p1 = ar.prod(c[0], v[0]), p2 = ar.prod(c[8], v[8]);
#pragma unroll
                    for (int u = 1; u < 8; ++u) {
                        p1 = ar.fma(p1, c[u], v[u]);
                        p2 = ar.fma(p2, c[8 + u], v[8 + u]);
                    }
                    sum = ar.add(sum, ar.add(ar.reduce(p1), ar.reduce(p2)));
                }
            if (q >= s)
                *own = sum;  // (t = t0 twice: the same value again)
        }
        xstage += nullity * xstride;
        __syncthreads();
        if (tid < rank)
            del[ps[tid]] += 1;
        __syncthreads();
        // length: a row multiplied by x with a coefficient past the old one
        if (basis && d0 + out > len && q > s) {
            const int d = d0 - w + q;
            if (d >= len)
                for (int r = tg; r < rank; r += TG) {
                    const int i = ps[r];
                    if (Y[i * kTile + q - del[i]] != 0)
                        top = d + 1;
                }
        }
    }
    __syncthreads();
    if (basis && d0 + out > len) {
        for (int d = 32; d > 0; d >>= 1)
            top = max(top, __shfl_xor(top, d));
        if (lane == 0)
            del[m + tid / 64] = top;
        __syncthreads();
        if (tid == 0) {
            for (int k = 0; k < kUpdateThreads / 64; ++k)
                top = max(top, del[m + k]);
            if (top > len)  // (at most two tiles of a column reach past len)
                a.lens[2 * j + (tile & 1)] = top;
        }
    }
    for (int idx = tid; idx < m * kTile; idx += kUpdateThreads) {
        const int i = idx / kTile, qq = idx % kTile, d = d0 - w + qq;
        if (qq < w || d >= lout)
            continue;
        const uint64_t v = Y[i * kTile + qq - del[i]];
        const size_t e = (size_t)i * cols + j;
        dst[e * stride + d] = v;
        if (!basis && d < ord0 + w + wnext)
            a.Rn[(size_t)(d - ord0 - w) * m * n + e] = v;  // the coming window
    }
}

// base + sum_r X[t][r] * src[row piv[r], column j, coefficient d].  All loads
// of a group of terms (32 words below 2^30, or 16 64-bit words: one L2 round
// trip) are issued before its products, with no branch between them: terms
// past the rank read row piv[r] of the LDS row list (padded with row 0 up to
// kMaxM; rank <= kMaxN) and X words past the row (X carries kXPad words of
// padding), and their X coefficient is zeroed by a select after the load.
template <typename Arith>
__device__ __forceinline__ typename Arith::V row_combo(const Arith &ar, const uint64_t *src,
                                                       const typename Arith::V *xr, const int *piv,
                                                       int rank, int stride, int cols, int j, int d,
                                                       typename Arith::V base)
{
    using V = typename Arith::V;
    const uint64_t *sj = src + (size_t)j * stride + d;
    const size_t rstride = (size_t)cols * stride;
    constexpr int G = sizeof(V) == 4 ? 32 : 16;
    V acc = base;
    for (int r = 0; r < rank; r += G) {
        V sv[G], xv[G];
#pragma unroll
        for (int u = 0; u < G; ++u) {
            sv[u] = Arith::load(sj + (size_t)piv[r + u] * rstride);
            const V x = xr[r + u];
            xv[u] = r + u < rank ? x : (V)0;
        }
#pragma unroll
        for (int h = 0; h < G; h += 8) {  // eight products, the most one reduction takes
            typename Arith::Acc part = ar.prod(xv[h], sv[h]);
#pragma unroll
            for (int u = 1; u < 8; ++u)
                part = ar.fma(part, xv[h + u], sv[h + u]);
            acc = ar.add(acc, ar.reduce(part));
        }
    }
    return acc;
}

// The same for single orders: a thread per coefficient of appbas and of the
// residual's later coefficients, read from and written to memory.  There is
// nothing to keep in LDS between orders, no halo and no place of a tile past the
// basis's length, and the kernel rows spread over the chip, where a tile takes
// all of a column's.  Step plus update per order, single orders / windows of 2 as
// the tiles take them: 78 / 127 us (192 x 24, 64-bit words), 30 / 81 (256 x 1, the
// same), 90 / 125 (100 x 25, p > 2^62).
template <typename Arith>
__global__ void __launch_bounds__(256) mbasis_update1_kernel(LeafArgs a, int ord)
{
    // The control words, the order's row list and its factor D are all
    // requested at entry, before any branch on them.
    using V = typename Arith::V;
    static_assert(kMaxM == 256, "one row-list entry per thread of the 256-thread workgroup");
    const int m = a.m, n = a.n, cap = a.cap, tx = threadIdx.x;
    const int steps = a.ctl[C_STEPS], cur = a.ctl[C_CUR], L = a.ctl[C_LEN], rank = a.ctl[C_RANK];
    const V D = (V)a.scale[m];
    const int piv_t = tx < m ? a.piv[tx] : 0;  // groups read up to kMaxM entries
    if (steps == 0)
        return;
    const unsigned tstride = gridDim.x * blockDim.x;
    const unsigned t0 = blockIdx.x * blockDim.x + tx;
    const uint64_t *rs = a.R[cur];
    if (rank == 0) {
        // residual unchanged: the coming order's coefficient is ord + 1
        if (ord + 1 < a.ordL)
            for (unsigned e = t0; e < (unsigned)(m * n); e += tstride)
                a.Rn[e] = rs[(size_t)e * a.ordL + ord + 1];
        return;
    }
    __shared__ int piv[kMaxM], role[kMaxM];  // role: t of a kernel row, -1 of a pivot row
    piv[tx] = piv_t;
    if (tx < m)
        role[piv_t] = tx < rank ? -1 : tx - rank;
    __syncthreads();
    const Arith ar(a.mc);
    const V *X = reinterpret_cast<const V *>(a.X);
    const uint64_t *src = a.app[cur];
    uint64_t *dst = a.app[cur ^ 1], *rd = a.R[cur ^ 1];
    const unsigned L1 = (unsigned)(L + 1 <= cap ? L + 1 : cap);
    const unsigned items = (unsigned)(m * m) * L1;
    const int spn = a.ordL - ord - 1;
    const unsigned span = spn > 0 ? (unsigned)spn : 0u;
    const unsigned ritems = (unsigned)(m * n) * span;
    // one index space, basis items then residual items: with the grid sized
    // for both, a thread has one item
    for (unsigned idx = t0; idx < items + ritems; idx += tstride) {
        if (idx < items) {
            const unsigned e = idx / L1;
            const int d = (int)(idx - e * L1);
            const int i = (int)(e / (unsigned)m), j = (int)(e - (unsigned)i * m);
            const int t = role[i];
            const uint64_t *x = src + (size_t)e * cap + d;
            uint64_t v;
            if (t >= 0) {
                v = d < L ? row_combo<Arith>(ar, src, X + (size_t)t * m, piv, rank, cap, m, j, d,
                                             ar.mul(D, Arith::load(x)))
                          : 0;
            } else {
                v = d >= 1 ? x[-1] : 0;
                if (d == L && v != 0)
                    a.lens[0] = L + 1;
            }
            dst[(size_t)e * cap + d] = v;
        } else {
            const unsigned k = idx - items;
            const unsigned e = k / span;
            const int d = ord + 1 + (int)(k - e * span);
            const int i = (int)(e / (unsigned)n), j = (int)(e - (unsigned)i * n);
            const int t = role[i];
            const uint64_t *x = rs + (size_t)e * a.ordL + d;
            const uint64_t v = t >= 0 ? row_combo<Arith>(ar, rs, X + (size_t)t * m, piv, rank, a.ordL, n, j, d,
                                                         ar.mul(D, Arith::load(x)))
                                      : x[-1];
            rd[(size_t)e * a.ordL + d] = v;
            if (d == ord + 1)
                a.Rn[e] = v;  // the coming order's coefficient
        }
    }
}

// appbas <- x^s appbas (entries of capacity cap, length len before), into dst
__global__ void leaf_shift_kernel(uint64_t *__restrict__ dst, const uint64_t *__restrict__ src, int64_t cap,
                                  int64_t entries, int64_t len, int64_t s)
{
    const int64_t items = entries * (len + s);
    for (int64_t idx = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; idx < items;
         idx += (int64_t)gridDim.x * blockDim.x) {
        const int64_t e = idx / (len + s), d = idx - e * (len + s);
        dst[e * cap + d] = d >= s ? src[e * cap + d - s] : 0;
    }
}

// scale[i] <- 1 / scale[i] as a plain residue (the scales are Montgomery
// residues, nonzero as products of pivots)
template <typename Arith>
__global__ void __launch_bounds__(kMaxM) leaf_scale_inv_kernel(LeafArgs a)
{
    const Arith ar(a.mc);
    const int i = threadIdx.x;
    if (i < a.m)
        a.scale[i] = ar.from(ar.inv((typename Arith::V)a.scale[i]));
}

// coefficients [0, len) of the m x m basis (entries of capacity cap) times
// their row's inverse scale
__global__ void __launch_bounds__(256) leaf_rescale_kernel(uint64_t *__restrict__ P, int64_t cap, int m,
                                                           int64_t len, const uint64_t *__restrict__ iscale,
                                                           ModConst mc)
{
    const int64_t items = (int64_t)m * m * len;
    for (int64_t idx = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; idx < items;
         idx += (int64_t)gridDim.x * blockDim.x) {
        const int64_t e = idx / len, d = idx - e * len;
        const int row = (int)(e / m);
        P[e * cap + d] = mulmod_g(P[e * cap + d], iscale[row], mc);
    }
}

// appbas <- identity (capacity cap), R <- F truncated to ordL, control reset
__global__ void leaf_init_kernel(LeafArgs a, const uint64_t *__restrict__ F, int64_t strideF,
                                 int64_t lenF, int w)
{
    const int m = a.m, n = a.n, cap = a.cap;
    const int64_t tstride = (int64_t)gridDim.x * blockDim.x;
    const int64_t t0 = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    const int64_t itemsA = (int64_t)m * m * cap;
    for (int64_t idx = t0; idx < itemsA; idx += tstride) {
        const int64_t e = idx / cap;
        const int d = (int)(idx - e * cap);
        const int i = (int)(e / m), j = (int)(e - (int64_t)i * m);
        a.app[0][idx] = (d == 0 && i == j) ? 1 : 0;
    }
    const int64_t itemsR = (int64_t)m * n * a.ordL;
    for (int64_t idx = t0; idx < itemsR; idx += tstride) {
        const int64_t e = idx / a.ordL;
        const int d = (int)(idx - e * a.ordL);
        const uint64_t v = d < lenF ? F[e * strideF + d] : 0;
        a.R[0][idx] = v;
        if (d < w)
            a.Rn[(size_t)d * m * n + e] = v;
    }
    for (int64_t idx = t0; idx < C_WORDS + 2 * m; idx += tstride)  // ctl, lens
        a.ctl[idx] = idx == C_LEN ? 1 : 0;
}

// copies an m x m x L block between two capacities (entry-major)
__global__ void copy_poly_kernel(uint64_t *__restrict__ dst, int64_t dcap,
                                 const uint64_t *__restrict__ src, int64_t scap, int64_t entries,
                                 int64_t len)
{
    const int64_t items = entries * len;
    for (int64_t idx = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; idx < items;
         idx += (int64_t)gridDim.x * blockDim.x) {
        const int64_t e = idx / len, d = idx - e * len;
        dst[e * dcap + d] = src[e * scap + d];
    }
}

template <typename T>
struct Tag {
    using type = T;
};

unsigned grid_for(int64_t items)
{
    int64_t b = (items + 255) / 256;
    if (b < 1)
        b = 1;
    if (b > 4096)
        b = 4096;
    return (unsigned)b;
}

// Bump allocator over one device buffer; results are moved down to the
// caller's mark so that temporaries of a recursion level are reclaimed.
struct Arena {
    char *base = nullptr;
    size_t size = 0, top = 0;
    uint64_t *alloc(size_t words)
    {
        size_t bytes = (words * 8 + 255) & ~(size_t)255;
        if (top + bytes > size)
            return nullptr;
        uint64_t *p = reinterpret_cast<uint64_t *>(base + top);
        top += bytes;
        return p;
    }
};

struct Poly {
    uint64_t *d;
    int64_t cap, len;
};

constexpr int kPmbasisThres = 32;  // PMBASIS_THRES, nmod_poly_mat_approximant.h:101

// M-Basis of F (m x n, entries at F + e*strideF, length lenF) at order ordL;
// the result is placed at the arena mark.
pmlg_status leaf(pmlg_ctx ctx, Arena &ar, const uint64_t *F, int64_t strideF, int64_t lenF,
                 int m, int n, int ordL, int64_t *dShift, Poly *out, hipStream_t s)
{
    const size_t mark = ar.top;
    const int cap = ordL + 1;
    LeafArgs a{};
    a.m = m;
    a.n = n;
    a.ordL = ordL;
    a.cap = cap;
    a.app[0] = ar.alloc((size_t)m * m * cap);
    a.app[1] = ar.alloc((size_t)m * m * cap);
    a.R[0] = ar.alloc((size_t)m * n * (ordL > 0 ? ordL : 1));
    a.R[1] = ar.alloc((size_t)m * n * (ordL > 0 ? ordL : 1));
    // p = 2 has no Montgomery form (p must be odd): plain residues as for p >= 2^62
    const bool big = ctx->p >= ((uint64_t)1 << 62) || ctx->p == 2;
    const bool small = !big && ctx->p < ((uint64_t)1 << 30);
    const size_t wbytes = small ? 4 : 8;
    if (step_lds_bytes(m, n, wbytes) > kStepLdsMax)
        return fail(PMLG_ERR_UNSUPPORTED, "M-Basis: an m x n residual of this size does not fit "
                                          "the step kernel's LDS");
    const int W = mbasis_window(small ? BASIS_W32 : big ? BASIS_ANY : BASIS_W64, m, n, ordL,
                                window_orders(m, n, wbytes));
    a.window = W;
    a.Rn = ar.alloc((size_t)m * n * W);
    a.scale = ar.alloc((size_t)m + kWindow);
    a.X = ar.alloc((size_t)m * m * W + kXPad);
    uint64_t *ints = ar.alloc(((size_t)m * (kWindow + 2) + C_WORDS) / 2 + 8);
    if (!a.app[0] || !a.app[1] || !a.R[0] || !a.R[1] || !a.Rn || !a.scale || !a.X || !ints)
        return fail(PMLG_ERR_ALLOC, "pmbasis: device arena exhausted");
    a.ctl = reinterpret_cast<int *>(ints);
    a.lens = a.ctl + C_WORDS;
    a.piv = a.lens + 2 * m;
    a.shift = dShift;
    a.mc = ctx->mc;
    const int64_t lt = lenF < ordL ? lenF : ordL;
    hipLaunchKernelGGL(leaf_init_kernel, dim3(grid_for((int64_t)m * m * cap + (int64_t)m * n * ordL)),
                       dim3(256), 0, s, a, F, strideF, lt, W);
    HIP_TRY(hipGetLastError(), "leaf_init_kernel");
    {
        const void *kernels[] = {(const void *)mbasis_step_kernel<Mont64Arith, 1>,
                                 (const void *)mbasis_step_kernel<Mont64Arith, 2>,
                                 (const void *)mbasis_step_kernel<Mont32Arith, 1>,
                                 (const void *)mbasis_step_kernel<Mont32Arith, 2>,
                                 (const void *)mbasis_step_kernel<BigArith, 1>,
                                 (const void *)mbasis_step_kernel<BigArith, 2>,
                                 (const void *)mbasis_update_kernel<Mont64Arith>,
                                 (const void *)mbasis_update_kernel<Mont32Arith>,
                                 (const void *)mbasis_update_kernel<BigArith>};
        constexpr int nk = sizeof(kernels) / sizeof(kernels[0]);
        static std::atomic<uint64_t> raised[nk];
        for (int i = 0; i < nk; ++i)
            HIP_TRY(raise_lds_limit(kernels[i], kLds, raised[i]), "hipFuncSetAttribute(mbasis kernels)");
    }
    // rows of the transposed residual per lane of the composing wave
    const bool one_row = n <= 64;
    const size_t ulds = update_lds_bytes(m, wbytes) + staged_words(m, n) * W * wbytes;
    const unsigned grid1 = grid_for((int64_t)m * m * cap + (int64_t)m * n * ordL);
    for (int ord = 0; ord < ordL; ord += W) {
        const int w = std::min(W, ordL - ord), wnext = std::min(W, ordL - ord - w);
        const size_t lds = window_lds_bytes(m, n, w, wbytes);
        // tiles of appbas (length at most ord + w + 1 after the window) and of
        // the residual's later coefficients
        const int out = kTile - w;
        const int tilesB = (std::min(cap, ord + w + 1) + out - 1) / out;
        const int tilesR = (std::max(ordL - ord - w, 0) + out - 1) / out;
        const dim3 ugrid((unsigned)(m * tilesB + n * tilesR));
        auto launch = [&](auto arith) {
            using A = decltype(arith);
            hipLaunchKernelGGL((one_row ? mbasis_step_kernel<typename A::type, 1>
                                        : mbasis_step_kernel<typename A::type, 2>),
                               dim3(1), dim3(kStepThreads), lds, s, a, ord, w);
            if (W == 1)
                hipLaunchKernelGGL(mbasis_update1_kernel<typename A::type>, dim3(grid1), dim3(256), 0, s, a, ord);
            else
                hipLaunchKernelGGL(mbasis_update_kernel<typename A::type>, ugrid, dim3(kUpdateThreads), ulds, s,
                                   a, ord, w, wnext, tilesB, tilesR);
        };
        if (small)
            launch(Tag<Mont32Arith>{});
        else if (big)
            launch(Tag<BigArith>{});
        else
            launch(Tag<Mont64Arith>{});
    }
    HIP_TRY(hipGetLastError(), "mbasis kernels");
    int ctl[C_WORDS + 2 * kMaxM];  // the lengths as well
    HIP_TRY(hipMemcpyAsync(ctl, a.ctl, (C_WORDS + 2 * m) * sizeof(int), hipMemcpyDeviceToHost, s), "D2H(ctl)");
    HIP_TRY(hipStreamSynchronize(s), "leaf sync");
    int res = ctl[C_CUR] ^ ctl[C_FLIP];
    int L = std::max(1, *std::max_element(ctl + C_WORDS, ctl + C_WORDS + 2 * m));
    if (ctl[C_DONE]) {
        // full-rank residual met: the basis times the rest of the power of x
        const int sft = ctl[C_SHIFT];
        hipLaunchKernelGGL(leaf_shift_kernel, dim3(grid_for((int64_t)m * m * (L + sft))), dim3(256), 0, s,
                           a.app[res ^ 1], a.app[res], (int64_t)cap, (int64_t)m * m, (int64_t)L, (int64_t)sft);
        HIP_TRY(hipGetLastError(), "leaf_shift_kernel");
        res ^= 1;
        L += sft;
    }
    if (ordL > 0) {
        // divide the row scales out of the basis
        if (small)
            hipLaunchKernelGGL(leaf_scale_inv_kernel<Mont32Arith>, dim3(1), dim3(kMaxM), 0, s, a);
        else if (big)
            hipLaunchKernelGGL(leaf_scale_inv_kernel<BigArith>, dim3(1), dim3(kMaxM), 0, s, a);
        else
            hipLaunchKernelGGL(leaf_scale_inv_kernel<Mont64Arith>, dim3(1), dim3(kMaxM), 0, s, a);
        hipLaunchKernelGGL(leaf_rescale_kernel, dim3(grid_for((int64_t)m * m * L)), dim3(256), 0, s,
                           a.app[res], (int64_t)cap, m, (int64_t)L, a.scale, ctx->mc);
        HIP_TRY(hipGetLastError(), "leaf_rescale_kernel");
    }
    // result to the mark (app[0] sits there; move app[1] down if needed)
    out->d = a.app[0];
    out->cap = cap;
    out->len = L;
    if (res == 1) {
        hipLaunchKernelGGL(copy_poly_kernel, dim3(grid_for((int64_t)m * m * L)), dim3(256), 0, s,
                           a.app[0], (int64_t)cap, a.app[1], (int64_t)cap, (int64_t)m * m, (int64_t)L);
        HIP_TRY(hipGetLastError(), "copy_poly_kernel");
    }
    ar.top = mark + (((size_t)m * m * cap * 8 + 255) & ~(size_t)255);
    return PMLG_OK;
}

// PM-Basis recursion (approximant_basis.c:33-69); result at the arena mark.
pmlg_status pmb_rec(pmlg_ctx ctx, Arena &ar, const uint64_t *F, int64_t strideF, int64_t lenF,
                    int m, int n, int64_t order, int64_t *dShift, int method, int thres, Poly *out,
                    hipStream_t s)
{
    const int64_t lt = lenF < order ? lenF : order;
    if (order <= thres)
        return leaf(ctx, ar, F, strideF, lt, m, n, (int)order, dShift, out, s);
    const size_t mark = ar.top;
    const int64_t order1 = order >> 1, order2 = order - order1;
    Poly P1;
    pmlg_status st = pmb_rec(ctx, ar, F, strideF, lt, m, n, order1, dShift, method, thres, &P1, s);
    if (st != PMLG_OK)
        return st;
    // residual = (P1 * F mod x^order) div x^order1
    uint64_t *Rz = ar.alloc((size_t)m * n * order2);
    if (!Rz)
        return fail(PMLG_ERR_ALLOC, "pmbasis: device arena exhausted");
    st = mulmid_dev_strided(ctx, Rz, order2, P1.d, P1.cap, F, strideF, m, m, n, P1.len, lt, order1,
                            order, method, s);
    if (st != PMLG_OK)
        return st;
    Poly P2;
    st = pmb_rec(ctx, ar, Rz, order2, order2, m, n, order2, dShift, method, thres, &P2, s);
    if (st != PMLG_OK)
        return st;
    // appbas = P2 * P1
    const int64_t L = P1.len + P2.len - 1;
    uint64_t *P = ar.alloc((size_t)m * m * L);
    if (!P)
        return fail(PMLG_ERR_ALLOC, "pmbasis: device arena exhausted");
    st = mulmid_dev_strided(ctx, P, L, P2.d, P2.cap, P1.d, P1.cap, m, m, m, P2.len, P1.len, 0, L,
                            method, s);
    if (st != PMLG_OK)
        return st;
    // move the result down to the mark (P1, Rz and P2 are dead)
    uint64_t *dst = reinterpret_cast<uint64_t *>(ar.base + mark);
    hipLaunchKernelGGL(copy_poly_kernel, dim3(grid_for((int64_t)m * m * L)), dim3(256), 0, s, dst, L,
                       P, L, (int64_t)m * m, L);
    HIP_TRY(hipGetLastError(), "copy_poly_kernel");
    ar.top = mark + (((size_t)m * m * L * 8 + 255) & ~(size_t)255);
    out->d = dst;
    out->cap = L;
    out->len = L;
    return PMLG_OK;
}

size_t arena_bytes(int64_t m, int64_t n, int64_t order, int64_t ordleaf)
{
    // generous bound: a few copies of every level's operands
    const double lvl = (double)m * m * (order + 2) * 4 + (double)m * n * (order + 1) * 2;
    const double leafb =
        (double)m * m * (ordleaf + 2) * 2 + (double)m * n * (ordleaf + 2) * 2 +
        (double)kWindow * (m * m + m * n + m) + 256;
    return (size_t)((2.5 * lvl + leafb + 4096.0) * 8.0);
}

// M-Basis / PM-Basis crossover.  The basis does not depend on it: the second
// half of the recursion repeats, on the residual of the first half's basis,
// the steps that M-Basis would take from that basis on (each step depends only
// on the current residual coefficient and shifts, and the basis updates are
// row operations that commute with the product by the first half's basis), so
// the leaf order is a pure speed choice.  Threshold t against 2t differs only
// at the nodes of order 2t, split into two leaves of order t plus a middle
// product and a product, or solved as one leaf: both are timed on seeded
// synthetic input of the caller's shape, first for t = 32 (the reference's
// threshold), then for t = 16 if the split won there, else for t = 64, and
// then for t = 128 if the leaf of 128 won too.  Measured once per context and
// (m, n, method), for orders of at least kTuneMinOrder (below it the
// reference's threshold is used as it is).
constexpr int kMaxLeafOrder = 256;
constexpr int64_t kTuneMinOrder = 512;

int64_t tune_leaf_bytes(int64_t m, int64_t n)
{
    return (int64_t)arena_bytes(m, n, kMaxLeafOrder, kMaxLeafOrder) + (m * n * kMaxLeafOrder + m) * 8 + 4096;
}

pmlg_status tune_leaf_order(pmlg_ctx ctx, int m, int n, int method, hipStream_t s, int *out)
{
    const uint64_t key = ((uint64_t)m << 16) | ((uint64_t)n << 8) | (uint64_t)(method & 0xff);
    auto it = ctx->leaf_orders.find(key);
    if (it != ctx->leaf_orders.end()) {
        *out = it->second;
        return PMLG_OK;
    }
    HIP_TRY(ctx->arena.ensure((size_t)tune_leaf_bytes(m, n)), "hipMalloc(arena)");
    Arena ar;
    ar.base = static_cast<char *>(ctx->arena.ptr);
    ar.size = ctx->arena.bytes;
    const int64_t len = kMaxLeafOrder;
    uint64_t *dF = ar.alloc((size_t)(m * n * len));
    int64_t *dShift = reinterpret_cast<int64_t *>(ar.alloc((size_t)m));
    if (!dF || !dShift)
        return fail(PMLG_ERR_ALLOC, "pmbasis: device arena exhausted");
    std::vector<uint64_t> F((size_t)(m * n * len));
    uint64_t x = 0x9e3779b97f4a7c15ull ^ key;
    for (uint64_t &v : F) {
        x ^= x << 13;
        x ^= x >> 7;
        x ^= x << 17;
        v = x % ctx->p;
    }
    HIP_TRY(hipMemcpyAsync(dF, F.data(), F.size() * 8, hipMemcpyHostToDevice, s), "H2D(tuning input)");
    const std::vector<int64_t> zero((size_t)m, 0);
    const size_t mark = ar.top;
    // best of three runs (the first also loads the transform tables)
    auto run = [&](int64_t order, int thres, double *sec) -> pmlg_status {
        *sec = 1e30;
        for (int r = 0; r < 3; ++r) {
            HIP_TRY(hipMemcpyAsync(dShift, zero.data(), (size_t)m * 8, hipMemcpyHostToDevice, s),
                    "H2D(shift)");
            HIP_TRY(hipStreamSynchronize(s), "sync");
            const auto t0 = std::chrono::steady_clock::now();
            Poly P;
            pmlg_status st = pmb_rec(ctx, ar, dF, len, len, m, n, order, dShift, method, thres, &P, s);
            if (st != PMLG_OK)
                return st;
            HIP_TRY(hipStreamSynchronize(s), "sync");
            *sec = std::min(*sec, std::chrono::duration<double>(std::chrono::steady_clock::now() - t0).count());
            ar.top = mark;
        }
        return PMLG_OK;
    };
    // true when two leaves of order t (and the products) beat one of order 2t
    auto split_wins = [&](int t, bool *wins) -> pmlg_status {
        double leaf_s = 0, split_s = 0;
        pmlg_status st = run(2 * t, 2 * t, &leaf_s);
        if (st == PMLG_OK)
            st = run(2 * t, t, &split_s);
        *wins = split_s < leaf_s;
        return st;
    };
    bool w32 = false, w = false;
    pmlg_status st = split_wins(32, &w32);
    if (st == PMLG_OK)
        st = split_wins(w32 ? 16 : 64, &w);
    if (st != PMLG_OK)
        return st;
    int best = w32 ? (w ? 16 : 32) : (w ? 64 : 0);
    if (best == 0) {
        st = split_wins(128, &w);
        if (st != PMLG_OK)
            return st;
        best = w ? 128 : 256;
    }
    ctx->leaf_orders[key] = best;
    *out = best;
    return PMLG_OK;
}

}  // namespace

pmlg_status basis_common(pmlg_ctx ctx, uint64_t *dP, int64_t capP, int64_t *lenP,
                         int64_t *shift, const uint64_t *dF, int64_t strideF, int64_t m, int64_t n,
                         int64_t lenF, int64_t order, int method, bool iterative, hipStream_t s,
                         uint64_t *hP)
{
    if (m <= 0 || n <= 0 || m > kMaxM || n > kMaxN || order < 0 || lenF < 0)
        return fail(PMLG_ERR_ARG, "approximant basis: 1 <= m <= 256, 1 <= n <= 128, order >= 0");
    if (step_lds_bytes((int)m, (int)n, ctx->p < ((uint64_t)1 << 30) && ctx->p != 2 ? 4 : 8) >
        kStepLdsMax)
        return fail(PMLG_ERR_UNSUPPORTED,
                    "approximant basis: the m x n residual exceeds one workgroup's LDS (n (m | 1) "
                    "words plus the step's buffers: e.g. m = 256 allows n <= 62 for p >= 2^30)");
    if (!ctx->is_prime && ctx->p != 2)
        return fail(PMLG_ERR_UNSUPPORTED, "approximant bases need a prime modulus");
    if (capP < order + 1)
        return fail(PMLG_ERR_ARG, "approximant basis: output capacity must be at least order + 1");
    int thres = ctx->leaf_order > 0 ? ctx->leaf_order : kPmbasisThres;
    if (!iterative && ctx->leaf_order == 0 && order >= kTuneMinOrder) {
        pmlg_status st = tune_leaf_order(ctx, (int)m, (int)n, method, s, &thres);
        if (st != PMLG_OK)
            return st;
    }
    // the M-Basis kernels index one leaf's items in 32 bits
    const int64_t ordleaf = iterative ? order : std::min<int64_t>(order, thres);
    if (m * m * (ordleaf + 1) + m * n * ordleaf >= ((int64_t)1 << 31))
        return fail(PMLG_ERR_UNSUPPORTED, "M-Basis: m^2 (order + 1) + m n order must stay below 2^31 "
                                          "(use PM-Basis for this order)");
    // device arena
    size_t need = arena_bytes(m, n, order, ordleaf) +
                  (size_t)(m * m * (ordleaf + 2) * 2 + m * n * (ordleaf + 1) * 2) * 8;
    HIP_TRY(ctx->arena.ensure(need), "hipMalloc(arena)");
    Arena ar;
    ar.base = static_cast<char *>(ctx->arena.ptr);
    ar.size = ctx->arena.bytes;
    int64_t *dShift = reinterpret_cast<int64_t *>(ar.alloc((size_t)m));
    HIP_TRY(hipMemcpyAsync(dShift, shift, (size_t)m * 8, hipMemcpyHostToDevice, s), "H2D(shift)");
    Poly P;
    pmlg_status st;
    if (iterative)
        st = leaf(ctx, ar, dF, strideF, std::min(lenF, order), (int)m, (int)n, (int)order, dShift, &P,
                  s);
    else
        st = pmb_rec(ctx, ar, dF, strideF, lenF, (int)m, (int)n, order, dShift, method, thres, &P, s);
    if (st != PMLG_OK)
        return st;
    HIP_TRY(hipMemcpyAsync(shift, dShift, (size_t)m * 8, hipMemcpyDeviceToHost, s), "D2H(shift)");
    const int64_t L = std::min<int64_t>(P.len, capP);
    if (hP) {
        // entries packed to the computed length on the device (stride L)
        const uint64_t *src = P.cap == L ? P.d : nullptr;
        if (!src) {
            uint64_t *packed = ar.alloc((size_t)(m * m * L));
            if (packed) {
                hipLaunchKernelGGL(copy_poly_kernel, dim3(grid_for(m * m * L)), dim3(256), 0, s, packed,
                                   (int64_t)L, P.d, P.cap, (int64_t)(m * m), L);
                HIP_TRY(hipGetLastError(), "copy_poly_kernel");
                src = packed;
            }
        }
        int64_t Ln = 0;
        if (src) {
            // through the pinned staging chunks: each entry trimmed of its zero
            // top coefficients and zero-filled up to capP; the normalised
            // length is the longest entry's (the basis has degree at most order)
            std::vector<uint64_t *> ptr((size_t)(m * m));
            std::vector<int64_t> len((size_t)(m * m));
            for (int64_t e = 0; e < m * m; ++e)
                ptr[(size_t)e] = hP + e * capP;
            pmlg_status st2 = stage_download(ctx, ptr.data(), len.data(), src, m * m, L, s, capP);
            if (st2 != PMLG_OK)
                return st2;
            HIP_TRY(hipStreamSynchronize(s), "sync");  // the shifts' read-back
            for (int64_t e = 0; e < m * m; ++e)
                Ln = std::max(Ln, len[(size_t)e]);
        } else {
            // no arena room to pack: one transfer of the entries at capacity
            std::vector<uint64_t> tmp((size_t)(m * m * P.cap));
            HIP_TRY(hipMemcpyAsync(tmp.data(), P.d, tmp.size() * 8, hipMemcpyDeviceToHost, s), "D2H(P)");
            HIP_TRY(hipStreamSynchronize(s), "sync");
            for (int64_t e = 0; e < m * m; ++e)
                for (int64_t d = L - 1; d >= Ln; --d)
                    if (tmp[(size_t)(e * P.cap + d)]) {
                        Ln = d + 1;
                        break;
                    }
            for (int64_t e = 0; e < m * m; ++e) {
                std::memcpy(hP + e * capP, tmp.data() + e * P.cap, (size_t)Ln * 8);
                std::memset(hP + e * capP + Ln, 0, (size_t)(capP - Ln) * 8);
            }
        }
        *lenP = Ln;
    } else {
        hipLaunchKernelGGL(copy_poly_kernel, dim3(grid_for(m * m * L)), dim3(256), 0, s, dP, capP, P.d,
                           P.cap, (int64_t)(m * m), L);
        HIP_TRY(hipGetLastError(), "copy_poly_kernel");
        HIP_TRY(hipStreamSynchronize(s), "sync");
        *lenP = L;
    }
    return PMLG_OK;
}

}  // namespace pmlg

using namespace pmlg;

extern "C" {

pmlg_status pmlg_pmbasis_dev(pmlg_ctx ctx, uint64_t *dP, int64_t capP, int64_t *lenP,
                             int64_t *shift, const uint64_t *dF, int64_t m, int64_t n,
                             int64_t lenF, int64_t order, int method, void *stream)
{
    pmlg_status st = check_ctx(ctx);
    if (st != PMLG_OK)
        return st;
    std::lock_guard<std::mutex> lk(ctx->mu);
    DeviceGuard g(ctx->device);
    hipStream_t s = stream ? (hipStream_t)stream : ctx->stream;
    return basis_common(ctx, dP, capP, lenP, shift, dF, lenF, m, n, lenF, order, method, false, s,
                        nullptr);
}

static pmlg_status basis_host(pmlg_ctx ctx, uint64_t *P, int64_t *lenP, int64_t *shift,
                              const uint64_t *F, int64_t m, int64_t n, int64_t lenF, int64_t order,
                              int64_t capP, int method, bool iterative)
{
    pmlg_status st = check_ctx(ctx);
    if (st != PMLG_OK)
        return st;
    if (m <= 0 || n <= 0 || lenF < 0 || !P || !lenP || !shift || (lenF > 0 && !F))
        return fail(PMLG_ERR_ARG, "approximant basis: bad arguments");
    std::lock_guard<std::mutex> lk(ctx->mu);
    DeviceGuard g(ctx->device);
    hipStream_t s = ctx->stream;
    const size_t fb = (size_t)(m * n * (lenF > 0 ? lenF : 1)) * 8;
    HIP_TRY(ctx->in_a.ensure(fb), "hipMalloc(F)");
    if (lenF > 0) {
        // through the pinned staging chunks, entry by entry
        std::vector<const uint64_t *> ptr((size_t)(m * n));
        std::vector<int64_t> len((size_t)(m * n), lenF);
        for (int64_t e = 0; e < m * n; ++e)
            ptr[(size_t)e] = F + e * lenF;
        st = stage_upload(ctx, static_cast<uint64_t *>(ctx->in_a.ptr), ptr.data(), len.data(), m * n,
                          lenF);
        if (st != PMLG_OK)
            return st;
    }
    return basis_common(ctx, nullptr, capP, lenP, shift, static_cast<const uint64_t *>(ctx->in_a.ptr),
                        lenF, m, n, lenF, order, method, iterative, s, P);
}

pmlg_status pmlg_pmbasis(pmlg_ctx ctx, uint64_t *P, int64_t *lenP, int64_t *shift,
                         const uint64_t *F, int64_t m, int64_t n, int64_t lenF, int64_t order,
                         int64_t capP, int method)
{
    return basis_host(ctx, P, lenP, shift, F, m, n, lenF, order, capP, method, false);
}

pmlg_status pmlg_mbasis(pmlg_ctx ctx, uint64_t *P, int64_t *lenP, int64_t *shift,
                        const uint64_t *F, int64_t m, int64_t n, int64_t lenF, int64_t order,
                        int64_t capP)
{
    return basis_host(ctx, P, lenP, shift, F, m, n, lenF, order, capP, PMLG_METHOD_AUTO, true);
}

pmlg_status pmlg_pmbasis_set_leaf_order(pmlg_ctx ctx, int64_t order)
{
    pmlg_status st = check_ctx(ctx);
    if (st != PMLG_OK)
        return st;
    if (order < 0 || order > kMaxLeafOrder)
        return fail(PMLG_ERR_ARG, "pmbasis leaf order must be 0 (measured) or in [1, 256]");
    std::lock_guard<std::mutex> lk(ctx->mu);
    ctx->leaf_order = (int)order;
    return PMLG_OK;
}

pmlg_status pmlg_pmbasis_leaf_order(pmlg_ctx ctx, int64_t m, int64_t n, int method, int64_t *order)
{
    pmlg_status st = check_ctx(ctx);
    if (st != PMLG_OK)
        return st;
    if (m <= 0 || n <= 0 || m > kMaxM || n > kMaxN || !order)
        return fail(PMLG_ERR_ARG, "pmbasis leaf order: 1 <= m <= 256, 1 <= n <= 128");
    if (!ctx->is_prime && ctx->p != 2)
        return fail(PMLG_ERR_UNSUPPORTED, "approximant bases need a prime modulus");
    std::lock_guard<std::mutex> lk(ctx->mu);
    if (ctx->leaf_order > 0) {
        *order = ctx->leaf_order;
        return PMLG_OK;
    }
    DeviceGuard g(ctx->device);
    int t = kPmbasisThres;
    st = tune_leaf_order(ctx, (int)m, (int)n, method, ctx->stream, &t);
    *order = t;
    return st;
}

}  // extern "C"

// ===========================================================================
// Constant matrices and evaluation (used by the approximant-basis certificate)
// ===========================================================================
namespace pmlg {
namespace {

// Gaussian elimination of an r x c matrix held in device memory, by one
// workgroup (the matrix is modified in place; fcol holds r words of scratch):
// rank, and the determinant when r == c (product of the pivots, sign of the
// row swaps).  Barriers order the global-memory updates of one workgroup.
__global__ void __launch_bounds__(1024) const_gauss_kernel(uint64_t *A, uint64_t *fcol, int r, int c,
                                                           int *out_rank, uint64_t *out_det,
                                                           ModConst mc)
{
    __shared__ int s_pr;
    __shared__ uint64_t s_inv;
    const int tid = threadIdx.x;
    const uint64_t p = mc.p;
    int rank = 0;
    uint64_t det = 1 % p;
    bool neg = false;
    for (int col = 0; col < c && rank < r; ++col) {
        if (tid == 0) {
            int pr = -1;
            for (int i = rank; i < r; ++i)
                if (A[(size_t)i * c + col]) {
                    pr = i;
                    break;
                }
            s_pr = pr;
            if (pr >= 0)
                s_inv = invmod_g(A[(size_t)pr * c + col], mc);
        }
        __syncthreads();
        const int pr = s_pr;
        if (pr < 0) {
            det = 0;
            __syncthreads();
            continue;
        }
        if (pr != rank) {
            for (int j = tid; j < c; j += blockDim.x) {
                const uint64_t t = A[(size_t)pr * c + j];
                A[(size_t)pr * c + j] = A[(size_t)rank * c + j];
                A[(size_t)rank * c + j] = t;
            }
            neg = !neg;
        }
        __syncthreads();
        det = mulmod_g(det, A[(size_t)rank * c + col], mc);
        for (int i = tid; i < r; i += blockDim.x)
            fcol[i] = mulmod_g(A[(size_t)i * c + col], s_inv, mc);
        __syncthreads();
        for (int64_t idx = (int64_t)(rank + 1) * c + tid; idx < (int64_t)r * c; idx += blockDim.x) {
            const int i = (int)(idx / c), j = (int)(idx - (int64_t)i * c);
            A[idx] = submod_g(A[idx], mulmod_g(fcol[i], A[(size_t)rank * c + j], mc), p);
        }
        ++rank;
        __syncthreads();
    }
    if (tid == 0) {
        *out_rank = rank;
        if (out_det)
            *out_det = (r == c && rank == r) ? (neg && det ? p - det : det) : 0;
    }
}

// out[e] = sum_d A[e*len + d] x^d (Horner), one thread per entry
__global__ void eval_kernel(uint64_t *out, const uint64_t *A, int64_t entries, int64_t len,
                            uint64_t x, ModConst mc)
{
    for (int64_t e = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; e < entries;
         e += (int64_t)gridDim.x * blockDim.x) {
        uint64_t v = 0;
        for (int64_t d = len - 1; d >= 0; --d) {
            v = addmod_any(mulmod_g(v, x, mc), A[e * len + d], mc.p);
        }
        out[e] = v;
    }
}

}  // namespace

pmlg_status const_rank_dev(pmlg_ctx ctx, uint64_t *dM, uint64_t *dScratch, int64_t r, int64_t c,
                           int64_t *rank, hipStream_t s)
{
    int *drank = reinterpret_cast<int *>(dScratch + r);
    hipLaunchKernelGGL(const_gauss_kernel, dim3(1), dim3(1024), 0, s, dM, dScratch, (int)r, (int)c,
                       drank, nullptr, ctx->mc);
    HIP_TRY(hipGetLastError(), "const_gauss_kernel");
    int hr = 0;
    HIP_TRY(hipMemcpyAsync(&hr, drank, sizeof(int), hipMemcpyDeviceToHost, s), "D2H(rank)");
    HIP_TRY(hipStreamSynchronize(s), "sync");
    *rank = hr;
    return PMLG_OK;
}

}  // namespace pmlg

extern "C" {

pmlg_status pmlg_const_rank_det(pmlg_ctx ctx, const uint64_t *M, int64_t r, int64_t c,
                                int64_t *rank, uint64_t *det)
{
    pmlg_status st = check_ctx(ctx);
    if (st != PMLG_OK)
        return st;
    if (r < 0 || c < 0 || r > (1 << 16) || c > (1 << 16) || r * c > (1 << 22) || !rank ||
        (r * c > 0 && !M))
        return fail(PMLG_ERR_ARG, "const_rank_det: at most 2^22 entries");
    std::lock_guard<std::mutex> lk(ctx->mu);
    DeviceGuard g(ctx->device);
    hipStream_t s = ctx->stream;
    const size_t words = (size_t)(r * c) + (size_t)r + 4;
    HIP_TRY(ctx->in_b.ensure(words * 8), "hipMalloc");
    uint64_t *dM = static_cast<uint64_t *>(ctx->in_b.ptr);
    uint64_t *dcol = dM + r * c;
    uint64_t *ddet = dcol + r;
    int *drank = reinterpret_cast<int *>(ddet + 1);
    if (r * c)
        HIP_TRY(hipMemcpyAsync(dM, M, (size_t)(r * c) * 8, hipMemcpyHostToDevice, s), "H2D");
    hipLaunchKernelGGL(const_gauss_kernel, dim3(1), dim3(1024), 0, s, dM, dcol, (int)r, (int)c,
                       drank, ddet, ctx->mc);
    HIP_TRY(hipGetLastError(), "const_gauss_kernel");
    int hr = 0;
    uint64_t hd = 0;
    HIP_TRY(hipMemcpyAsync(&hr, drank, sizeof(int), hipMemcpyDeviceToHost, s), "D2H");
    HIP_TRY(hipMemcpyAsync(&hd, ddet, 8, hipMemcpyDeviceToHost, s), "D2H");
    HIP_TRY(hipStreamSynchronize(s), "sync");
    *rank = hr;
    if (det)
        *det = hd;
    return PMLG_OK;
}

pmlg_status pmlg_polmat_eval(pmlg_ctx ctx, uint64_t *out, const uint64_t *A, int64_t r, int64_t c,
                             int64_t len, uint64_t x)
{
    pmlg_status st = check_ctx(ctx);
    if (st != PMLG_OK)
        return st;
    if (r < 0 || c < 0 || len < 0 || !out || (r * c * len > 0 && !A))
        return fail(PMLG_ERR_ARG, "polmat_eval: bad arguments");
    std::lock_guard<std::mutex> lk(ctx->mu);
    DeviceGuard g(ctx->device);
    hipStream_t s = ctx->stream;
    const size_t ab = (size_t)(r * c * len) * 8, ob = (size_t)(r * c) * 8;
    HIP_TRY(ctx->in_a.ensure(ab ? ab : 8), "hipMalloc");
    HIP_TRY(ctx->out_c.ensure(ob ? ob : 8), "hipMalloc");
    if (ab)
        HIP_TRY(hipMemcpyAsync(ctx->in_a.ptr, A, ab, hipMemcpyHostToDevice, s), "H2D");
    hipLaunchKernelGGL(eval_kernel, dim3(grid_for(r * c)), dim3(256), 0, s,
                       static_cast<uint64_t *>(ctx->out_c.ptr),
                       static_cast<const uint64_t *>(ctx->in_a.ptr), r * c, len, x % ctx->p, ctx->mc);
    HIP_TRY(hipGetLastError(), "eval_kernel");
    if (ob)
        HIP_TRY(hipMemcpyAsync(out, ctx->out_c.ptr, ob, hipMemcpyDeviceToHost, s), "D2H");
    HIP_TRY(hipStreamSynchronize(s), "sync");
    return PMLG_OK;
}

}  // extern "C"
