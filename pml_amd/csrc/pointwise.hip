// Pointwise modular matrix products at every evaluation point:
//   C_hat[i][j][q] = sum_k A_hat[i][k][q] * B_hat[k][j][q] mod p.
//
// Two kernels:
//  * plain: each lane owns one point q and a TM x TN block of outputs; the
//    dot products are accumulated exactly in 128 bits (64-bit words) or
//    64 bits (32-bit words) and folded once per 15 terms;
//  * mfma: residues are split into balanced signed 8-bit digits
//    (x = sum_t l_t 2^(8t), l_t in [-128,127], 8 of them for 64-bit words and
//    4 for 32-bit ones); for every weight w the int8 MFMA chain
//    T_w = sum_{s+t=w} A_s * B_t accumulates exactly in int32 over the whole
//    k, the T_w are folded into three (or two) signed 64-bit partial sums,
//    and the exact dot product is rebuilt in 128 bits and reduced.
// 64-bit words leave V 2^-64 mod p (Montgomery REDC; the inverse transform's
// scaling carries the 2^64), below 4p for p < 2^60 and below 2p above, as the
// inverse's lazy and strict butterflies need; 32-bit words are reduced to [0, p) by
// Barrett steps.  No floating point is involved.
#include "internal.hpp"
#include "rules.hpp"

namespace pmlg {

namespace {

constexpr int kThreads = 256;
// Shapes that an explicit request for the MFMA kernel accepts: int8 planes of
// A and B at one point, padded to multiples of 32, within 128 KiB.  The
// kernel itself has no such limit (mfma_exact), and the automatic choice
// uses it beyond.
constexpr int64_t kMfmaPlanes = 128 * 1024;

typedef int v4i __attribute__((ext_vector_type(4)));

// waves per SIMD of the MFMA kernel: two with its usual points per task
// (about 200 registers), four with fewer
template <int PT, typename W>
constexpr int kMfmaWaves = PT * sizeof(W) < 16 ? 4 : 2;

// ---------------------------------------------------------------------------
// plain kernel
// ---------------------------------------------------------------------------
// Outputs per lane: TM x TN, TM = 2 or 4 (plain_rows).  A lane works on one
// point, so the wave's 64 lanes read 16 (8) neighbouring runs of each entry and
// the lines' other entries come with the next kk or column from L1.  Four rows
// read less per product; two leave registers for twice the waves, which hide the
// loads' latency, and waste less on a few rows.
constexpr int TN = 4;

// V 2^-64 mod p of a 128-bit sum of at most 15 products and a residue
// (Montgomery REDC; the inverse transform's scaling undoes the 2^-64): below
// 2p.  V < 15 p^2 + p, so for p < 2^60 the high word is below p; above, it is
// reduced first.
__device__ __forceinline__ uint64_t plain_redc(uint64_t hi, uint64_t lo, const ModConst &mc)
{
    if (mc.bits > 60)
        hi = barrett(hi, mc.bm, mc.p);
    const uint64_t mm = lo * mc.pinvneg;
    return hi + mulhi64(mm, mc.p) + (lo != 0 ? 1u : 0u);
}

// Lane (point q, output tile `tile` of TM x TN entries) of the plain product.
// Rows and columns past the matrix are not stored; tiles of four rows read the
// last ones instead, tiles of two none.
template <typename W, int TM>
__device__ __forceinline__ void plain_body(const W *__restrict__ Ah, const W *__restrict__ Bh,
                                           W *__restrict__ Ch, int m, int k, int n, int64_t N,
                                           int logP, int logPc, const ModConst &mc, int64_t q,
                                           int tile)
{
    const int tiles_n = (n + TN - 1) / TN;
    const int i0 = (tile / tiles_n) * TM;
    const int j0 = (tile % tiles_n) * TN;
    if (q >= N || i0 >= m)
        return;
    const int64_t run = q >> logP;
    const int off = (int)(q & ((1 << logP) - 1));
    const W *pa[TM], *pb[TN];
#pragma unroll
    for (int r = 0; r < TM; ++r)
        pa[r] = Ah + (((run * m + (TM == 4 ? min(i0 + r, m - 1) : i0 + r)) * k) << logP) + off;
#pragma unroll
    for (int c = 0; c < TN; ++c)
        pb[c] = Bh + ((run * k * n + (TM == 4 ? min(j0 + c, n - 1) : j0 + c)) << logP) + off;
    const int64_t bstep = (int64_t)n << logP;
    uint64_t hi[TM][TN], lo[TM][TN];  // 32-bit words: lo only
#pragma unroll
    for (int r = 0; r < TM; ++r)
#pragma unroll
        for (int c = 0; c < TN; ++c)
            hi[r][c] = lo[r][c] = 0;
    for (int k0 = 0; k0 < k; k0 += 15) {
        // 15 products (64-bit words: below 2^124 each, 32-bit: 2^60) plus a
        // residue below p do not overflow
        if (k0 > 0) {
#pragma unroll
            for (int r = 0; r < TM; ++r)
#pragma unroll
                for (int c = 0; c < TN; ++c) {
                    if constexpr (sizeof(W) == 8) {
                        lo[r][c] = reduce128(hi[r][c], lo[r][c], mc);
                        hi[r][c] = 0;
                    } else {
                        lo[r][c] = barrett(lo[r][c], mc.bm, mc.p);
                    }
                }
        }
        const int k1 = min(k0 + 15, k);
#pragma unroll 2
        for (int kk = k0; kk < k1; ++kk) {
            W a[TM], b[TN];
#pragma unroll
            for (int r = 0; r < TM; ++r)
                a[r] = TM == 4 || i0 + r < m ? pa[r][(int64_t)kk << logP] : (W)0;
#pragma unroll
            for (int c = 0; c < TN; ++c)
                b[c] = TM == 4 || j0 + c < n ? pb[c][kk * bstep] : (W)0;
#pragma unroll
            for (int r = 0; r < TM; ++r)
#pragma unroll
                for (int c = 0; c < TN; ++c) {
                    if constexpr (sizeof(W) == 8)
                        mac128(hi[r][c], lo[r][c], a[r], b[c]);
                    else
                        lo[r][c] += (uint64_t)a[r] * b[c];
                }
        }
    }
    W *cp = Ch + (((q >> logPc) * m * n) << logPc) + (q & ((1 << logPc) - 1));
#pragma unroll
    for (int r = 0; r < TM; ++r)
#pragma unroll
        for (int c = 0; c < TN; ++c)
            if (i0 + r < m && j0 + c < n) {
                W v;
                if constexpr (sizeof(W) == 8)
                    v = plain_redc(hi[r][c], lo[r][c], mc);
                else
                    v = (W)barrett(lo[r][c], mc.bm, mc.p);
                cp[((int64_t)(i0 + r) * n + j0 + c) << logPc] = v;
            }
}

// grid: x = 64-point chunks, y = groups of 4 output tiles (one per wave)
template <typename W, int TM>
__global__ void __launch_bounds__(kThreads)
pw_plain(const W *__restrict__ Ah, const W *__restrict__ Bh, W *__restrict__ Ch, int m, int k,
         int n, int64_t N, int logP, int logPc, ModConst mc)
{
    const int64_t q = (int64_t)blockIdx.x * 64 + (threadIdx.x & 63);
    const int tile = blockIdx.y * (kThreads / 64) + (threadIdx.x >> 6);
    plain_body<W, TM>(Ah, Bh, Ch, m, k, n, N, logP, logPc, mc, q, tile);
}

// ---------------------------------------------------------------------------
// int8-limb MFMA kernel
// ---------------------------------------------------------------------------

// Balanced signed base-256 digits: with C = 0x80..80 (one 0x80 per byte),
// y = x + C has ordinary digits b_t and x = sum (b_t - 128) 256^t, so the
// signed digit l_t = b_t - 128 is the byte b_t ^ 0x80, i.e. byte t of
// (x + C) ^ C.  Valid while x + C does not overflow (x < 2^61 for 8 limbs,
// x < 2^30 for 4 limbs).
__device__ __forceinline__ uint64_t limb_bytes(uint64_t x)
{
    const uint64_t C = 0x8080808080808080ull;
    return (x + C) ^ C;
}
__device__ __forceinline__ uint32_t limb_bytes(uint32_t x)
{
    const uint32_t C = 0x80808080u;
    return (x + C) ^ C;
}

// bytes of x in reverse order
__device__ __forceinline__ uint32_t rev_bytes(uint32_t x)
{
    return __builtin_amdgcn_perm(0, x, 0x00010203u);
}

// Position s (byte s) of the result holds digit w - s of the word whose
// reversed digits are r (zero where w - s is outside 0..3)
template <int w>
__device__ __forceinline__ uint32_t conv_word(uint32_t r)
{
    return w <= 3 ? r >> (8 * (3 - w)) : r << (8 * (w - 3));
}

// PT consecutive words at src (aligned to the PT words, 16 bytes at most)
template <typename W, int PT>
__device__ __forceinline__ void load_points(const W *__restrict__ src, W (&v)[PT])
{
    if constexpr (PT * sizeof(W) == 16) {
        const uint4 x = *reinterpret_cast<const uint4 *>(src);
        if constexpr (sizeof(W) == 8) {
            v[0] = ((uint64_t)x.y << 32) | x.x;
            v[1] = ((uint64_t)x.w << 32) | x.z;
        } else {
            v[0] = x.x;
            v[1] = x.y;
            v[2] = x.z;
            v[3] = x.w;
        }
    } else if constexpr (PT == 2) {
        const uint2 x = *reinterpret_cast<const uint2 *>(src);
        v[0] = x.x;
        v[1] = x.y;
    } else {
#pragma unroll
        for (int t = 0; t < PT; ++t)
            v[t] = src[t];
    }
}

template <typename W, int PT>
__device__ __forceinline__ void store_points(W *dst, const W (&v)[PT])
{
    if constexpr (PT * sizeof(W) == 16) {
        uint4 u;
        if constexpr (sizeof(W) == 8) {
            u.x = (uint32_t)v[0];
            u.y = (uint32_t)(v[0] >> 32);
            u.z = (uint32_t)v[1];
            u.w = (uint32_t)(v[1] >> 32);
        } else {
            u.x = v[0];
            u.y = v[1];
            u.z = v[2];
            u.w = v[3];
        }
        *reinterpret_cast<uint4 *>(dst) = u;
    } else if constexpr (PT == 2) {
        *reinterpret_cast<uint2 *>(dst) = make_uint2(v[0], v[1]);
    } else {
#pragma unroll
        for (int t = 0; t < PT; ++t)
            dst[t] = v[t];
    }
}

// One task: a 16 x 16 tile of outputs at PT consecutive points, by one wave,
// with no LDS and no barrier.
//
// The contraction runs over (kk, s), s the digit index within a 32-bit half
// word: a lane's A fragment is the balanced digits of four kk as they lie in
// memory (16 bytes), and the B fragment of weight w holds at position s the
// digit w - s, i.e. the reversed digits of the B word shifted by 8 |w - 3|
// bits.  So the digits are never transposed: A costs an add and an xor, B a
// byte reversal and six shifts per half word, and both come straight from
// the evaluations into registers.  The order of the kk within a chunk of 16
// is free; load u of lane group g takes kk = 4 u + g, so that the four groups
// read neighbouring entries of A (one 128-byte line per row and load, not
// four).  The price is matrix work, 112
// digit products instead of 64 (7 weights x 4 positions for each of the four
// half-word products), which the matrix cores have to spare: they are busy
// for a third of the time in which the vector ALUs prepare, fold and reduce.
// For each weight the chain accumulates exactly in int32 over the whole k
// (|T_w| <= 8 k 2^14 < 2^30 for k <= 4064).
//
// 16 x 16 x 64 tiles: lane l holds A[row l % 16][bytes 16 (l / 16) ..], B the
// same by column; output register r of lane l is row 4 (l / 16) + r, column
// l % 16.
template <typename W, int PT>
struct MfmaTile {
    static constexpr int H = sizeof(W) == 8 ? 2 : 1;  // half words
    static constexpr int NW = 8 * H - 1;              // weights: 15 or 7
    v4i acc[PT][NW];

    // one chunk of 16 kk: xa, xb the lane's four words of A and B per point
    template <bool FIRST>
    __device__ __forceinline__ void chunk(const W (&xa)[4][PT], const W (&xb)[4][PT])
    {
#pragma unroll
        for (int pt = 0; pt < PT; ++pt) {
            v4i fa[H];
            uint32_t rb[H][4];
#pragma unroll
            for (int u = 0; u < 4; ++u) {
                const W za = limb_bytes(xa[u][pt]), zb = limb_bytes(xb[u][pt]);
                fa[0][u] = (int)(uint32_t)za;
                rb[0][u] = rev_bytes((uint32_t)zb);
                if constexpr (H == 2) {
                    fa[H - 1][u] = (int)(uint32_t)(za >> 32);
                    rb[H - 1][u] = rev_bytes((uint32_t)(zb >> 32));
                }
            }
            weights<FIRST, 0>(acc[pt], fa, rb);
        }
    }

    template <bool FIRST, int w>
    __device__ __forceinline__ void weights(v4i (&t)[NW], const v4i (&fa)[H], const uint32_t (&rb)[H][4])
    {
        const v4i zero = {0, 0, 0, 0};
        v4i fb[H];
#pragma unroll
        for (int h = 0; h < H; ++h)
#pragma unroll
            for (int u = 0; u < 4; ++u)
                fb[h][u] = (int)conv_word<w>(rb[h][u]);
        // half-word products of weight 2^(8 w), 2^(8 w + 32), 2^(8 w + 64); the
        // first product into an accumulator of the first chunk starts from
        // zero: low x low for weights 0..3 (all seven with one half-word), the
        // cross products for 4..7, high x high for 8..14
        constexpr bool Z = FIRST && (w < 4 || H == 1);
        t[w] = __builtin_amdgcn_mfma_i32_16x16x64_i8(fa[0], fb[0], Z ? zero : t[w], 0, 0, 0);
        if constexpr (H == 2) {
            t[w + 4] = __builtin_amdgcn_mfma_i32_16x16x64_i8(fa[0], fb[H - 1], Z ? zero : t[w + 4], 0, 0, 0);
            t[w + 4] = __builtin_amdgcn_mfma_i32_16x16x64_i8(fa[H - 1], fb[0], t[w + 4], 0, 0, 0);
            t[w + 8] = __builtin_amdgcn_mfma_i32_16x16x64_i8(fa[H - 1], fb[H - 1], FIRST ? zero : t[w + 8], 0, 0, 0);
        }
        if constexpr (w < 6)
            weights<FIRST, w + 1>(t, fa, rb);
    }
};

// sum of five (or fewer) consecutive weights, T_0 + T_1 2^8 + ... + T_4 2^32
// (below 2^62 in magnitude): multiply-adds by the powers of two kept in
// scalar registers (hidden from the compiler, which would otherwise turn
// each into a sign extension, a shift and an add)
struct Pow2 {
    int c0, c8, c16, c24;
    __device__ Pow2() : c0(1), c8(1 << 8), c16(1 << 16), c24(1 << 24)
    {
        asm volatile("" : "+s"(c0), "+s"(c8), "+s"(c16), "+s"(c24));
    }
};
template <int CNT>
__device__ __forceinline__ int64_t fold_weights(int t0, int t1, int t2, int t3, int t4, const Pow2 &c)
{
    int64_t g = (int64_t)t0 * c.c0;
    g += (int64_t)t1 * c.c8;
    g += (int64_t)t2 * c.c16;
    if constexpr (CNT > 3)
        g += (int64_t)t3 * c.c24;
    if constexpr (CNT > 4)
        g = (int64_t)(((uint64_t)((uint32_t)((uint64_t)g >> 32) + (uint32_t)t4) << 32) | (uint32_t)g);
    return g;
}

// V = g0 + g1 2^40 + g2 2^80 as a nonnegative 128-bit integer (hi, lo): each
// sum hands what exceeds its 40 bits to the next, then the bytes are put
// together
__device__ __forceinline__ void join_sums(int64_t g0, int64_t g1, int64_t g2, uint64_t &hi, uint64_t &lo)
{
    const uint64_t u = (uint64_t)(g1 + (g0 >> 40));
    const uint64_t v = (uint64_t)(g2 + ((int64_t)u >> 40));
    const uint32_t ul = (uint32_t)u, uh = (uint32_t)(u >> 32), vl = (uint32_t)v, vh = (uint32_t)(v >> 32);
    // v_perm_b32(s0, s1, sel): selector 0-3 picks bytes of s1, 4-7 bytes of s0
    const uint32_t l1 = __builtin_amdgcn_perm(ul, (uint32_t)((uint64_t)g0 >> 32), 0x06050400u);
    const uint32_t h0 = __builtin_amdgcn_perm(vl, __builtin_amdgcn_alignbit(uh, ul, 24), 0x05040100u);
    lo = ((uint64_t)l1 << 32) | (uint32_t)g0;
    hi = ((uint64_t)__builtin_amdgcn_alignbit(vh, vl, 16) << 32) | h0;
}

// (hi 2^64 + lo + m p) / 2^64 with m = -lo / p mod 2^64 (Montgomery REDC), one
// 32-bit word of m at a time: below hi + p + 1
__device__ __forceinline__ uint64_t redc_words(uint64_t hi, uint64_t lo, const ModConst &mc)
{
    const uint32_t pi = (uint32_t)mc.pinvneg, p0 = (uint32_t)mc.p, p1 = (uint32_t)(mc.p >> 32);
    const uint32_t m0 = (uint32_t)lo * pi;
    const uint64_t c0 = ((uint64_t)m0 * p0 + (uint32_t)lo) >> 32;
    const uint64_t t = (uint64_t)m0 * p1 + (lo >> 32) + c0;  // no overflow: 2^64 - 1 at most
    const uint32_t m1 = (uint32_t)t * pi;
    const uint64_t c1 = ((uint64_t)m1 * p0 + (uint32_t)t) >> 32;
    return hi + ((uint64_t)m1 * p1 + (t >> 32) + c1);
}

template <typename W, int PT>
__device__ __forceinline__ void mfma_task(const W *__restrict__ Ah, const W *__restrict__ Bh,
                                          W *__restrict__ Ch, int m, int k, int n, int logP,
                                          int logPc, const ModConst &mc, int64_t q0, int mt, int nt)
{
    const int lane = threadIdx.x & 63;
    const int lr = lane & 15, g = lane >> 4;
    // rows and columns past the matrix read its last one; their outputs are
    // not stored.  kk past k reads the last one and A counts as zero there.
    const int row = min(mt * 16 + lr, m - 1), col = min(nt * 16 + lr, n - 1);
    const int64_t run = q0 >> logP;
    const int off = (int)(q0 & ((1 << logP) - 1));
    // uniform bases of the chunk and the lane's byte offsets from them (the
    // entries of one run fit 32 bits of offset, see mfma_exact): a whole chunk
    // needs no address arithmetic on the vector ALUs
    const char *pa = reinterpret_cast<const char *>(Ah + ((run * m * k) << logP) + off);
    const char *pb = reinterpret_cast<const char *>(Bh + ((run * k * n) << logP) + off);
    const int sh = logP + (sizeof(W) == 8 ? 3 : 2);  // bytes of a run
    const int64_t astep = (int64_t)16 << sh, bstep = (int64_t)(16 * n) << sh;
    uint32_t oa[4], ob[4];
#pragma unroll
    for (int u = 0; u < 4; ++u) {
        oa[u] = (uint32_t)(row * k + 4 * u + g) << sh;
        ob[u] = (uint32_t)((4 * u + g) * n + col) << sh;
    }
    auto load = [&](int kc, W (&xa)[4][PT], W (&xb)[4][PT]) __attribute__((always_inline)) {
        if (kc + 16 <= k) {
#pragma unroll
            for (int u = 0; u < 4; ++u) {
                load_points<W, PT>(reinterpret_cast<const W *>(pa + oa[u]), xa[u]);
                load_points<W, PT>(reinterpret_cast<const W *>(pb + ob[u]), xb[u]);
            }
        } else {
#pragma unroll
            for (int u = 0; u < 4; ++u) {
                // signed: a chunk's first entries may lie above the last one
                const int back = max(kc + 4 * u + g - (k - 1), 0);
                load_points<W, PT>(reinterpret_cast<const W *>(pa + ((int64_t)oa[u] - ((int64_t)back << sh))), xa[u]);
                load_points<W, PT>(reinterpret_cast<const W *>(pb + ((int64_t)ob[u] - ((int64_t)back * n << sh))), xb[u]);
#pragma unroll
                for (int pt = 0; pt < PT; ++pt)
                    xa[u][pt] = back > 0 ? (W)0 : xa[u][pt];
            }
        }
        pa += astep;
        pb += bstep;
    };
    MfmaTile<W, PT> tile;
    W xa[4][PT], xb[4][PT];
    load(0, xa, xb);
    {
        W ya[4][PT], yb[4][PT];
        if (k > 16)
            load(16, ya, yb);  // in flight during the first chunk's products
        tile.template chunk<true>(xa, xb);
        for (int kc = 16; kc < k; kc += 16) {
#pragma unroll
            for (int u = 0; u < 4; ++u)
#pragma unroll
                for (int pt = 0; pt < PT; ++pt) {
                    xa[u][pt] = ya[u][pt];
                    xb[u][pt] = yb[u][pt];
                }
            if (kc + 16 < k)
                load(kc + 16, ya, yb);
            tile.template chunk<false>(xa, xb);
        }
    }
    const Pow2 c2;
    W res[4][PT];
#pragma unroll
    for (int r = 0; r < 4; ++r)
#pragma unroll
        for (int pt = 0; pt < PT; ++pt) {
            const auto &t = tile.acc[pt];
            if constexpr (sizeof(W) == 8) {
                // exact V, 0 <= V < 2^128, then REDC: V 2^-64 mod p (the 2^-64 is
                // undone by the inverse transform's scaling)
                const int64_t g0 = fold_weights<5>(t[0][r], t[1][r], t[2][r], t[3][r], t[4][r], c2);
                const int64_t g1 = fold_weights<5>(t[5][r], t[6][r], t[7][r], t[8][r], t[9][r], c2);
                const int64_t g2 = fold_weights<5>(t[10][r], t[11][r], t[12][r], t[13][r], t[14][r], c2);
                uint64_t hi, lo;
                join_sums(g0, g1, g2, hi, lo);
                res[r][pt] = (W)redc_words(hi, lo, mc);
            } else {
                // V = G0 + G1 2^32 < k p^2 < 2^72: hi < 2^8, hi * (2^64 mod p) < 2^38
                const int64_t g0 = fold_weights<4>(t[0][r], t[1][r], t[2][r], t[3][r], 0, c2);
                const int64_t g1 = fold_weights<3>(t[4][r], t[5][r], t[6][r], 0, 0, c2) + (g0 >> 32);
                const uint64_t lo = ((uint64_t)g1 << 32) | (uint32_t)g0;
                const uint64_t hi = (uint64_t)(g1 >> 32);
                res[r][pt] = (W)barrett(barrett_lazy(lo, mc.bm, mc.p) + hi * mc.c64, mc.bm, mc.p);
            }
        }
    // small k p: the REDC outputs are within the inverse's range already;
    // otherwise a Barrett step to below 2p (they are below 2^64)
    if (sizeof(W) == 8 && !mc.redc_small) {
#pragma unroll
        for (int r = 0; r < 4; ++r)
#pragma unroll
            for (int pt = 0; pt < PT; ++pt)
                res[r][pt] = (W)barrett_lazy((uint64_t)res[r][pt], mc.bm, mc.p);
    }
    // all outputs are formed before the first conditional store: independent
    // chains in one basic block
#pragma unroll
    for (int r = 0; r < 4; ++r)
#pragma unroll
        for (int pt = 0; pt < PT; ++pt)
            asm volatile("" : "+v"(res[r][pt]));
    const int ocol = nt * 16 + lr, orow = mt * 16 + 4 * g;
    // (PT <= 2^logP <= 2^logPc: the points lie within one run of C)
    char *pc = reinterpret_cast<char *>(Ch + (((q0 >> logPc) * m * n) << logPc) +
                                        (q0 & ((1 << logPc) - 1)));
    const int shc = logPc + (sizeof(W) == 8 ? 3 : 2);
#pragma unroll
    for (int r = 0; r < 4; ++r)
        if (orow + r < m && ocol < n)
            store_points<W, PT>(reinterpret_cast<W *>(pc + ((uint32_t)((orow + r) * n + ocol) << shc)),
                                res[r]);
}

// Tasks of one product, in the order point group, row tile, column tile (the
// tiles of one point group read the same entries, so they stay together)
struct MfmaTasks {
    uint32_t tn, tiles;
    int64_t total;  // below 2^32: an evaluation array of that many tiles has 2^40 words
    __host__ __device__ MfmaTasks(int m, int n, int64_t N, int pt)
        : tn((uint32_t)(n + 15) >> 4), tiles(((uint32_t)(m + 15) >> 4) * tn), total(N / pt * tiles)
    {
    }
};

// Workgroups b, b + 8, b + 16, ... run on one XCD (round-robin dispatch):
// each XCD takes one contiguous eighth of the blocks, so that the tasks of
// one point group, and neighbouring groups, which share lines, meet in one
// L2.  Launch indices run over xcd_grid(blocks); those with no block get -1.
__host__ __device__ inline int64_t xcd_grid(int64_t blocks)
{
    return (blocks + 7) & ~(int64_t)7;
}
__device__ __forceinline__ int64_t xcd_block(int64_t b, int64_t blocks)
{
    const int64_t per = (blocks + 7) >> 3;
    const int64_t u = (b & 7) * per + (b >> 3);
    return u < blocks ? u : -1;
}

template <typename W, int PT>
__device__ __forceinline__ void mfma_wave(const W *Ah, const W *Bh, W *Ch, int m, int k, int n,
                                          int64_t N, int logP, int logPc, const ModConst &mc,
                                          int64_t task)
{
    const MfmaTasks ts(m, n, N, PT);
    if (task >= ts.total)
        return;
    const uint32_t grp = (uint32_t)task / ts.tiles;
    const uint32_t tile = (uint32_t)task - grp * ts.tiles;
    const uint32_t mt = tile / ts.tn;
    mfma_task<W, PT>(Ah, Bh, Ch, m, k, n, logP, logPc, mc, (int64_t)grp * PT, (int)mt,
                     (int)(tile - mt * ts.tn));
}

constexpr int kWaves = kThreads / 64;

template <typename W, int PT>
__global__ void __launch_bounds__(kThreads) __attribute__((amdgpu_waves_per_eu(kMfmaWaves<PT, W>)))
pw_mfma_kernel(const W *__restrict__ Ah, const W *__restrict__ Bh, W *__restrict__ Ch, int m,
               int k, int n, int64_t N, int64_t blocks, int logP, int logPc, ModConst mc)
{
    const int64_t b = xcd_block(blockIdx.x, blocks);
    if (b < 0)
        return;
    // the task is uniform across the wave
    const int64_t task = b * kWaves + __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    mfma_wave<W, PT>(Ah, Bh, Ch, m, k, n, N, logP, logPc, mc, task);
}

// ---------------------------------------------------------------------------
// persistent segment-table launches (batched products)
// ---------------------------------------------------------------------------
template <typename W>
__device__ __forceinline__ const PwSeg<W> &pw_seg_of(const PwSeg<W> *segs, int nseg, int64_t b)
{
    int lo = 0, hi = nseg - 1;
    while (lo < hi) {
        const int mid = (lo + hi + 1) >> 1;
        if (segs[mid].block0 <= b)
            lo = mid;
        else
            hi = mid - 1;
    }
    return segs[lo];
}

// Every workgroup walks the block list from its own index on, in steps of
// the grid (a multiple of 8, so that it stays on its XCD's share); a block is
// one task per wave.
template <typename W, int PT>
__global__ void __launch_bounds__(kThreads) __attribute__((amdgpu_waves_per_eu(kMfmaWaves<PT, W>)))
pw_mfma_segs(const PwSeg<W> *__restrict__ segs, int nseg, int64_t blocks, ModConst mc)
{
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    for (int64_t i = blockIdx.x; i < xcd_grid(blocks); i += gridDim.x) {
        const int64_t b = xcd_block(i, blocks);
        if (b < 0)
            continue;
        const PwSeg<W> &sg = pw_seg_of(segs, nseg, b);
        ModConst mcs = mc;
        mcs.redc_small = __builtin_amdgcn_readfirstlane(sg.redc_small);
        mfma_wave<W, PT>(as_global(sg.Ah), as_global(sg.Bh), as_global(sg.Ch),
                         __builtin_amdgcn_readfirstlane(sg.m), __builtin_amdgcn_readfirstlane(sg.k),
                         __builtin_amdgcn_readfirstlane(sg.n), uniform(sg.N),
                         __builtin_amdgcn_readfirstlane(sg.logP), __builtin_amdgcn_readfirstlane(sg.logPc),
                         mcs, (b - uniform(sg.block0)) * kWaves + wave);
    }
}

// task = (64-point chunk, group of 4 output tiles) of one product
template <typename W, int TM>
__global__ void __launch_bounds__(kThreads)
pw_plain_segs(const PwSeg<W> *__restrict__ segs, int nseg, int64_t blocks, ModConst mc)
{
    for (int64_t b = blockIdx.x; b < blocks; b += gridDim.x) {
        const PwSeg<W> &sg = pw_seg_of(segs, nseg, b);
        const int64_t gx = (sg.N + 63) >> 6;
        const int64_t lb = b - sg.block0;
        const int64_t by = lb / gx;
        const int64_t q = (lb - by * gx) * 64 + (threadIdx.x & 63);
        const int tile = (int)by * kWaves + (threadIdx.x >> 6);
        plain_body<W, TM>(as_global(sg.Ah), as_global(sg.Bh), as_global(sg.Ch), sg.m, sg.k, sg.n, sg.N, sg.logP,
                      sg.logPc, mc, q, tile);
    }
}

template <typename W, int PT>
hipError_t launch_mfma_pt(const W *Ah, const W *Bh, W *Ch, int m, int k, int n, int64_t N,
                          int logP, int logPc, const ModConst &mc, hipStream_t s)
{
    const int64_t blocks = (MfmaTasks(m, n, N, PT).total + kWaves - 1) / kWaves;
    const int64_t grid = xcd_grid(blocks);
    if (grid > INT32_MAX)
        return hipErrorInvalidValue;
    hipLaunchKernelGGL((pw_mfma_kernel<W, PT>), dim3((unsigned)grid), dim3(kThreads), 0, s, Ah, Bh,
                       Ch, m, k, n, N, blocks, logP, logPc, mc);
    return hipGetLastError();
}

// groups of kWaves output tiles of `rows` rows
inline int64_t plain_groups(int m, int n, int rows)
{
    return ((int64_t)((m + rows - 1) / rows) * ((n + TN - 1) / TN) + kWaves - 1) / kWaves;
}

template <typename W, int TM>
hipError_t launch_plain(const W *Ah, const W *Bh, W *Ch, int m, int k, int n, int64_t N, int logP,
                        int logPc, const ModConst &mc, hipStream_t s)
{
    const dim3 grid((unsigned)((N + 63) / 64), (unsigned)plain_groups(m, n, TM));
    hipLaunchKernelGGL((pw_plain<W, TM>), grid, dim3(kThreads), 0, s, Ah, Bh, Ch, m, k, n, N, logP, logPc,
                       mc);
    return hipGetLastError();
}

// points of one task: 16 bytes of a run, or one point where runs are shorter
template <typename W>
constexpr int kPoints = 16 / sizeof(W);

template <typename W>
hipError_t launch_pointwise_w(PointwiseKind kind, const W *Ah, const W *Bh, W *Ch, int m, int k,
                              int n, int64_t N, int logP, int logPc, const ModConst &mc,
                              hipStream_t s)
{
    if (kind == PW_MFMA) {
        if (mc.limbs != (int)sizeof(W) || !mfma_exact(m, k, n, mc.limbs, mc.p))
            return hipErrorInvalidValue;
        if ((1 << logP) >= kPoints<W>)
            return launch_mfma_pt<W, kPoints<W>>(Ah, Bh, Ch, m, k, n, N, logP, logPc, mc, s);
        return launch_mfma_pt<W, 1>(Ah, Bh, Ch, m, k, n, N, logP, logPc, mc, s);
    }
    if (plain_rows(m, N, plain_waves(m, n, N)) == 4)
        return launch_plain<W, 4>(Ah, Bh, Ch, m, k, n, N, logP, logPc, mc, s);
    return launch_plain<W, 2>(Ah, Bh, Ch, m, k, n, N, logP, logPc, mc, s);
}

}  // namespace

bool mfma_exact(int m, int k, int n, int limbs, uint64_t p)
{
    // the signed partial sums stay below 2^62 for K <= 4064; the exact
    // recombination needs the dot product k (p-1)^2 below 2^128
    if (m <= 0 || k <= 0 || n <= 0 || k > 4064 || limbs <= 0)
        return false;
    // byte offsets within one run of an operand (at most 32 bytes an entry)
    // fit 32 bits
    const int64_t most = (int64_t)1 << 26;
    if ((int64_t)m * k >= most || (int64_t)(k + 16) * n >= most || (int64_t)m * n >= most)
        return false;
    // REDC needs V + (p+1) 2^64 <= 2^128 (8 limbs); 4 limbs only needs V < 2^72
    const unsigned __int128 sq = (unsigned __int128)(p - 1) * (p - 1);
    const unsigned __int128 lim =
        limbs == 8 ? (~(unsigned __int128)0) - ((unsigned __int128)(p + 1) << 64)
                   : ((unsigned __int128)1 << 72);
    return sq == 0 || (unsigned __int128)k <= lim / sq;
}

bool mfma_supported(int m, int k, int n, int limbs, uint64_t p)
{
    const int64_t Mp = (m + 31) & ~31, Kp = (k + 31) & ~31, Np = (n + 31) & ~31;
    return mfma_exact(m, k, n, limbs, p) && limbs * (Mp * Kp + Np * Kp) <= kMfmaPlanes;
}

template <>
hipError_t launch_pointwise<uint64_t>(PointwiseKind kind, const uint64_t *Ah, const uint64_t *Bh,
                                      uint64_t *Ch, int m, int k, int n, int64_t N, int logP,
                                      int logPc, const ModConst &mc, hipStream_t s)
{
    return launch_pointwise_w<uint64_t>(kind, Ah, Bh, Ch, m, k, n, N, logP, logPc, mc, s);
}

template <>
hipError_t launch_pointwise<uint32_t>(PointwiseKind kind, const uint32_t *Ah, const uint32_t *Bh,
                                      uint32_t *Ch, int m, int k, int n, int64_t N, int logP,
                                      int logPc, const ModConst &mc, hipStream_t s)
{
    return launch_pointwise_w<uint32_t>(kind, Ah, Bh, Ch, m, k, n, N, logP, logPc, mc, s);
}

// ---------------------------------------------------------------------------
// batched launches
// ---------------------------------------------------------------------------
int pw_plain_rows(int m, int64_t N)
{
    // (the other products of the launch fill the chip)
    return plain_rows(m, N, INT64_MAX);
}

int64_t pw_seg_blocks(PointwiseKind kind, int pt, int m, int n, int64_t N)
{
    if (kind == PW_MFMA)
        return (MfmaTasks(m, n, N, pt).total + kWaves - 1) / kWaves;
    return ((N + 63) / 64) * plain_groups(m, n, pt);
}

template <typename W>
hipError_t launch_pointwise_segs(PointwiseKind kind, int pt, const PwSeg<W> *segs, int nseg,
                                 int64_t blocks, int grid, const ModConst &mc, hipStream_t s)
{
    if (nseg <= 0 || blocks <= 0)
        return hipSuccess;
    if (kind == PW_PLAIN) {
        if (grid <= 0 || grid > blocks)
            grid = (int)(blocks < (1 << 30) ? blocks : (1 << 30));
        if (pt == 4)
            hipLaunchKernelGGL((pw_plain_segs<W, 4>), dim3((unsigned)grid), dim3(kThreads), 0, s, segs,
                               nseg, blocks, mc);
        else if (pt == 2)
            hipLaunchKernelGGL((pw_plain_segs<W, 2>), dim3((unsigned)grid), dim3(kThreads), 0, s, segs,
                               nseg, blocks, mc);
        else
            return hipErrorInvalidValue;
        return hipGetLastError();
    }
    if (mc.limbs != (int)sizeof(W))
        return hipErrorInvalidValue;
    const int64_t all = xcd_grid(blocks);
    if (grid <= 0 || grid > all)
        grid = (int)(all < (1 << 30) ? all : (1 << 30));
    grid = (int)xcd_grid(grid);
    if (pt == kPoints<W>)
        hipLaunchKernelGGL((pw_mfma_segs<W, kPoints<W>>), dim3((unsigned)grid), dim3(kThreads), 0, s,
                           segs, nseg, blocks, mc);
    else if (pt == kPoints<W> / 2)
        hipLaunchKernelGGL((pw_mfma_segs<W, kPoints<W> / 2>), dim3((unsigned)grid), dim3(kThreads), 0, s,
                           segs, nseg, blocks, mc);
    else if (pt == 1)
        hipLaunchKernelGGL((pw_mfma_segs<W, 1>), dim3((unsigned)grid), dim3(kThreads), 0, s, segs,
                           nseg, blocks, mc);
    else
        return hipErrorInvalidValue;
    return hipGetLastError();
}

template hipError_t launch_pointwise_segs<uint64_t>(PointwiseKind, int, const PwSeg<uint64_t> *,
                                                    int, int64_t, int, const ModConst &, hipStream_t);
template hipError_t launch_pointwise_segs<uint32_t>(PointwiseKind, int, const PwSeg<uint32_t> *,
                                                    int, int64_t, int, const ModConst &, hipStream_t);

}  // namespace pmlg
