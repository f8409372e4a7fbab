// Rules on sizes that pick between exact variants of one computation.  Host code,
// plain integers in and out, so that they can be tested without a device.
#pragma once

#include <stdint.h>

#include <algorithm>

namespace pmlg {

// Waves of the plain pointwise kernel for m x n outputs at N points in tiles of 4 x 4.
inline int64_t plain_waves(int m, int n, int64_t N)
{
    return (N + 63) / 64 * ((m + 3) / 4) * ((n + 3) / 4);
}

// Rows of a lane's tile in the plain kernel at N points.  Two below 2048 waves of
// four rows (two per SIMD) or with idle lanes, where the loads' latency bounds it,
// and for up to 6 rows.
// Microseconds, four / two rows, 64-bit words: 1 x 64 x 1 at 2^16 points 80 / 34,
// 4 x 32 x 4 at 2^16 53 / 37, 64 x 64 x 64 at 2^8 71 / 61; 12 x 8 x 12 at 2^16 63 /
// 66, 64 x 32 x 64 at 2^12 334 / 364; 200 x 200 x 200 at one point (transforms
// included) 515 / 415; 32-bit words: 64 x 64 x 64 at 2^10 43 / 61.
// (Two rows were the old kernel's; four everywhere had cost the small products
// up to half their speed.)
inline int plain_rows(int m, int64_t N, int64_t waves)
{
    return N >= 64 && waves >= 2048 && m > 6 ? 4 : 2;
}

// Points per task of the MFMA kernel, for words of elem_bytes in runs of 2^logP
// points: 16 bytes of a run, or 8 (half), or one point where the run is shorter.
// Half of it takes twice the waves per SIMD and reads as many bytes in half the
// requests that single points take; with one point for 32-bit words configuration 6
// took 2960 us for 16 products 32 x 32 x 32 of length 4096 (30-bit prime), with two
// 2160.
inline int pw_points(int elem_bytes, int logP, bool half)
{
    const int pt = (half ? 8 : 16) / elem_bytes;
    return (1 << logP) < pt ? 1 : pt;
}

// Whether the MFMA kernel is the faster one where both are exact: its time and the
// plain kernel's in nanoseconds, a start and a chain (the loads of a step of 16, or
// of one, of the inner dimension, one after another) plus what each task (a tile of
// 16 x 16 outputs at 16 bytes of points) or wave adds.  Fitted (least squares) to
// 1280 shapes from 1 x 2 x 1 to 64 x 64 x 64 at 2 to 2^16 points, on which the rule
// takes the slower kernel by more than 15% and 2 us nine times.  Without the starts
// and chains products too small to fill the chip took the plain kernel where MFMA is
// up to five times as fast (us, plain / MFMA, 64-bit words: 4 x 200 x 4 at 2 points
// 147 / 13, 8 x 8 x 8 at 2 points 13 / 4; 8 x 8 x 8 at 2^16 points 28 / 59, 32 x 32 x
// 32 at 2^13 175 / 48; 32-bit words: 4 x 64 x 5 at 2^12 21 / 7, 8 x 8 x 8 at 2^16
// 13 / 38).
inline bool mfma_pays(int m, int k, int n, int64_t N, int limbs)
{
    const double steps = (k + 15) / 16;
    const double tasks = (double)((m + 15) / 16) * ((n + 15) / 16) * std::max<int64_t>(1, limbs == 8 ? N / 2 : N / 4);
    const double waves = (double)plain_waves(m, n, N);
    if (limbs == 8)
        return 2740 + 790 * steps + tasks * (1.07 + 0.50 * steps) < 2630 + 540.0 * k + waves * (1.49 + 0.26 * k);
    return 2900 + 510 * steps + tasks * (1.65 + 0.41 * steps) < 2310 + 259.0 * k + waves * (1.02 + 0.079 * k);
}

// Orders per launch of the M-Basis step kernel (1: single orders, applied by a
// thread per coefficient instead of in LDS tiles) for m x n residuals, in a leaf
// of order ordL, when at most `most` fit LDS.
//
// Microseconds per order that a window of w costs over single orders, for the
// arithmetic of 32-bit words, 64-bit words below 2^62, and others:
//   launch   spared: the launches, first loads and last stores of w - 1 orders;
//   update   the step kernel's own update of the window's later coefficients, which
//            one workgroup does alone, per 10^4 products and order ahead;
//   round    the tiles' chains: a round of 32 kernel rows by 16 pivots;
//   rounds   those of the tiles that one compute unit takes one after another;
//   empty    256 tiles past the basis's length, launched since only the device
//            knows it;
//   words    spared: 10^6 coefficients read and written once per order;
//   terms    spared: 10^7 terms of kernel rows read from memory, not from LDS.
// Fitted (least squares, nonnegative) to 330 measurements of single orders and
// windows of 2 to 4: m from 4 to 256, n from 1 to m - 1 up to 128, orders 32 and
// 128, some of 512 and 1500.  The rule's choices take 1.008, 1.004 and 1.002 times
// the best ones' time on average.  Microseconds an order, single orders / windows
// of 4 (of 2 where marked): 32-bit words 64 x 32 at order 128 25.3 / 21.2, 192 x 24
// 41.5 / 54.9; 64-bit words 16 x 8 17.9 / 13.1, 64 x 48 73.3 / 92.2, 100 x 25 57.4 /
// 86.8, 128 x 1 17.8 / 27.5, 128 x 32 at order 1500 232 / 213 (2); others 64 x 32
// 70.5 / 90.4, 128 x 1 19.2 / 44.6.
enum BasisWords { BASIS_W32, BASIS_W64, BASIS_ANY };

inline int mbasis_window(BasisWords words, int m, int n, int64_t ordL, int most)
{
    struct Cost {
        double launch, update, round, rounds, empty, words, terms;
        double margin;  // a window has to win by this much
    };
    static const Cost kCost[3] = {{7.6, 0.40, 0.57, 0.0, 0.5, 3.2, 2.5, 0.6},
                                  {8.1, 2.1, 1.6, 0.51, 1.7, 5.8, 2.8, 0.7},
                                  {7.6, 5.4, 2.7, 1.3, 2.8, 17.0, 0.0, 1.5}};
    const Cost &c = kCost[words];
    const double rank = std::min(m, n), kernel = m - rank;  // of a generic residual
    const double pad = 16 * (double)(((int)rank + 15) / 16);
    const double chain = (((int)kernel + 31) / 32) * (pad / 16);
    // averages over the leaf: tiles of 12 coefficients of the basis (length order
    // n / m) and of the residual, and of what the basis could reach
    const double tiles = (m * std::max(1.0, (double)ordL * n / m / 24) + (double)n * ordL / 24) / 256;
    const double launched = (double)m * ordL / 24 / 256;
    const double spared = c.words * m * n * ordL / 1e6 + c.terms * n * ordL * kernel * pad / 1e7;
    int best = 1;
    double least = -c.margin;
    for (int w = 2; w <= most; ++w) {
        const double d = -c.launch * (1 - 1.0 / w) + c.update * kernel * rank * n * (w - 1) / 2 / 1e4 +
                         c.round * chain + c.rounds * chain * tiles + c.empty * launched / w - spared;
        if (d < least) {
            least = d;
            best = w;
        }
    }
    return best;
}

}  // namespace pmlg
