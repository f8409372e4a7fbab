// Rules on sizes that pick between exact variants of one computation.  Host code,
// plain integers in and out, so that they can be tested without a device.
#pragma once

#include <stdint.h>

#include <algorithm>

namespace pmlg {

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
