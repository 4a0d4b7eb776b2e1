// mc_log_shape.h - how the estimators' words are divided into the ranges of
// the deposit log (mc_deposit.h), and which sweeps it is for.
#pragma once
#include <stddef.h>

namespace mcl {

constexpr int kRange = 16384;            // words summed by one workgroup (128 KB of LDS)
constexpr int kMaxBins = 7936;           // with half a block's entries, 4 bytes each, they fill half the LDS of a CU
constexpr int kMaxShift = 16;

// `words` estimator words in at most kMaxBins bins of 2^shift; a bin is one
// range of kRange words, or up to four, each of which reads all of it.  With
// eight the log gains nothing any more: H+He octants on the cold start's
// tables, 2e7 packets, logged and with atomics: 64^3 cells (1.6e8 words, two
// ranges to a bin) 17.4, 30.0 ms, 88^3 (4.1e8, four) 31.9, 37.1, 100^3 (6e8,
// eight) 46.0, 39.3; a full 100^3 grid 24.4, 24.9.
struct Shape {
    unsigned words;
    int shift, bins;
};

// The shape of `words` words, or bins = 0 if the log does not take that many.
inline Shape shape(size_t words)
{
    Shape s = { 0, 14, 0 };
    if (words == 0 || words > (size_t)kMaxBins << kMaxShift) return s;
    while (((words - 1) >> s.shift) + 1 > (size_t)kMaxBins) ++s.shift;
    s.words = (unsigned)words;
    s.bins = (int)(((words - 1) >> s.shift) + 1);
    return s;
}

// The fewest deposits the log is for.  Sorting and planning have a cost of
// their own, and so has every range that a deposit falls in (128 KB of LDS
// cleared and added).  Deposits where both sides take the same, by words
// (octants and full grids of 11^3 to 90^3 cells, H+He, seven elements, dust):
// 1e6 2e6-3e6, 5e6 4e6-1e7, 2e7 6e6-3e7, 6e7 2e7, 9e7 1e7-4e7, 1.3e8 3e7, 1.6e8
// 4e7, 2.2e8 4e7-5e7, 4.1e8 1e8.  On either side of the line, logged and with
// atomics: 45^3 octant of 6.3e7 words, 4e6 deposits 0.52, 0.43 ms, 3.2e7 1.24,
// 1.52; 88^3 octant of 4.1e8 words, 4e6 1.05, 0.62, 3.2e7 2.35, 1.68, 1e8 3.66,
// 3.70.
inline double least_deposits(const Shape &s) { return 3.e6 + 0.2 * s.words; }

}  // namespace mcl
