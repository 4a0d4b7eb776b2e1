// mc_deposit.h - the deposit log of a sweep and the two kernels that add it
// to the estimators.
//
// Memory-side FP64 atomics run at about 2e10 64-byte requests per second on
// the whole chip, and a sweep whose every segment was one (merged two to a
// request, where a packet stays in a brick) spent two thirds of its time
// waiting for them.  The log takes 8 bytes a deposit in the order they come
// (coalesced stores) instead; then each block of kBlock entries is sorted by
// the range of estimator words it adds to, in place, and each range is summed
// in LDS in FP64.
#pragma once
#include <hip/hip_runtime.h>
#include <stddef.h>
#include <stdint.h>

#include "mc_kernels.h"

namespace mcl {

constexpr int kBlock = 16384;            // entries sorted together
constexpr int kBlockChunks = kBlock / mcd::kLogChunk;
constexpr int kGroup = 16;               // blocks whose run tables lie together
constexpr int kRange = 16384;            // words summed by one workgroup (128 KB of LDS)
constexpr int kMaxBins = 7936;           // with half a block's entries, 4 bytes each, they fill half the LDS of a CU
constexpr int kMaxShift = 16;

// `words` estimator words in at most kMaxBins bins of 2^shift; a bin is one
// range of kRange words, or up to four, each of which reads all of it.  With
// eight the log loses to atomics: H+He on 100^3 cells, 6e8 words, 2e8 packets,
// 220 ms against 199; with four it gains still: 88^3, 4.1e8 words, 2e7
// packets, 15.5 ms against 20.0; with two, 64^3, 1.6e8 words, 13.1 against 22.3.
struct Shape {
    unsigned words;
    int shift, bins;
};

struct Log {
    mcd::LogEntry *entries;              // [chunks * kLogChunk]
    unsigned *count;                     // [chunks] (what the sweep left in each)
    const unsigned *next;                // chunks the sweep asked for
    unsigned chunks;
    unsigned short *runs;                // [groups][bins + 1][kGroup]: where a block's run of a bin starts
    // the plan: per bin its entries and the slices it is read in (several
    // workgroups sum a bin with many entries); the work items, bin | range of
    // the bin << 13 | slice << 16; their number
    unsigned long long *total;           // [kMaxBins]
    unsigned *slices, *items, *n_items;
};
constexpr int kParts = 1024;             // a slice is at most about 1/kParts of the log
constexpr int kMaxItems = (kMaxBins + kParts) << (kMaxShift - 14);
constexpr size_t kPlanWords = 3 * kMaxBins + kMaxItems + 1;

// The shape of `words` words, or bins = 0 if the log does not take that many.
Shape shape(size_t words);
size_t run_entries(unsigned chunks, const Shape &s);

}  // namespace mcl

// Sort the log's blocks, then add it: words below j_words to J, the others to
// esc.  Both kernels read the number of chunks in use from the device.
hipError_t mcl_sort(const mcl::Log &L, const mcl::Shape &s, int cus, hipStream_t st);
hipError_t mcl_reduce(const mcl::Log &L, const mcl::Shape &s, double *J, double *esc, unsigned j_words, int cus,
                      hipStream_t st);
