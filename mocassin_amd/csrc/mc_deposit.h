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
#include "mc_log_shape.h"

namespace mcl {

constexpr int kBlock = 16384;            // entries sorted together
constexpr int kBlockChunks = kBlock / mcd::kLogChunk;
constexpr int kGroup = 16;               // blocks whose run tables lie together
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

size_t run_entries(unsigned chunks, const Shape &s);

}  // namespace mcl

// Sort the log's blocks, then add it: words below j_words to J, the others to
// esc.  Both kernels read the number of chunks in use from the device.
hipError_t mcl_sort(const mcl::Log &L, const mcl::Shape &s, int cus, hipStream_t st);
hipError_t mcl_reduce(const mcl::Log &L, const mcl::Shape &s, double *J, double *esc, unsigned j_words, int cus,
                      hipStream_t st);
