// mc_kernels.h - launch arguments shared by the host library and kernels.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

namespace mcd {

struct Grid;
struct J3Shape;

// A deposit: `val` to be added to word w of an estimator (J3, then esc).
struct alignas(8) LogEntry { unsigned w; float val; };
constexpr int kLogChunk = 2048;

// Per-launch arguments of the transport kernel.
struct RunArgs {
    int istar;                          // 1-based source index (random stream id)
    long long npackets;
    unsigned long long packet_offset;
    unsigned long long *next_packet;    // global refill counter (zeroed per launch)
    int *error;                         // first fail-stop code (atomicMax)
    unsigned long long *counts;         // 8 event counters, then walk passes and lanes, emission passes and lanes
    double *qphot;
    float deltaE;
    float px, py, pz;                   // source position [cm]
    int sx, sy, sz;                     // source cell (1-based)
    int star_cell;                      // its active index
    int emit_min;                       // emission pass when >= this many lanes wait
    int walk_steps;                     // walk passes between emission checks
    // the deposit log (log_kernel): chunks of kLogChunk entries, taken by
    // wavefronts from *log_next; when they run out a wavefront saves its
    // packets in `save` and ends, to go on in a launch with `resume` set
    LogEntry *log;
    unsigned *log_count;                // [log_chunks] entries of each chunk
    unsigned *log_next;
    unsigned log_chunks;
    uint32_t *save;                     // kSaveWords per wavefront
    int *suspended;
    int resume;
};

// Per-model arguments of a batched launch (device memory).  share[i] is the
// work of the models before model i (share[models]: of all).
struct BatchArgs {
    const Grid *G;                      // [models]
    const RunArgs *RA;                  // [models]
    const double *share;                // [models + 1]
    int models;
};

}  // namespace mcd

hipError_t mcd_launch_batch(const mcd::BatchArgs &B, size_t lds_bytes, int blocks, hipStream_t s);
// The transport kernels: one packet per lane, and one per lane with a pool of
// 32 packets per wavefront in LDS.  The pool kernel packs a packet's cell and
// bin and keeps 32-bit indices of the tables: it takes grids of at most 2047 x
// 2047 x 1023 cells, 65535 bins and 2^32 - 1 table words; other grids run the
// first whatever kernel is asked for, which there is no slower (2e7 packets,
// 240^3 octant of 320 bins, 4.4e9 words: 109 ms, and 115 with a pool of 64-bit
// indices; 200^3 of 300, 2.4e9 words: 108, and 110 with this pool).
// The log kernel is the pool kernel with the deposits written to the log of
// its RunArgs instead of added to the estimators.  The thin kernel is the
// first with shorter rings, for axes that leave no room for more.
enum { MCD_KERNEL_ONE = 1, MCD_KERNEL_POOL = 3, MCD_KERNEL_LOG = 4, MCD_KERNEL_THIN = 5 };
// the first kernel's tables and rings fit a CU's LDS
bool mcd_transport_fits(const mcd::Grid &G, int threads);
size_t mcd_save_words(int blocks, int threads);
bool mcd_pool_fits(const mcd::Grid &G);
size_t mcd_pool_lds(const mcd::Grid &G, int threads);
hipError_t mcd_launch_transport(const mcd::Grid &G, const mcd::RunArgs &RA, int blocks, int threads, int kernel,
                                hipStream_t s);
hipError_t mcd_densify(const float *compact, const int *active, const mcd::J3Shape &js, int nc1, int nbins,
                       float *dense, hipStream_t s);
hipError_t mcd_guides(const float *cdf, int rows, int nbins, unsigned short *guide, hipStream_t s);
hipError_t mcd_compact(const double *J3, const int *active, const mcd::J3Shape &js, int nc1, int nbins,
                       double *out, hipStream_t s);
hipError_t mcd_launch_replay(const mcd::Grid &G, int n, const float *pos, const float *dir,
                             const int *cell, int *cell_seq, float *ds_seq, int *seq_len,
                             int *status, int max_len, hipStream_t s);
