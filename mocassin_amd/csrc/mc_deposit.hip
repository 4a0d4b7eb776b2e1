// mc_deposit.hip - sort and reduce of the deposit log (mc_deposit.h).
#include "mc_deposit.h"

namespace mcl {

constexpr int kThreads = 1024;
constexpr int kWaves = kThreads / 64;
constexpr int kPer = kBlock / kThreads;                       // entries a thread
constexpr int kBinsPer = (kMaxBins + kThreads - 1) / kThreads; // bins a thread

// In LDS: half of each of a block's entries (first their words, then their
// values) in sorted order, the bins' counts (then starts), two to a word, and
// the wavefront sums of the scan.  A place and a bin more take what is no
// entry (a branch each would cost registers).
constexpr size_t kSortLds = sizeof(unsigned) * (kBlock + 4 + kMaxBins / 2 + 4 + kWaves);
static_assert(kSortLds <= 80 * 1024, "sort: two workgroups fill a CU's LDS");
static_assert(kMaxBins % kBinsPer == 0 && kBinsPer == 8, "a thread scans four words of counts");

__device__ __forceinline__ unsigned chunks_used(const Log &L) { return min(*L.next, L.chunks); }
__device__ __forceinline__ unsigned blocks_of(unsigned chunks) { return (chunks + kBlockChunks - 1) / kBlockChunks; }

// One workgroup sorts a block of 16384 entries by bin, in place: a counting
// sort whose ranks come from LDS atomics with a result.  HBM bound: 8 bytes
// read and written per entry.  Workgroup i runs on XCD i mod 8; the 16 blocks
// of a group go to 16 workgroups of one XCD at the same time, so that their
// run tables, 32 bytes a bin, meet in its L2.
// A workgroup goes through phases (load, rank, scan, place, store) of which
// only the first and the last use the HBM.  One workgroup a CU, entries whole
// in 128 KB of LDS and counts in 32 KB, ran at 2.7 TB/s (a copy runs at 4.8).
// Entries placed half by half through 64 KB and counts of 16 bits let two
// share a CU, one in the HBM while the other is in its LDS: 45^3 octant, a full
// log, 3.9 -> 2.5 ms; 60^3 cells with dust, 3.2 -> 2.0 ms (4.2 TB/s).  With 32 wavefronts a CU there are 64 registers: the entries
// take 32, packed ranks and the bins' counts 8 each, and what the compiler
// would keep beside them is made again where it is used.
__global__ void __launch_bounds__(kThreads) __attribute__((amdgpu_waves_per_eu(8)))
sort_kernel(Log L, Shape s)
{
    extern __shared__ __align__(16) unsigned char dyn[];
    unsigned *half = reinterpret_cast<unsigned *>(dyn), *hist = half + kBlock + 4, *wsum = hist + kMaxBins / 2 + 4;
    const auto start = [&](unsigned bin) { return hist[bin >> 1] >> (bin & 1) * 16 & 0xffffu; };
    unsigned t = threadIdx.x;
    const unsigned lane = t & 63, wave = __builtin_amdgcn_readfirstlane((int)(t >> 6));
    const unsigned used = __builtin_amdgcn_readfirstlane((int)chunks_used(L)), blocks = blocks_of(used);
    const unsigned groups = (blocks + kGroup - 1) / kGroup;
    const unsigned x = blockIdx.x % 8, j = blockIdx.x / 8, teams = gridDim.x / (8 * kGroup);
    unsigned mine[kBinsPer] = {};                   // entries of this thread's bins in the workgroup's blocks
    const unsigned b0 = t * kBinsPer, nbins = (unsigned)s.bins;
    const unsigned k = j % kGroup;
    for (unsigned g = (j / kGroup) * 8 + x; g < groups; g += teams * 8) {
        unsigned b = g * kGroup + k;
        asm("" : "+v"(t), "+s"(b));                 // addresses are made in place: kept, they spill
        mcd::LogEntry *at = L.entries + (size_t)b * kBlock;
        unsigned short *run = L.runs + (size_t)g * (nbins + 1) * kGroup + k;
        if (b >= blocks) {                          // the last group's missing blocks: empty runs
            for (unsigned i = t; i <= nbins; i += kThreads) run[i * kGroup] = 0;
            continue;
        }
        // the block's entries, 0xffffffff in place of those its chunks lack
        // (what is beyond a chunk's count is read all the same, and the first row
        // for a chunk that was not asked for)
        constexpr unsigned rows = mcd::kLogChunk / kThreads;           // thread rows of a chunk
        const unsigned c0 = b * kBlockChunks, counts = lane < kBlockChunks && c0 + lane < used ? L.count[c0 + lane] : 0;
        mcd::LogEntry e[kPer];
#pragma unroll
        for (unsigned i = 0; i < kPer; ++i)
            e[i] = (at + (c0 + i / rows < used ? i : 0) * kThreads)[t];
        for (unsigned i = t; i < kMaxBins / 2; i += kThreads) hist[i] = 0;
        if (t == 0) hist[kMaxBins / 2] = 0;
        __syncthreads();
        unsigned word[kPer], val[kPer], rank[kPer / 2];       // two ranks to a word
#pragma unroll
        for (int i = 0; i < kPer; ++i) {
            // out of the pairs that the loads took, which stay pairs otherwise
            asm("v_mov_b32 %0, %2\n\tv_mov_b32 %1, %3" : "=&v"(word[i]), "=&v"(val[i]) : "v"(e[i].w), "v"(e[i].val));
            if (i % rows * kThreads + t >= (unsigned)__builtin_amdgcn_readlane((int)counts, i / rows)) word[i] = 0xffffffffu;
            const unsigned bin = min(word[i] >> s.shift, (unsigned)kMaxBins), up = (bin & 1) * 16;
            const unsigned r = atomicAdd(&hist[bin >> 1], 1u << up) >> up & 0xffffu;
            rank[i / 2] = i & 1 ? rank[i / 2] | r << 16 : r;
            asm("" : "+v"(rank[i / 2]));            // packed here
            if (i % 4 == 3) __builtin_amdgcn_sched_barrier(0);          // registers
        }
        __syncthreads();
        // exclusive scan of the counts, kBinsPer bins a thread
        unsigned n[kBinsPer / 2] = {}, sum = 0;
        if (b0 < kMaxBins) {
            const uint4 v = reinterpret_cast<const uint4 *>(hist)[t];
            n[0] = v.x; n[1] = v.y; n[2] = v.z; n[3] = v.w;
        }
#pragma unroll
        for (int i = 0; i < kBinsPer / 2; ++i) {
            mine[2 * i] += n[i] & 0xffffu;
            mine[2 * i + 1] += n[i] >> 16;
            asm("" : "+v"(mine[2 * i]), "+v"(mine[2 * i + 1]));
            sum += (n[i] & 0xffffu) + (n[i] >> 16);
        }
        const unsigned own = sum;
#pragma unroll
        for (int o = 1; o < 64; o <<= 1) {
            const unsigned v = __shfl_up(sum, o);
            if (lane >= (unsigned)o) sum += v;
        }
        if (lane == 63) wsum[wave] = sum;
        __syncthreads();
        // lanes 0 to 15: the sums up to each wavefront's end
        unsigned ends = lane < kWaves ? wsum[lane] : 0;
#pragma unroll
        for (int o = 1; o < kWaves; o <<= 1) {
            const unsigned v = __shfl_up(ends, o);
            if (lane >= (unsigned)o) ends += v;
        }
        const unsigned total = __builtin_amdgcn_readlane((int)ends, kWaves - 1);
        unsigned before = sum - own + (wave ? __builtin_amdgcn_readlane((int)ends, wave - 1) : 0);
        if (b0 < kMaxBins) {
#pragma unroll
            for (int i = 0; i < kBinsPer / 2; ++i) {
                const unsigned mid = before + (n[i] & 0xffffu), next = mid + (n[i] >> 16);
                n[i] = before | mid << 16;
                before = next;
            }
            reinterpret_cast<uint4 *>(hist)[t] = make_uint4(n[0], n[1], n[2], n[3]);
        }
        __syncthreads();
        for (unsigned i = t; i <= nbins; i += kThreads)
            run[i * kGroup] = (unsigned short)(i < nbins ? start(i) : total);
        // the words into their places, and into registers again in order
#pragma unroll
        for (int i = 0; i < kPer; ++i) {
            asm("" : "+v"(word[i]));                // its bin again: kept from the ranks, it would spill
            const unsigned own = start(min(word[i] >> s.shift, (unsigned)kMaxBins)) + (rank[i / 2] >> 16 * (i & 1) & 0xffffu);
            const unsigned p = word[i] != 0xffffffffu ? own : kBlock;
            rank[i / 2] = i & 1 ? (rank[i / 2] & 0xffffu) | p << 16 : (rank[i / 2] & ~0xffffu) | p;
            asm("" : "+v"(rank[i / 2]));
            half[p] = word[i];
            if (i % 4 == 3) __builtin_amdgcn_sched_barrier(0);          // registers
        }
        __syncthreads();
#pragma unroll
        for (int i = 0; i < kPer; ++i) word[i] = half[i * kThreads + t];
        __syncthreads();
        // the values
#pragma unroll
        for (int i = 0; i < kPer; ++i) {
            const unsigned p = rank[i / 2] >> 16 * (i & 1) & 0xffffu;
            half[p] = val[i];
        }
        __syncthreads();
#pragma unroll
        for (int i = 0; i < kPer; ++i) {
            if (i * kThreads + t < total)
                (at + i * kThreads)[t] = { word[i], __uint_as_float(half[i * kThreads + t]) };
        }
    }
#pragma unroll
    for (int i = 0; i < kBinsPer; ++i) {
        asm("" : "+v"(mine[i]));                    // 32 bits until here
        if (mine[i]) atomicAdd(&L.total[b0 + i], (unsigned long long)mine[i]);
    }
}

// Work items: a bin's ranges, each in slices of at most 1/kParts of the log,
// so that the bins next to the source, which a large part of all segments
// falls in, do not hold up the end.
__global__ void __launch_bounds__(kThreads) plan_kernel(Log L, Shape s)
{
    __shared__ unsigned long long all;
    __shared__ unsigned scan[kThreads];
    const int t = threadIdx.x;
    const unsigned subs = 1u << (s.shift - 14);
    static_assert(kMaxBins <= 1 << 13 && kMaxShift - 14 <= 3, "packed work items");
    if (t == 0) all = 0;
    __syncthreads();
    unsigned long long n[kBinsPer], sum = 0;
#pragma unroll
    for (int i = 0; i < kBinsPer; ++i) {
        n[i] = t * kBinsPer + i < s.bins ? L.total[t * kBinsPer + i] : 0;
        sum += n[i];
    }
    if (sum) atomicAdd(&all, sum);
    __syncthreads();
    // at most kParts slices more than bins
    const unsigned long long most = all / kParts + 1 > 16384 ? all / kParts + 1 : 16384;
    unsigned k[kBinsPer], items = 0;
#pragma unroll
    for (int i = 0; i < kBinsPer; ++i) {
        k[i] = (unsigned)((n[i] + most - 1) / most);
        items += k[i] * subs;
    }
    scan[t] = items;
    __syncthreads();
    for (int o = 1; o < kThreads; o <<= 1) {
        const unsigned v = t >= o ? scan[t - o] : 0;
        __syncthreads();
        scan[t] += v;
        __syncthreads();
    }
    unsigned at = scan[t] - items;
    if (t == kThreads - 1) *L.n_items = scan[t];
#pragma unroll
    for (int i = 0; i < kBinsPer; ++i) {
        const unsigned bin = t * kBinsPer + i;
        if (bin >= (unsigned)s.bins) continue;
        L.slices[bin] = k[i];
        for (unsigned q = 0; q < k[i]; ++q)
            for (unsigned r = 0; r < subs; ++r) L.items[at++] = bin | r << 13 | q << 16;
    }
}

// Where word w is summed: the 64 points of a tile row turned by their bin, so
// that one cell's words of all frequencies (the source's cell has a share of
// every packet) do not lie in one LDS bank.
__device__ __forceinline__ unsigned place(unsigned w)
{
    return (w & (kRange - 64)) | ((w + (w >> 6)) & 63u);
}

// acc[w] += v of the lanes with `has`.  Lanes that share a word add one after
// another, some 64 cycles each, so in a range with many entries up to two
// words that four lanes or more share are summed across the lanes first.
__device__ __forceinline__ void add(double *acc, bool has, unsigned w, double v, bool hot, int lane)
{
    for (int k = 0; hot && k < 2; ++k) {
        const uint64_t m = __ballot(has);
        if (!m) return;
        const int leader = __ffsll((unsigned long long)m) - 1;
        const unsigned wl = (unsigned)__builtin_amdgcn_readlane((int)w, leader);
        const bool same = has && w == wl;
        const uint64_t ms = __ballot(same);
        if (__popcll(ms) < 4) break;
        double sum = same ? v : 0.0;
        for (int o = 32; o >= 1; o >>= 1) sum += __shfl_xor(sum, o);
        if (lane == leader) unsafeAtomicAdd(&acc[place(w)], sum);
        has = has && !same;
    }
    if (has) unsafeAtomicAdd(&acc[place(w)], v);
}

// A work item is a range of kRange words and a slice of its bin (the same
// part of every block's run): one workgroup reads the slice and adds the
// entries of its words in LDS, then adds the sums to the estimator (atomics
// where slices of a range meet there, 8 words to a request).  32 consecutive
// items go to the CUs of one XCD, which read neighbouring runs out of the
// same lines.  A run has kBlock / bins entries on average, a few, so a
// wavefront lays the runs of 64 blocks end to end and reads them 64 entries
// at a time (marks in LDS of where runs begin give each lane its run), kAhead
// loads in flight.
constexpr int kAhead = 4;
struct Reader { unsigned mark[64 * kAhead]; int delta[64]; };
constexpr size_t kReduceLds = sizeof(double) * kRange + sizeof(Reader) * kWaves;

// set bits of m below this lane
__device__ __forceinline__ int rank_below(uint64_t m)
{
    return (int)__builtin_amdgcn_mbcnt_hi((unsigned)(m >> 32), __builtin_amdgcn_mbcnt_lo((unsigned)m, 0u));
}

// orders a wavefront's LDS accesses (the LDS serves them in order)
__device__ __forceinline__ void wave_order()
{
    __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
    __builtin_amdgcn_wave_barrier();
}

__global__ void __launch_bounds__(kThreads) reduce_kernel(Log L, Shape s, double *J, double *esc, unsigned j_words)
{
    extern __shared__ __align__(16) double acc[];
    const int t = threadIdx.x, lane = t & 63, wave = t >> 6;
    static_assert(kRange == 1 << 14, "a range is 2^14 words");
    Reader &R = reinterpret_cast<Reader *>(acc + kRange)[wave];
    unsigned *mark = R.mark;
    int *delta = R.delta;
    const unsigned blocks = blocks_of(chunks_used(L)), groups = (blocks + kGroup - 1) / kGroup;
    const unsigned items = *L.n_items;
    const unsigned x = blockIdx.x % 8, per = gridDim.x / 8;
    // with fewer than 64 blocks a wavefront, several share them, a part each
    const unsigned stripes = (groups + 3) / 4;
    const unsigned parts = stripes >= (unsigned)kWaves ? 1 : kWaves / (stripes ? stripes : 1);
    const unsigned part = (unsigned)wave % parts, first = (unsigned)wave / parts, step = kWaves / parts;
    for (int i = t; i < kRange; i += kThreads) acc[i] = 0.0;
    __syncthreads();
    for (unsigned y = blockIdx.x / 8; (y / per * 8 + x) * per < items; y += per) {
        const unsigned item = (y / per * 8 + x) * per + y % per;
        if (item >= items) continue;
        const unsigned what = L.items[item];
        const unsigned bin = what & 0x1fffu, sub = what >> 13 & 7u, slices = L.slices[bin];
        const size_t w0 = ((size_t)bin << s.shift) + (size_t)sub * kRange;
        if (w0 >= s.words) continue;
        const unsigned range = (unsigned)(w0 >> 14);
        const bool hot = slices > 1;
        const unsigned cut = (what >> 16) * parts + part, cuts = slices * parts;
        // start | end << 16 of this item's part of the run in this lane's block
        const auto descriptor = [&](unsigned g) -> unsigned {
            if (g >= groups) return 0;
            const unsigned short *r = L.runs + ((size_t)g * (s.bins + 1) + bin) * kGroup + (lane & 15);
            const unsigned a = r[0], n = r[kGroup] - a;
            return cuts == 1 ? a | (a + n) << 16 : (a + n * cut / cuts) | (a + n * (cut + 1) / cuts) << 16;
        };
        unsigned d = descriptor(4 * first + (lane >> 4));
        for (unsigned g0 = 4 * first; g0 < groups && first < stripes; g0 += 4 * step) {
            const unsigned now = d;
            d = descriptor(g0 + 4 * step + (lane >> 4));
            if (!__any((now & 0xffffu) != now >> 16)) continue;
            // the runs end to end: run r begins at position p
            const int n = (int)(now >> 16) - (int)(now & 0xffffu);
            int p = n;
#pragma unroll
            for (int o = 1; o < 64; o <<= 1) {
                const int v = __shfl_up(p, o);
                if (lane >= o) p += v;
            }
            const int all = __builtin_amdgcn_readlane(p, 63);
            p -= n;
            const uint64_t some = __ballot(n > 0);
            // of the non-empty runs in order: entry index less position
            if (n > 0) delta[rank_below(some)] = (int)(lane * kBlock + (now & 0xffffu)) - p;
            const mcd::LogEntry *from = L.entries + (size_t)g0 * kGroup * kBlock;
            int begun = 0;                             // runs that begin before this batch of positions
            for (int f0 = 0; f0 < all; f0 += 64 * kAhead) {
#pragma unroll
                for (int j = 0; j < kAhead; ++j) mark[64 * j + lane] = 0;
                wave_order();
                if (n > 0 && p >= f0 && p < f0 + 64 * kAhead) mark[p - f0] = 1;
                wave_order();
                mcd::LogEntry e[kAhead];
#pragma unroll
                for (int j = 0; j < kAhead; ++j) {
                    const unsigned own = mark[64 * j + lane];
                    const uint64_t m = __ballot(own != 0);
                    const int r = begun + rank_below(m) + (int)own - 1;
                    begun += __popcll(m);
                    const int f = f0 + 64 * j + lane;
                    e[j].w = 0xffffffffu;
                    if (f < all) e[j] = from[delta[r] + f];
                }
#pragma unroll
                for (int j = 0; j < kAhead; ++j) add(acc, e[j].w >> 14 == range, e[j].w, (double)e[j].val, hot, lane);
                wave_order();
            }
        }
        __syncthreads();
        for (int i = t; i < kRange; i += kThreads) {
            const size_t w = w0 + i;
            const unsigned at = place((unsigned)w);
            const double v = acc[at];
            acc[at] = 0.0;
            if (v == 0.0) continue;
            double *to = w < j_words ? &J[w] : &esc[w - j_words];
            if (slices > 1) unsafeAtomicAdd(to, v);
            else *to += v;
        }
        __syncthreads();
    }
}

size_t run_entries(unsigned chunks, const Shape &s)
{
    const size_t blocks = (chunks + kBlockChunks - 1) / kBlockChunks;
    return (blocks + kGroup - 1) / kGroup * kGroup * (size_t)(s.bins + 1);
}

}  // namespace mcl

static hipError_t lds_of(const void *f, size_t bytes)
{
    return hipFuncSetAttribute(f, hipFuncAttributeMaxDynamicSharedMemorySize, (int)bytes);
}

// whole teams of an XCD
static unsigned grid_of(int cus, int per) { return (unsigned)((cus + per - 1) / per * per); }

hipError_t mcl_sort(const mcl::Log &L, const mcl::Shape &s, int cus, hipStream_t st)
{
    const hipError_t e = lds_of((const void *)mcl::sort_kernel, mcl::kSortLds);
    if (e != hipSuccess) return e;
    hipLaunchKernelGGL(mcl::sort_kernel, dim3(grid_of(2 * cus, 8 * mcl::kGroup)), dim3(mcl::kThreads), mcl::kSortLds, st, L, s);
    return hipGetLastError();
}

hipError_t mcl_reduce(const mcl::Log &L, const mcl::Shape &s, double *J, double *esc, unsigned j_words, int cus,
                      hipStream_t st)
{
    const size_t lds = mcl::kReduceLds;
    const hipError_t e = lds_of((const void *)mcl::reduce_kernel, lds);
    if (e != hipSuccess) return e;
    hipLaunchKernelGGL(mcl::plan_kernel, dim3(1), dim3(mcl::kThreads), 0, st, L, s);
    hipLaunchKernelGGL(mcl::reduce_kernel, dim3(grid_of(cus, 8)), dim3(mcl::kThreads), lds, st, L, s, J, esc, j_words);
    return hipGetLastError();
}
