// mc_transport.hip - persistent packet-transport kernels and geometry replay
// kernel for MI355X (gfx950).
//
// Transport: wavefronts take packets from a counter in stocks.  Packet
// events are split in two classes and scheduled per wavefront so that SIMD
// lanes stay coherent:
//   walk      one cell segment of pathSegment (three reciprocal products, one
//             opacity gather, one deposit): the common event;
//   emission  creation of a stellar packet or re-emission of an absorbed one
//             (Philox draws, CDF search, direction, optical-depth draw):
//             about ten times the instructions of a walk step.
// Four kernels share that code.  log_kernel runs large sweeps: a pool of
// packets per wavefront in LDS keeps the lanes walking, and deposits go to a
// log that mc_deposit.hip sums by range.  pool_kernel is the same with FP64
// atomics (small sweeps, crossing counts); transport_kernel keeps one packet
// per lane (any lattice); batch_kernel is the pool over several models.  The
// axes' walls and word offsets live in LDS.  J_nu and the opacity tables are
// stored in 2x2x2 bricks of 4x4x4 tiles (mc_device.h).  Where deposits are
// atomics each lane queues them in a ring in LDS, and a full ring flushes
// every lane's ring, one packet's consecutive updates to an instruction, so
// that adds sharing a 64-byte line travel as one request.
//
// What bounds them: an FP64 atomic add goes to the memory side as one 64-byte
// request, 2e10 of them a second, which was 2/3 of a sweep's time; a logged
// deposit is 8 bytes written and read three times.  The walk itself is bound
// by its instructions at 16 and more wavefronts a CU.  One sweep of 1e8
// packets on a 45^3 octant of 800 bins (1.8e9 deposits): 64.8 ms before (the
// pool with atomics and divisions), 39.0 now (walk and log 22.6, sort 8.4,
// sums 7.8); 4e7 packets in dust and gas 60^3: 67.4 ms before, 42.0 now; 8
// models of 20^3 to 50^3 cells, 2.8e5 to 2e6 packets, in one launch: 5.9-6.6 ms.
#include <algorithm>

#include "mc_device.h"
#include "mc_kernels.h"

#pragma clang fp contract(off)

namespace mcd {

// LDS of a staged grid: parts | walls.  The tables of an axis follow those
// of the one before.
template <bool WIDE>
__device__ __forceinline__ void stage_axes(const Grid &G, float *lds, Axes &A)
{
    const int n3[3] = { G.nx, G.ny, G.nz };
    const int na = G.nx + G.ny + G.nz;
    AxisPart *parts = reinterpret_cast<AxisPart *>(lds);
    float *walls = lds + 2 * na;
    for (int k = 0, o = 0; k < 3; o += n3[k], ++k) {
        const float *ax = G.axis + o, *mid = G.mid + o - k;
        const int n = n3[k];
        for (int i = threadIdx.x; i <= n; i += blockDim.x) {
            walls[o + k + i] = i == 0 ? ax[0] : i < n ? mid[i - 1] : ax[n - 1];
            if (i < n) parts[o + i] = AxisPart{ G.dfac[o + i], axis_word<WIDE>(G, k, i) };
        }
    }
    __syncthreads();
    A.wx = walls; A.wy = walls + G.nx + 1; A.wz = walls + G.nx + G.ny + 2;
    A.px = parts; A.py = parts + G.nx; A.pz = parts + G.nx + G.ny;
}

__host__ __device__ inline size_t lds_floats(int nx, int ny, int nz)
{
    return (size_t)3 * (nx + ny + nz) + 3;
}

// A launch's grid and run arguments in memory, at wavefront-uniform
// addresses of the constant address space (scalar loads; they do not change
// in a launch).  The walk keeps the few fields it needs in scalar registers;
// everything else is loaded by the pass that uses it: kept in registers over
// the whole launch the arguments spilled.
struct Args {
    uint64_t g, r;          // addresses of the Grid and the RunArgs
};

template <class T>
__device__ __forceinline__ T scalar_copy(uint64_t at)
{
    asm volatile("" : "+s"(at));               // a load of its own, not one hoisted to the top of the kernel
    return *(const T *)(const __attribute__((address_space(4))) T *)at;
}

// lanes below this one in m
__device__ __forceinline__ int lane_rank(uint64_t m, int)
{
    return (int)__builtin_amdgcn_mbcnt_hi((unsigned)(m >> 32), __builtin_amdgcn_mbcnt_lo((unsigned)m, 0u));
}

// Orders the wavefront's LDS accesses on either side (the compiler may not
// move them across; the LDS serves one wavefront's instructions in order).
__device__ __forceinline__ void wave_lds_order()
{
    __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
    __builtin_amdgcn_wave_barrier();
}

// ------------------------------------------------ J update queue (per wave)
// Each lane keeps its last D updates (word of J3, value) in a ring of its own
// at the start of the wavefront's dynamic LDS, entry k of lane L at
// L * (D + 1) + k (rows padded by one entry against bank conflicts); wide
// tables (2^32 words or more) keep the point there and the bin in a second
// array behind.  When a lane's ring is full the wavefront flushes every ring,
// lane-major: atomic instruction j carries the rings of lanes (64 / D) j ..
// (64 / D)(j + 1) - 1.  Adds of one instruction that fall in one 64-byte line
// travel to memory as one request, and with J3's 2x2x2 bricks a packet's next
// segment stays in the line after half of its steps, so keeping a packet's
// updates in one instruction turns those pairs into single requests.
struct JEntry { unsigned w; float val; };
template <int D, bool WIDE>
struct JRing {
    static_assert(D == 4 || D == 8, "rings of 4 or 8 updates");
    static constexpr int kRow = D + 1;
    static constexpr int kEntries = 64 * kRow;
    static constexpr int kFloats = kEntries * 2 + (WIDE ? kEntries / 2 : 0);
};
constexpr int kJDepth = 8;

struct JQ {
    JEntry *e;
    unsigned short *nu;   // wide tables only
    int n;                // this lane's queued updates
};

template <int D, bool WIDE>
__device__ __forceinline__ JQ jq_at(float *lds, int wave)
{
    float *b = lds + (size_t)wave * JRing<D, WIDE>::kFloats;
    JQ Q;
    Q.e = reinterpret_cast<JEntry *>(b);
    Q.nu = reinterpret_cast<unsigned short *>(b + 2 * JRing<D, WIDE>::kEntries);
    Q.n = 0;
    return Q;
}

// the J3 point of a word (crossing counts)
template <bool WIDE>
__device__ __forceinline__ unsigned point_of(const Grid &G, unsigned w)
{
    return WIDE ? w : w / ((unsigned)G.nbins * kJTile) * kJTile + w % kJTile;
}

// Crossing counts.  Adds to one line are served one after another, and every
// packet crosses the source's surroundings: so a wavefront counts the points of
// the source's tile in LDS, in the words that pad its rings (point i in lane
// i's; the tile beside the count), and adds them when it ends.  3e6 packets, 5^3
// to 30^3 cells: 13.7 to 23.3 ms with an add for each crossing, 1.8 to 9.9 now.
// The counts are a loop of their own: within the flush's they cost sweeps
// without them up to 8 %.
template <int D, bool WIDE>
__device__ __forceinline__ JEntry &near_count(const JQ &Q, unsigned point)
{
    return Q.e[point % kJTile * JRing<D, WIDE>::kRow + D];
}
template <int D, bool WIDE>
__device__ __forceinline__ void crossings_open(const Grid &G, const RunArgs &RA, const JQ &Q, int lane)
{
    const unsigned tile = j3_point(G.js, RA.sx - 1, RA.sy - 1, RA.sz - 1) / kJTile;
    near_count<D, WIDE>(Q, (unsigned)lane) = JEntry{ 0u, __uint_as_float(tile) };
    wave_lds_order();
}
// the lane's own queued updates
template <int D, bool WIDE>
__device__ __forceinline__ void count_crossings(const Grid &G, const JQ &Q, int lane)
{
    const unsigned tile = __float_as_uint(near_count<D, WIDE>(Q, 0).val);
    for (int k = 0; k < Q.n; ++k) {
        const unsigned point = point_of<WIDE>(G, Q.e[lane * JRing<D, WIDE>::kRow + k].w);
        atomicAdd(point / kJTile == tile ? &near_count<D, WIDE>(Q, point).w : &G.cross[point], 1u);
    }
}
template <int D, bool WIDE>
__device__ __forceinline__ void crossings_close(const Grid &G, const JQ &Q, int lane)
{
    wave_lds_order();
    const JEntry e = near_count<D, WIDE>(Q, (unsigned)lane);
    if (e.w) atomicAdd(&G.cross[(size_t)__float_as_uint(e.val) * kJTile + lane], e.w);
}

// every queued update: instruction j takes entry lane % D of lane
// (64 / D) j + lane / D's ring
template <int D, bool WIDE>
__device__ __forceinline__ void jq_flush(const Grid &G, JQ &Q, int lane)
{
    constexpr int per = 64 / D;                       // rings per instruction
    __builtin_amdgcn_wave_barrier();
    const int k = lane % D;
    for (int j = 0; j < D; ++j) {
        const int owner = per * j + lane / D;
        const int cnt = __shfl(Q.n, owner);
        if (k < cnt) {
            const int slot = owner * JRing<D, WIDE>::kRow + k;
            const JEntry e = Q.e[slot];
            const unsigned nu0 = WIDE ? Q.nu[slot] : 0;
            unsafeAtomicAdd(&G.J3[Word<WIDE>::index(G, e.w, nu0)], (double)e.val);
        }
    }
    __builtin_amdgcn_wave_barrier();
    if (G.flags & F_CROSS) count_crossings<D, WIDE>(G, Q, lane);
    Q.n = 0;
}

// the J update of each lane with `has` (path length times deltaE over dV,
// photon_mod.f90:1563-1574, 1822-1833), flushed when a lane's ring is full
template <int D, bool WIDE>
__device__ __forceinline__ void jq_push(const Grid &G, JQ &Q, bool has, unsigned w, unsigned nu0, float v, int lane)
{
    if (has) {
        const int slot = lane * JRing<D, WIDE>::kRow + Q.n;
        Q.e[slot] = JEntry{ w, v };
        if (WIDE) Q.nu[slot] = (unsigned short)nu0;
        Q.n += 1;
    }
    if (__any(Q.n == D)) jq_flush<D, WIDE>(G, Q, lane);
}

// ------------------------------------------------------------ replay kernel
__global__ void __launch_bounds__(256) walk_replay_kernel(Grid G, int n, const float *pos,
                                                          const float *dir, const int *cell,
                                                          int *cell_seq, float *ds_seq, int *seq_len,
                                                          int *status, int max_len)
{
    extern __shared__ float lds[];
    Axes A;
    stage_axes<true>(G, lds, A);
    int p = blockIdx.x * blockDim.x + threadIdx.x;
    if (p >= n) return;
    Walker W;
    W.rx = pos[3 * p]; W.ry = pos[3 * p + 1]; W.rz = pos[3 * p + 2];
    W.vx = dir[3 * p]; W.vy = dir[3 * p + 1]; W.vz = dir[3 * p + 2];
    W.x = cell[3 * p] - 1; W.y = cell[3 * p + 1] - 1; W.z = cell[3 * p + 2] - 1;
    W.absTau = 0.f; W.passProb = 0.f;
    flight_reciprocals(G, W);
    mirror_start(G, W);
    int len = 0, st = 3;
    for (int i = 1; i <= kSafeLimit; ++i) {
        Segment S;
        int err = 0;
        int r = walk_step<true, true>(G, A, W, 0, S, err);
        if (r == ST_ERROR) { st = -err; break; }
        if (r == ST_LOST) { st = 2; break; }
        if (len < max_len) {
            size_t o = (size_t)p * max_len + len;
            const int xyz = j3_lattice(G.js, S.w);
            cell_seq[3 * o] = xyz % G.nx + 1;
            cell_seq[3 * o + 1] = xyz / G.nx % G.ny + 1;
            cell_seq[3 * o + 2] = xyz / (G.nx * G.ny) + 1;
            ds_seq[o] = S.len;
        }
        ++len;
        if (r == ST_ESCAPED) { st = 1; break; }
    }
    seq_len[p] = len;
    status[p] = st;
}

// ----------------------------------------------------------- transport kernel
// PH_INTERACT: at an interaction point, to be absorbed (then re-emitted) or
// scattered; PH_ESCAPED: left the grid, its viewing-angle bins still to be
// taken.  Both wait for an emission pass.
enum Phase { PH_IDLE = 0, PH_STELLAR = 1, PH_INTERACT = 2, PH_WALK = 3, PH_ESCAPED = 4 };

// A packet.  enPacket%direction (the direction at the start of the flight or
// the last scatter) has the magnitudes of the walker's components, which the
// octant's mirrors only turn over, so its signs (bits 0..2 of dsign) are all
// that is kept of it.
struct Lane {
    Walker W;
    uint32_t plo, phi, draws;   // packet id and draws taken from its stream
    int nuP, origin;
    int steps, runs, phase, dsign;
};

__device__ __forceinline__ float flight_direction(float v, int dsign, int k)
{
    return __uint_as_float((__float_as_uint(v) & 0x7fffffffu) | ((uint32_t)(dsign >> k) << 31));
}

// wave-uniform event counters (scalar registers; emptied into the launch's
// 64-bit totals long before one could overflow, see kFlushLanes)
struct WaveCounts {
    unsigned seg, abs, sca, esc, lost, line, trapped, flights;
    unsigned wpass, wlanes, epass, elanes;              // passes and the lanes in them
};
constexpr unsigned kFlushLanes = 1u << 31;

__device__ __forceinline__ unsigned wcount(bool p)
{
    return (unsigned)__popcll(__ballot(p));
}

// An escape of a packet whose flight direction (enPacket%direction) is d:
// its theta and phi bins, then the viewing-angle planes they feed, as every
// escape site of pathSegment and energyPacketRun does
// (photon_mod.f90:1582-1666, 370-465), as a bit mask.  err 60/61: the
// reference's stops on a bin out of range.  The bin tables were
// range-checked on the host.
__device__ __forceinline__ unsigned esc_planes(const Grid &G, float dx, float dy, float dz, int &err)
{
    const View *V = G.view;
    if (!V) return 1u;
    const bool sym = (G.flags & F_SYM) != 0;
    const float q = mcf_acosf(sym ? fabsf(dz) : dz) / V->dTheta;
    if (isnan(q)) { err = 60; return 0; }
    int it = (int)q + 1;
    if (it > V->totT) it = V->totT;
    if (it < 1) { err = 60; return 0; }
    int ip;
    if (fabsf(dx) < 1.e-35f) ip = 0;
    else if (sym) ip = (int)(mcf_atanf(fabsf(dy) / fabsf(dx)) / V->dPhi);
    else ip = (int)(mcf_atanf(dy / dx) / V->dPhi);
    if (ip < 0) ip = V->totP + ip;
    ip = ip + 1;
    if (ip > V->totP) ip = V->totP;
    if (ip < 1) { err = 61; return 0; }
    const int t = V->Pt[it], ph = V->Pp[ip];
    if (t > 0 && V->vph[t] < 0.f) return 1u | 1u << t;
    if (t == ph || V->vth[ph] == V->vth[t] || V->vph[t] == V->vph[ph]) return 1u | 1u << t;
    return 1u;
}

__device__ __forceinline__ unsigned esc_planes(const Grid &G, const Lane &L, int &err)
{
    return esc_planes(G, flight_direction(L.W.vx, L.dsign, 0), flight_direction(L.W.vy, L.dsign, 1),
                      flight_direction(L.W.vz, L.dsign, 2), err);
}

// the word of plane a of esc for a packet
__device__ __forceinline__ size_t esc_index(const Grid &G, int a, const Lane &L)
{
    return ((size_t)a * (size_t)(G.nbins + 1) + (size_t)L.nuP) * (size_t)(G.nCells + 1) + L.origin;
}

// ------------------------------------------------------------------- sinks
// Where a wavefront's deposits go.  segment(): the J update of the lanes with
// `has`; escape(): dE to the planes in each lane's mask.  ready(): room for
// one more pass (at most three deposits a lane).

// FP64 atomics, J's through the rings.
template <int D, bool WIDE>
struct AddSink {
    JQ Q;
    __device__ __forceinline__ void begin(const Grid &G, const RunArgs &RA, int lane)
    {
        if (G.flags & F_CROSS) crossings_open<D, WIDE>(G, RA, Q, lane);
    }
    __device__ __forceinline__ bool ready(const Args &, int) { return true; }
    __device__ __forceinline__ void segment(const Grid &G, bool has, unsigned w, unsigned nu0, float v, int lane)
    {
        jq_push<D, WIDE>(G, Q, has, w, nu0, v, lane);
    }
    __device__ __forceinline__ void escape(const Grid &G, unsigned planes, const Lane &L, float dE, int)
    {
        for (int a = 0; a < 3; ++a)
            if (planes >> a & 1u) unsafeAtomicAdd(&G.esc[esc_index(G, a, L)], (double)dE);
    }
    __device__ __forceinline__ void close(const Grid &G, const Args &, int lane)
    {
        jq_flush<D, WIDE>(G, Q, lane);
        if (G.flags & F_CROSS) crossings_close<D, WIDE>(G, Q, lane);
    }
};

// The deposit log: 8 bytes a deposit, in the order they come.  A wavefront
// queues them in LDS and writes kLogFlush at a time to chunks of its own: a
// store in every pass would be waited for by the next pass's opacity gather
// (loads and stores count down together).  45^3 octant, 1e8 packets: the walk
// takes 14 ms with this sink, 45 with atomics (AddSink).
constexpr int kLogQueue = 512;           // entries in LDS per wavefront
constexpr int kLogFlush = 256;
struct LogSink {
    LogEntry *q;             // the queue
    LogEntry *at;            // the chunk
    unsigned n, chunk, used; // queued entries; the chunk's index and entries
    bool open;
    __device__ __forceinline__ void begin(const Grid &, const RunArgs &, int) {}
    __device__ __forceinline__ void put(bool has, unsigned w, float v, int lane)
    {
        const uint64_t m = __ballot(has);
        if (has) q[n + lane_rank(m, lane)] = LogEntry{ w, v };
        n += (unsigned)__popcll(m);
    }
    // the first kLogFlush entries (or all) to the chunk; the rest move down
    __device__ __forceinline__ void flush(unsigned count, int lane)
    {
        wave_lds_order();
        for (unsigned i = lane; i < count; i += 64) at[used + i] = q[i];
        used += count;
        n -= count;
        for (unsigned i = lane; i < n; i += 64) {
            const LogEntry e = q[count + i];
            wave_lds_order();
            q[i] = e;
        }
        wave_lds_order();
    }
    __device__ __forceinline__ bool ready(const Args &P, int lane)
    {
        if (n + 3 * 64 <= (unsigned)kLogQueue) return true;
        if (!open || used + kLogFlush > (unsigned)kLogChunk) {
            const RunArgs RA = scalar_copy<RunArgs>(P.r);
            unsigned c = 0;
            if (lane == 0) {
                if (open) RA.log_count[chunk] = used;
                c = atomicAdd(RA.log_next, 1u);
            }
            chunk = (unsigned)__builtin_amdgcn_readfirstlane((int)c);
            open = chunk < RA.log_chunks;
            at = RA.log + (size_t)chunk * kLogChunk;
            used = 0;
            if (!open) return false;
        }
        flush(kLogFlush, lane);
        return true;
    }
    __device__ __forceinline__ void segment(const Grid &, bool has, unsigned w, unsigned, float v, int lane)
    {
        put(has, w, v, lane);
    }
    __device__ __forceinline__ void escape(const Grid &G, unsigned planes, const Lane &L, float dE, int lane)
    {
        for (int a = 0; a < 3; ++a) {
            const bool has = planes >> a & 1u;
            if (a == 0 || (G.flags & F_VIEW)) put(has, G.esc_word + (unsigned)esc_index(G, a, L), dE, lane);
        }
    }
    // What is queued goes to the end of the chunk, or (a wavefront whose
    // packets are few, or that found the log full) to the estimators.
    __device__ __forceinline__ void close(const Grid &G, const Args &P, int lane)
    {
        if (open && used + n <= (unsigned)kLogChunk) flush(n, lane);
        wave_lds_order();
        for (unsigned i = lane; i < n; i += 64) {
            const LogEntry e = q[i];
            double *to = e.w < G.esc_word ? G.J3 + e.w : G.esc + (e.w - G.esc_word);
            unsafeAtomicAdd(to, (double)e.val);
        }
        n = 0;
        if (open && lane == 0) scalar_copy<RunArgs>(P.r).log_count[chunk] = used;
        open = false;
    }
};

// What ends or continues a packet in a pass.
struct Events {
    bool absorbed = false, scattered = false, lost = false, escaped = false, line = false, flight = false;
    unsigned planes = 0;     // of an escape
};

// The start of a flight in direction d: reciprocals, the octant's mirror and
// the optical depth to the next interaction (photon_mod.f90:1176-1184).
__device__ __forceinline__ void start_flight(Lane &L, const Grid &G, Rng &R, float dx, float dy, float dz)
{
    L.W.vx = dx; L.W.vy = dy; L.W.vz = dz;
    L.dsign = (int)((__float_as_uint(dx) >> 31) | (__float_as_uint(dy) >> 31) << 1 | (__float_as_uint(dz) >> 31) << 2);
    flight_reciprocals(G, L.W);
    mirror_start(G, L.W);
    L.W.absTau = 0.f;
    const float random = draw(R, G);
    L.W.passProb = -mcf_logf(1.f - random);
    L.phase = PH_WALK;
}

// A packet at its interaction point (photon_mod.f90:1577-1797): beyond R_out
// it has escaped, grains scatter or absorb it, gas absorbs it.  Returns true
// when it is absorbed and due for its re-emission.
template <bool WIDE>
__device__ __forceinline__ bool interact(Lane &L, const Grid &G, const Axes &A, Rng &R, Events &E, int &err)
{
    const float rx = L.W.rx / 1.e10f, ry = L.W.ry / 1.e10f, rz = L.W.rz / 1.e10f;
    if (sqrtf(rx * rx + ry * ry + rz * rz) * 1.e10f >= G.R_out && G.R_out > 0.f) {
        E.planes = esc_planes(G, L, err);
        E.escaped = true;
        L.phase = PH_IDLE;
        return false;
    }
    if (G.flags & F_DUST) {
        const unsigned nu0 = (unsigned)(L.nuP - 1);
        const size_t i = Word<WIDE>::index(G, Word<WIDE>::of(A.px[L.W.x], A.py[L.W.y], A.pz[L.W.z], nu0), nu0);
        const float probSca = G.sca3[i] / G.opac3[i];
        const float u = 1.f - draw(R, G);
        if (u > probSca) {
            E.absorbed = true;
            if (!(G.flags & F_GAS)) { err = 41; return false; }           // dustEmi needs dust PDFs
        } else if (u <= probSca) {
            E.scattered = true;                               // 1720-1797
            L.origin = act(G, L.W);
            float dx = flight_direction(L.W.vx, L.dsign, 0), dy = flight_direction(L.W.vy, L.dsign, 1),
                  dz = flight_direction(L.W.vz, L.dsign, 2);
            if (G.flags & F_ISO) {
                new_direction(R, G, false, dx, dy, dz);
            } else {
                for (int ihg = 1; ihg <= 10; ++ihg)
                    if (hg(R, G, L.nuP, dx, dy, dz) == 0) break;
            }
            start_flight(L, G, R, dx, dy, dz);
        } else {
            err = 39;
            return false;
        }
    } else {
        E.absorbed = true;
    }
    // safeLimit (2838-2846); recursionLimit (120-126)
    if (L.steps >= kSafeLimit) {
        E.lost = true;
        L.phase = PH_IDLE;
    }
    if (L.phase == PH_INTERACT && L.runs >= kRecursionLimit) L.phase = PH_IDLE;
    return L.phase == PH_INTERACT;
}

// newPhotonPacket + initPhotonPacket + the start of pathSegment
// (photon_mod.f90:768-1059, 491-684) for stellar packets and re-emissions at
// an absorption point.
__device__ __forceinline__ void emit(Lane &L, const Grid &G, const RunArgs &RA, Rng &R, double &qphot,
                                     Events &E, int &err)
{
    const bool stellar = (L.phase == PH_STELLAR);
    const float *cdf;
    const unsigned short *guide;
    int a;
    if (stellar) {
        L.runs = 1;
        L.W.x = RA.sx - 1; L.W.y = RA.sy - 1; L.W.z = RA.sz - 1;
        L.W.rx = RA.px; L.W.ry = RA.py; L.W.rz = RA.pz;
        a = RA.star_cell;
        cdf = G.specCDF + (size_t)(RA.istar - 1) * G.nbins;
        guide = G.specGuide + (size_t)(RA.istar - 1) * (kGuide + 1);
    } else {
        L.runs++;
        a = act(G, L.W);
        if (!(G.flags & F_GAS)) { err = 13; return; }
        if (a <= 0) { err = 14; return; }
        float random = 1.f - draw(R, G);
        if (random <= G.totalLines[a]) {                 // line packet (923-956)
            E.line = true;
            L.phase = PH_IDLE;
            return;
        }
        cdf = G.recCDF + (size_t)a * G.nbins;
        guide = G.recGuide + (size_t)a * (kGuide + 1);
    }
    int nuP = getnu2(R, G, cdf, guide, G.nbins, err);
    if (err) return;
    if (nuP < 1 || nuP >= G.nbins) { err = stellar ? 11 : 15; return; }
    L.nuP = nuP;
    float dx, dy, dz;
    new_direction(R, G, stellar && (G.flags & (F_SYM | F_MULTI)) == F_SYM, dx, dy, dz);
    L.origin = a;
    const float nu = G.nuArray[nuP - 1];
    if (stellar && nu > 1.f) qphot += (double)(RA.deltaE / (2.1799153e-11f * nu));
    if (!(G.flags & F_DUST) && nu < G.ionEdge1) {        // escapes at birth (370-465)
        E.planes = esc_planes(G, dx, dy, dz, err);
        E.escaped = true;
        L.phase = PH_IDLE;
        return;
    }
    start_flight(L, G, R, dx, dy, dz);
    L.steps = 0;
    E.flight = true;
}

__device__ __forceinline__ bool pending(const Lane &L)
{
    return L.phase != PH_IDLE && L.phase != PH_WALK;
}

// An emission pass of the wavefront: every lane whose packet waits runs it
// together.  Escapes and interactions end or turn their packets first; then
// new and absorbed packets are emitted.  Taking the interactions here keeps
// their divisions, square root and draws out of the walk passes, nearly all
// of which have a lane or two that interacts.  Counts events into C.
template <bool WIDE, class Sink>
__device__ __forceinline__ void emission_pass(Lane &L, const Args &P, const Axes &A, WaveCounts &C, double &qphot,
                                              int &err, Sink &K, int lane)
{
    const Grid G = scalar_copy<Grid>(P.g);
    const RunArgs RA = scalar_copy<RunArgs>(P.r);
    Events E;
    Rng R = rng_at(L.plo, L.phi, (uint32_t)RA.istar, L.draws);
    bool emits = L.phase == PH_STELLAR;
    if (L.phase == PH_ESCAPED) {
        E.planes = esc_planes(G, L, err);
        L.phase = PH_IDLE;
    } else if (L.phase == PH_INTERACT) {
        emits = interact<WIDE>(L, G, A, R, E, err);
    }
    bool ends = E.escaped || (E.absorbed && L.phase == PH_IDLE) || E.lost;
    if (emits) {
        emit(L, G, RA, R, qphot, E, err);
        ends = E.line || E.escaped;
    }
    if (err) L.phase = PH_IDLE;
    L.draws = R.k;
    if (__any(E.planes != 0)) K.escape(G, E.planes, L, RA.deltaE, lane);
    C.epass += 1;
    C.elanes += wcount(emits);
    C.abs += wcount(E.absorbed);
    C.sca += wcount(E.scattered);
    C.lost += wcount(E.lost);
    C.line += wcount(E.line);
    C.esc += wcount(E.escaped);
    C.flights += wcount(E.flight);
    // energyPacketDriver counts the packet whose last run is the
    // recursionLimit-th as trapped (photon_mod.f90:126)
    C.trapped += wcount(!err && ends && L.runs >= kRecursionLimit);
}

// One walk pass of the wavefront: every lane whose packet walks takes one
// step of pathSegment.  Counts events into C, queues the J updates.
template <bool WIDE, class Sink>
__device__ __forceinline__ void walk_pass(Lane &L, const Grid &G, const Axes &A, float dE, WaveCounts &C, int &err,
                                          Sink &K, int lane)
{
    bool seg = false;
    float jv = 0.f;
    Segment S;
    S.w = 0;
    const unsigned nu0 = (unsigned)(L.nuP - 1);
    bool escaped = false, lost = false;
    C.wpass += 1;
    C.wlanes += wcount(L.phase == PH_WALK);
    if (L.phase == PH_WALK) {
        L.steps++;
        int e = 0;
        const int r = walk_step<false, WIDE>(G, A, L.W, nu0, S, e);
        seg = r != ST_LOST && r != ST_ERROR;
        if (seg) jv = S.len * dE / S.dV;
        if (r == ST_ABSORBED) L.phase = PH_INTERACT;
        if (r == ST_ESCAPED) {
            escaped = true;
            L.phase = (G.flags & F_VIEW) ? PH_ESCAPED : PH_IDLE;
        }
        lost = r == ST_LOST || (r == ST_CONTINUE && L.steps >= kSafeLimit);   // safeLimit, 2838-2846
        if (lost || r == ST_ERROR) L.phase = PH_IDLE;
        if (e) err = e;
    }
    K.segment(G, seg, S.w, nu0, jv, lane);
    if (!(G.flags & F_VIEW) && __any(escaped)) K.escape(G, escaped ? 1u : 0u, L, dE, lane);
    C.seg += wcount(seg);
    C.esc += wcount(escaped);
    if (__any(lost)) C.lost += wcount(lost);
    if (__any((lost || escaped) && L.runs >= kRecursionLimit))
        C.trapped += wcount((lost || escaped) && L.runs >= kRecursionLimit);
}

// ------------------------------------------------ packet pool (per wave, LDS)
// A wavefront keeps a pool of P packets in LDS beside its 64 lanes: packets
// that walk (the walker stack, slots 0 .. nw-1 from the bottom) and packets
// that wait for an emission pass (the pending stack, slots P-npd .. P-1 from
// the top).  A lane whose flight ends takes a walker from the pool, leaving
// its own packet on the pending stack if it waits; an emission round moves
// walkers into the pool, so that the emission pass runs on a full wavefront,
// and the walkers come back as flights end.  The walk passes then stay nearly
// full between emissions.  Word k of slot s is at pw[k * P + s]; the cell
// indices are packed in one word (11, 11 and 10 bits: the host runs this
// kernel on lattices of at most 2047 x 2047 x 1023 points: an escaped packet's
// index is one past the last), the frequency
// bin, run count and phase in another (16, 13 and 3 bits), steps and direction
// signs in a third.  The stream is the launch's source, not stored, and a
// waiting packet's optical depths and reciprocals are of no use any more.
constexpr int kPoolWords = 18;
// Slots per wavefront: with 8-deep J rings, 4 workgroups of 256 per CU keep
// 32 slots within the CU's 160 KB of LDS (6.9 KB per wavefront, plus the
// staged tables).
constexpr int kPoolSlots = 32;
constexpr int kLogSlots = 32;    // log_kernel
static_assert(kSafeLimit < (1 << 20) && kRecursionLimit < (1 << 13), "packed packet words");

template <int P>
__device__ __forceinline__ void pool_put(uint32_t *pw, int s, const Lane &L)
{
    uint32_t *q = pw + s;
    q[0 * P] = L.plo; q[1 * P] = L.phi; q[2 * P] = L.draws;
    q[3 * P] = __float_as_uint(L.W.rx); q[4 * P] = __float_as_uint(L.W.ry); q[5 * P] = __float_as_uint(L.W.rz);
    q[6 * P] = __float_as_uint(L.W.vx); q[7 * P] = __float_as_uint(L.W.vy); q[8 * P] = __float_as_uint(L.W.vz);
    q[9 * P] = (uint32_t)L.W.x | ((uint32_t)L.W.y << 11) | ((uint32_t)L.W.z << 22);
    q[10 * P] = (uint32_t)L.nuP | ((uint32_t)L.runs << 16) | ((uint32_t)L.phase << 29);
    q[11 * P] = (uint32_t)L.origin;
    q[12 * P] = (uint32_t)L.steps | ((uint32_t)L.dsign << 20);
    if (L.phase == PH_WALK) {
        q[13 * P] = __float_as_uint(L.W.absTau); q[14 * P] = __float_as_uint(L.W.passProb);
        q[15 * P] = __float_as_uint(L.W.qx); q[16 * P] = __float_as_uint(L.W.qy); q[17 * P] = __float_as_uint(L.W.qz);
    }
}

template <int P, bool WALKER>
__device__ __forceinline__ void pool_get(const uint32_t *pw, int s, Lane &L)
{
    const uint32_t *q = pw + s;
    L.plo = q[0 * P]; L.phi = q[1 * P]; L.draws = q[2 * P];
    L.W.rx = __uint_as_float(q[3 * P]); L.W.ry = __uint_as_float(q[4 * P]); L.W.rz = __uint_as_float(q[5 * P]);
    L.W.vx = __uint_as_float(q[6 * P]); L.W.vy = __uint_as_float(q[7 * P]); L.W.vz = __uint_as_float(q[8 * P]);
    const uint32_t c = q[9 * P];
    L.W.x = (int)(c & 2047u); L.W.y = (int)((c >> 11) & 2047u); L.W.z = (int)(c >> 22);
    const uint32_t f = q[10 * P];
    L.nuP = (int)(f & 65535u); L.runs = (int)((f >> 16) & 8191u); L.phase = WALKER ? PH_WALK : (int)(f >> 29);
    L.origin = (int)q[11 * P];
    const uint32_t t = q[12 * P];
    L.steps = (int)(t & 0xfffffu); L.dsign = (int)(t >> 20);
    if (WALKER) {
        L.W.absTau = __uint_as_float(q[13 * P]); L.W.passProb = __uint_as_float(q[14 * P]);
        L.W.qx = __uint_as_float(q[15 * P]); L.W.qy = __uint_as_float(q[16 * P]); L.W.qz = __uint_as_float(q[17 * P]);
    }
}

// Lanes that do not walk take walkers from the pool (the first nw of them in
// lane order); a taker whose packet waits for an emission pass leaves it on
// the pending stack first, if the pool has a free slot for it.  The pending
// slots written lie in the free region, the walker slots read below it.
template <int P>
__device__ __forceinline__ void pool_settle(Lane &L, uint32_t *pw, int &nw, int &npd, int lane)
{
    if (nw == 0) return;
    const bool nonw = L.phase != PH_WALK;
    if (!__any(nonw)) return;
    const int F = P - nw - npd;
    const bool pend = pending(L);
    const uint64_t mp = __ballot(pend);
    const bool elig = nonw && (!pend || lane_rank(mp, lane) < F);
    const uint64_t me = __ballot(elig);
    const int re = lane_rank(me, lane);
    const bool take = elig && re < nw;
    const uint64_t mt = __ballot(take);
    const uint64_t mtp = mt & mp;
    if (mtp) {
        if (take && pend) pool_put<P>(pw, P - npd - 1 - lane_rank(mtp, lane), L);
        npd += __popcll(mtp);
        wave_lds_order();
    }
    if (take) pool_get<P, true>(pw, nw - 1 - re, L);
    nw -= __popcll(mt);
    wave_lds_order();
}

// The packets a wavefront holds: indices next .. end - 1 of the launch.  It
// takes them from the launch's counter many at a time, 1/8 of its share of
// what is left (64 to 2048).  Atomics with a result on one address are served
// one every 12 ns: taking the packets of each emission round alone, the 4096
// wavefronts of a sweep waited 49 us a round for one another.
struct Stock {
    unsigned long long next = 0, end = 0;
    bool last = false;           // nothing left at the counter
    __device__ __forceinline__ bool empty() const { return last && next >= end; }
};

// Fresh packets for the lanes with `need`.
__device__ __forceinline__ void take_fresh(Lane &L, const Args &P, bool need, Stock &S, int lane)
{
    uint64_t m = __ballot(need);
    if (!m) return;
    const RunArgs RA = scalar_copy<RunArgs>(P.r);
    const unsigned long long total = (unsigned long long)RA.npackets;
    while (m) {
        if (S.next >= S.end) {
            if (S.last) break;
            const unsigned long long waves = (unsigned long long)gridDim.x * (blockDim.x >> 6);
            const unsigned long long share = (total - S.end) / (8 * waves) & ~63ull;
            const unsigned long long n = share < 64 ? 64 : share > 2048 ? 2048 : share;
            unsigned long long base = 0;
            if (lane == 0) base = atomicAdd(RA.next_packet, n);
            base = (unsigned long long)(unsigned)__builtin_amdgcn_readfirstlane((int)(base >> 32)) << 32 |
                   (unsigned)__builtin_amdgcn_readfirstlane((int)base);
            S.next = base < total ? base : total;
            S.end = base + n < total ? base + n : total;
            S.last = base + n >= total;
            continue;
        }
        const unsigned long long id = S.next + (unsigned long long)lane_rank(m, lane);
        const bool mine = ((m >> lane) & 1ull) && id < S.end;
        if (mine) {
            const uint64_t packet = RA.packet_offset + id;
            L.plo = (uint32_t)packet;
            L.phi = (uint32_t)(packet >> 32);
            L.draws = 0;
            L.phase = PH_STELLAR;
        }
        const uint64_t took = __ballot(mine);
        S.next += (unsigned long long)__popcll(took);
        m &= ~took;
    }
}

// An emission round of the pool kernel: walkers move to the pool (as many
// as the candidates for an emission exceed the lanes that do not walk, and
// as fit), idle lanes take packets from the pending stack, then fresh
// packets, and the emission pass runs.
template <int P, bool WIDE, class Sink>
__device__ __forceinline__ void pool_emission_round(Lane &L, uint32_t *pw, int &nw, int &npd, Stock &S,
                                                    const Args &A_, const Axes &A, WaveCounts &C, double &qphot,
                                                    int &err, Sink &K, int lane)
{
    const bool walk = L.phase == PH_WALK;
    const uint64_t mw = __ballot(walk);
    const int nwalk = __popcll(mw);
    const int npl = (int)wcount(pending(L));
    const int cand = npl + npd + (S.empty() ? 0 : 64);
    const int k = max(0, min(min(nwalk, P - nw - npd), cand - (64 - nwalk)));
    if (k > 0) {
        const int rw = lane_rank(mw, lane);
        if (walk && rw < k) {
            pool_put<P>(pw, nw + rw, L);
            L.phase = PH_IDLE;
        }
        nw += k;
        wave_lds_order();
    }
    if (npd > 0) {
        const bool idle = L.phase == PH_IDLE;
        const uint64_t mi = __ballot(idle);
        const int ri = lane_rank(mi, lane);
        if (idle && ri < npd) pool_get<P, false>(pw, P - npd + ri, L);
        npd -= min(__popcll(mi), npd);
        wave_lds_order();
    }
    if (!S.empty()) take_fresh(L, A_, L.phase == PH_IDLE, S, lane);
    if (__any(pending(L))) emission_pass<WIDE>(L, A_, A, C, qphot, err, K, lane);
}

__device__ __forceinline__ Lane idle_lane()
{
    Lane L;
    L.W.rx = L.W.ry = L.W.rz = L.W.vx = L.W.vy = L.W.vz = L.W.qx = L.W.qy = L.W.qz = 0.f;
    L.W.x = L.W.y = L.W.z = 0;
    L.W.absTau = L.W.passProb = 0.f;
    L.plo = L.phi = L.draws = 0;
    L.nuP = 1; L.origin = 0; L.steps = 0; L.runs = 0; L.phase = PH_IDLE; L.dsign = 0;
    return L;
}

// Add a wavefront's counters to its model's totals and clear them.
__device__ __forceinline__ void flush_counts(const Args &P, WaveCounts &C)
{
    const RunArgs RA = scalar_copy<RunArgs>(P.r);
    if ((threadIdx.x & 63) == 0) {
        const unsigned v[12] = { C.seg, C.abs, C.sca, C.esc, C.lost, C.line, C.trapped, C.flights,
                                 C.wpass, C.wlanes, C.epass, C.elanes };
        for (int i = 0; i < 12; ++i) atomicAdd(&RA.counts[i], (unsigned long long)v[i]);
    }
    C = WaveCounts{0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0};
}

__device__ __forceinline__ void flush_qphot(const Args &P, double qphot)
{
    for (int o = 32; o >= 1; o >>= 1) qphot += __shfl_xor(qphot, o);
    if ((threadIdx.x & 63) == 0) unsafeAtomicAdd(scalar_copy<RunArgs>(P.r).qphot, qphot);
}

// A fail-stop code goes to the launch's error word.
__device__ __forceinline__ void report(const Args &P, int &err)
{
    if (__any(err != 0)) {
        if (err) atomicMax(scalar_copy<RunArgs>(P.r).error, err);
        err = 0;
    }
}

// The arguments of the single-model kernels, read in place from the launch's
// argument block.
struct LaunchArgs { Grid G; RunArgs RA; };

__device__ __forceinline__ Args kernel_args()
{
    const uint64_t at = (uint64_t)__builtin_amdgcn_kernarg_segment_ptr();
    return Args{ at, at + offsetof(LaunchArgs, RA) };
}

// One packet per lane, for lattices the pool kernel does not take (64-bit
// table indices).  An emission pass runs when at least emit_min lanes (or as
// many as are walking) wait for one, then walk_steps walk passes.  Rings of
// D: in a batch, lattices with axes too long for four wavefronts' rings of
// eight beside their tables run one-wavefront workgroups with rings of four.
template <int D>
__global__ void __launch_bounds__(256) transport_kernel(LaunchArgs)
{
    extern __shared__ float lds[];
    const Args P = kernel_args();
    const Grid G = scalar_copy<Grid>(P.g);
    const RunArgs RA = scalar_copy<RunArgs>(P.r);
    Axes A;
    const int nwaves = (int)(blockDim.x >> 6);
    stage_axes<true>(G, lds + (size_t)nwaves * JRing<D, true>::kFloats, A);
    const int lane_id = threadIdx.x & 63;
    AddSink<D, true> K{ jq_at<D, true>(lds, (int)(threadIdx.x >> 6)) };
    K.begin(G, RA, lane_id);

    Lane L = idle_lane();
    Stock S;
    WaveCounts C = {0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0};
    double qphot = 0.0;
    int err = 0;

    for (;;) {
        if (!S.empty()) take_fresh(L, P, L.phase == PH_IDLE, S, lane_id);
        const int npend = (int)wcount(pending(L));
        const int nwalk = (int)wcount(L.phase == PH_WALK);
        if (npend + nwalk == 0) {
            if (S.empty()) break;
            continue;
        }
        if (npend >= RA.emit_min || npend >= nwalk) emission_pass<true>(L, P, A, C, qphot, err, K, lane_id);
        for (int s = 0; s < RA.walk_steps; ++s) walk_pass<true>(L, G, A, RA.deltaE, C, err, K, lane_id);
        report(P, err);
        if (C.wlanes >= kFlushLanes) flush_counts(P, C);
    }
    K.close(G, P, lane_id);
    flush_counts(P, C);
    flush_qphot(P, qphot);
}

// A suspended wavefront's packets: its lanes (kPoolWords words each, phase
// included), its pool's slots, nw, npd and its stock.
template <int P>
struct Save {
    static constexpr int kWords = kPoolWords * (64 + P) + 64;
    static __device__ __forceinline__ void put(uint32_t *at, const Lane &L, const uint32_t *pw, int nw, int npd,
                                               const Stock &S, int lane)
    {
        pool_put<64>(at, lane, L);
        for (int i = lane; i < kPoolWords * P; i += 64) at[kPoolWords * 64 + i] = pw[i];
        if (lane == 0) {
            uint32_t *t = at + kPoolWords * (64 + P);
            t[0] = (uint32_t)nw; t[1] = (uint32_t)npd; t[2] = S.last;
            t[3] = (uint32_t)S.next; t[4] = (uint32_t)(S.next >> 32); t[5] = (uint32_t)S.end; t[6] = (uint32_t)(S.end >> 32);
        }
    }
    static __device__ __forceinline__ void get(const uint32_t *at, Lane &L, uint32_t *pw, int &nw, int &npd,
                                               Stock &S, int lane)
    {
        pool_get<64, true>(at, lane, L);
        L.phase = (int)(at[10 * 64 + lane] >> 29);
        for (int i = lane; i < kPoolWords * P; i += 64) pw[i] = at[kPoolWords * 64 + i];
        uint32_t t[7];
        for (int i = 0; i < 7; ++i)
            t[i] = (uint32_t)__builtin_amdgcn_readfirstlane((int)at[kPoolWords * (64 + P) + i]);
        nw = (int)t[0];
        npd = (int)t[1];
        S.last = t[2] != 0;
        S.next = t[3] | (unsigned long long)t[4] << 32;
        S.end = t[5] | (unsigned long long)t[6] << 32;
        wave_lds_order();
    }
};

// One model's packets on one wavefront, with a packet pool of P slots in LDS
// (one packet per lane in registers).  An emission round runs when at least
// emit_min lanes do not walk (or none does); every walk pass is followed by a
// settle from the pool.  A sink that runs out of room suspends the wavefront.
template <int P, class Sink>
__device__ __forceinline__ void pool_run(const Args &K, const Axes &A, uint32_t *pw, Sink &D, int lane_id)
{
    const Grid G = scalar_copy<Grid>(K.g);
    const RunArgs RA = scalar_copy<RunArgs>(K.r);
    Lane L = idle_lane();
    int nw = 0, npd = 0;
    Stock S;
    bool room = true;
    WaveCounts C = {0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0};
    double qphot = 0.0;
    int err = 0;
    const size_t save = (size_t)(blockIdx.x * (blockDim.x >> 6) + (threadIdx.x >> 6)) * Save<P>::kWords;
    if (RA.resume) Save<P>::get(RA.save + save, L, pw, nw, npd, S, lane_id);
    D.begin(G, RA, lane_id);
    for (;;) {
        pool_settle<P>(L, pw, nw, npd, lane_id);
        const int nwalk = (int)wcount(L.phase == PH_WALK);
        if (nwalk == 0 && nw == 0 && npd == 0 && S.empty() && !__any(pending(L))) break;
        room = D.ready(K, lane_id);
        if (!room) break;
        if (64 - nwalk >= RA.emit_min || nwalk == 0)
            pool_emission_round<P, false>(L, pw, nw, npd, S, K, A, C, qphot, err, D, lane_id);
        for (int s = 0; s < RA.walk_steps; ++s) {
            // on with the next round early when fewer than half the lanes
            // walk and there are packets to fill an emission pass with
            const int walking = (int)wcount(L.phase == PH_WALK);
            if (walking == 0 || (s > 0 && walking < 32 &&
                                 (!S.empty() || npd + (int)wcount(pending(L)) >= 16))) break;
            room = D.ready(K, lane_id);
            if (!room) break;
            walk_pass<false>(L, G, A, RA.deltaE, C, err, D, lane_id);
            pool_settle<P>(L, pw, nw, npd, lane_id);
        }
        report(K, err);
        if (C.wlanes >= kFlushLanes) flush_counts(K, C);
        if (!room) break;
    }
    D.close(G, K, lane_id);
    flush_counts(K, C);
    flush_qphot(K, qphot);
    if (!room) {
        const RunArgs RB = scalar_copy<RunArgs>(K.r);
        Save<P>::put(RB.save + save, L, pw, nw, npd, S, lane_id);
        if (lane_id == 0) *RB.suspended = 1;
    } else if (RA.save && lane_id == 0) {
        // done: nothing to go on with in a further launch
        uint32_t *t = scalar_copy<RunArgs>(K.r).save + save + kPoolWords * (64 + P);
        t[0] = 0; t[1] = 0; t[2] = 1;
        t[3] = 0; t[4] = 0; t[5] = 0; t[6] = 0;
    }
    if (room && RA.save) scalar_copy<RunArgs>(K.r).save[save + 10 * 64 + lane_id] = 0;
}

// The single-model kernel with atomic deposits (small sweeps, crossing
// counts, no memory for the log).
__global__ void __launch_bounds__(256) pool_kernel(LaunchArgs)
{
    extern __shared__ float lds[];
    const Args K = kernel_args();
    Axes A;
    const int nwaves = (int)(blockDim.x >> 6), wave = (int)(threadIdx.x >> 6);
    uint32_t *pools = reinterpret_cast<uint32_t *>(lds + (size_t)nwaves * JRing<kJDepth, false>::kFloats);
    stage_axes<false>(scalar_copy<Grid>(K.g), reinterpret_cast<float *>(pools + (size_t)nwaves * kPoolSlots * kPoolWords),
                      A);
    AddSink<kJDepth, false> D{ jq_at<kJDepth, false>(lds, wave) };
    pool_run<kPoolSlots>(K, A, pools + (size_t)wave * kPoolSlots * kPoolWords, D, (int)(threadIdx.x & 63));
}

// The single-model kernel with its deposits in the log: 78 VGPRs, six
// wavefronts a SIMD as far as its LDS (queue and pool, 6.3 KB a wavefront) allows.
__global__ void __launch_bounds__(256) log_kernel(LaunchArgs)
{
    extern __shared__ float lds[];
    const Args K = kernel_args();
    Axes A;
    const int nwaves = (int)(blockDim.x >> 6), wave = (int)(threadIdx.x >> 6);
    LogEntry *queues = reinterpret_cast<LogEntry *>(lds);
    uint32_t *pools = reinterpret_cast<uint32_t *>(queues + (size_t)nwaves * kLogQueue);
    stage_axes<false>(scalar_copy<Grid>(K.g), reinterpret_cast<float *>(pools + (size_t)nwaves * kLogSlots * kPoolWords),
                      A);
    LogSink D{ queues + (size_t)wave * kLogQueue, nullptr, 0, 0, 0, false };
    pool_run<kLogSlots>(K, A, pools + (size_t)wave * kLogSlots * kPoolWords, D, (int)(threadIdx.x & 63));
}

// Many models in one persistent launch.  A workgroup runs one model at a
// time with the single-model kernel's pool: it starts with the model its
// share of the launch falls to (shares by packets and lattice size, so that
// the models run side by side and few workgroups change model), and when
// that model has no packets left goes through the others in turn, helping
// those that still have some.  Each packet keeps its own random stream, so
// results equal those of the models' separate runs.  Every workgroup visits
// every model at most once, which bounds the loop.  128 VGPRs: with two more
// three wavefronts fit a SIMD instead of four (8 models of 20^3 to 50^3 cells:
// 6.76 ms against 6.18).
__global__ void __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(4))) batch_kernel(BatchArgs B)
{
    extern __shared__ float lds[];
    __shared__ int s_left;
    const int nwaves = (int)(blockDim.x >> 6), wave = (int)(threadIdx.x >> 6);
    uint32_t *pools = reinterpret_cast<uint32_t *>(lds + (size_t)nwaves * JRing<kJDepth, false>::kFloats);
    float *tab = reinterpret_cast<float *>(pools + (size_t)nwaves * kPoolSlots * kPoolWords);
    // the last model whose share begins at or before this workgroup's
    int first = 0;
    {
        const double at = ((double)blockIdx.x + 0.5) / (double)gridDim.x * B.share[B.models];
        while (first + 1 < B.models && B.share[first + 1] <= at) ++first;
    }
    for (int t = 0; t < B.models; ++t) {
        const int m = __builtin_amdgcn_readfirstlane((first + t) % B.models);
        const Args K = { (uint64_t)(B.G + m), (uint64_t)(B.RA + m) };
        __syncthreads();                       // the last model's tables and s_left are done with
        if (threadIdx.x == 0) {
            const RunArgs RA = scalar_copy<RunArgs>(K.r);
            s_left = __hip_atomic_load(RA.next_packet, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) <
                     (unsigned long long)RA.npackets;
        }
        __syncthreads();
        if (!__builtin_amdgcn_readfirstlane(s_left)) continue;
        Axes A;
        stage_axes<false>(scalar_copy<Grid>(K.g), tab, A);
        AddSink<kJDepth, false> D{ jq_at<kJDepth, false>(lds, wave) };
        pool_run<kPoolSlots>(K, A, pools + (size_t)wave * kPoolSlots * kPoolWords, D, (int)(threadIdx.x & 63));
    }
}

// ------------------------------------------------------- table preparation
// opac3 in the J3 layout: the value of lattice point p at bin nu is
// opacity(active(xyz(p)), nu) (reference layout in: [nu][cell]); padding
// points hold 0.  Written in layout order (coalesced stores).
__global__ void densify_kernel(const float *compact, const int *active, J3Shape js, int nc1, int nbins,
                               float *dense)
{
    size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    const size_t tot = j3_size(js, nbins);
    for (; i < tot; i += (size_t)gridDim.x * blockDim.x) {
        const size_t tile = i / ((size_t)nbins * kJTile);
        const int nu = (int)((i / kJTile) % (size_t)nbins);
        const int xyz = j3_lattice(js, (unsigned)(tile * kJTile + i % kJTile));
        dense[i] = xyz < 0 ? 0.f : compact[(size_t)nu * nc1 + active[xyz]];
    }
}

// guide[row][j] for every row of a [rows][nbins] CDF table
__global__ void guide_kernel(const float *cdf, int rows, int nbins, unsigned short *guide)
{
    size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    size_t tot = (size_t)rows * (kGuide + 1);
    for (; i < tot; i += (size_t)gridDim.x * blockDim.x) {
        int r = (int)(i / (kGuide + 1)), j = (int)(i % (kGuide + 1));
        guide[i] = guide_entry(cdf + (size_t)r * nbins, nbins, j);
    }
}

// J(cell,nu) = value at the (x,y,z) of that cell; row 0 collects every
// inactive position, as the reference's Jste(0,:) does.  out must be zero.
// Bound by memory: 16 bytes a word.  setMotherGrid numbers cells z fastest, so
// a thread takes one (x,y,z) of a column of bricks, z fastest, and goes
// through the bins: a wavefront's stores are runs of the column's length, and
// its workgroup reads whole rows of the bricks.  In the lattice's order (x
// fastest) every store was a request of its own: 27^3 cells 448 -> 21 us, 19^3
// octant 96 -> 11.
constexpr int kCompact = 512;
__global__ void __launch_bounds__(kCompact)
compact_kernel(const double *__restrict__ J3, const int *__restrict__ active, J3Shape js, int nc1, int nbins, int per,
               double *__restrict__ out)
{
    const unsigned parts = (16u * (unsigned)js.nz + kCompact - 1) / kCompact;
    const unsigned column = blockIdx.x / parts, e = blockIdx.x % parts * kCompact + threadIdx.x;
    const int xy = (int)(e / (unsigned)js.nz), z = (int)(e % (unsigned)js.nz);
    const int x = (int)(column % (unsigned)js.tx) * 4 + (xy & 3), y = (int)(column / (unsigned)js.tx) * 4 + (xy >> 2);
    const bool in = xy < 16 && x < js.nx && y < js.ny;
    const int a = in ? active[x + js.nx * (y + js.ny * z)] : 0;
    const int nu0 = (int)blockIdx.y * per, nu1 = min(nu0 + per, nbins);
    const double *from = J3 + (in ? j3_index(nbins, 0, j3_point(js, x, y, z)) : 0);
    const auto store = [&](int nu, double v) {
        if (a > 0) {
            out[(size_t)nu * nc1 + a] = v;
            v = 0.0;
        }
        if (__any(v != 0.0)) {
            for (int o = 32; o >= 1; o >>= 1) v += __shfl_xor(v, o);
            if ((threadIdx.x & 63) == 0) unsafeAtomicAdd(&out[(size_t)nu * nc1], v);
        }
    };
    // four loads in flight
    int nu = nu0;
    for (; nu + 4 <= nu1; nu += 4) {
        double v[4];
        for (int k = 0; k < 4; ++k) v[k] = in ? from[(size_t)(nu + k) * kJTile] : 0.0;
        for (int k = 0; k < 4; ++k) store(nu + k, v[k]);
    }
    for (; nu < nu1; ++nu) store(nu, in ? from[(size_t)nu * kJTile] : 0.0);
}

}  // namespace mcd

// ---------------------------------------------------------------- launchers
size_t mcd_pool_lds(const mcd::Grid &G, int threads)
{
    return sizeof(float) * ((size_t)(threads / 64) * (mcd::JRing<mcd::kJDepth, false>::kFloats +
                                                      (size_t)mcd::kPoolSlots * mcd::kPoolWords) +
                            mcd::lds_floats(G.nx, G.ny, G.nz));
}

size_t mcd_save_words(int blocks, int threads)
{
    return (size_t)blocks * (threads / 64) * mcd::Save<mcd::kLogSlots>::kWords;
}

bool mcd_pool_fits(const mcd::Grid &G)
{
    return G.nx <= 2047 && G.ny <= 2047 && G.nz <= 1023 && G.nbins <= 65535 &&
           mcd::j3_size(G.js, G.nbins) <= 0xffffffffull;
}

// dynamic LDS of transport_kernel
template <int D>
static size_t transport_lds(const mcd::Grid &G, int threads)
{
    return sizeof(float) * ((size_t)(threads / 64) * mcd::JRing<D, true>::kFloats + mcd::lds_floats(G.nx, G.ny, G.nz));
}

bool mcd_transport_fits(const mcd::Grid &G, int threads)
{
    return transport_lds<mcd::kJDepth>(G, threads) <= 160 * 1024;
}

hipError_t mcd_launch_batch(const mcd::BatchArgs &B, size_t lds_bytes, int blocks, hipStream_t s)
{
    hipLaunchKernelGGL(mcd::batch_kernel, dim3(blocks), dim3(256), lds_bytes, s, B);
    return hipGetLastError();
}

hipError_t mcd_launch_transport(const mcd::Grid &G, const mcd::RunArgs &RA, int blocks, int threads, int kernel,
                                hipStream_t s)
{
    if (kernel == MCD_KERNEL_LOG) {
        const size_t lds = sizeof(float) * ((size_t)(threads / 64) * (mcd::kLogSlots * mcd::kPoolWords + 2 * mcd::kLogQueue) +
                                            mcd::lds_floats(G.nx, G.ny, G.nz));
        hipLaunchKernelGGL(mcd::log_kernel, dim3(blocks), dim3(threads), lds, s, mcd::LaunchArgs{ G, RA });
    } else if (kernel == MCD_KERNEL_POOL && mcd_pool_fits(G)) {
        hipLaunchKernelGGL(mcd::pool_kernel, dim3(blocks), dim3(threads), mcd_pool_lds(G, threads), s,
                           mcd::LaunchArgs{ G, RA });
    } else if (kernel == MCD_KERNEL_THIN) {
        hipLaunchKernelGGL(mcd::transport_kernel<4>, dim3(blocks), dim3(threads), transport_lds<4>(G, threads), s,
                           mcd::LaunchArgs{ G, RA });
    } else {
        hipLaunchKernelGGL(mcd::transport_kernel<mcd::kJDepth>, dim3(blocks), dim3(threads),
                           transport_lds<mcd::kJDepth>(G, threads), s, mcd::LaunchArgs{ G, RA });
    }
    return hipGetLastError();
}

hipError_t mcd_launch_replay(const mcd::Grid &G, int n, const float *pos, const float *dir,
                             const int *cell, int *cell_seq, float *ds_seq, int *seq_len,
                             int *status, int max_len, hipStream_t s)
{
    size_t lds = sizeof(float) * mcd::lds_floats(G.nx, G.ny, G.nz);
    int threads = 256, blocks = (n + threads - 1) / threads;
    hipLaunchKernelGGL(mcd::walk_replay_kernel, dim3(blocks), dim3(threads), lds, s, G, n, pos,
                       dir, cell, cell_seq, ds_seq, seq_len, status, max_len);
    return hipGetLastError();
}

hipError_t mcd_densify(const float *compact, const int *active, const mcd::J3Shape &js, int nc1, int nbins,
                       float *dense, hipStream_t s)
{
    hipLaunchKernelGGL(mcd::densify_kernel, dim3(2048), dim3(256), 0, s, compact, active, js, nc1, nbins, dense);
    return hipGetLastError();
}

hipError_t mcd_guides(const float *cdf, int rows, int nbins, unsigned short *guide, hipStream_t s)
{
    hipLaunchKernelGGL(mcd::guide_kernel, dim3(2048), dim3(256), 0, s, cdf, rows, nbins, guide);
    return hipGetLastError();
}

hipError_t mcd_compact(const double *J3, const int *active, const mcd::J3Shape &js, int nc1, int nbins,
                       double *out, hipStream_t s)
{
    // bins a workgroup: some 2048 workgroups, or one bin each
    const unsigned parts = (16u * (unsigned)js.nz + mcd::kCompact - 1) / mcd::kCompact;
    const size_t blocks = (size_t)js.tx * js.ty * parts;
    const int per = (int)std::max<size_t>({ 1, blocks * (size_t)nbins / 2048, ((size_t)nbins + 65534) / 65535 });
    hipLaunchKernelGGL(mcd::compact_kernel, dim3((unsigned)blocks, (nbins + per - 1) / per), dim3(mcd::kCompact), 0, s, J3,
                       active, js, nc1, nbins, per, out);
    return hipGetLastError();
}
