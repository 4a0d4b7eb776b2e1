// mc_opacity.hip - opacity tables on the device (ionizationDriver and
// addOpacity, ionization_mod.f90:26-484; the dust add of iterateMC,
// iteration_mod.f90:164-228), written straight into the transport's dense
// [nu][xyz] tables.
//
// One lane per lattice point, one wavefront per 64 consecutive points, so
// every bin's row of opac3 is written in one coalesced 256-byte store.  A
// lane forms its cell's ion densities in its LDS column once, then walks the
// bins; each bin's cross-section entries are the same for every lane, in
// addOpacity's order, and are added in FP32 in that order, so the tables
// equal the reference's bit for bit.  The entries of successive bins follow
// each other in memory, each bin's filled up to a multiple of four with
// entries that never count: a wavefront loads 64 of them at a time, one a
// lane and the next 64 ahead, and reads them out of the lanes four by four
// (scalar loads would be waited for together with the densities' LDS reads).
// The wavefronts of a tile share its bins by their cost: nearly all entries lie
// in the last fourth of them, and equal ranges left one wavefront the work.
// Bound by the instructions of the entries on large grids and by the chain of
// bins on small ones.  45^3 octant, 800 bins: 0.78 ms with loads where a bin
// needed them, 0.25 now; 21^3: 0.49, 0.05 now.  Bin 1 also
// carries the free-free term: addOpacity assigns FFOpacity at i = 1 only
// (ionization_mod.f90:369-393), with the Gaunt factor of the cell's own Te
// (Hummer 1988, getGauntFF, 195-318).
#include "mc_opacity.h"

#pragma clang fp contract(off)

namespace mco {

constexpr float kTe1Ryd = 1.578866e5f;   // constants_mod.f90:23

// Hummer's Chebyshev coefficients d(8,11), column-major (ionization_mod.f90:213-242)
__constant__ double kHummer[88] = {
    8.986940175e+00, -4.009515855e+00, 8.808871266e-01, 2.640245111e-02, -4.580645915e-02,
    -3.568055702e-03, 2.827798067e-03, 3.365860195e-04, -8.006936989e-01, 9.466021705e-01,
    9.043402532e-02, -9.608451450e-02, -1.885629865e-02, 1.050313890e-02, 2.800889961e-03,
    -1.078209202e-03, -3.781305103e-01, 1.102726332e-01, -1.543619180e-02, 8.310561114e-03,
    2.179620525e-02, 4.259726289e-03, -4.181588794e-03, -1.770208330e-03, 1.877213132e-02,
    -1.004885705e-01, -5.483366378e-02, -4.520154409e-03, 8.366530426e-03, 3.700273930e-03,
    6.889320423e-04, 9.460313195e-05, 7.300158392e-02, 3.576785497e-03, -4.545307025e-03,
    -1.017965604e-02, -9.530211924e-03, -3.450186162e-03, 1.040482914e-03, 1.407073544e-03,
    -1.744671550e-03, 2.864013856e-02, 1.903394837e-02, 7.091074494e-03, -9.668371391e-04,
    -2.999107465e-03, -1.820642230e-03, -3.874082085e-04, -1.707268366e-02, -4.694254776e-03,
    1.311691517e-03, 5.316703136e-03, 5.178193095e-03, 2.451228935e-03, -2.277321615e-05,
    -8.182359057e-04, 2.567331664e-04, -9.155339970e-03, -6.997479192e-03, -3.571518641e-03,
    -2.096101038e-04, 1.553822487e-03, 1.509584686e-03, 6.212627837e-04, 4.098322531e-03,
    1.635218463e-03, -5.918883504e-04, -2.333091048e-03, -2.484138313e-03, -1.359996060e-03,
    -5.371426147e-05, 5.553549563e-04, 3.837562402e-05, 2.938325230e-03, 2.393747064e-03,
    1.328839809e-03, 9.135013312e-05, -7.137252303e-04, -7.656848158e-04, -3.504683798e-04,
    -8.491991820e-04, -3.615327726e-04, 3.148015257e-04, 8.909207650e-04, 9.869737522e-04,
    6.134671184e-04, 1.068883394e-04, -2.046080100e-04};

// getGauntFF at one frequency for nuclear charge 10^z (ionization_mod.f90:195-318)
__device__ float gaunt_ff(float z, float log10Te, float xlf)
{
    float xlrkt;
    if (log10Te < 2.5f) xlrkt = 5.1983649f - 2.5f;
    else if (log10Te > 8.f) xlrkt = 5.1983649f - 8.f;
    else xlrkt = 5.1983649f - log10Te;
    const float txg = 0.66666667f * (2.0f * z + xlrkt);
    const float gamma2 = powf(10.f, txg * 1.5f);
    const float con = 0.72727273f * xlrkt + 0.90909091f;
    float c[9];
    for (int j = 1; j <= 8; ++j) {
        // Clenshaw recurrence b(ir) over ir = 11..1, three terms live
        float b2 = (float)kHummer[10 * 8 + j - 1];                              // b(11)
        float b1 = (float)((double)(txg * b2) + kHummer[9 * 8 + j - 1]);        // b(10)
        float bb1 = 0.f, bb3 = 0.f;
        for (int ir = 9; ir >= 1; --ir) {
            const float b0 = (float)((double)(txg * b1 - b2) + kHummer[(ir - 1) * 8 + j - 1]);
            if (ir == 3) bb3 = b0;
            if (ir == 1) bb1 = b0;
            b2 = b1;
            b1 = b0;
        }
        c[j] = 0.25f * (bb1 - bb3);
    }
    const float txu = 0.72727273f * xlf + con;
    const float u = powf(10.f, (txu - .90909091f) / .72727273f);
    float g = 0.f;
    if (fabsf(txu) <= 2.0f) {
        float b2 = c[8];
        float b1 = txu * b2 + c[7];
        float bb1 = 0.f, bb3 = 0.f;
        for (int ir = 6; ir >= 1; --ir) {
            const float b0 = txu * b1 - b2 + c[ir];
            if (ir == 3) bb3 = b0;
            if (ir == 1) bb1 = b0;
            b2 = b1;
            b1 = b0;
        }
        g = bb1 - bb3;
    } else if (log10f(u) < -4.0f && gamma2 < 0.3f) {
        g = 0.551329f * logf(2.24593f / u);
    } else if (log10f(u) < -4.0f && gamma2 >= 0.3f) {
        g = 0.551329f * logf(0.944931f / u / sqrtf(gamma2));
    } else if (txu > 2.0f) {
        if (log10f(gamma2) < -3.f) {
            g = sqrtf(0.9549297f / u);
        } else if (log10f(gamma2) < 0.0f) {
            const float slope = (sqrtf(12.f * gamma2 / u) - sqrtf(0.9549297f / u)) / 3.0f;
            g = sqrtf(12.f * gamma2 / u) + slope * log10f(gamma2);
        } else {
            g = sqrtf(12.f * gamma2 / u);
            g = 1.05f < g ? 1.05f : g;
        }
    }
    return g;
}

__global__ void __launch_bounds__(64) opacity_kernel(OpacArgs a, int parts)
{
    extern __shared__ float lds[];               // [nslot][64] densities, then [ndrow][64] weights
    const int lane = threadIdx.x;
    // `parts` wavefronts share a tile of 64 lattice points, each writing one
    // contiguous range of bins (more wavefronts in flight to hide latency)
    const int tile = blockIdx.x / parts, part = blockIdx.x % parts;
    const int xyz = mcd::j3_lattice(a.js, (unsigned)(tile * 64 + lane));   // -1: a padding point
    const bool in = xyz >= 0;
    const int cell = in ? a.active[xyz] : 0;
    // row nslot: zero, of the entries that never count
    float *dens = lds, *wr = lds + (a.nslot + 1) * 64;
    dens[a.nslot * 64 + lane] = 0.f;
    float ff1 = 0.f;
    if (cell <= 0)
        for (int q = 0; q < a.nslot; ++q) dens[q * 64 + lane] = 0.f;
    if (cell > 0) {
        const float *s = a.st + (size_t)cell * a.ldst;
        const float T = s[0], N = s[1], H = s[2];
        float eSum = 0.f, d22 = 0.f;
        for (int q = 0; q < a.nslot; ++q) {
            const float d = s[3 + q] * a.slot_abun[q] * H;
            dens[q * 64 + lane] = d;
            if (a.slot_efac[q] != 0.f) eSum = eSum + a.slot_efac[q] * d;
            if (q == a.slot_he2) d22 = d;
        }
        if (part == 0) {                          // bin 1's free-free term
            const float log10Te = log10f(T);
            const float sqrTe = sqrtf(T);
            const float expo = (kTe1Ryd / T) + a.nu1;
            const float cb1 = expo > 84.f ? 0.f : expf(-expo);
            const float g1 = gaunt_ff(0.f, log10Te, a.xlf1);
            // (density(1,2) + density(2,2) + 4 density(2,3) + eDenFFSum): the
            // H+ and He++ densities are never set in ionizationDriver's loop
            float t = 0.f + d22;
            t = t + 4.f * 0.f;
            t = t + eSum;
            const float fac1 = (N / 1.e10f) * (t / 1.e10f) / sqrTe;
            const float fac2 = fac1 * kTe1Ryd / T;
            if (cb1 < 0.995f) ff1 = (a.brems1 * (1.f - cb1) * g1) * fac1;
            else ff1 = (a.brems1 * a.nu1 * g1) * fac2;
        }
        if (a.ndrow) {
            const float *Td = a.Tdust + (size_t)cell * (a.nsMax + 1) * (a.nSizes + 1);
            for (int r = 0; r < a.ndrow; ++r) {
                const int sp = r / a.nSizes + 1, ai = r % a.nSizes + 1;
                const float td = Td[sp + (a.nsMax + 1) * ai];
                wr[r * 64 + lane] = (td < a.tsub[r]) ? a.dw[r] * a.ndust[cell] : -1.f;
            }
        }
    }
    const int *cut = a.cuts + (parts - 1) * (parts + 2) / 2 + part;
    const int i0 = cut[0], i1 = cut[1];
    if (i0 >= i1) return;
    if (!__any(cell > 0)) {
        for (int i = i0; i < i1; ++i) {
            const size_t o = ((size_t)tile * a.nb + i) * 64 + lane;
            a.opac3[o] = 0.f;
            if (a.sca3) a.sca3[o] = 0.f;
        }
        return;
    }
    int bound = a.bin_start[min(i0 + lane, a.nb)];       // where bin i0 + lane begins
    int e = __builtin_amdgcn_readlane(bound, 0), r = 0;
    const int2 *E = reinterpret_cast<const int2 *>(a.ent) + lane;
    int2 now = E[e], next = E[e + 64];
    for (int i = i0; i < i1; ++i) {
        const int b = (i - i0 + 1) & 63;
        if (b == 0) bound = a.bin_start[min(i + 1 + lane, a.nb)];
        const int e1 = __builtin_amdgcn_readlane(bound, b);
        float acc = i == 0 ? 0.f + ff1 : 0.f, sca = 0.f;
        for (; e < e1; e += 4, r += 4) {
            if (r == 64) {
                now = next;
                next = E[e + 64];
                r = 0;
            }
            int qk[4];
            float sigma[4], d[4];
#pragma unroll
            for (int k = 0; k < 4; ++k) {
                qk[k] = __builtin_amdgcn_readlane(now.x, r + k);
                sigma[k] = __uint_as_float((unsigned)__builtin_amdgcn_readlane(now.y, r + k));
                d[k] = dens[(qk[k] >> 1) * 64 + lane];
            }
            // a heavy ion (qk odd) counts only where its density is above zero
#pragma unroll
            for (int k = 0; k < 4; ++k)
                if (!(qk[k] & 1) || d[k] > 0.f) acc = acc + sigma[k] * d[k];
        }
        if (cell > 0) {
            if (a.ndrow) {
                float ab = 0.f;
                for (int r = 0; r < a.ndrow; ++r) {
                    const float w = wr[r * 64 + lane];
                    if (w < 0.f) continue;
                    sca = sca + w * a.dsca[(size_t)r * a.nb + i];
                    ab = ab + w * a.dabs[(size_t)r * a.nb + i];
                }
                acc = acc + (sca + ab);
            }
        } else {
            acc = 0.f;
        }
        const size_t o = ((size_t)tile * a.nb + i) * 64 + lane;   // padding points get 0
        a.opac3[o] = acc;
        if (a.sca3) a.sca3[o] = sca;
    }
}

__global__ void state_kernel(const double *Te, const double *Ne, const double *Hden, const double *ion, int nE,
                             int nst1, const int *slot_e, const int *slot_stage, int nslot, int nc, float *st,
                             int ldst)
{
    const int cell = blockIdx.x * blockDim.x + threadIdx.x;
    if (cell > nc) return;
    float *s = st + (size_t)cell * ldst;
    s[0] = (float)Te[cell];
    s[1] = (float)Ne[cell];
    s[2] = (float)Hden[cell];
    const double *x = ion + (size_t)cell * nE * nst1;
    for (int q = 0; q < nslot; ++q) s[3 + q] = (float)x[slot_e[q] * nst1 + slot_stage[q]];
}

__global__ void f32_kernel(const double *in, size_t n, float *out)
{
    const size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) out[i] = (float)in[i];
}

}  // namespace mco

hipError_t mco_launch_opacity(const mco::OpacArgs &a, size_t lds_bytes, hipStream_t s)
{
    const unsigned tiles = (unsigned)(mcd::j3_points(a.js) / 64);
    // wavefronts for the chip (16 a CU), at least four a tile; each lays out
    // the tile's densities for itself, which eight a tile repeated too often
    // (0.18 against 0.15 ms for H and He on 45^3; 0.25 against 0.31 with 80
    // segments, at twice the cost of a bin)
    const unsigned want = (4096 + tiles - 1) / tiles;
    const unsigned parts = want < 4 ? 4 : want > mco::kMaxParts ? mco::kMaxParts : want;
    hipLaunchKernelGGL(mco::opacity_kernel, dim3(tiles * parts), dim3(64), lds_bytes, s, a, (int)parts);
    return hipGetLastError();
}

hipError_t mco_launch_state(const double *Te, const double *Ne, const double *Hden, const double *ion, int nE,
                            int nst1, const int *slot_e, const int *slot_stage, int nslot, int nc, float *st,
                            int ldst, hipStream_t s)
{
    hipLaunchKernelGGL(mco::state_kernel, dim3((nc + 1 + 255) / 256), dim3(256), 0, s, Te, Ne, Hden, ion, nE, nst1,
                       slot_e, slot_stage, nslot, nc, st, ldst);
    return hipGetLastError();
}

hipError_t mco_launch_f32(const double *in, size_t n, float *out, hipStream_t s)
{
    if (n == 0) return hipSuccess;
    hipLaunchKernelGGL(mco::f32_kernel, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, s, in, n, out);
    return hipGetLastError();
}

namespace mco {
__global__ void gather_kernel(const float *t3, mcd::J3Shape js, const int *cell_xyz, int nc, int nb, float *out)
{
    const size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    const size_t nc1 = (size_t)nc + 1;
    if (i >= nc1 * nb) return;
    const size_t cell = i % nc1, nu = i / nc1;
    out[i] = cell == 0 ? 0.f : t3[mcd::j3_index(nb, (int)nu, mcd::j3_point_of(js, cell_xyz[cell]))];
}
}  // namespace mco

namespace mco {
// A tiled table as rows [cell][nb]: a tile's 64 points by 64 bins through
// LDS, lanes over points on the way in and over bins on the way out.
__global__ void __launch_bounds__(256) rows_kernel(const float *t3, mcd::J3Shape js, const int *active, int nb, float *out)
{
    __shared__ float v[64][65];
    __shared__ int cell[64];
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6, nu0 = blockIdx.y * 64;
    const unsigned p0 = blockIdx.x * 64u;
    if (w == 0) {
        const int xyz = mcd::j3_lattice(js, p0 + (unsigned)lane);
        cell[lane] = xyz >= 0 ? active[xyz] : 0;
    }
    const float *t = t3 + mcd::j3_index(nb, 0, p0) + lane;
    for (int q = w; q < 64 && nu0 + q < nb; q += 4) v[lane][q] = t[(size_t)(nu0 + q) * mcd::kJTile];
    __syncthreads();
    for (int q = w; q < 64; q += 4)
        if (cell[q] > 0 && nu0 + lane < nb) out[(size_t)cell[q] * nb + nu0 + lane] = v[q][lane];
}
}  // namespace mco

namespace mco {
// Rows [cell][nb] as the host's columns (0:nc, nb), 64 cells by 64 bins through
// LDS.  Bound by the copy to the host that follows.  The whole build call of a
// 36^3 octant, H and He on 400 bins (39 MB of columns): 13.3 ms with one host
// thread laying them out, 2.2 now.
__global__ void __launch_bounds__(256) columns_kernel(const float *__restrict__ rows, size_t nc1, int nb,
                                                      float *__restrict__ out)
{
    __shared__ float v[64][65];
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6, nu0 = blockIdx.y * 64;
    const size_t c0 = (size_t)blockIdx.x * 64;
    for (int q = w; q < 64 && c0 + q < nc1; q += 4)
        if (nu0 + lane < nb) v[q][lane] = rows[(c0 + q) * nb + nu0 + lane];
    __syncthreads();
    for (int q = w; q < 64 && nu0 + q < nb; q += 4)
        if (c0 + lane < nc1) out[c0 + lane + nc1 * (nu0 + q)] = v[lane][q];
}
}  // namespace mco

hipError_t mco_launch_columns(const float *rows, size_t nc1, int nb, float *out, hipStream_t s)
{
    hipLaunchKernelGGL(mco::columns_kernel, dim3((unsigned)((nc1 + 63) / 64), (unsigned)((nb + 63) / 64)), dim3(256), 0, s,
                       rows, nc1, nb, out);
    return hipGetLastError();
}

hipError_t mco_launch_rows(const float *t3, const mcd::J3Shape &js, const int *active, int nb, float *out, hipStream_t s)
{
    hipLaunchKernelGGL(mco::rows_kernel, dim3((unsigned)(mcd::j3_points(js) / 64), (unsigned)((nb + 63) / 64)), dim3(256),
                       0, s, t3, js, active, nb, out);
    return hipGetLastError();
}

hipError_t mco_launch_gather(const float *t3, const mcd::J3Shape &js, const int *cell_xyz, int nc, int nb,
                             float *out, hipStream_t s)
{
    const size_t n = ((size_t)nc + 1) * nb;
    hipLaunchKernelGGL(mco::gather_kernel, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, s, t3, js, cell_xyz, nc,
                       nb, out);
    return hipGetLastError();
}
