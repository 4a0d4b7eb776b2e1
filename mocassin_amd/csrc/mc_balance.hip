// mc_balance.hip - per-cell ionisation and thermal balance (MOCASSIN's
// updateCell, update_mod.f90:15-525) on MI355X, FP64.
//
// One 64-lane wavefront per cell (one wavefront per workgroup), or several
// cells to a wavefront where there are no model ions; cell state in LDS.
// Lanes share the work of each stage of the reference's schedule:
//   * photoionisation rates and heating integrals: a kernel of their own
//     before the balance, lanes over lattice points (update_mod.f90:184-269,
//     1146-1234);
//   * recombination fits, charge exchange, ion ratios: lanes over the
//     (elem, ion) channels (calcAlpha, radRecFit, dielectronic, ionBalance);
//   * CEL cooling: the n-level systems of four model ions at a time, one in
//     each row of 16 lanes (mc_cel.h);
//   * the bracketed false-position T iteration and the fixed-point ion
//     iteration run uniformly on the wavefront (iterateT, ionBalance).
// The collision-strength spline second derivatives depend only on the
// atomic data, so they are computed once at setup (the reference recomputes
// them on every call; the values are the same).
#include "mc_balance.h"
#include "mc_cel.h"
#include "mc_device.h"
#include "mc_grid_limit.h"
#include "mc_mlp.h"

#include <algorithm>
#include <cstdarg>
#include <cstdio>

#pragma clang fp contract(off)

namespace mcb {

constexpr int W = 64;

// A cell's state in LDS, sized by the atomic data: what stays through the
// balance, then a block that serves the ion fixed point first and the level
// solves after it, then the grains'.
struct Scalars { double Te, Ne, Hden, red; };
struct Lds {
    Scalars *v;
    double *ion;                     // [nE][ns1]
    double *nPhot, *heatNu;          // [nch]
    double *ratio, *den, *diO;       // [nch], [nE], [ns1]: ion fixed point
    void *cel;                       // the solves' block
    int ns1;
};
// the solves' block: records [ncel], cooling [ncel], rates [most]
__host__ __device__ inline size_t cel_bytes(int ncel, int most)
{
    return ((size_t)ncel * (sizeof(CelRec) + sizeof(double)) + 15) / 16 * 16 + (size_t)most * sizeof(double2);
}
__host__ __device__ inline size_t state_bytes(int nE, int ns1, int nch)
{
    return (sizeof(Scalars) + sizeof(double) * ((size_t)nE * ns1 + 2 * nch) + 15) / 16 * 16;
}
__host__ __device__ inline size_t shared_bytes(int ncel, int most, int nE, int ns1, int nch)
{
    const size_t cel = cel_bytes(ncel, most), ions = sizeof(double) * ((size_t)nch + nE + ns1);
    return ncel > 0 && cel > ions ? cel : ions;
}
__device__ __forceinline__ Lds lds_of_cell(const Atomic &A, char *at)
{
    Lds S;
    const int ns1 = A.nstages + 1, nch = A.nch;
    S.ns1 = ns1;
    S.v = reinterpret_cast<Scalars *>(at);
    S.ion = reinterpret_cast<double *>(S.v + 1);
    S.nPhot = S.ion + A.nE * ns1;
    S.heatNu = S.nPhot + nch;
    S.cel = at + state_bytes(A.nE, ns1, nch);
    S.ratio = static_cast<double *>(S.cel);
    S.den = S.ratio + nch;
    S.diO = S.den + A.nE;
    return S;
}

// orders the LDS accesses of a wavefront, the whole of a workgroup here (its
// cells' groups of lanes may stand at different places)
__device__ __forceinline__ void wave_order()
{
    __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
    __builtin_amdgcn_wave_barrier();
}

__device__ double rad_rec(const Channel &c, double Te)
{
    if (c.rr_kind == 0) {
        double tt = sqrt(Te / c.rr[2]);
        return c.rr[0] / (tt * pow(tt + 1.0, 1.0 - c.rr[1]) * pow(1.0 + sqrt(Te / c.rr[3]), 1.0 + c.rr[1]));
    }
    double tt = Te * 1.e-4;
    if (c.rr_kind == 2) return c.rr[0] / pow(tt, c.rr[1] + c.rr[2] * log10(tt));
    return c.rr[0] / pow(tt, c.rr[1]);
}

// dielectronic (update_mod.f90:1782-1834) for one (elem, ion): the last
// satisfying Nussbaumer-Storey row, else (or above 6e4 K) Aldrovandi-Pequignot
__device__ double di_rec(const Atomic &A, int ndr, const int *dr, int ap, double Te)
{
    double v = 0.0;
    double t = Te / 10000.;
    for (int r = 0; r < ndr; ++r) {
        const int i = dr[r];
        const int g = A.dr_g[i];
        if (g == 0 || (g == 1 && Te < 20000.) || (g == 2 && Te >= 20000.)) {
            const double *c = A.dr_real[i];
            v = 1.e-12 * (c[0] / t + c[1] + c[2] * t + c[3] * (t * t)) * pow(t, -1.5) * exp(-c[4] / t);
        }
    }
    if (Te > 60000. || v == 0.0) {
        if (ap >= 0) {
            const double *c = A.ap_real[ap];
            v = c[0] * pow(Te, -1.5) * exp(-c[2] / Te) * (1.0 + c[1] * exp(-c[3] / Te));
        } else {
            v = 0.0;
        }
    }
    return v;
}

// total cooling at temperature T for the cell's current ionisation and Ne
// (thermBalance, update_mod.f90:933-1113: H and He free-free and
// recombination fits, H collisional excitation, CEL lines); valid on lane 0.
// Cells on fewer lanes than a wavefront have no model ions.
template <int G>
__device__ __forceinline__ double cooling(const Atomic &A, const Lds &S, int lane, double T)
{
    double cool = 0.0;
    if constexpr (G == W) {
        CelRec *rec = static_cast<CelRec *>(S.cel);
        double *ions = reinterpret_cast<double *>(rec + A.ncel);
        double2 *rate = reinterpret_cast<double2 *>(static_cast<char *>(S.cel) + cel_bytes(A.ncel, 0));
        const double sqrTe = sqrt(T), log10Te = log10(T);
        for (int k = lane; k < A.ncel; k += W) {
            const CelIon &ci = A.cel[k];
            const double xi = S.ion[ci.eidx * S.ns1 + ci.ion];
            const double up = (ci.ion < A.nstages) ? S.ion[ci.eidx * S.ns1 + ci.ion + 1] / xi : 0.0;
            rec[A.cel_place[k]] = cel_record(A, ci, T, log10Te, up, A.el[ci.eidx].abun, xi);
        }
        wave_order();
        // CEL cooling of each model ion [erg/s per H] from its levels 1..10
        // (forLines, equilibrium and the cooling sum of thermBalance), its terms
        // added in the reference's order
        for (int b = 0; b < A.ncelb; ++b) {
            const CelBatch &B = A.celb[b];
            const CelRec *R = rec + kCelSlots * b;
            const CelLevels L = cel_levels(A, b, R, rate, lane, T, sqrTe, S.v->Ne);
            const int g = lane >> 4, r = lane & 15, n = B.most;
            const bool mine = r < B.rows[g];
            const double part = L.y / L.sum, s1 = R[mine ? g : 0].ab, s2 = R[mine ? g : 0].x;
            const double kE = 1.9865e-16;
            const double *ae = A.cel_ae + (size_t)b * kMaxLev * 64 + lane;
            const int *term = A.cel_term + (size_t)b * kMaxLev * 64 + lane;
            double cool = 0.0;
            static_for<0, 9>([&](auto Lo) {
                constexpr int lo = decltype(Lo)::value;          // lower level lo + 1, upper r + 2 <= 10
                if (lo < n) {
                    const double f = ae[64 * lo] * part * s1 * s2 * kE;
                    const double t = term[64 * lo] >= 0 ? f : 0.0;
                    static_for<lo, 9>([&](auto Up) {
                        constexpr int up = decltype(Up)::value;
                        cool = cool + row_lane<up>(t);
                    });
                }
            });
            if (r == 0 && mine) ions[B.ion[g]] = R[g].skip ? 0.0 : cool;
        }
        wave_order();
        for (int k = 0; k < A.ncel; ++k) cool = cool + ions[k];
        wave_order();
    }
    if (lane != 0) return 0.0;
    const double Ne = S.v->Ne, kB = 1.380658e-16, hcRyd = 2.1799153e-11;
    const double lg = log10(T), Te4 = T / 1.e4;
    double Np = S.ion[0 * S.ns1 + 2] * A.el[0].abun;
    double bFF = 1.0108464E-11 + 9.7930778E-13 * lg - 6.6433144E-13 * lg * lg +
                 2.4793747E-13 * lg * lg * lg - 2.3938215E-14 * lg * lg * lg * lg;
    double coolFF = Np * Ne * bFF * kB * T / sqrt(T);
    double bRec = 9.4255985E-11 - 4.04794384E-12 * lg - 1.0055237E-11 * lg * lg +
                  1.99266862E-12 * lg * lg * lg - 1.06681387E-13 * lg * lg * lg * lg;
    double coolRec = Np * Ne * bRec * kB * T / sqrt(T);
    // (with two stages there is no He++, nor a word for it in the row)
    Np = S.ns1 > 3 ? S.ion[1 * S.ns1 + 3] * A.el[1].abun : 0.0;
    const double ls = log10(T / 4.);
    bFF = 2. * (1.0108464E-11 + 9.7930778E-13 * ls - 6.6433144E-13 * ls * ls +
                2.4793747E-13 * ls * ls * ls - 2.3938215E-14 * ls * ls * ls * ls);
    coolFF = coolFF + Np * Ne * bFF * kB * T / sqrt(T / 4.);
    bRec = 2. * (9.4255985E-11 - 4.04794384E-12 * ls - 1.0055237E-11 * ls * ls +
                 1.99266862E-12 * ls * ls * ls - 1.06681387E-13 * ls * ls * ls * ls);
    coolRec = coolRec + Np * Ne * bRec * kB * T / sqrt(T / 4.);
    Np = S.ion[1 * S.ns1 + 2] * A.el[1].abun;
    bFF = 1.070073e-11 - 2.5730207e-13 * lg + 2.109134e-13 * lg * lg;
    coolFF = coolFF + Np * Ne * bFF * kB * T / sqrt(T);
    bRec = 9.4255985E-11 - 4.04794384E-12 * lg - 1.0055237E-11 * lg * lg +
           1.99266862E-12 * lg * lg * lg - 1.06681387E-13 * lg * lg * lg * lg;
    coolRec = coolRec + Np * Ne * bRec * kB * T / sqrt(T);
    double coolColl = 0.0;
    if (T > 5000.)
        coolColl = (2.47e-8 * exp(-118338. / T) * pow(Te4, -0.228) +
                    1.32e-8 * exp(-140252. / T) * pow(Te4, -0.460)) *
                   hcRyd * S.ion[0 * S.ns1 + 1] * Ne;
    coolColl = coolColl + cool;
    return coolFF + coolRec + coolColl;
}

// ---- grains: charge, photoelectric heating, gas-grain collisions ---------
// (update_mod.f90:527-932).  Per temperature iteration, after the ion fixed
// point: every grain row's potential (setGrainPotential's secant iteration,
// at most 100 steps), then the photoelectric heating and cooling
// (setPhotoelHeatCool) and the collision terms (setDustGasCollHeatCool).
// The rows are independent, and each step of a row's iteration waits for the
// one before: so all rows iterate at once, each on its own group of lanes
// (the cell's lanes over the next power of two of the rows), instead of one
// after another on all of them.  The sums over frequency are linear in the
// potential for every bin above the threshold (yield Y (1 - V/d) with d = nu
// - vn, photoelectron energy Y (d - V^2/d) / 2), so the cell's suffix sums of
// u, u/d and u d (u = Y sigma flux) over 16 chunks of bins are formed once,
// and a step adds up the bins of the threshold's chunk alone.  Bound by the
// latency of the steps: the balance kernel of the dust and gas 60^3 grid (10
// rows, 160 bins) took 38 ms with one row at a time over all bins, 11.5 with
// all rows at once, 6.3 with four cells to a wavefront besides.
constexpr double kPiR = (double)3.141592654f;             // constants_mod.f90:32 (REAL)
constexpr double kFourPiR = (double)(4.f * 3.141592654f);
constexpr double kHcRyd = 2.1799153e-11, kRyd2erg = 2.1799e-11, kKB = 1.380658e-16;
constexpr double kAmu = 1.66053e-24, kMe = 9.109382e-28;
constexpr int kChunks = 16;              // of the frequency bins

// a cell's grain block
struct GrainLds {
    double *pf;                      // [nbins] photon flux
    double *w;                       // [nch] n(ion) v_mean of each channel's ion
    double *nu0;                     // [kChunks] first bin of each chunk
    double *gdc, *peh, *hg, *gg;     // [K]
    double *tot;                     // gas-grain cooling, photoelectric heating
    double *sums;                    // [3][kChunks + 1][K]
};
__host__ __device__ inline size_t grain_bytes(int nb, int nch, int K)
{
    return sizeof(double) * ((size_t)nb + nch + kChunks + 4 * K + 2 + 3 * (kChunks + 1) * (size_t)K);
}
__device__ __forceinline__ GrainLds grain_lds(int nb, int nch, int K, char *at)
{
    GrainLds L;
    L.pf = reinterpret_cast<double *>(at);
    L.w = L.pf + nb;
    L.nu0 = L.w + nch;
    L.gdc = L.nu0 + kChunks;
    L.peh = L.gdc + K;
    L.hg = L.peh + K;
    L.gg = L.hg + K;
    L.tot = L.gg + K;
    L.sums = L.tot + 2;
    return L;
}

__device__ __forceinline__ double minr(double a, double b) { return a < b ? a : b; }
__device__ __forceinline__ double maxr(double a, double b) { return a > b ? a : b; }

// The rows' geometry: lane `sub` of the n lanes of row `row` (the last row
// again on lanes without one, which are not live).
struct RowLane {
    int n, row, sub;
    bool live;
};
template <int G>
__device__ __forceinline__ RowLane row_lanes(int K, int lane)
{
    RowLane R;
    R.n = G;
    while (G / R.n < K) R.n >>= 1;
    R.row = lane / R.n;
    R.sub = lane % R.n;
    R.live = R.row < K;
    if (!R.live) R.row = K - 1;
    return R;
}

// sum over a row's n lanes, on each of them (every lane active)
__device__ __forceinline__ double row_sum(double v, int n)
{
    if (n > 1) v += __builtin_amdgcn_update_dpp(0.0, v, 0xB1, 0xf, 0xf, true);      // quad_perm 1 0 3 2
    if (n > 2) v += __builtin_amdgcn_update_dpp(0.0, v, 0x4E, 0xf, 0xf, true);      // quad_perm 2 3 0 1
    if (n > 4) v += __builtin_amdgcn_update_dpp(0.0, v, 0x141, 0xf, 0xf, true);     // row_half_mirror
    if (n > 8) v += __builtin_amdgcn_update_dpp(0.0, v, 0x140, 0xf, 0xf, true);     // row_mirror
    if (n > 16) v += __shfl_xor(v, 16);
    if (n > 32) v += __shfl_xor(v, 32);
    return v;
}

// The spectrum's part of a row: bins above x = max(vn + V, vn), which locate
// (interpolation_mod.f90:48-81) finds on the increasing mesh; its answer 1
// for x equal to the last bin is `whole`.
struct Spectrum {
    const double *nu, *pf, *yn, *ax, *qa, *sums;
    double vn;
    int nb, K, row, size;             // size: bins of a chunk
    // chunk of x: the last whose first bin is at or below x, -1 before all
    __device__ __forceinline__ int chunk(const GrainLds &L, double x) const
    {
        int lo = 0, hi = kChunks;     // nu0 is infinite beyond the mesh
        while (lo < hi) {
            const int mid = (lo + hi) >> 1;
            if (L.nu0[mid] > x) hi = mid; else lo = mid + 1;
        }
        return lo - 1;
    }
    __device__ __forceinline__ double sum(int q, int c) const { return sums[(q * (kChunks + 1) + c) * K + row]; }
};

// getGrainEmission (update_mod.f90:601-651) at potential V: this lane's part
__device__ __forceinline__ double grain_emission(const Spectrum &P, const GrainLds &L, double perArea, double V,
                                                 const RowLane &R)
{
    const double x = maxr(P.vn + V, P.vn);
    const int c = P.chunk(L, x);
    double sum = 0.0;
    for (int u = R.sub; u < P.size; u += R.n) {
        const int f = c * P.size + u;
        if (c >= 0 && f < P.nb && P.nu[f] > x) {
            const double Yhat = P.yn[f] * minr(1., maxr(0., 1. - V / (P.nu[f] - P.vn)));
            sum = sum + Yhat * (P.pf[f] * kFourPiR) * P.qa[f];
        }
    }
    if (R.sub == 0) {
        const double a = P.sum(0, c + 1);
        sum = sum + (V < 0. ? a : a - V * P.sum(1, c + 1)) * perArea;
    }
    if (__any(x == P.nu[P.nb - 1])) {
        double all = 0.0;
        for (int f = 1 + R.sub; f < P.nb; f += R.n)
            all = all + P.yn[f] * minr(1., maxr(0., 1. - V / (P.nu[f] - P.vn))) * (P.pf[f] * kFourPiR) * P.qa[f];
        sum = x == P.nu[P.nb - 1] ? all : sum;
    }
    return sum;
}

// getGrainRecombination (update_mod.f90:656-733), the ions' part of this lane
__device__ __forceinline__ double grain_ions(const Atomic &A, const GrainLds &L, double kT, double V, const RowLane &R)
{
    double ions = 0.0;
    for (int k = R.sub; k < A.nch; k += R.n) {
        double et = (double)A.ch[k].ion * V / kT;
        et = et <= 0. ? 1. - et : exp(-et);
        ions = ions + L.w[k] * et;
    }
    return ions;
}
__device__ __forceinline__ double grain_electrons(double kT, double eNe, double V)
{
    double eta = -(V / kT);
    eta = eta <= 0. ? 1. - eta : exp(-eta);
    return eNe * eta;
}

// the suffix sums of a cell's spectrum, once per cell
template <int N>
__device__ __forceinline__ void grain_sums(const Atomic &A, const Grains &G, const GrainLds &L, int lane)
{
    const double *pf = L.pf;
    double *sums = L.sums;
    const int nb = A.nbins, K = G.K, size = (nb + kChunks - 1) / kChunks;
    for (int c = lane; c < kChunks; c += N) L.nu0[c] = c * size < nb ? A.nu[c * size] : __builtin_inf();
    for (int t = lane; t < K * kChunks; t += N) {
        const int k = t % K, c = t / K, s = k / G.nSizes;
        const double vn = G.vn[s];
        const double *ax = G.absx + (size_t)k * nb, *yn = G.yn + (size_t)s * nb;
        double a = 0.0, b = 0.0, e = 0.0;
        for (int f = c * size; f < min(nb, (c + 1) * size); ++f) {
            const double d = A.nu[f] - vn;
            if (!(d > 0.)) continue;
            const double u = yn[f] * ax[f] * pf[f];
            a = a + u;
            b = b + u / d;
            e = e + u * d;
        }
        sums[(0 * (kChunks + 1) + c) * K + k] = a;
        sums[(1 * (kChunks + 1) + c) * K + k] = b;
        sums[(2 * (kChunks + 1) + c) * K + k] = e;
    }
    wave_order();
    for (int t = lane; t < 3 * K; t += N) {
        double *p = sums + (t / K) * (kChunks + 1) * K + t % K;
        double v = 0.0;
        p[kChunks * K] = 0.0;
        for (int c = kChunks - 1; c >= 0; --c) {
            v = v + p[c * K];
            p[c * K] = v;
        }
    }
    wave_order();
}

// the grain block of iterateT after ionBalance (update_mod.f90:367-388) and
// the two heat/cool terms it adds to thermBalance (1252-1255)
template <int N>
__device__ __forceinline__ void grain_terms(const Atomic &A, const Grains &G, const GrainLds &L, const Lds &S, int lane, int cell)
{
    const double *pf = L.pf, *sums = L.sums;
    const int nb = A.nbins, K = G.K, nch = A.nch;
    const double Te = S.v->Te, Ne = S.v->Ne, Hden = S.v->Hden;
    const double kT = 6.336e-6 * Te, e8 = 1.1045e-15 * Te / kPiR;
    // n(ion) v_mean of the ions; electrons ((Ne vmean) S) with S = 1
    for (int k = lane; k < nch; k += N) {
        const int e = A.ch[k].eidx, st = A.ch[k].ion + 1;
        const double cpDen = S.ion[e * S.ns1 + st] * A.el[e].abun * Hden;
        const double vm = sqrt(e8 / (G.aweight[A.el[e].z - 1] * kAmu));
        L.w[k] = cpDen * vm * 1.;
    }
    wave_order();
    const double eNe = Ne * sqrt(e8 / kMe) * 1.;
    const RowLane R = row_lanes<N>(K, lane);
    const int k = R.row, s = k / G.nSizes, ai = k % G.nSizes;
    const double vn = G.vn[s], rad = G.radius[ai];
    const Spectrum P{ A.nu, pf, G.yn + (size_t)s * nb, G.absx + (size_t)k * nb, G.qa + (size_t)k * nb, sums, vn, nb, K,
                      k, (nb + kChunks - 1) / kChunks };
    const double perArea = kFourPiR / (1.e-8 * rad * rad);
    // setGrainPotential: secant on emission - recombination, from 0 V
    double slope = 0., potOld = 0.;
    double emiOld = row_sum(grain_emission(P, L, perArea, 0., R), R.n);
    double recOld = grain_electrons(kT, eNe, 0.) - row_sum(grain_ions(A, L, kT, 0., R), R.n);
    double pot = potOld + 0.05;
    bool done = !R.live;
    for (int n = 1; n <= 100 && __any(!done); ++n) {
        const double threshold = maxr(vn + pot, vn);
        const double emi = row_sum(grain_emission(P, L, perArea, pot, R), R.n);
        const double rec = grain_electrons(kT, eNe, pot) - row_sum(grain_ions(A, L, kT, pot, R), R.n);
        double delta = emi - rec;
        double delta1 = fabs(delta / (0.5 * maxr(1.e-35, emi + rec)));
        done = done || delta1 < 0.005;
        if (!done) {
            if (pot != potOld) {
                const double fac = (emi - emiOld) - (rec - recOld);
                if (fac != 0.) slope = fac / (pot - potOld);
            }
            potOld = pot;
            recOld = rec;
            emiOld = emi;
            delta1 = -(delta / slope);
            delta = minr(fabs(delta1), 0.05 * threshold);
            delta = signbit(delta1) ? -fabs(delta) : fabs(delta);
            pot = pot + delta;
        }
    }
    // setPhotoelHeatCool.  The photoelectron energy is zero below vn + |V|,
    // and the bin that locate returns (the last at or below the threshold,
    // which can lie below vn) counts too.
    {
        const double x = maxr(vn + pot, vn), x2 = vn + fabs(pot);
        const int c = P.chunk(L, x), c2 = P.chunk(L, x2);
        double hE = 0.0, hY = 0.0;
        for (int u = R.sub; u < P.size; u += R.n) {
            const int f = c * P.size + u, f2 = c2 * P.size + u;
            if (c >= 0 && f < nb) {
                const double nu = A.nu[f], q = P.ax[f] * pf[f], d = nu - vn;
                const bool last = !(nu > x) && (f == nb - 1 || A.nu[f + 1] > x);
                if (nu > x || last) hY = hY + q * (P.yn[f] * minr(1., maxr(0., 1. - pot / d)));
                if (last) hE = hE + q * (P.yn[f] * 0.5 * minr(d, maxr(0., (d * d - pot * pot) / d)));
            }
            if (c2 >= 0 && f2 < nb && A.nu[f2] > x2) {
                const double d = A.nu[f2] - vn;
                hE = hE + P.ax[f2] * pf[f2] * (P.yn[f2] * 0.5 * minr(d, maxr(0., (d * d - pot * pot) / d)));
            }
        }
        if (R.sub == 0) {
            hY = hY + (P.sum(0, c + 1) - maxr(pot, 0.) * P.sum(1, c + 1));
            hE = hE + 0.5 * (P.sum(2, c2 + 1) - pot * pot * P.sum(1, c2 + 1));
        }
        // x at the last bin (locate gives the first), or a potential that is
        // no number: bin by bin
        const bool whole = x == A.nu[nb - 1] || pot != pot;
        if (__any(whole)) {
            double aE = 0.0, aY = 0.0;
            for (int f = R.sub; f < nb; f += R.n) {
                const double d = A.nu[f] - vn, q = P.ax[f] * pf[f];
                aY = aY + q * (P.yn[f] * minr(1., maxr(0., 1. - pot / d)));
                aE = aE + q * (P.yn[f] * 0.5 * minr(d, maxr(0., (d * d - pot * pot) / d)));
            }
            hE = whole ? aE : hE;
            hY = whole ? aY : hY;
        }
        hE = row_sum(hE, R.n);
        hY = row_sum(hY, R.n);
        if (R.live && R.sub == 0) {
            L.peh[k] = hE * kHcRyd / kPiR;
            L.hg[k] = (hE - hY * pot) * G.gabun[s] * G.weight[ai];
        }
    }
    // setDustGasCollHeatCool: a row's lanes over the channels, each with its
    // ionised stage, the first of an element with the neutral one too.  The
    // neutral stage sees the ionisation potential of the stage before it in
    // the reference's order (0 at the start).
    double gd = 0.0, gg = 0.0;
    const double ms = G.msurf[s], nd = G.ndust[cell];
    const double Td = G.Tdust[(size_t)cell * (G.nsMax + 1) * (G.nSizes + 1) + (s + 1) + (G.nsMax + 1) * (ai + 1)];
    auto stage = [&](int e, int st, int from) {
        const double mcp = G.aweight[A.el[e].z - 1] * kAmu;
        const double vmean = sqrt(e8 / mcp);
        const double Z = (double)(st - 1), IPerg = from >= 0 ? A.nu[A.ch[from].ip - 1] * kRyd2erg : 0.0;
        const double S_ = st == 1 ? 2. * mcp * ms / ((mcp + ms) * (mcp + ms)) : 1.;
        const double psi = Z * pot / kT;
        double eta, xi;
        if (psi <= 0.) { eta = 1. - psi; xi = 1. - psi / 2.; }
        else { eta = exp(-psi); xi = (1. + psi / 2.) * eta; }
        const double x = S.ion[e * S.ns1 + st], ab = A.el[e].abun;
        gd = gd + x * ab * Hden * kPiR * rad * rad * 1.e-8 * S_ * vmean *
                      (2. * kT * kRyd2erg * xi - eta * (Z * pot * kRyd2erg - IPerg + 2. * kKB * Td));
        gg = gg + x * G.weight[ai] * G.gabun[s] * nd * ab * kPiR * rad * rad * 1.e-8 * S_ * vmean *
                      (2. * kT * kRyd2erg * xi - eta * 2. * kKB * Td);
    };
    for (int j = R.sub; j < nch; j += R.n) {
        const Channel &ch = A.ch[j];
        if (ch.ion == 1) stage(ch.eidx, 1, j - 1);
        stage(ch.eidx, ch.ion + 1, j);
    }
    if (R.sub == 0) {
        // electrons
        const double vme = sqrt(e8 / kMe), Z = -1.;
        const double psi = Z * pot / kT;
        double eta, xi;
        if (psi <= 0.) { eta = 1. - psi; xi = 1. - psi / 2.; }
        else { eta = exp(-psi); xi = (1. + psi / 2.) * eta; }
        gd = gd + Ne * kPiR * rad * rad * 1.e-8 * 1. * vme * (2. * kT * kRyd2erg * xi - eta * (Z * pot * kRyd2erg));
        gg = gg + Ne * G.weight[ai] * G.gabun[s] * nd * kPiR * rad * rad * 1.e-8 * 1. * vme *
                  (2. * kT * kRyd2erg * xi) / Hden;
    }
    gd = row_sum(gd, R.n);
    gg = row_sum(gg, R.n);
    if (R.live && R.sub == 0) {
        L.gdc[k] = gd / kFourPiR;
        L.gg[k] = gg;
    }
    wave_order();
    if (lane == 0) {
        double p = 0.0, q = 0.0;
        for (int r = 0; r < K; ++r) { p = p + L.hg[r]; q = q + L.gg[r]; }
        L.tot[1] = p * nd * kHcRyd / Hden;
        L.tot[0] = q / kFourPiR;
    }
    wave_order();
}

// G lanes a cell.  Registers for three wavefronts a SIMD with model ions (5.6
// ms on the 45^3 octant; two take 6.6; for four more would spill than the 71
// registers that do), for two without (the chain of steps bounds it: dust and
// gas 60^3 6.3 ms against 7.0 for three and 8.0 for four).
template <bool PE, int G>
__global__ void __launch_bounds__(64) __attribute__((amdgpu_waves_per_eu(G == 64 ? 3 : 2))) balance_kernel(const Atomic *__restrict__ Ap, CellArgs a)
{
    extern __shared__ __align__(16) char dyn[];
    const Atomic &A = *Ap;
    const int lane = threadIdx.x % G;
    const int slot = (int)blockIdx.x * (W / G) + (int)threadIdx.x / G;
    if (slot >= a.ncells) return;
    const int cell = a.order ? a.order[slot] : slot + 1;
    const int ns = A.nstages, nE = A.nE, nch = A.nch;
    char *mine = dyn + (size_t)(threadIdx.x / G) * a.cell_lds;
    const Lds S = lds_of_cell(A, mine);
    double *ionOut = a.ion + (size_t)cell * nE * (ns + 1);

    // hit test (update_mod.f90:104-154) and the channel integrals, both
    // from integrals_kernel
    if (!a.hit[cell]) {
        if (lane == 0) { a.flags[cell] = 16; a.nIter[cell] = 0; }
        return;
    }
    if (lane == 0) {
        S.v->Te = a.Te[cell];
        S.v->Ne = a.Ne[cell];
        S.v->Hden = a.Hden[cell];
    }
    for (int i = lane; i < nE * (ns + 1); i += G) S.ion[(i / (ns + 1)) * S.ns1 + i % (ns + 1)] = ionOut[i];
    for (int k = lane; k < nch; k += G) {
        S.nPhot[k] = 1.e-20 + a.Rint[(size_t)cell * nch + k];
        S.heatNu[k] = a.Hint[(size_t)cell * nch + k];
    }
    GrainLds GL{};
    if (PE) {
        // the cell's photon flux J/(h c Ryd nu) (getGrainEmission, setPhotoelHeatCool)
        const Grains &D = *a.grains;
        GL = grain_lds(A.nbins, nch, D.K, mine + state_bytes(nE, ns + 1, nch) + shared_bytes(A.ncel, A.cel_most, nE, ns + 1, nch));
        const unsigned pt = mcd::j3_point_of(mcd::j3_shape(D.nx, D.ny, D.nz), D.cell_xyz[cell]);
        for (int f = lane; f < A.nbins; f += G)
            GL.pf[f] = D.J3[mcd::j3_index(A.nbins, f, pt)] * a.jscale / (kHcRyd * A.nu[f]);
        wave_order();
        grain_sums<G>(A, D, GL, lane);
    }
    wave_order();
    // lgConverged compares with the caller's H0 fraction (update_mod.f90:510-515)
    const double XOldHI = a.ion0 ? a.ion0[(size_t)cell * nE * (ns + 1) + 1] : S.ion[0 * S.ns1 + 1];

    const bool on = lane < nch;
    const Channel &c = A.ch[on ? lane : 0];
    const double abun = A.el[c.eidx].abun;
    const int ch0 = A.el[lane < nE ? lane : 0].ch0, chn = A.el[lane < nE ? lane : 0].nch;
    int nIterT = 0, flags = 0, lgIBConv = 1, nTot = 0;
    for (int attempt = 0;; ++attempt) {
        nIterT = 0;
        flags = 0;
        lgIBConv = 1;
        double rHigh = 0., rLow = 0., Thigh = 0., Tlow = 0.;        // reference schedule
        double Tp = 0., fp = 0., Tlo = 0., Thi = 0.;                // secant iteration
        bool havep = false, haveLo = false, haveHi = false;
        for (;;) {
            nIterT++;
            const double Te = S.v->Te;
            // calcAlpha: radiative + dielectronic (oxygen rows fill empty entries)
            for (int i = 1 + lane; i < ns; i += G)
                S.diO[i] = di_rec(A, A.odr_n[i], A.odr[i], A.oap[i], Te);
            wave_order();
            // a lane's channel (no cell has more channels than lanes): its
            // recombination and charge-exchange coefficients, and what the
            // fixed point adds to its rates that depends on Te alone
            double al = 0.0, cx = 0.0, coll = 0.0, back = 0.0;
            if (on) {
                al = rad_rec(c, Te);
                if (c.elem >= 3) {
                    double d = di_rec(A, c.ndr, c.dr, c.ap, Te);
                    if (d == 0.0) d = S.diO[c.ion];
                    al = al + d;
                }
                // charge-exchange rate coefficient (ionBalance, 1448-1455)
                const double t4 = Te / 10000.;
                cx = c.chex[0] * pow(t4, c.chex[1]) * (1. + c.chex[2] * exp(c.chex[3] * t4));
                if (cx < 0.) cx = 0.;
                if (Te < 6000. || Te > 5.e4) cx = 0.;
                if (lane == 0) {
                    double expFact = 157893.94 / Te;
                    if (expFact > 75.) expFact = 75.;
                    coll = 2.75E-16 * Te * sqrt(Te) * (157893.94 / Te + 2.) * exp(-expFact);
                }
                if (c.dEk > 1.0) back = exp(-c.dEk / Te);
            }
            // ionBalance fixed point (1320-1622).  It is a chain of steps
            // that wait for each other, up to 25 of them: so a step keeps
            // its rates in registers, forms an element's products in one
            // pass and sums Ne on every lane.
            int nIterX = 1;
            double Ne = S.v->Ne;
            const double Hden = S.v->Hden;
            for (;;) {
                const double HIOld = S.ion[1], HeIOld = S.ion[S.ns1 + 1], HeIIOld = S.ion[S.ns1 + 2];
                const double xH0 = HIOld;
                if (on) {
                    double revRate = 0.0;
                    if (c.dEk > 1.0) revRate = cx * (1. - xH0) * Hden * 2. * back / c.g0g1;
                    S.ratio[lane] = (S.nPhot[lane] + coll + revRate) / (Ne * al + cx * Hden * xH0);
                }
                wave_order();
                if (lane < nE) {
                    double r[kMaxStage - 1], den = 1.0, p = 1.0;
#pragma unroll
                    for (int i = 0; i < kMaxStage - 1; ++i) r[i] = S.ratio[ch0 + (i < chn ? i : 0)];
#pragma unroll
                    for (int i = 0; i < kMaxStage - 1; ++i)
                        if (i < chn) {
                            p = p * r[i];
                            den = den + p;
                            S.ratio[ch0 + i] = p;
                        }
                    S.den[lane] = den;
                }
                wave_order();
                if (on) {
                    const double den = S.den[c.eidx];
                    double v = S.ratio[lane] / den;
                    if (v > 0.99999) v = 0.99999;
                    if (v < 1.e-20) v = 1.e-20;
                    S.ion[c.eidx * S.ns1 + c.ion + 1] = v;
                    // the electrons of this stage
                    S.ratio[lane] = v >= 1.e-10 ? (double)c.ion * abun * v : 0.0;
                    if (c.ion == 1) {
                        v = 1.0 / den;
                        if (v > 0.99999) v = 0.99999;
                        if (v < 1.e-20) v = 1.e-20;
                        S.ion[c.eidx * S.ns1 + 1] = v;
                    }
                }
                wave_order();
                Ne = 0.0;
                for (int k = 0; k < nch; ++k) Ne = Ne + S.ratio[k];
                Ne = Ne * Hden;
                if (Ne == 0.0) Ne = 1.0;
                const double dHI = (S.ion[1] - HIOld) / HIOld;
                const double dHeI = (S.ion[S.ns1 + 1] - HeIOld) / HeIOld;
                const double dHeII = (S.ion[S.ns1 + 2] - HeIIOld) / HeIIOld;
                wave_order();
                const bool big = fabs(dHI) > a.ion_tol || fabs(dHeI) > a.ion_tol || fabs(dHeII) > a.ion_tol;
                if (big && nIterX < 25) { nIterX++; continue; }
                lgIBConv = !(big && nIterX == 25);
                break;
            }
            // the heating of each channel, summed in order
            if (on) S.ratio[lane] = S.heatNu[lane] * S.ion[c.eidx * S.ns1 + c.ion] * abun;
            if (lane == 0) S.v->Ne = Ne;
            wave_order();
            double heat = 0.0;
            for (int k = 0; k < nch; ++k) heat = heat + S.ratio[k];
            wave_order();
            if (PE) grain_terms<G>(A, *a.grains, GL, S, lane, cell);
            // thermBalance (933-1258)
            double cool = cooling<G>(A, S, lane, S.v->Te);
            if (lane == 0) S.v->red = cool;
            wave_order();
            cool = S.v->red;
            if (PE) {
                // the grain terms of thermBalance (1252-1255)
                cool = cool + GL.tot[0];
                heat = heat + GL.tot[1];
            }
            wave_order();
            // iterateT false-position update (398-458)
            const double res = heat - cool;
            double Tn = S.v->Te;
            bool again = false;
            if (a.solver == 0) {
                if (fabs(res) >= 0.01 * heat) {
                    if (nIterT < 25) {
                        if (res < 0.) {
                            rLow = res; Tlow = Tn;
                            Tn = (Thigh != 0.) ? Tlow - (Thigh - Tlow) * rLow / (rHigh - rLow) : Tn / 1.2;
                        } else {
                            rHigh = res; Thigh = Tn;
                            Tn = (Tlow != 0.) ? Tlow - (Thigh - Tlow) * rLow / (rHigh - rLow) : Tn * 1.2;
                        }
                        if (nIterT >= 6 && fabs(Thigh - Tlow) <= 0.002 * (Thigh + Tlow)) {
                            if (res < 0.) { Tn = Thigh - 100.; Thigh = 0.; }
                            else { Tn = Tlow + 100.; Tlow = 0.; }
                        }
                        if (Tn <= 0.) Tn = 1.;
                        again = true;
                    } else {
                        if (Thigh == 0.) Tn = Tlow;
                        else if (Tlow == 0.) Tn = Thigh;
                        else Tn = (Thigh + Tlow) * 0.5;
                        flags |= 2 | 4;
                    }
                }
            } else if (fabs(res) > a.tol * heat) {
                // secant steps on f(T) = heat - cool, kept inside the bracket
                // once both signs have been seen (f > 0: heating wins, T rises)
                const double f = res, T = Tn;
                if (f > 0.) { Tlo = T; haveLo = true; } else { Thi = T; haveHi = true; }
                const double bl = fmin(Tlo, Thi), bh = fmax(Tlo, Thi);
                // a warm-started attempt gets warm_iter iterations before
                // the restart from the caller's state
                const int cap = (attempt == 0 && a.Te0) ? min(a.max_iter, a.warm_iter) : a.max_iter;
                if (nIterT >= cap) {
                    if (haveLo && haveHi) Tn = 0.5 * (bl + bh);
                    flags |= 2 | 4;
                } else if (haveLo && haveHi && bh - bl <= 1.e-7 * T) {
                    Tn = 0.5 * (bl + bh);
                } else {
                    // first trial: a step of the relative residual (cooling
                    // grows about linearly with T near balance), divided by
                    // the expected slope d(f/heat)/d ln T, at most step0
                    const double d0 = fmin(a.step0, fmax(fabs(f) / heat / a.slope0, 1.e-4));
                    double Tc = (havep && f != fp) ? T - f * (T - Tp) / (f - fp)
                                                   : (f > 0. ? T * (1. + d0) : T / (1. + d0));
                    if (haveLo && haveHi) {
                        if (!(Tc > bl && Tc < bh)) Tc = 0.5 * (bl + bh);
                    } else {
                        if (f > 0. && !(Tc > T)) Tc = T * 1.2;
                        if (f < 0. && !(Tc < T)) Tc = T / 1.2;
                        Tc = fmin(fmax(Tc, T / 1.5), T * 1.5);
                    }
                    Tp = T;
                    fp = f;
                    havep = true;
                    Tn = Tc;
                    again = true;
                }
            }
            wave_order();
            if (lane == 0) S.v->Te = Tn;
            wave_order();
            if (!again) break;
        }
        nTot += nIterT;
        const bool failed = (flags & 4) != 0 || !lgIBConv;
        if (failed && attempt == 0 && a.Te0) {
            // restart from the caller's state (the reference's starting point)
            const double *src = a.ion0 + (size_t)cell * nE * (ns + 1);
            for (int i = lane; i < nE * (ns + 1); i += G) S.ion[(i / (ns + 1)) * S.ns1 + i % (ns + 1)] = src[i];
            if (lane == 0) { S.v->Te = a.Te0[cell]; S.v->Ne = a.Ne0[cell]; }
            wave_order();
            continue;
        }
        if (attempt > 0) flags |= 32;
        break;
    }
    if (!lgIBConv) flags |= 2 | 8;
    const double dXHI = (S.ion[0 * S.ns1 + 1] - XOldHI) / XOldHI;
    if (fabs(dXHI) <= (double)A.XHILimit) flags |= 1;
    for (int i = lane; i < nE * (ns + 1); i += G) ionOut[i] = S.ion[(i / (ns + 1)) * S.ns1 + i % (ns + 1)];
    if (PE && lane < a.grains->K) {
        // terms of the last temperature iteration, for getDustT
        const Grains &D = *a.grains;
        D.gdc[(size_t)cell * D.K + lane] = GL.gdc[lane];
        D.peh[(size_t)cell * D.K + lane] = GL.peh[lane];
    }
    if (lane == 0) {
        a.Te[cell] = S.v->Te;
        a.Ne[cell] = S.v->Ne;
        a.flags[cell] = flags;
        a.nIter[cell] = nTot;
    }
}

// Per lattice point (one lane each, so that every read of J3[nu][xyz] is
// coalesced across the wavefront): the photoionisation rate and heating
// integrals of every channel (update_mod.f90:184-269, 1146-1234), the hit
// flag (104-154) and, when X is given, the warm-start network's features of
// the cell (row cell-1 of X [nCells][72]): log10 of J summed over 64
// contiguous groups of bins, log10 nH, log10 abundances of its seven
// elements (-30 when absent).
//
// A wavefront takes kIntCh channels of one tile of 64 points; the wavefronts
// of a tile follow each other on one XCD, so that its L2 serves the tile's J
// to all but the first.  The coefficients of a channel are wavefront-uniform
// and come by scalar loads, 16 bins at a time, which leaves LDS out of the
// loop.  Bound by the FP64 products for large grids and by the chain of bins
// for small ones.  45^3 octant, 800
// bins, 31 channels: 1.61 ms with all channels in one wavefront, 0.23 now;
// 21^3: 1.39, 0.15 now (two or eight channels, or eight bins: 0.30 to 0.43 and
// 0.15 to 0.39).
constexpr int kIntCh = 4, kIntBins = 16;

struct Coeffs { double v[kIntBins]; };
__device__ __forceinline__ Coeffs uniform_row(const double *p)
{
    typedef const __attribute__((address_space(4))) Coeffs *Row;
    return *(const Coeffs *)(Row)(uint64_t)p;
}

__global__ void __launch_bounds__(64) integrals_kernel(const Atomic *__restrict__ Ap, CellArgs a,
                                                       const double *__restrict__ J3,
                                                       const int *__restrict__ active, mcd::J3Shape js, int groups,
                                                       unsigned tile0, double *__restrict__ Rint, double *__restrict__ Hint,
                                                       int *__restrict__ hit, float *__restrict__ X)
{
    const Atomic &A = *Ap;
    const int lane = threadIdx.x;
    const unsigned i = blockIdx.x >> 3, tile = tile0 + (i / groups) * 8 + (blockIdx.x & 7);
    const int g0 = (int)(i % groups) * kIntCh;
    if (tile >= mcd::j3_points(js) / mcd::kJTile) return;
    const int xyz = mcd::j3_lattice(js, tile * 64u + (unsigned)lane);
    const int cell = xyz >= 0 ? active[xyz] : 0;
    if (!__any(cell > 0)) return;
    const int nb = A.nbins, nch = A.nch;
    // this wavefront's tile of J3: [nu][64 points], contiguous
    const double *Jp = J3 + mcd::j3_index(nb, 0, tile * 64u) + lane;
    const int ng = nch - g0 < kIntCh ? nch - g0 : kIntCh;
    double r[kIntCh], h[kIntCh];
    for (int k = 0; k < kIntCh; ++k) { r[k] = 0.0; h[k] = 0.0; }
    // the first group visits every bin (hit flag, band sums)
    int jlo = nb + 1, jhi = 0;
    for (int k = 0; k < ng; ++k) {
        const Channel &c = A.ch[g0 + k];
        jlo = c.ip < jlo ? c.ip : jlo;
        const int hi = c.hiR > c.hiH ? c.hiR : c.hiH;
        jhi = hi > jhi ? hi : jhi;
    }
    float *brow = nullptr;
    if (g0 == 0) {
        jlo = 1;
        jhi = nb;
        if (X && cell > 0) brow = X + (size_t)(cell - 1) * mcm::kIn;
    }
    double band = 0.0;
    int any = 0, b = 0, bend = nb / mcm::kBands;
    double next[kIntBins];
    for (int u = 0; u < kIntBins; ++u)
        next[u] = jlo + u <= jhi ? Jp[(size_t)(jlo + u - 1) * mcd::kJTile] : 0.0;
    for (int j0 = jlo; j0 <= jhi; j0 += kIntBins) {
        double J[kIntBins];
        for (int u = 0; u < kIntBins; ++u) {
            J[u] = next[u] * a.jscale;
            const int j = j0 + kIntBins + u;
            next[u] = j <= jhi ? Jp[(size_t)(j - 1) * mcd::kJTile] : 0.0;
        }
        if (j0 + kIntBins - 1 <= jhi) {
#pragma unroll
            for (int k = 0; k < kIntCh; ++k)
                if (k < ng) {
                    const size_t o = (size_t)(g0 + k) * nb + j0 - 1;
                    const Coeffs cr = uniform_row(A.cR + o), ch = uniform_row(A.cH + o);
#pragma unroll
                    for (int u = 0; u < kIntBins; ++u) {
                        r[k] = __builtin_fma(J[u], cr.v[u], r[k]);
                        h[k] = __builtin_fma(J[u], ch.v[u], h[k]);
                    }
                }
        } else {
#pragma unroll
            for (int u = 0; u < kIntBins; ++u)
                if (j0 + u <= jhi) {
#pragma unroll
                    for (int k = 0; k < kIntCh; ++k)
                        if (k < ng) {
                            const size_t o = (size_t)(g0 + k) * nb + j0 - 1 + u;
                            r[k] = __builtin_fma(J[u], A.cR[o], r[k]);
                            h[k] = __builtin_fma(J[u], A.cH[o], h[k]);
                        }
                }
        }
        if (g0 == 0)
#pragma unroll
            for (int u = 0; u < kIntBins; ++u) {
                any |= J[u] > 0.0;
                band += J[u];
                if (j0 + u == bend) {
                    if (brow) brow[b] = (float)log10(fmax(band, 1.e-30));
                    band = 0.0;
                    ++b;
                    // (no bin beyond the mesh ends a band)
                    bend = b < mcm::kBands ? (b + 1) * nb / mcm::kBands : 0;
                }
            }
    }
    if (cell <= 0) return;
#pragma unroll
    for (int k = 0; k < kIntCh; ++k)
        if (k < ng) {
            Rint[(size_t)cell * nch + g0 + k] = r[k];
            Hint[(size_t)cell * nch + g0 + k] = h[k];
        }
    if (g0 != 0) return;
    hit[cell] = any;
    if (brow) {
        float *row = brow;
        row[mcm::kBands] = (float)log10(a.Hden[cell]);
        for (int k = 0; k < 7; ++k) {
            float v = -30.f;
            for (int e = 0; e < A.nE; ++e)
                if (A.el[e].z == mcm::kSlotsZ[k] && A.el[e].abun > 0.0) v = (float)log10(A.el[e].abun);
            row[mcm::kBands + 1 + k] = v;
        }
    }
}

// Warm start of reached cells from the network's (unscaled) outputs Y
// [nCells][ldy]: Te = 10^y0, the seven elements' fractions 10^y normalised
// per element and clamped as ionBalance clamps them, Ne from them.
__global__ void warm_kernel(const Atomic *__restrict__ Ap, CellArgs a, const float *__restrict__ Y, int ldy,
                            const int *__restrict__ hit)
{
    const Atomic &A = *Ap;
    const int cell = blockIdx.x * blockDim.x + threadIdx.x + 1;
    if (cell > a.ncells || !hit[cell]) return;
    const int ns = A.nstages, nE = A.nE;
    const float *y = Y + (size_t)(cell - 1) * ldy;
    double *ion = a.ion + (size_t)cell * nE * (ns + 1);
    a.Te[cell] = fmin(fmax(pow(10.0, (double)y[0]), 500.0), 2.e5);
    int base = 1;
    for (int k = 0; k < 7; ++k) {
        const int z = mcm::kSlotsZ[k], nslot = z + 1 < mcm::kStageMax ? z + 1 : mcm::kStageMax;
        for (int e = 0; e < nE; ++e) {
            if (A.el[e].z != z) continue;
            const int nst = A.el[e].nst;
            double v[kMaxStage], sum = 0.0;
            for (int st = 1; st <= nst; ++st) {
                v[st] = st <= nslot ? pow(10.0, fmin((double)y[base + st - 1], 0.0)) : 0.0;
                sum += v[st];
            }
            for (int st = 1; st <= nst; ++st) {
                double x = sum > 0.0 ? v[st] / sum : (st == 1 ? 1.0 : 0.0);
                x = fmin(fmax(x, 1.e-20), 0.99999);
                ion[e * (ns + 1) + st] = x;
            }
        }
        base += nslot;
    }
    double Ne = 0.0;
    for (int e = 0; e < nE; ++e)
        for (int st = 2; st <= A.el[e].nst; ++st) {
            const double x = ion[e * (ns + 1) + st];
            if (x >= 1.e-10) Ne = Ne + (double)(st - 1) * A.el[e].abun * x;
        }
    a.Ne[cell] = Ne * a.Hden[cell] > 0.0 ? Ne * a.Hden[cell] : 1.0;
}

// ---- analytic line luminosities (outputGas, output_mod.f90:302-520) -----
// One wavefront per block of consecutive cells.  Per batch of four model
// ions (outer loop, so that a lane's sums stay in registers: its upper level,
// 16 lower ones): every cell's level populations (mc_cel.h), then forLines'
// emissivity times Hden * getVolume.  The records of kLineCells cells are made
// together, one lane each.  Each block writes its sums to its own row of
// `part`; lines_reduce_kernel adds the rows in block order, so the result
// does not depend on scheduling.
constexpr int kLineCells = W / kCelSlots;

__device__ __forceinline__ float line_volume(const LineArgs &a, int cell)
{
    // getVolume (grid_mod.f90:2876-2964) of the cell's lattice point: the
    // per-axis widths over 1e15 multiplied in FP32 as (dx * dy) * dz
    const int l = a.cell_xyz[cell];
    const int ix = l % a.nx, iy = (l / a.nx) % a.ny, iz = l / (a.nx * a.ny);
    return (a.dfac[ix] * a.dfac[a.nx + iy]) * a.dfac[a.nx + a.ny + iz];
}

__global__ void __launch_bounds__(64) lines_kernel(const Atomic *__restrict__ Ap, LineArgs a)
{
    __shared__ CelRec recs[W];                   // [cell][slot]
    __shared__ float hds[kLineCells], dvs[kLineCells], tes[kLineCells], nes[kLineCells];
    __shared__ double hsum;
    extern __shared__ __align__(16) double2 rate[];
    const Atomic &A = *Ap;
    const int lane = threadIdx.x;
    const int nE = A.nE, ns = A.nstages;
    const int c0 = 1 + blockIdx.x * a.cells_per_blk;
    const int c1 = min(a.ncells, c0 + a.cells_per_blk - 1);
    double *out = a.part + (size_t)blockIdx.x * a.ldp;
    // forLines' 1.9865e9 is a REAL literal
    const double kL = (double)1.9865e9f;
    const int g = lane >> 4, r = lane & 15;
    for (int b = 0; b < A.ncelb; ++b) {
        const CelBatch &B = A.celb[b];
        const bool mine = r < B.rows[g];
        const double *ae = A.cel_ae + (size_t)b * kMaxLev * 64 + lane;
        const int *term = A.cel_term + (size_t)b * kMaxLev * 64 + lane;
        double acc[16];
        for (int l = 0; l < 16; ++l) acc[l] = 0.0;
        for (int cc = c0; cc <= c1; cc += kLineCells) {
            __syncthreads();
            {
                const int cell = cc + lane / kCelSlots, k = B.ion[lane % kCelSlots];
                if (cell <= c1) {
                    // the state as the host grid stores it (REAL)
                    const float te = (float)a.Te[cell];
                    if (k >= 0) {
                        const CelIon &ci = A.cel[k];
                        const double *ion = a.ion + ((size_t)cell * nE + ci.eidx) * (ns + 1);
                        const float x = (float)ion[ci.ion];
                        const float up = (ci.ion < ns) ? (float)ion[ci.ion + 1] / x : 0.f;
                        recs[lane] = cel_record(A, ci, (double)te, log10((double)te), (double)up,
                                                (double)(float)A.el[ci.eidx].abun, (double)x);
                    }
                    if (lane % kCelSlots == 0) {
                        const int u = lane / kCelSlots;
                        tes[u] = te;
                        nes[u] = (float)a.Ne[cell];
                        hds[u] = (float)a.Hden[cell];
                        dvs[u] = line_volume(a, cell);
                    }
                }
            }
            __syncthreads();
            for (int cell = cc; cell <= min(c1, cc + kLineCells - 1); ++cell) {
                if (a.black && (a.black[cell] & a.black_mask)) continue;
                const int u = cell - cc;
                const CelRec *R = recs + kCelSlots * u;
                const double Te = (double)tes[u], hd = (double)hds[u], dv = (double)dvs[u];
                const CelLevels L = cel_levels(A, b, R, rate, lane, Te, sqrt(Te), (double)nes[u]);
                const double part = L.y / L.sum;
                const double abun = R[mine ? g : 0].ab, x = R[mine ? g : 0].x;
                const bool on = mine && !R[mine ? g : 0].skip;
                static_for<0, 16>([&](auto Lo) {
                    constexpr int lo = decltype(Lo)::value;
                    if (lo < B.most) {
                        double f = ae[64 * lo] * part;
                        f = f * abun * x;
                        f = f * kL;
                        const double t = acc[lo] + f * hd * dv;
                        acc[lo] = on && term[64 * lo] >= 0 ? t : acc[lo];
                    }
                });
            }
        }
        for (int s = 0; s < kCelSlots; ++s)
            for (int e = lane; e < kLineEnt; e += W)
                if (B.ion[s] >= 0 && (e % kMaxLev >= e / kMaxLev || e / kMaxLev > B.rows[s]))
                    out[(size_t)B.ion[s] * kLineEnt + e] = 0.0;
        for (int lo = 0; lo < 16; ++lo)
            if (mine && lo <= r) out[(size_t)B.ion[g] * kLineEnt + (r + 1) * kMaxLev + lo] = acc[lo];
    }
    // RecLinesEmission's Hbeta (output_mod.f90:2065-2079), HIRecLines(4,2) =
    // (fh/hb) * Hbeta = Hbeta, times Hden * dV
    double hb = 0.0;
    const double abunH = (double)(float)A.el[0].abun;
    for (int cell = c0 + lane; cell <= c1; cell += W) {
        if (a.black && (a.black[cell] & a.black_mask)) continue;
        const float te = (float)a.Te[cell], ne = (float)a.Ne[cell], hd = (float)a.Hden[cell];
        const float xp = (float)a.ion[((size_t)cell * nE) * (ns + 1) + 2];
        float h = 2530.f / powf(te, 0.833f);
        h = h * ne * xp * (float)abunH;
        hb = hb + (double)h * (double)hd * (double)line_volume(a, cell);
    }
    // lanes in order: a fixed summation order
    if (lane == 0) hsum = 0.0;
    __syncthreads();
    for (int l = 0; l < W; ++l) {
        if (lane == l) hsum = hsum + hb;
        __syncthreads();
    }
    if (lane == 0) out[(size_t)A.ncel * kLineEnt] = hsum;
}

// out[t] = sum over blocks b (in order) of part[b][t]; four wavefronts per
// 64 outputs, each over every fourth block, combined in wavefront order
__global__ void __launch_bounds__(256) lines_reduce_kernel(const double *__restrict__ part, int ldp, int nblk,
                                                           int n, double *__restrict__ out)
{
    __shared__ double red[4][W];
    const int lane = threadIdx.x % W, w = threadIdx.x / W;
    const int t = blockIdx.x * W + lane;
    double sum = 0.0;
    if (t < n)
        for (int b = w; b < nblk; b += 4) sum = sum + part[(size_t)b * ldp + t];
    red[w][lane] = sum;
    __syncthreads();
    if (w == 0 && t < n) out[t] = ((red[0][lane] + red[1][lane]) + red[2][lane]) + red[3][lane];
}

}  // namespace mcb

hipError_t mcb_launch_balance(const mcb::Atomic *dA, const mcb::CellArgs &a, hipStream_t s)
{
    if (a.ncells <= 0) return hipSuccess;
    // A cell has a wavefront, or without model ions 16 lanes (at most 16
    // channels, elements and grain rows) or 4 (at most 4, no grains): cells
    // side by side instead of idle lanes.  172000 cells of H and He, reference
    // schedule: 7.2 ms with a wavefront a cell, 1.1 with 4 lanes; secant from
    // the network's prediction, bound by the slowest cell's steps: 3.1 and
    // 1.7.  The same with grains, dust and gas 60^3: 11.5 and 6.3 (16 lanes).
    // Grains on many bins or rows have a wavefront a cell again: a row's few
    // lanes then sum long chunks one after another, and four cells' LDS lets
    // few wavefronts on a CU (with 4096 bins and 16 rows it is more than a CU
    // has).  Both grow alike, so the line is drawn by the LDS.  30000 cells,
    // 16 lanes against 64, ms, by the KB of four cells: 10 rows 160 bins (25)
    // 2.5, 3.6, 320 bins (30) 4.4, 4.3, 640 bins (40) 8.7, 6.0; 16 rows 96
    // bins (33) 3.7, 4.0, 240 bins (37) 5.8, 4.9; 5 rows 640 bins (31) 2.9, 3.1.
    const int K = a.grains ? a.grains_rows : 0, most = std::max(a.nch, a.nE);
    constexpr size_t kSideBySide = 32 * 1024;
    mcb::CellArgs b = a;
    b.cell_lds = (mcb::state_bytes(a.nE, a.ns1, a.nch) + mcb::shared_bytes(a.ncel, a.cel_most, a.nE, a.ns1, a.nch) +
                  (K ? mcb::grain_bytes(a.grains_nb, a.nch, K) : 0) + 7) / 8 * 8;
    const bool wide = a.ncel > 0 || most > 16 || K > 16 || (K > 0 && 4 * b.cell_lds > kSideBySide);
    const int lanes = wide ? 64 : most > 4 || K > 0 ? 16 : 4;
    // an odd number of words apart, the cells' equal words lie in different banks
    if (lanes < 64 && b.cell_lds % 16 == 0) b.cell_lds += 8;
    const int per = 64 / lanes;
    const dim3 grid((a.ncells + per - 1) / per);
    const size_t lds = b.cell_lds * per;
    auto *kernel = K ? (lanes == 64 ? mcb::balance_kernel<true, 64> : mcb::balance_kernel<true, 16>)
                     : lanes == 64 ? mcb::balance_kernel<false, 64>
                                   : lanes == 16 ? mcb::balance_kernel<false, 16> : mcb::balance_kernel<false, 4>;
    hipLaunchKernelGGL(kernel, grid, dim3(64), lds, s, dA, b);
    return hipGetLastError();
}

hipError_t mcb_launch_integrals(const mcb::Atomic *dA, const mcb::CellArgs &a, const double *J3, const int *active,
                               int nx, int ny, int nz, double *Rint, double *Hint, int *hit, float *X, hipStream_t s)
{
    const mcd::J3Shape js = mcd::j3_shape(nx, ny, nz);
    const unsigned tiles = (unsigned)(mcd::j3_points(js) / mcd::kJTile);
    const int groups = a.nch > mcb::kIntCh ? (a.nch + mcb::kIntCh - 1) / mcb::kIntCh : 1;
    const unsigned most = mcb::tiles_per_launch((unsigned)groups);
    for (unsigned t = 0; t < tiles; t += most) {
        const unsigned n = std::min(most, tiles - t);
        hipLaunchKernelGGL(mcb::integrals_kernel, dim3((n + 7) / 8 * 8 * groups), dim3(64), 0, s, dA, a, J3, active, js,
                           groups, t, Rint, Hint, hit, X);
        const hipError_t e = hipGetLastError();
        if (e != hipSuccess) return e;
    }
    return hipSuccess;
}

hipError_t mcb_launch_warm(const mcb::Atomic *dA, const mcb::CellArgs &a, const float *Y, int ldy, const int *hit,
                           hipStream_t s)
{
    if (a.ncells <= 0) return hipSuccess;
    hipLaunchKernelGGL(mcb::warm_kernel, dim3((a.ncells + 255) / 256), dim3(256), 0, s, dA, a, Y, ldy, hit);
    return hipGetLastError();
}

hipError_t mcb_launch_lines(const mcb::Atomic *dA, const mcb::LineArgs &a, int nblk, int ncel, double *out,
                            hipStream_t s)
{
    if (nblk <= 0) return hipSuccess;
    hipLaunchKernelGGL(mcb::lines_kernel, dim3(nblk), dim3(64), a.cel_most * sizeof(double2), s, dA, a);
    const int n = ncel * mcb::kLineEnt + 1;
    hipLaunchKernelGGL(mcb::lines_reduce_kernel, dim3((n + 63) / 64), dim3(256), 0, s, a.part, a.ldp, nblk, n, out);
    return hipGetLastError();
}

// ------------------------------------------------------------ host tables
namespace mcb {
namespace {

// Charge-exchange fits (elem, ion, a, b, c, d) with a in units of 1e-9
// cm^3 s^-1, in the order ionBalance assigns them (update_mod.f90:1389-1446):
// the second Ar II/III pair replaces the first, as there.
struct ChexRow { int elem, ion; double a, b, c, d; };
const ChexRow kChex[] = {
    {2, 1, 7.47e-6, 2.06, 9.93, -3.89},    {2, 2, 1.e-5, 0., 0., 0.},
    {3, 2, 1.26, 0.96, 3.02, -0.65},       {3, 3, 1.e-5, 0., 0., 0.},
    {4, 2, 1.e-5, 0., 0., 0.},             {4, 3, 1.e-5, 0., 0., 0.},
    {4, 4, 5.17, 0.82, -.69, -1.12},       {5, 2, 2.e-2, 0., 0., 0.},
    {5, 3, 1.e-5, 0., 0., 0.},             {5, 4, 5.27e-1, 0.76, -0.63, -1.17},
    {6, 1, 1.76e-9, 8.33, 4278.78, -6.41}, {6, 2, 1.67e-4, 2.79, 304.72, -4.07},
    {6, 3, 3.25, 0.21, 0.19, -3.29},       {6, 4, 332.46, -0.11, -0.995, -1.58e-3},
    {7, 1, 1.01e-3, -0.29, -0.92, -8.38},  {7, 2, 3.05e-1, 0.60, 2.65, -0.93},
    {7, 3, 4.54, 0.57, -0.65, -0.89},      {7, 4, 3.28, 0.52, -0.52, -0.19},
    {8, 1, 1.04, 3.15e-2, -0.61, -9.73},   {8, 2, 1.04, 0.27, 2.02, -5.92},
    {8, 3, 3.98, 0.26, 0.56, -2.62},       {8, 4, 2.52e-1, 0.63, 2.08, -4.16},
    {9, 2, 1.e-5, 0., 0., 0.},             {9, 3, 9.86, 0.29, -0.21, -1.15},
    {9, 4, 7.15e-1, 1.21, -0.70, -0.85},   {10, 2, 1.e-5, 0., 0., 0.},
    {10, 3, 14.73, 4.52e-2, -0.84, -0.31}, {10, 4, 6.47, 0.54, 3.59, -5.22},
    {11, 2, 1.e-5, 0., 0., 0.},            {11, 3, 1.33, 1.15, 1.20, -0.32},
    {11, 4, 1.01e-1, 1.34, 10.05, -6.41},  {12, 2, 8.58e-5, 2.49e-3, 2.93e-2, -4.33},
    {12, 3, 6.49, 0.53, 2.82, -7.63},      {12, 4, 6.36, 0.55, 3.86, -5.19},
    {13, 2, 1.e-5, 0., 0., 0.},            {13, 3, 7.11e-5, 4.12, 1.72e4, -22.24},
    {13, 4, 7.52e-1, 0.77, 6.24, -5.67},   {14, 2, 1.23, 0.24, 3.17, 4.18e-3},
    {14, 3, 4.900e-1, -8.74e-2, -0.36, -0.79}, {14, 4, 7.58, 0.37, 1.06, -4.09},
    {16, 1, 3.82e-7, 11.10, 2.57e4, -8.22}, {16, 2, 1.e-5, 0., 0., 0.},
    {16, 3, 2.29, 4.02e-2, 1.59, -6.06},   {16, 4, 6.44, 0.13, 2.69, -5.69},
    {18, 2, 1.e-5, 0., 0., 0.},            {18, 3, 4.57, 0.27, -0.18, -1.57},
    {18, 4, 6.37, 2.12, 10.21, -6.22},     {18, 3, 3.17e-2, 2.12, 12.06, -0.40},
    {18, 4, 2.68, 0.69, -0.68, -4.47},     {26, 2, 1.26, 7.72e-2, -0.41, -7.31},
    {26, 3, 3.42, 0.51, -2.06, -8.99},
};

int err(char *e, size_t n, int code, const char *fmt, ...)
{
    va_list ap;
    va_start(ap, fmt);
    vsnprintf(e, n, fmt, ap);
    va_end(ap);
    return code;
}

// natural cubic spline second derivatives (spline, interpolation_mod.f90:
// 182-266, with zero end derivatives of second order)
void spline_nat(const double *xa, const double *ya, int n, double *y2)
{
    double u[kMaxTemp];
    y2[0] = 0.0;
    u[0] = 0.0;
    for (int i = 1; i < n - 1; ++i) {
        const double sig = (xa[i] - xa[i - 1]) / (xa[i + 1] - xa[i - 1]);
        const double p = sig * y2[i - 1] + 2.0;
        y2[i] = (sig - 1.0) / p;
        double v = ya[i + 1];
        v = v - ya[i];
        v = v / (xa[i + 1] - xa[i]);
        v = v - (ya[i] - ya[i - 1]) / (xa[i] - xa[i - 1]);
        u[i] = (6.0 * v / (xa[i + 1] - xa[i - 1]) - sig * u[i - 1]) / p;
    }
    y2[n - 1] = 0.0;
    for (int k = n - 2; k >= 0; --k) y2[k] = y2[k] * y2[k + 1] + u[k];
}

// dielectronic rows (direc_coeffs, aldropequi_coeffs) that fill (z, ion)
// (dielectronic, update_mod.f90:1782-1834); returns their number, or -1
// with a message in e
int dr_rows(const mc_atomic *in, int ns, int z, int ion, int *rows, int *ap, char *e, size_t n)
{
    int nr = 0;
    for (int i = 0; i < 25; ++i) {
        const int el = in->dr_int[3 * i], nn = in->dr_int[3 * i + 1];
        const int io = el + 1 - nn;
        if (el != z || io != ion || io > ns || io < 1) continue;
        if (nr == kMaxDr) {
            err(e, n, MC_ETABLE, "more than %d dielectronic rows for Z=%d ion %d", kMaxDr, z, ion);
            return -1;
        }
        rows[nr++] = i;
    }
    *ap = -1;
    for (int i = 0; i < 167; ++i) {
        const int el = in->ap_int[2 * i], nn = in->ap_int[2 * i + 1];
        const int io = el + 1 - nn;
        if (el == z && io == ion && io >= 1 && io <= ns) *ap = i;
    }
    return nr;
}

// The batches of model ions and the tables their lanes read (mc_cel.h) from
// each ion's levels (energies, then A(up, lo) at up + nl lo) and weights.
void cel_batches(Prepared &P, const std::vector<const double *> &lev, const std::vector<const float *> &wgt,
                 const std::vector<int> &term0)
{
    Atomic &A = P.A;
    std::vector<int> order(A.ncel);
    for (int k = 0; k < A.ncel; ++k) order[k] = k;
    std::stable_sort(order.begin(), order.end(), [&](int u, int v) { return A.cel[u].nl > A.cel[v].nl; });
    A.ncelb = (A.ncel + kCelSlots - 1) / kCelSlots;
    A.cel_most = 0;
    P.cel_at.assign((size_t)A.ncelb * (kMaxLev + 1) * 64, 0.0);
    P.cel_ae.assign((size_t)A.ncelb * kMaxLev * 64, 0.0);
    P.cel_term.assign((size_t)A.ncelb * kMaxLev * 64, -1);
    for (int b = 0; b < A.ncelb; ++b) {
        CelBatch &B = A.celb[b];
        B = CelBatch{};
        B.pair0 = (int)P.cel_pair.size();
        double *at = P.cel_at.data() + (size_t)b * (kMaxLev + 1) * 64;
        double *ae = P.cel_ae.data() + (size_t)b * kMaxLev * 64;
        int *term = P.cel_term.data() + (size_t)b * kMaxLev * 64;
        for (int s = 0; s < kCelSlots; ++s) {
            B.ion[s] = -1;
            if (kCelSlots * b + s >= A.ncel) continue;
            const int k = order[kCelSlots * b + s], nl = A.cel[k].nl;
            const double *E = lev[k], *a = E + nl;
            A.cel_place[k] = kCelSlots * b + s;
            B.ion[s] = k;
            B.rows[s] = nl - 1;
            B.base[s] = B.npair;
            B.most = std::max(B.most, nl - 1);
            int t = term0[k];
            for (int lo = 0, p = 0; lo < nl - 1; ++lo)
                for (int up = lo + 1; up < nl; ++up, ++p) {
                    const double av = a[up + nl * lo];
                    P.cel_pair.push_back(s + 4 * p);
                    P.cel_de.push_back((E[lo] - E[up]) * 1.4388463);
                    P.cel_glo.push_back((double)wgt[k][lo]);
                    P.cel_gup.push_back((double)wgt[k][up]);
                    // level L (from 0) of slot s is lane 16 s + L - 1
                    at[64 * (lo + 1) + 16 * s + up - 1] = av;
                    if (lo > 0) at[64 * (up + 1) + 16 * s + lo - 1] = av;
                    ae[64 * lo + 16 * s + up - 1] = av * (E[up] - E[lo]);
                    if (av != 0.0) term[64 * lo + 16 * s + up - 1] = t++;
                }
            B.npair += nl * (nl - 1) / 2;
        }
        A.cel_most = std::max(A.cel_most, B.npair);
    }
}

}  // namespace

int prepare(const mc_atomic *in, int nb, const float *nuArray, Prepared &P, char *e, size_t n)
{
    if (!in || !in->elemOn || !in->xref || !in->abun || !in->ch_meta || !in->ch_sigma || !in->rrec ||
        !in->rnew || !in->fe || !in->dr_int || !in->dr_real || !in->ap_int || !in->ap_real ||
        (in->ncel > 0 && (!in->cel_meta || !in->cel_dbl || !in->cel_flt)))
        return err(e, n, MC_EINVAL, "atomic descriptor has null arrays");
    const int ns = in->nstages;
    if (ns < 2 || ns > kMaxStage - 1) return err(e, n, MC_EUNSUP, "nstages %d outside 2..%d", ns, kMaxStage - 1);
    if (nb > kMaxNb || nb < mcm::kBands)
        return err(e, n, MC_EUNSUP, "nbins %d outside %d..%d", nb, mcm::kBands, kMaxNb);
    if (!in->elemOn[0] || !in->elemOn[1]) return err(e, n, MC_EUNSUP, "H and He must be switched on");
    Atomic &A = P.A;
    A = Atomic{};
    A.nbins = nb;
    A.nstages = ns;
    A.XHILimit = in->XHILimit;
    for (auto *v : { &P.sigma, &P.cR, &P.cH, &P.cel_s, &P.cel_t, &P.cel_de, &P.cel_glo, &P.cel_gup, &P.cel_at,
                     &P.cel_ae })
        v->clear();
    P.cel_pair.clear();
    P.nu.assign(nuArray, nuArray + nb);
    // elements in atomic-number order, their channels ion = 1..min(z, ns-1)
    int eidx_of_z[31];
    for (int z = 0; z <= 30; ++z) eidx_of_z[z] = -1;
    int nE = 0, nch = 0;
    P.eidx_xref.clear();
    for (int z = 1; z <= 30; ++z) {
        if (!in->elemOn[z - 1]) continue;
        if (nE == kMaxElem) return err(e, n, MC_EUNSUP, "more than %d elements", kMaxElem);
        const int xr = in->xref[z - 1];
        if (xr < 1 || xr > in->nElemUsed) return err(e, n, MC_ETABLE, "elementXref(%d) = %d", z, xr);
        Element &E = A.el[nE];
        E.z = z;
        E.nst = std::min(z + 1, ns);
        E.ch0 = nch;
        E.nch = std::min(z, ns - 1);
        E.abun = (double)in->abun[z - 1];
        if (nch + E.nch > kMaxCh) return err(e, n, MC_EUNSUP, "more than %d channels", kMaxCh);
        for (int ion = 1; ion <= E.nch; ++ion) {
            Channel &c = A.ch[nch];
            c.elem = z; c.ion = ion; c.eidx = nE;
            c.ip = 1; c.hiR = 0; c.hiH = 0;
            int g0 = 0, g1 = 0, row = -1;
            for (int k = 0; k < in->nch; ++k)
                if (in->ch_meta[8 * k] == z && in->ch_meta[8 * k + 1] == ion) row = k;
            std::vector<double> sig(nb, 0.0);
            if (row >= 0) {
                const int32_t *m = in->ch_meta + 8 * row;
                g0 = m[2]; g1 = m[3];
                c.ip = m[4]; c.hiR = m[5]; c.hiH = m[6];
                if (c.ip < 1 || c.ip > nb || c.hiR > nb || c.hiH > nb)
                    return err(e, n, MC_ETABLE, "channel Z=%d ion %d: bins %d..%d/%d outside 1..%d", z, ion,
                               c.ip, c.hiR, c.hiH, nb);
                for (int j = 0; j < nb; ++j) sig[j] = (double)in->ch_sigma[(size_t)row * nb + j];
                // the heating integral stops at the first cross section below 1e-35
                for (int j = c.ip; j <= c.hiH; ++j)
                    if (sig[j - 1] < 1.e-35) { c.hiH = j - 1; break; }
            }
            // coefficients of the rate and heating integrals per bin:
            // rate J sigma / (h c Ryd nu) over ip..hiRate where sigma >= 1e-35,
            // heating J sigma (nu - nu_ip) / nu over ip..hiHeat
            {
                const double hcRyd = 2.1799153e-11;
                const double nuIP = (double)nuArray[c.ip - 1];
                for (int j = 1; j <= nb; ++j) {
                    const double nu = (double)nuArray[j - 1], ph = sig[j - 1];
                    P.cR.push_back(j >= c.ip && j <= c.hiR && ph >= 1.e-35 ? ph / (hcRyd * nu) : 0.0);
                    P.cH.push_back(j >= c.ip && j <= c.hiH ? ph * (nu - nuIP) / nu : 0.0);
                }
            }
            P.sigma.insert(P.sigma.end(), sig.begin(), sig.end());
            c.g0g1 = (double)g0 / (double)g1;
            // radiative recombination fit (radRecFit, update_mod.f90:1674-1780)
            const int nn = z - ion + 1;
            if (nn <= 3 || nn == 11 || (z > 5 && z < 9) || z == 10 || (z == 26 && nn > 11)) {
                c.rr_kind = 0;
                for (int i = 0; i < 4; ++i) c.rr[i] = (double)in->rnew[(z - 1) * 120 + (nn - 1) * 4 + i];
            } else if (z == 26 && nn <= 13) {
                c.rr_kind = 2;
                for (int i = 0; i < 3; ++i) c.rr[i] = (double)in->fe[(nn - 4) * 3 + i];
            } else {
                c.rr_kind = 1;
                for (int i = 0; i < 2; ++i) c.rr[i] = (double)in->rrec[(z - 1) * 60 + (nn - 1) * 2 + i];
            }
            const int nr = dr_rows(in, ns, z, ion, c.dr, &c.ap, e, n);
            if (nr < 0) return MC_ETABLE;
            c.ndr = nr;
            // charge exchange
            for (const ChexRow &r : kChex)
                if (r.elem == z && r.ion == ion) {
                    c.chex[0] = r.a * 1.e-9; c.chex[1] = r.b; c.chex[2] = r.c; c.chex[3] = r.d;
                }
            c.dEk = (z == 7 && ion == 1) ? 10863. : (z == 8 && ion == 1) ? 2205. : 0.;
            ++nch;
        }
        eidx_of_z[z] = nE;
        P.eidx_xref.push_back(xr);
        ++nE;
    }
    A.nE = nE;
    A.nch = nch;
    if (A.ch[0].elem != 1 || A.ch[0].ion != 1) return err(e, n, MC_EUNSUP, "first channel is not H I");
    for (int ion = 1; ion < ns; ++ion) {
        const int nr = dr_rows(in, ns, 8, ion, A.odr[ion], &A.oap[ion], e, n);
        if (nr < 0) return MC_ETABLE;
        A.odr_n[ion] = nr;
    }
    for (int i = 0; i < 25; ++i) {
        for (int k = 0; k < 5; ++k) A.dr_real[i][k] = (double)in->dr_real[5 * i + k];
        A.dr_g[i] = in->dr_int[3 * i + 2];
    }
    for (int i = 0; i < 167; ++i)
        for (int k = 0; k < 4; ++k) A.ap_real[i][k] = (double)in->ap_real[4 * i + k];
    // CEL model ions
    if (in->ncel < 0 || in->ncel > kMaxCel) return err(e, n, MC_EUNSUP, "more than %d CEL ions", kMaxCel);
    A.ncel = in->ncel;
    size_t od = 0, of = 0;
    std::vector<const double *> lev(in->ncel);
    std::vector<const float *> wgt(in->ncel);
    std::vector<int> term0(in->ncel);             // the ion's first radiating pair
    int nterm = 0;
    for (int k = 0; k < in->ncel; ++k) {
        const int32_t *m = in->cel_meta + 6 * k;
        const int z = m[0], ion = m[1], nl = m[4], nt = m[5];
        if (z < 1 || z > 30 || eidx_of_z[z] < 0 || ion < 1 || ion > ns)
            return err(e, n, MC_ETABLE, "CEL ion %d: Z=%d ion %d not switched on", k, z, ion);
        if (nl < 2 || nl > kMaxLev || nt < 1 || nt > kMaxTemp)
            return err(e, n, MC_EUNSUP, "CEL ion %d: %d levels, %d temperatures", k, nl, nt);
        const double *ev = in->cel_dbl + od;
        const double *av = ev + nl;
        const double *qv = av + (size_t)nl * nl;
        const float *lt = in->cel_flt + of;
        const float *gv = lt + nt;
        CelIon &ci = A.cel[k];
        ci.eidx = eidx_of_z[z]; ci.ion = ion; ci.nl = nl; ci.nt = nt;
        ci.br = (double)gv[nl];
        ci.z = (double)gv[nl + 1];
        for (int i = 0; i < 4; ++i) ci.a_r[i] = (double)gv[nl + 2 + i];
        for (int i = 0; i < 5; ++i) ci.a_d[i] = (double)gv[nl + 6 + i];
        ci.off_s = (int)(P.cel_s.size() / 2);
        ci.off_t = (int)P.cel_t.size();
        lev[k] = ev;
        wgt[k] = gv;
        term0[k] = nterm;
        for (int lo = 0; lo < nl; ++lo)
            for (int up = lo + 1; up < nl; ++up) nterm += av[up + nl * lo] != 0.0;
        std::vector<double> xa(nt);
        for (int t = 0; t < nt; ++t) xa[t] = (double)lt[t];
        for (int t = 1; t < nt; ++t)
            if (!(xa[t] > xa[t - 1])) return err(e, n, MC_ETABLE, "CEL ion %d: log T not increasing", k);
        P.cel_t.insert(P.cel_t.end(), xa.begin(), xa.end());
        // collision strengths of each pair (lo < up) and their spline curvature
        double qq[kMaxTemp], y2[kMaxTemp];
        const int npair = nl * (nl - 1) / 2;
        P.cel_s.resize(P.cel_s.size() + (size_t)2 * nt * npair);
        double *s2 = P.cel_s.data() + 2 * (size_t)ci.off_s;
        for (int lo = 1, p = 0; lo <= nl - 1; ++lo)
            for (int up = lo + 1; up <= nl; ++up, ++p) {
                for (int t = 0; t < nt; ++t) qq[t] = qv[t + (size_t)nt * ((lo - 1) + (size_t)nl * (up - 1))];
                if (nt >= 3) spline_nat(xa.data(), qq, nt, y2);
                else for (int t = 0; t < nt; ++t) y2[t] = 0.0;
                for (int t = 0; t < nt; ++t) {
                    s2[2 * ((size_t)t * npair + p)] = qq[t];
                    s2[2 * ((size_t)t * npair + p) + 1] = y2[t];
                }
            }
        od += (size_t)nl + (size_t)nl * nl + (size_t)nt * nl * nl;
        of += (size_t)nt + nl + 2 + 4 + 5;
    }
    A.nterm = nterm;
    cel_batches(P, lev, wgt, term0);
    return MC_OK;
}

}  // namespace mcb
