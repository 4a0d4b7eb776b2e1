// mc_emission.hip - the re-emission tables on MI355X: emissionDriver's gas
// part and setDiffusePDF (emission_mod.f90:32-1311) for every active cell,
// written into the transport's recPDF rows ([cell][nu]) and totalLines.
//
// One 64-lane wavefront per cell, in two kernels: forbidden_kernel sums the
// forbidden-line terms from the balance's n-level solve (FP64), and
// emission_kernel does the rest without the registers of those solves.  Lanes
// over frequency bins evaluate the free-bound, free-free and two-photon
// coefficients and the cell's partial sums (sumDiffuseHI/HeI/HeII and the
// dust term) into LDS; lanes over lines evaluate the recombination terms.
// The sums the reference forms in REAL, in a fixed order (normHI, normRec,
// normFor, the cumulative recPDF), are taken in that order, each on a lane of
// its own, so the tables follow the reference's rounding.
//
// Bound by the FP64 exponentials and powers of the bins (one per bin and
// heavy ion above its edge, three of the recombination continua, up to three
// of the tabulated ones).  45^3 octant, 800 bins: 10.4 ms at first, 5.0 with
// four model ions to a wavefront, 3.9 in the two kernels (1.4 + 2.5);
// dust and gas 60^3, 160 bins: 2.6, then 3.0, now 2.0.
#include "mc_cel.h"
#include "mc_emission.h"

#pragma clang fp contract(off)

namespace mce {

constexpr int W = 64;
constexpr float kHcRydK = 157893.94f;   // continuum_mod.f90:10
constexpr float kHcRyd = 2.1799153e-11f; // continuum_mod.f90:11
constexpr float kCRyd = 3.2898423e15f;   // continuum_mod.f90:12
constexpr float kHPlanck = 6.6262e-27f;  // constants_mod.f90:14
constexpr float kPi = 3.141592654f;      // constants_mod.f90:32
constexpr int kLev = mcb::kMaxLev;

// A heavy-ion free-bound channel of the cell (fb_ff).
struct FreeBound {
    int first, end, off;          // bins first .. end - 1, its cross-sections
    float edge, g, x, abun;       // nu of the first bin, g0/g1, ion fraction, elemAbun
};

// The dynamic LDS of a wavefront: the per-bin partial sums s1, s2, s3 (and
// the grains' sD), the free-bound channels, the log-gamma rows, the
// recombination-line terms.
__host__ __device__ inline int padded(int nb) { return (nb + 3) / 4 * 4; }
__host__ __device__ inline size_t sums_bytes(const EmArgs &a)
{
    return (size_t)(a.dabs ? 4 : 3) * padded(a.nb) * sizeof(float);
}
__host__ __device__ inline size_t fb_bytes(const EmArgs &a)
{
    return ((size_t)a.nfb * sizeof(FreeBound) + 15) / 16 * 16;
}
constexpr size_t kRestBytes = sizeof(float) * (3 * kMaxLim + kMaxRec + 4);

// The part of hydro2phot that depends on the bin alone, gNu 1e27 of H I (Z =
// 1) or He II; the tables of every bin are made once at setup.
__device__ float two_photon_shape(float nu, int Z)
{
    const float z6 = 64.f;
    const float y = nu / (Z == 1 ? 0.7496f : 3.00f);
    float gNu;
    if (Z == 1) {
        const float Ay = 202.0f * (y * (1.f - y) * (1.f - powf(4.f * y * (1.f - y), 0.8f)) +
                                   0.88f * powf(y * (1.f - y), 1.53f) * powf(4.f * y * (1.f - y), 0.8f));
        gNu = kHPlanck * y * Ay / 8.2249f;
    } else {
        const float Ay = z6 * 0.9994667f * 202.0f *
                         (y * (1.f - y) * (1.f - powf(4.f * y * (1.f - y), 0.8f)) +
                          0.88f * powf(y * (1.f - y), 1.53f) * powf(4.f * y * (1.f - y), 0.8f));
        const float A2qZ = 8.226f * z6;
        gNu = kHPlanck * y * Ay / A2qZ;
    }
    return gNu * 1e27f;
}

__global__ void two_photon_kernel(const float *__restrict__ nu, int nb, float *__restrict__ shape)
{
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= nb) return;
    shape[i] = nu[i] < 0.7496f ? two_photon_shape(nu[i], 1) : 0.f;
    shape[nb + i] = nu[i] < 3.00f ? two_photon_shape(nu[i], 2) : 0.f;
}

// The part that depends on the cell: alpha of each, and H I's collisional
// de-excitation 1 + Ne Q / 8.23
struct TwoPhoton { float alpha1, quench1, alpha2; };
// hydro2phot (emission_mod.f90:553-663), REAL arithmetic
__device__ __forceinline__ TwoPhoton two_photon(float Te, float Ne)
{
    TwoPhoton T;
    float factor;
    T.alpha1 = 0.8368f * powf(Te * 1.e-4f, -0.723f);
    float Q;
    if (Te <= 10000.f) Q = 5.31e-4f;
    else if (Te >= 20000.f) Q = 4.71e-4f;
    else {
        factor = log10f(4.71e-4f / 5.31e-4f) / log10f(2.f);
        Q = powf(10.f, log10f(5.31e-4f) + factor * log10f(Te / 10000.f));
    }
    T.quench1 = 1.f + (Ne * Q) / 8.23f;
    if (Te <= 5000.f) T.alpha2 = 6.161f;
    else if (Te >= 30000.f) T.alpha2 = 2.035f;
    else if (Te > 5000.f && Te <= 10000.f) {
        factor = log10f(4.091f / 6.161f) / log10f(2.f);
        T.alpha2 = powf(10.f, log10f(6.161f) + factor * log10f(Te / 5000.f));
    } else if (Te > 10000.f && Te <= 15000.f) {
        factor = log10f(3.189f / 4.091f) / log10f(1.5f);
        T.alpha2 = powf(10.f, log10f(4.091f) + factor * log10f(Te / 10000.f));
    } else {
        factor = log10f(2.035f / 3.189f) / log10f(2.f);
        T.alpha2 = powf(10.f, log10f(3.189f) + factor * log10f(Te / 15000.f));
    }
    return T;
}

// ffCoeff (emission_mod.f90:726-742); expF = exp(-h nu / k Te)
__device__ __forceinline__ double ffcoeff(float Z, float g, double expF, float sqrTe)
{
    return (double)(4.f * kPi * 54.43f * Z * Z * g) * expF / (double)sqrTe;
}

// getFlux's blackbody (continuum_mod.f90:359-400): the Planck function over h
__device__ __forceinline__ float blackbody(float energy, float T)
{
    const float constant = 0.5250229f / kHPlanck;
    if (kHcRydK * energy / T > 86.f)
        return (float)((double)(constant * energy * energy * energy) * exp((double)(-kHcRydK * energy / T)));
    const float den = expf(kHcRydK * energy / T) - 1.f;
    if (den <= 0.f) return 3.32154e-6f * energy * energy * T / kHPlanck;
    return constant * energy * energy * energy / den;
}

// locate (interpolation_mod.f90:48-81) of Te in the increasing tkGamma
__device__ int locate_tk(const float *xa, int n, float x)
{
    if (x > xa[n - 1]) return n;
    if (x < xa[0]) return 0;
    int p = 0;
    float bd = 0.f;
    for (int i = 0; i < n; ++i) {
        const float d = xa[i] - x;
        if (d > 0.f && (p == 0 || d < bd)) { p = i + 1; bd = d; }
    }
    return p - 1 > 1 ? p - 1 : 1;
}

#define XION(e, st) ((float)ionc[(e) * a.ns1 + (st)])

// normFor of every cell
__global__ void __launch_bounds__(64) forbidden_kernel(const mcb::Atomic *__restrict__ Ap, EmArgs a)
{
    extern __shared__ __align__(16) unsigned char dyn[];
    const mcb::Atomic &A = *Ap;
    const int cell = blockIdx.x + 1;
    const int lane = threadIdx.x;
    double2 *rate = reinterpret_cast<double2 *>(dyn);
    mcb::CelRec *rec = reinterpret_cast<mcb::CelRec *>(rate + a.cel_most);
    float *fterm = reinterpret_cast<float *>(rec + a.ncel);

    // the state as the host grid stores it (REAL)
    const float Te = (float)a.Te[cell], NeIn = (float)a.Ne[cell];
    const double *ionc = a.ion + (size_t)cell * a.nE * a.ns1;
    const float NeUsed = NeIn < 1.e-5f ? 1.e-5f : NeIn;
    // a state emission_kernel refuses
    if (!(Te > 0.f) || !isfinite(Te) || !isfinite(NeIn)) return;

    float normFor = 0.f;
    // forbidden lines (forLines): the terms above 1e-35 of every model ion's
    // radiating pairs, summed ion by ion, lower level outer, upper inner, as
    // setDiffusePDF does
    const double kL = (double)1.9865e9f;
    const double TeD = (double)Te, sqrTeD = sqrt(TeD), log10TeD = log10(TeD);
    for (int k = lane; k < A.ncel; k += W) {
        const mcb::CelIon &ci = A.cel[k];
        const float x = XION(ci.eidx, ci.ion);
        const float up = (ci.ion < a.ns1 - 1) ? XION(ci.eidx, ci.ion + 1) / x : 0.f;
        rec[A.cel_place[k]] = mcb::cel_record(A, ci, TeD, log10TeD, (double)up, (double)(float)A.el[ci.eidx].abun,
                                              (double)x);
    }
    __syncthreads();
    for (int b = 0; b < A.ncelb; ++b) {
        const mcb::CelBatch &B = A.celb[b];
        const mcb::CelRec *R = rec + mcb::kCelSlots * b;
        const mcb::CelLevels L = mcb::cel_levels(A, b, R, rate, lane, TeD, sqrTeD, (double)NeUsed);
        const int g = lane >> 4;
        const bool mine = (lane & 15) < B.rows[g];
        const double part = L.y / L.sum, ab = R[mine ? g : 0].ab, x = R[mine ? g : 0].x;
        const bool none = R[mine ? g : 0].skip;
        const double *ae = A.cel_ae + (size_t)b * kLev * 64 + lane;
        const int *term = A.cel_term + (size_t)b * kLev * 64 + lane;
        for (int lo = 0; lo < B.most; ++lo) {
            double f = ae[64 * lo] * part;
            f = f * ab * x;
            f = f * kL;
            const int t = term[64 * lo];
            if (t >= 0) fterm[t] = !none && f > (double)1.e-35f ? (float)f : 0.f;
        }
    }
    __syncthreads();
    for (int t = 0; t < A.nterm; ++t) normFor = normFor + fterm[t];
    if (lane == 0) a.forbidden[cell] = normFor;
}

__global__ void __launch_bounds__(64) emission_kernel(EmArgs a)
{
    extern __shared__ __align__(16) unsigned char dyn[];
    const int cell = blockIdx.x + 1;
    const int lane = threadIdx.x;
    const int nb = a.nb, ld = padded(nb);
    const float *nu = a.nu;
    const bool dust = a.dabs != nullptr;
    float *s1 = reinterpret_cast<float *>(dyn), *s2 = s1 + ld, *s3 = s1 + 2 * ld, *sD = s1 + 3 * ld;
    FreeBound *fb = reinterpret_cast<FreeBound *>(dyn + sums_bytes(a));
    unsigned char *rest = dyn + sums_bytes(a) + fb_bytes(a);
    float (*loc)[kMaxLim] = reinterpret_cast<float (*)[kMaxLim]>(rest);
    float *rterm = reinterpret_cast<float *>(rest + sizeof(float) * 3 * kMaxLim);
    float *red = rterm + kMaxRec;

    // the state as the host grid stores it (REAL)
    const float Te = (float)a.Te[cell], NeIn = (float)a.Ne[cell];
    const double *ionc = a.ion + (size_t)cell * a.nE * a.ns1;
    float NeUsed = NeIn;
    const float sqrTe = sqrtf(Te);
    const float log10Te = log10f(Te);
    if (NeUsed < 1.e-5f) NeUsed = 1.e-5f;
    const float xHp = XION(a.eH, 2), xHe1 = XION(a.eHe, 2), xHe2 = XION(a.eHe, 3);
    if (!(Te > 0.f) || !isfinite(Te) || !isfinite(NeIn)) {
        // not a state the balance leaves (its floor is 1 K): refused
        if (lane == 0) a.err[cell] = 1;
        return;
    }

    for (int c = lane; c < a.nfb; c += W) {
        const int *m = a.fb_i + 4 * c;
        fb[c] = FreeBound{ m[2], m[3], a.fb_off[c], nu[m[2] - 1], a.fb_f[2 * c], XION(m[0], m[1]), a.fb_f[2 * c + 1] };
    }
    const TwoPhoton tp = two_photon(Te, NeUsed);

    // log gamma rows at Te (fb_ff, emission_mod.f90:306-336)
    for (int s = 0; s < 3; ++s)
        for (int i = lane; i < a.nlim[s]; i += W) {
            const float *g = a.lg[s];
            const int ntk = a.ntk;
            float v;
            if (Te <= a.tk[0]) v = g[ntk * i];
            else if (Te >= a.tk[ntk - 1]) v = g[(ntk - 1) + ntk * i];
            else {
                const int t = locate_tk(a.tk, ntk, Te);
                const double factor = (double)log10f(Te / a.tk[t - 1]);
                const double aFit = (double)((g[t + ntk * i] - g[(t - 1) + ntk * i]) / log10f(a.tk[t] / a.tk[t - 1]));
                v = g[(t - 1) + ntk * i] + (float)(aFit * factor);
            }
            loc[s][i] = v;
        }
    __syncthreads();

    // per bin: emission coefficients and the partial sums of setDiffusePDF
    const double constant = (double)4.9874105e-6f;
    const float statW[3] = { 2.f, 0.5f, 2.f };
    const float alpha21 = 6.23f * powf(Te / 10000.f, -0.827f);
    for (int i = lane + 1; i <= nb; i += W) {
        const float nui = nu[i - 1];
        double g[3];
        for (int s = 0; s < 3; ++s) {
            g[s] = 0.0;
            const int k = a.pair[s][i - 1];
            if (k >= 0) {
                const int ilow = a.edge[s][2 * k], iup = a.edge[s][2 * k + 1];
                const double aFit = (double)((loc[s][2 * k + 1] - loc[s][2 * k]) / (nu[iup - 1] - nu[ilow - 1]));
                const double v = (double)loc[s][2 * k + 1] + aFit * (double)(nui - nu[iup - 1]);
                g[s] = pow(10.0, v);
            }
        }
        if (i >= a.ip[0]) {
            // the Milne relation above the H, He I and He II edges, plus free-free
            const double factor = (double)((nui * nui * nui) / (Te * sqrTe));
            double expF = exp((double)((-nui + nu[a.ip[0] - 1]) * kHcRydK / Te));
            const double expFF = exp((double)(-nui * kHcRydK / Te));
            g[0] = (double)(4.f * kPi) * (double)a.sig[0][i - a.i0[0]] * (double)statW[0] * (double)kHcRyd * constant *
                   factor * expF * (double)1.e20f * (double)1.e20f;
            g[0] = g[0] + ffcoeff(1.f, a.gff[i - 1], expFF, sqrTe);
            if (i >= a.i0[1]) {
                expF = exp((double)((-nui + nu[a.ip[1] - 1]) * kHcRydK / Te));
                g[1] = (double)(4.f * kPi) * (double)a.sig[1][i - a.i0[1]] * (double)statW[1] * (double)kHcRyd *
                       constant * factor * expF * (double)1.e20f * (double)1.e20f;
                g[1] = g[1] + ffcoeff(1.f, a.gff[i - 1], expFF, sqrTe);
                if (i >= a.i0[2]) {
                    expF = exp((double)((-nui + nu[a.ip[2] - 1]) * kHcRydK / Te));
                    g[2] = (double)(4.f * kPi) * (double)a.sig[2][i - a.i0[2]] * (double)statW[2] * (double)kHcRyd *
                           constant * factor * expF * (double)1.e20f * (double)1.e20f;
                    g[2] = g[2] + ffcoeff(2.f, a.gffHeII[i - 1], expFF, sqrTe);
                }
            }
        }
        // heavy-ion free-bound emission (fb_ff, emission_mod.f90:473-528)
        double gh = 0.0;
        for (int c = 0; c < a.nfb; ++c) {
            const FreeBound f = fb[c];
            if (i >= f.first && i < f.end) {
                const double expF = exp((double)((-nui + f.edge) * kHcRydK / Te));
                gh = gh + expF * (double)a.fb_sig[f.off + (i - f.first)] * (double)f.g * (double)f.x * (double)f.abun;
            }
        }
        {
            const float factor = nui * nui * nui / (Te * sqrTe);
            gh = gh * (double)(4.f * kPi) * constant * (double)kHcRyd * (double)factor * (double)1.e20f *
                 (double)1.e20f;
        }
        // two-photon continua (twoPhoton, HeI2photSub)
        const double tHI = nui < 0.7496f ? (double)(tp.alpha1 * a.shape[i - 1] / tp.quench1) : 0.0;
        const double tHeII = nui < 3.00f ? (double)(tp.alpha2 * a.shape[nb + i - 1]) : 0.0;
        double tHeI = 0.0;
        const int j = a.jHeI[i - 1];
        if (j > 0) {
            const float y = nui / 1.514f;
            const float fit1 = (a.Aydat[j] - a.Aydat[j - 1]) / (a.ydat[j] - a.ydat[j - 1]);
            const float fit2 = a.Aydat[j - 1] - a.ydat[j - 1] * fit1;
            float Ay = fit1 * y + fit2;
            if (Ay < 9.2163086E-03f) Ay = 0.f;
            tHeI = (double)(alpha21 * Ay * 0.66262f * y / 51.3f);
        }
        double eHI = (g[0] + tHI) * (double)a.abH * (double)xHp * (double)NeUsed + gh * (double)NeUsed;
        double eHeI = (g[1] + tHeI) * (double)a.abHe * (double)xHe1 * (double)NeUsed;
        double eHeII = (g[2] + tHeII) * (double)a.abHe * (double)xHe2 * (double)NeUsed;
        if (eHI < (double)1.e-15f) eHI = 0.0;
        if (eHeI < (double)1.e-15f) eHeI = 0.0;
        if (eHeII < (double)1.e-15f) eHeII = 0.0;
        const float cw = kCRyd * a.widFlx[i - 1];
        s1[i - 1] = (float)((double)cw * eHI / (double)1.e15f);
        s2[i - 1] = (float)((double)cw * eHeI / (double)1.e15f);
        s3[i - 1] = (float)((double)cw * eHeII / (double)1.e15f);
        if (dust) {
            // grains below their sublimation temperature, sizes outer and
            // species inner as setDiffusePDF loops
            float sd = 0.f;
            const size_t tb = (size_t)cell * (a.dnsMax + 1) * (a.dSizes + 1);
            for (int ai = 1; ai <= a.dSizes; ++ai)
                for (int sp = 1; sp <= a.dS; ++sp) {
                    const float td = (float)a.Tdust[tb + sp + (size_t)(a.dnsMax + 1) * ai];
                    if (!(td < a.dtsub[(sp - 1) * a.dSizes + ai - 1])) continue;
                    const float bb = blackbody(nui, td);
                    sd = sd + a.dabs[((size_t)(sp - 1) * a.dSizes + ai - 1) * nb + i - 1] * bb * a.widFlx[i - 1] *
                                  a.dweight[ai - 1] * a.dgabun[sp - 1];
                }
            sD[i - 1] = sd;
        }
    }

    // recombination-line terms in normRec's order (RecLinesEmission and
    // setDiffusePDF, emission_mod.f90:744-832, 1099-1117): H I 3..15 -> 2..8,
    // He II 3..30 -> 2..16, He I singlets
    {
        float Hbeta = powf(10.f, -0.870f * log10Te + 3.57f);
        Hbeta = Hbeta * NeUsed * xHp * a.abH;
        const float Lalpha = powf(10.f, -0.897f * log10Te + 5.05f);
        float h4686 = powf(10.f, -.997f * log10f(Te) + 5.16f);
        h4686 = h4686 * NeUsed * a.abHe * xHe2;
        const float T4 = Te / 10000.f;
        int denint;
        if (NeIn <= 100.f) denint = 0;
        else if (NeIn <= 1.e4f) denint = 1;
        else if (NeIn <= 1.e6f) denint = 2;
        else denint = 3;
        const float p100[4] = { 1.f, 100.f, 10000.f, 1.e6f };
        for (int t = lane; t < 70 + 315 + 34; t += W) {
            float v;
            if (t < 70) {
                int u = 3, r = t;
                while (r >= (u - 1 < 8 ? u - 1 : 8) - 1) { r -= (u - 1 < 8 ? u - 1 : 8) - 1; ++u; }
                const int l = 2 + r;
                double h = a.HIrec[(u - 3) + 28 * (l - 2)] * (double)Hbeta;
                if (u == 15 && l == 8) h = h + (double)(a.abH * xHp * NeUsed * Lalpha);
                v = (float)h;
            } else if (t < 70 + 315) {
                int u = 3, r = t - 70;
                while (r >= (u - 1 < 16 ? u - 1 : 16) - 1) { r -= (u - 1 < 16 ? u - 1 : 16) - 1; ++u; }
                const int l = 2 + r;
                v = (float)(a.HeIIrec[(u - 3) + 28 * (l - 2)] * (double)h4686);
            } else {
                const int i = t - 70 - 315 + 1;
#define HEIC(d, k) a.HeIc[((i) - 1) + 34 * (((d) - 1) + 3 * ((k) - 1))]
                double h;
                if (denint > 0 && denint < 3) {
                    const float x1 = HEIC(denint, 1) * powf(T4, HEIC(denint, 2)) * expf(HEIC(denint, 3) / T4);
                    const float x2 =
                        HEIC(denint + 1, 1) * powf(T4, HEIC(denint + 1, 2)) * expf(HEIC(denint + 1, 3) / T4);
                    h = (double)(x1 + ((x2 - x1) * (NeUsed - p100[denint]) / (p100[denint + 1] - p100[denint])));
                } else {
                    const int d = denint == 0 ? 1 : 3;
                    h = (double)(HEIC(d, 1) * powf(T4, HEIC(d, 2)) * expf(HEIC(d, 3) / T4));
                }
#undef HEIC
                h = h * (double)NeUsed * (double)a.abHe * (double)xHe1;
                v = (float)h;
            }
            rterm[t] = v;
        }
    }
    __syncthreads();
    // the sums in order, a lane each: bins of H I, He I, He II and grains,
    // recombination lines
    float sum = 0.f;
    {
        const float *p = lane < 4 ? s1 + (size_t)lane * ld : rterm;
        const int n = lane < (dust ? 4 : 3) ? nb : lane == 4 ? 70 + 315 + 34 : 0;
        for (int i = 0; i < n; i += 4) {
            const float4 v = *reinterpret_cast<const float4 *>(p + i);
            sum = sum + v.x;
            if (i + 1 < n) sum = sum + v.y;
            if (i + 2 < n) sum = sum + v.z;
            if (i + 3 < n) sum = sum + v.w;
        }
    }
    float nHI = __shfl(sum, 0), nHeI = __shfl(sum, 1), nHeII = __shfl(sum, 2), nD = __shfl(sum, 3);
    const float normRec = __shfl(sum, 4), normFor = a.ncel > 0 ? a.forbidden[cell] : 0.f;
    __syncthreads();
    // setDiffusePDF scales the raw grain sums by h 4 pi 1e25 cRyd Ndust /
    // Hden; the raw total is taken in bin order here (the reference adds
    // sizes, species, then bins)
    if (dust) {
        const float cst = kHPlanck * 4.f * kPi * 1.e25f * kCRyd;
        const float nd = a.ndust[cell], hd = (float)a.Hden[cell];
        for (int i = lane; i < nb; i += W) sD[i] = sD[i] * cst * nd / hd;
        nD = nD * cst * nd / hd;
    }
    // lane 0: the He lines able to ionise H and totalLines
    if (lane == 0) {
        const float T4 = Te * 1.e-4f;
        const float a2tS = 27.2f * powf(T4, -0.678f);
        const float corr = a2tS * NeUsed * a.abHe * xHe1 * 1.45673f * kHcRyd * 1e11f;
        s2[a.j2TsP - 1] = s2[a.j2TsP - 1] + corr;
        nHeI = nHeI + corr;
        float ly[kMaxLy];
        for (int k = 0; k < a.nly; ++k) ly[k] = a.lyData[k];
        ly[3] = powf(10.f, -0.792f * log10f(Te) + 6.01f);
        ly[3] = ly[3] * NeUsed * xHe2 * a.abHe;
        for (int k = 0; k < a.nly - 1; ++k) ly[k] = ly[k] * ly[3];
        for (int k = 0; k < a.nly; ++k) {
            s3[a.lyP[k] - 1] = s3[a.lyP[k] - 1] + ly[k];
            nHeII = nHeII + ly[k];
        }
        float normalize = nHI + nHeI + nHeII;
        if (dust) normalize = normalize + nD;
        const float tl = normRec + normFor;
        normalize = normalize + tl;
        // the reference's fraction; at a few tens of K its fits give inf*0
        // and it is NaN, which newPhotonPacket's test random <= totalLines
        // never passes (photon_mod.f90:925-929): the same as 0
        float f = tl / normalize;
        a.err[cell] = isnan(f) ? 2 : 0;
        if (isnan(f)) f = 0.f;
        a.totalLines[cell] = f;
    }
    __syncthreads();
    // the cumulative recPDF in bin order, in s1
    if (!dust) {
        for (int i = lane; i < nb; i += W) s1[i] = s1[i] + s2[i] + s3[i];
        __syncthreads();
    }
    if (lane == 0) {
        float r = 0.f;
        if (dust) {
            for (int i = 0; i < nb; ++i) {
                r = i == 0 ? s1[i] + s2[i] + s3[i] + sD[i] : r + s1[i] + s2[i] + s3[i] + sD[i];
                s1[i] = r;
            }
        } else {
            for (int i = 0; i < nb; i += 4) {
                float4 v = *reinterpret_cast<const float4 *>(s1 + i);
                r = i == 0 ? v.x : r + v.x;
                v.x = r;
                if (i + 1 < nb) { r = r + v.y; v.y = r; }
                if (i + 2 < nb) { r = r + v.z; v.z = r; }
                if (i + 3 < nb) { r = r + v.w; v.w = r; }
                *reinterpret_cast<float4 *>(s1 + i) = v;
            }
        }
        red[0] = r;
    }
    __syncthreads();
    // recPDF = cumulative / last (setDiffusePDF).  In barely lit cells the
    // iteration leaves at a few tens of K, the REAL cumulative sum
    // overflows (the Milne factor exp((nu_edge - nu) hcRyd/kT) of the bins
    // between a cross-section's start and its edge bin), so entries from the
    // overflow on are inf/inf = NaN; no finite total divides 0/0 = NaN
    // everywhere.  getNu2's scan (photon_mod.f90:745-752) stops at the
    // first entry random >= probDen fails, which a NaN entry fails as an
    // entry of 1 does: from the first NaN on the row is written 1, and the
    // transport draws the bins the reference draws.
    const float last = red[0];
    int m = nb;
    for (int i0 = 0; i0 < nb; i0 += W) {
        const int i = i0 + lane;
        const uint64_t bad = __ballot(i < nb && isnan(s1[i] / last));
        if (bad) { m = i0 + __ffsll((unsigned long long)bad) - 1; break; }
    }
    if (lane == 0 && m < nb) a.err[cell] = 2;
    float *row = a.rec + (size_t)cell * nb;
    for (int i = lane; i < nb; i += W) {
        float v = s1[i] / last;
        if (i >= m) v = 1.f;
        if (i == nb - 1) v = 1.f;
        if (v > 0.999998f) v = 1.f;
        row[i] = v;
    }
#undef XION
}

}  // namespace mce

size_t mce_mesh_bytes(int nb)
{
    return (4 * (size_t)nb * sizeof(float) + 15) / 16 * 16 + mce::kRestBytes;
}

hipError_t mce_two_photon(const float *nu, int nb, float *shape, hipStream_t s)
{
    hipLaunchKernelGGL(mce::two_photon_kernel, dim3((nb + 63) / 64), dim3(64), 0, s, nu, nb, shape);
    return hipGetLastError();
}

hipError_t mce_launch(const mcb::Atomic *dA, const mce::EmArgs &a, hipStream_t s)
{
    if (a.nc <= 0) return hipSuccess;
    if (a.ncel > 0) {
        const size_t lds = (size_t)a.cel_most * sizeof(double2) + (size_t)a.ncel * sizeof(mcb::CelRec) +
                           (size_t)a.nterm * sizeof(float);
        hipLaunchKernelGGL(mce::forbidden_kernel, dim3(a.nc), dim3(64), lds, s, dA, a);
        const hipError_t e = hipGetLastError();
        if (e != hipSuccess) return e;
    }
    hipLaunchKernelGGL(mce::emission_kernel, dim3(a.nc), dim3(64),
                       mce::sums_bytes(a) + mce::fb_bytes(a) + mce::kRestBytes, s, a);
    return hipGetLastError();
}
