// mc_cel.h - the n-level solves of the collisionally excited model ions
// (equilibrium, emission_mod.f90:1913-2114, with luSlv/lured/reslv
// 2119-2190), shared by the balance, line-luminosity and re-emission
// kernels.
//
// A 64-lane wavefront solves four ions at a time, one in each row of 16
// lanes: lane r of a row holds row r + 2 of the ion's rate matrix in
// registers (row 1 is all ones and needs no lane, so 17 levels fit), and a
// pivot row reaches the others by a DPP row broadcast.  Every entry gets the
// reference's operations in its order.  The work is bound by FP64
// instructions and by the serial chain of pivots; with one ion at a time,
// rows in LDS and the back substitution on one lane, 22 ions took 2.0e3
// vector instructions each and most of the time waited for LDS.  45^3 octant
// (46890 cells, 22 ions of 2 to 15 levels), before and now: line luminosities
// 9.3 -> 1.7 ms, the balance's reference schedule 24.6 -> 5.6 ms (with the
// shorter ion steps), re-emission tables 10.4 -> 3.8 ms (1.3 of it here).
// What depends on the atomic data alone (level differences, A times energy,
// which pairs radiate) is prepared once on the host, laid out as the lanes
// read it; the ions are sorted by size, so that a batch's ions are alike.
#pragma once
#include <hip/hip_runtime.h>

#include "mc_balance.h"

#pragma clang fp contract(off)

namespace mcb {

// What a solve needs of one ion at one temperature: the level recombination
// coefficient, ionDen(ion+1)/ionDen(ion), the spline weights of its
// collision strengths and where their rows begin, its abundance and fraction.
struct CelRec {
    double alev, up, ca, cb, h2, ab, x;
    int tab, step, mode, skip;
};

// The record of ion ci.  splint's bracket (interpolation_mod.f90:268-316) and
// the level recombination of emission_mod.f90:1991-2002 depend on the ion
// and the temperature only.  up NaN: no emission (equilibrium's test).
__device__ __forceinline__ CelRec cel_record(const Atomic &A, const CelIon &ci, double Te, double log10Te, double up,
                                             double ab, double x)
{
    CelRec R;
    R.alev = 0.0;
    if (ci.br > 0.0) {
        double t4 = Te * 1.e-4;
        double zz = ci.z;
        double x1 = t4 / (zz * zz);
        R.alev = 1.e-13 * ci.br * zz * ci.a_r[0] * pow(x1, ci.a_r[1]) /
                     (1. + ci.a_r[2] * pow(t4 / (zz * zz), ci.a_r[3])) +
                 1.0e-12 * ci.br * (ci.a_d[0] / t4 + ci.a_d[1] + ci.a_d[2] * Te * 1.e-4 + ci.a_d[3] * (t4 * t4)) *
                     pow(t4, -1.5) * exp(-(ci.a_d[4] * 1.e4 / Te));
    }
    const double *xa = A.cel_t + ci.off_t;
    const int n = ci.nt;
    int k = 0;
    R.mode = 0;
    R.ca = 1.0; R.cb = 0.0; R.h2 = 0.0;
    if (n == 2) {
        R.mode = 1;
        R.ca = xa[1] - xa[0];
        R.cb = log10Te - xa[0];
    } else if (n > 2 && log10Te >= xa[n - 1]) {
        k = n - 1;
    } else if (n > 2 && !(log10Te <= xa[0])) {
        int klo = 1, khi = n;
        while (khi - klo > 1) {
            int m = (khi + klo) / 2;
            if (xa[m - 1] > log10Te) khi = m; else klo = m;
        }
        const double h = xa[khi - 1] - xa[klo - 1];
        R.mode = 2;
        R.ca = (xa[khi - 1] - log10Te) / h;
        R.cb = (log10Te - xa[klo - 1]) / h;
        R.h2 = h * h;
        k = klo - 1;
    }
    const int npair = ci.nl * (ci.nl - 1) / 2;
    R.tab = ci.off_s + k * npair;
    R.step = R.mode ? npair : 0;
    R.up = up;
    R.ab = ab;
    R.x = x;
    R.skip = up != up;
    return R;
}

// Collision rates of a batch's pairs (emission_mod.f90:2004-2045), lanes
// over the pairs of its four ions together: rate[].x is q(lower, upper),
// rate[].y q(upper, lower).  rec: the batch's records by slot.
__device__ __forceinline__ void cel_rates(const Atomic &A, const CelBatch &B, const CelRec *rec, double2 *rate,
                                          int lane, double Te, double sqrTe)
{
    for (int p = lane; p < B.npair; p += 64) {
        const int at = A.cel_pair[B.pair0 + p], slot = at & 3, local = at >> 2;
        const CelRec &R = rec[slot];
        const double2 t0 = A.cel_s[R.tab + local], t1 = A.cel_s[R.tab + R.step + local];
        double cs = t0.x;
        if (R.mode == 2) {
            const double a = R.ca, b = R.cb;
            cs = a * t0.x + b * t1.x + ((a * a * a - a) * t0.y + (b * b * b - b) * t1.y) * R.h2 / 6.;
        } else if (R.mode == 1) {
            cs = t0.x + (t1.x - t0.x) / R.ca * R.cb;
        }
        const double expFac = exp(A.cel_de[B.pair0 + p] / Te);
        rate[p] = double2{ 8.63e-6 * cs * expFac / (A.cel_glo[B.pair0 + p] * sqrTe),
                           8.63e-6 * cs / (A.cel_gup[B.pair0 + p] * sqrTe) };
    }
}

// v of lane P of each row of 16 lanes (every lane active)
template <int P>
__device__ __forceinline__ double row_lane(double v)
{
    return __builtin_amdgcn_update_dpp(0.0, v, 0x150 + P, 0xf, 0xf, true);
}

template <int I> struct Const { static constexpr int value = I; };
template <int I, int N, class F>
__device__ __forceinline__ void static_for(F &&f)
{
    if constexpr (I < N) {
        f(Const<I>{});
        static_for<I + 1, N>(f);
    }
}

// Populations of a batch: the lane's level (r + 2), level 1 and the sum over
// levels, unnormalised.
struct CelLevels { double y, y1, sum; };

// N rows per ion at most (8 or 16).  Rows and columns an ion does not have
// are those of a unit matrix with a zero right side: they stay as they are.
template <int N>
__device__ __forceinline__ CelLevels cel_solve(const Atomic &A, int b, const CelBatch &B, const CelRec *rec,
                                               const double2 *rate, int lane, double Ne)
{
    const int g = lane >> 4, r = lane & 15, i = r + 2;
    const int rows = B.rows[g], nl = rows + 1, most = B.most;
    const bool mine = r < rows;
    const double *Aul = A.cel_at + (size_t)b * (kMaxLev + 1) * 64 + lane;
    const double2 *q = rate + B.base[g];
    // rate matrix row i in the reference's j order (emission_mod.f90:
    // 2047-2085); pairs (lower, upper) are numbered lower level outermost
    double x[N], x1, y, diag;
    {
        const double2 q1 = q[mine ? r : 0];
        const double a1 = Aul[64];
        x1 = mine ? 0.0 + Ne * q1.x : 0.0;
        diag = mine ? 0.0 - Ne * q1.y - a1 : 1.0;
    }
    const int own = (i - 1) * nl - (i - 1) * i / 2 - i - 1;      // pair (i, j) at own + j
    static_for<0, N / 4>([&](auto G) {
        constexpr int c0 = 4 * decltype(G)::value;
        if (c0 < most) {
            double2 qq[4];
            double a[4];
            for (int u = 0; u < 4; ++u) {
                const int j = c0 + u + 2;
                const bool on = mine && j <= nl && j != i;
                const int below = (j - 1) * nl - (j - 1) * j / 2 - j - 1;   // pair (j, i) at below + i
                qq[u] = q[on ? (j < i ? below + i : own + j) : 0];
                a[u] = Aul[64 * j];
            }
            for (int u = 0; u < 4; ++u) {
                const int j = c0 + u + 2;
                const bool on = mine && j <= nl && j != i, lower = j < i;
                const double in = 0.0 + Ne * (lower ? qq[u].x : qq[u].y);
                const double out = diag - Ne * (lower ? qq[u].y : qq[u].x);
                x[c0 + u] = on ? (lower ? in : in + a[u]) : 0.0;
                diag = on ? (lower ? out - a[u] : out) : diag;
            }
        } else {
            for (int u = 0; u < 4; ++u) x[c0 + u] = 0.0;
        }
    });
    y = mine ? -(Ne * rec[g].up * rec[g].alev) : 0.0;
    // the pivot of row 1, whose entries and right side are ones
    for (int c = 0; c < N; ++c) {
        x[c] = r == c ? diag : x[c];
        x[c] = mine && c < rows ? x[c] - x1 : x[c];
    }
    y = y - x1;
    // lured without pivoting, reslv's forward substitution with it
    static_for<0, N - 1>([&](auto P) {
        constexpr int p = decltype(P)::value;
        if (p < most - 1) {
            const double pivot = row_lane<p>(x[p]), yp = row_lane<p>(y);
            const double factor = x[p] / pivot, ynew = y - yp * x[p] / pivot;
            const bool update = r > p && mine;
            static_for<p / 4, N / 4>([&](auto G) {
                constexpr int c0 = 4 * decltype(G)::value;
                if (c0 < most) {
                    double t[4];
                    static_for<0, 4>([&](auto U) {
                        constexpr int u = decltype(U)::value;
                        if constexpr (c0 + u > p) t[u] = row_lane<p>(x[c0 + u]);
                    });
                    if (update) {
                        static_for<0, 4>([&](auto U) {
                            constexpr int u = decltype(U)::value;
                            if constexpr (c0 + u > p) x[c0 + u] = x[c0 + u] - t[u] * factor;
                        });
                    }
                }
            });
            y = update ? ynew : y;
        }
    });
    // reslv's back substitution; column k turns into the products with y(k)
    CelLevels L;
    static_for<0, N>([&](auto K) {
        constexpr int k = N - 1 - decltype(K)::value;
        if (k < most) {
            double t = y;
            static_for<k + 1, N>([&](auto C) {
                constexpr int c = decltype(C)::value;
                if (c < most) t = t - x[c];
            });
            t = t / x[k];
            y = r == k ? t : y;
            x[k] = row_lane<k>(t) * x[k];
        }
    });
    L.y = y;
    L.y1 = 1.0;
    static_for<0, N>([&](auto C) {
        constexpr int c = decltype(C)::value;
        if (c < most) L.y1 = L.y1 - row_lane<c>(y);
    });
    L.sum = 0.0 + L.y1;
    static_for<0, N>([&](auto C) {
        constexpr int c = decltype(C)::value;
        if (c < most) L.sum = L.sum + row_lane<c>(y);
    });
    return L;
}

__device__ __forceinline__ CelLevels cel_levels(const Atomic &A, int b, const CelRec *rec, double2 *rate, int lane,
                                                double Te, double sqrTe, double Ne)
{
    const CelBatch &B = A.celb[b];
    cel_rates(A, B, rec, rate, lane, Te, sqrTe);
    __syncthreads();
    const CelLevels L = B.most > 8 ? cel_solve<16>(A, b, B, rec, rate, lane, Ne)
                                   : cel_solve<8>(A, b, B, rec, rate, lane, Ne);
    __syncthreads();
    return L;
}

}  // namespace mcb
