// gamd_scf.hpp -- the SCF basis expansion on a GPU lane.
//
// Hernquist-Ostriker, Lowing+2011 real coefficients: the quantity gala computes
// term by term in bfe.cpp:114-189 with GSL calls per (n,l,m)
// (bfe_helper.cpp:24-90), reorganised:
//   * cos(m phi), sin(m phi) by the angle-addition recurrence from x/R, y/R;
//   * normalised Y_lm(cos theta) and dY_lm/dtheta by the standard stable
//     recurrences (one pass over l, m);
//   * per l, Gegenbauer C_n^{(2l+3/2)}(xi) and C_{n-1}^{(2l+5/2)}(xi) by their
//     three-term recurrences, giving phi_nl(s) and dphi_nl/ds for all n;
//   * the n-sums A_lm = sum_n phi_nl S_nlm (and T, and the s-derivatives)
//     are FMA chains over coefficients read with wave-uniform (scalar) loads.
//
// What bounds it is FP64 issue: 1,078 of ~2,500 vector instructions per
// evaluation at nmax 10, lmax 6 are those FMAs.  Left to itself the compiler
// interleaves the seven l and reads coefficients far ahead: 366 registers, one
// wave per SIMD, stalled 40 % of the time (262,144 Leapfrog orbits x 200
// steps: 7.40 ms).  Here one l is worked off at a time, its rows of
// coefficients read one batch ahead into scalar registers, its sums pinned
// before the next batch: 160 registers, three waves per SIMD, ~2,370 vector
// instructions instead of 3,270 (no T_nl0, sin(0 phi) = 0; C_n and its
// derivative share a product), the same results bit for bit, 3.71 ms.  Any
// other size runs the same code with n counted at run time (220 registers):
// 100,001 points of an nmax 6, lmax 4 expansion take 10 us for the value
// and 12 for the gradient, 115 and 135 with the expansion behind a call
// and its sums in scratch memory.
//
// The table is one stream of doubles in order of use, made by the host
// (scf_table in gamd_potential.hip).  Per l a block of
//   nmax + 1 rows  n + a - 1, n + 2a - 2, 1/n, n + 2a - 1, 1/(n - 1),
//                  S_nl0, S_nl1, T_nl1, ..., S_nll, T_nll      (a = 2l + 3/2)
//   one row        c_l, then for m < l: al, bl, d
// with Y_(l+1)(l+1) = c_l sin(theta) Y_ll, Y_lm = al (X Y_(l-1)m - bl Y_(l-2)m)
// (bl absent for m = l - 1), sin(theta) dY_lm/dtheta = l X Y_lm - d Y_(l-1)m.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

#include "gala_amd.h"

namespace gamd {

constexpr int SCF_ROW_HEAD = 5;
__host__ __device__ constexpr int scf_row(int l) { return SCF_ROW_HEAD + 1 + 2 * l; }
__host__ __device__ inline int scf_table_size(int nmax, int lmax) {
    int n = 0;
    for (int l = 0; l <= lmax; l++) n += (nmax + 1) * scf_row(l) + 1 + 3 * l;
    return n;
}

// a batch of table doubles into scalar registers: the table is read-only for
// the whole launch and every lane reads the same double, so through the
// constant address space these are scalar loads
typedef const __attribute__((address_space(4))) double *scf_cptr;
constexpr int SCF_BATCH = 26;
__device__ __forceinline__ void scf_load(double (&d)[SCF_BATCH], scf_cptr p, int count) {
#pragma unroll
    for (int i = 0; i < SCF_BATCH; i++)
        if (i < count) d[i] = p[i];
}

// what one evaluation carries from l to l + 1
template <int LB>
struct ScfState {
    scf_cptr p;                     // the table's block of l
    double s, X, sinth, cphi, sphi; // radius in r_s, angles
    double xi, inv_s, inv_ops, inv_ops2;
    double pre;                     // -sqrt(4 pi) s^l (1 + s)^(-2l - 1)
    double ymm;                     // Y_ll
    double cm[LB + 1], sm[LB + 1];  // cos(m phi), sin(m phi)
    double y1[LB + 1], y2[LB + 1];  // Y_(l-1)m, Y_(l-2)m
    double Phi, dr, dth, dph;
};

// the terms of one l, a constant once inlined.  NMAX < 0: nmax at run time.
template <int NMAX, int LB, bool VALUE, bool GRAD>
__device__ __forceinline__ void scf_terms(ScfState<LB> &q, int l, int nmax) {
    if (l > 0) {
        q.cm[l] = q.cm[l - 1] * q.cphi - q.sm[l - 1] * q.sphi;
        q.sm[l] = q.sm[l - 1] * q.cphi + q.cm[l - 1] * q.sphi;
    }
    const int RL = scf_row(l);
    // phi_nl = pre C_n^{a}(xi), a = 2l + 3/2
    // dphi_nl/ds = pre [ (l/s - (2l+1)/(1+s)) C_n^{a} + 2a C_{n-1}^{a+1} 2/(1+s)^2 ]
    const double a = 2.0 * l + 1.5, b = a + 1.0;
    const double dlog = (l == 0 ? 0.0 : l * q.inv_s) - (2.0 * l + 1.0) * q.inv_ops;
    const double chain = 4.0 * a * q.inv_ops2;
    double As[LB + 1], Bs[LB + 1], dAs[LB + 1], dBs[LB + 1];  // n-sums per m
    double c0 = 1.0, c1 = 0.0;  // C_n^a, C_{n-1}^a
    double e0 = 0.0, e1 = 0.0;  // C_{n-1}^{a+1}, C_{n-2}^{a+1}
    // row n (counted only as far as 3) of the sums; `next` asks for the rows
    // after it once this row has arrived (scalar loads return in any order, so
    // a wait is a wait for all of them)
    auto row_terms = [&](const double *row, int n, auto next) {
        double Cn = 1.0, En = 0.0;  // C_n^a(xi), C_{n-1}^{a+1}(xi)
        if (n == 1) {
            Cn = 2.0 * a * q.xi;
            En = 1.0;
        } else if (n > 1) {
            const double t = 2.0 * q.xi * row[0];
            Cn = (t * c0 - row[1] * c1) * row[2];
            if (GRAD) En = n == 2 ? 2.0 * b * q.xi : (t * e0 - row[3] * e1) * row[4];
        }
        c1 = c0;
        c0 = Cn;
        e1 = e0;
        e0 = En;
        const double phinl = q.pre * Cn;
        const double dphinl = n == 0   ? q.pre * dlog
                              : n == 1 ? q.pre * (dlog * Cn + chain)
                                       : q.pre * (dlog * Cn + chain * En);
        next();
        const double *st = row + SCF_ROW_HEAD;
#pragma unroll
        for (int m = 0; m <= l; m++) {
            const double S = st[m == 0 ? 0 : 2 * m - 1], T = st[2 * m];
            As[m] = n == 0 ? phinl * S : fma(phinl, S, As[m]);
            if (m > 0) Bs[m] = n == 0 ? phinl * T : fma(phinl, T, Bs[m]);
            if (GRAD) {
                dAs[m] = n == 0 ? dphinl * S : fma(dphinl, S, dAs[m]);
                if (m > 0) dBs[m] = n == 0 ? dphinl * T : fma(dphinl, T, dBs[m]);
            }
        }
    };
    double cur[SCF_BATCH], nxt[SCF_BATCH];
    if (NMAX >= 0) {
        // G rows per batch of loads: scalar registers for two batches
        const int G = RL <= 6 ? 4 : RL <= 8 ? 3 : RL <= 12 ? 2 : 1;
        scf_load(cur, q.p, (G < NMAX + 1 ? G : NMAX + 1) * RL);
#pragma unroll
        for (int n0 = 0; n0 <= NMAX; n0 += G) {
#pragma unroll
            for (int k = 0; k < G; k++) {
                if (n0 + k > NMAX) break;
                row_terms(cur + k * RL, n0 + k, [&] {
                    if (k > 0 || n0 + G > NMAX) return;
                    const int left = (NMAX + 1 - n0 - G) * RL;
                    __builtin_amdgcn_sched_barrier(0);
                    scf_load(nxt, q.p + (n0 + G) * RL, left < G * RL ? left : G * RL);
                    __builtin_amdgcn_sched_barrier(0);
                });
            }
            // the sums so far, here and not later: sunk below the next loads,
            // they would keep every batch in scalar registers
#pragma unroll
            for (int m = 0; m <= l; m++) {
                asm volatile("" : "+v"(As[m]));
                if (m > 0) asm volatile("" : "+v"(Bs[m]));
                if (GRAD) {
                    asm volatile("" : "+v"(dAs[m]));
                    if (m > 0) asm volatile("" : "+v"(dBs[m]));
                }
            }
            __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (int i = 0; i < SCF_BATCH; i++)
                if (i < G * RL) cur[i] = nxt[i];
        }
    } else {
        scf_load(cur, q.p, RL);
        row_terms(cur, 0, [] {});
        scf_cptr row = q.p;
        if (nmax >= 1) {
            scf_load(cur, row += RL, RL);
            row_terms(cur, 1, [] {});
        }
        if (nmax >= 2) {
            scf_load(cur, row += RL, RL);
            row_terms(cur, 2, [] {});
        }
#pragma unroll 1
        for (int n = 3; n <= nmax; n++) {
            scf_load(cur, row += RL, RL);
            row_terms(cur, 3, [] {});
        }
    }
    const scf_cptr ang = q.p + (nmax + 1) * RL;
#pragma unroll
    for (int m = 0; m <= l; m++) {
        double v;  // Y_lm(X), normalised, Condon-Shortley phase
        if (m == l)
            v = q.ymm;
        else if (m == l - 1)
            v = ang[1 + 3 * m] * q.X * q.y1[m];
        else
            v = ang[1 + 3 * m] * (q.X * q.y1[m] - ang[2 + 3 * m] * q.y2[m]);
        const double ac = m == 0 ? As[0] : As[m] * q.cm[m] + Bs[m] * q.sm[m];
        if (VALUE) q.Phi = fma(v, ac, q.Phi);
        if (GRAD) {
            const double dac = m == 0 ? dAs[0] : dAs[m] * q.cm[m] + dBs[m] * q.sm[m];
            q.dr = fma(v, dac, q.dr);
            double dy = l * q.X * v;
            if (NMAX >= 0 && l == 1 && m == 0) {
                // both factors are constants: one rounded product, not fused
                const double dY = ang[3] * q.y1[0];
                dy = dy - dY;
            } else if (m < l) {
                dy -= ang[3 + 3 * m] * q.y1[m];
            }
            q.dth = fma(dy, ac, q.dth);
            if (m > 0) q.dph = fma((double)m * v, Bs[m] * q.cm[m] - As[m] * q.sm[m], q.dph);
        }
        q.y2[m] = q.y1[m];
        q.y1[m] = v;
    }
    q.ymm = ang[0] * q.sinth * q.ymm;
    q.pre = q.pre * q.s * q.inv_ops2;
    q.p += (nmax + 1) * RL + 1 + 3 * l;
    // one l at a time: interleaved, their sums exceed the registers
    if (NMAX >= 0) {
        if (VALUE) asm volatile("" : "+v"(q.Phi));
        if (GRAD) asm volatile("" : "+v"(q.dr), "+v"(q.dth), "+v"(q.dph));
#pragma unroll
        for (int m = 0; m <= l; m++) asm volatile("" : "+v"(q.y1[m]));
    }
    __builtin_amdgcn_sched_barrier(0);
}

template <int l, int LB, bool VALUE, bool GRAD>
__device__ __forceinline__ void scf_terms_from(ScfState<LB> &q, int nmax, int lmax) {
    if constexpr (l <= LB) {
        if (l > lmax) return;
        scf_terms<-1, LB, VALUE, GRAD>(q, l, nmax);
        scf_terms_from<l + 1, LB, VALUE, GRAD>(q, nmax, lmax);
    }
}

// Phi (VALUE) and grad Phi (GRAD) of an expansion with table `table`.  NMAX <
// 0: any size with lmax <= LB; else exactly nmax = NMAX, lmax = LB.
template <int NMAX, int LB, bool VALUE, bool GRAD>
__device__ __forceinline__ void scf_field(const double *table, double G, double M, double rs,
                                          int nmax, int lmax, double x, double y, double z,
                                          double &phi, double &gx, double &gy, double &gz) {
    const double FOURPI_SQRT = 3.544907701811031;
    ScfState<LB> q;
    // opaque at each evaluation, so that a time loop does not lift the 900
    // loads out of itself and spill them
    q.p = (scf_cptr)table;
    asm volatile("" : "+s"(q.p));
    const double R2 = x * x + y * y;
    const double r2 = R2 + z * z;
    const double r = sqrt(r2);
    const double Rc = sqrt(R2);
    const double s = r / rs;
    q.s = s;
    q.X = z / r;         // cos(theta)
    q.sinth = Rc / r;    // sin(theta)
    q.cphi = 1.0;        // atan2(0, 0) = 0 on the axis, as gala
    q.sphi = 0.0;
    if (Rc > 0.0) {
        q.cphi = x / Rc;
        q.sphi = y / Rc;
    }
    const double ops = 1.0 + s;
    q.inv_ops = 1.0 / ops;
    q.inv_s = 1.0 / s;
    q.xi = (s - 1.0) * q.inv_ops;
    q.inv_ops2 = q.inv_ops * q.inv_ops;
    q.pre = -FOURPI_SQRT / ops;
    q.ymm = 1.0 / FOURPI_SQRT;
    q.Phi = q.dr = q.dth = q.dph = 0.0;
    q.cm[0] = 1.0;
    q.sm[0] = 0.0;
#pragma unroll
    for (int m = 0; m <= LB; m++) q.y1[m] = q.y2[m] = 0.0;
    if (NMAX >= 0) {
#pragma unroll
        for (int l = 0; l <= LB; l++) scf_terms<NMAX, LB, VALUE, GRAD>(q, l, NMAX);
    } else {
        scf_terms_from<0, LB, VALUE, GRAD>(q, nmax, lmax);
    }
    const double GMr = G * M / rs;
    if (VALUE) phi = q.Phi * GMr;
    if (GRAD) {
        // (d/dr, (1/r) d/dtheta, 1/(r sin theta) d/dphi) in units of r_s, then Cartesian
        const double g_r = q.dr;
        const double g_t = q.dth / (s * q.sinth);
        const double g_p = q.dph / (s * q.sinth);
        const double fac = G * M / (rs * rs);
        gx = (q.sinth * q.cphi * g_r + q.X * q.cphi * g_t - q.sphi * g_p) * fac;
        gy = (q.sinth * q.sphi * g_r + q.X * q.sphi * g_t + q.cphi * g_p) * fac;
        gz = (q.X * g_r - q.sinth * g_t) * fac;
    }
}

}  // namespace gamd
