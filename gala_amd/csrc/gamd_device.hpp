// gamd_device.hpp -- device-side potential table and FP64 force kernels.
//
// A potential is a small flat table (DevPot) passed BY VALUE as a kernel
// argument, so every wave reads it through scalar loads from the kernarg
// segment: the component type switch is wave-uniform (a scalar branch, no
// divergence) and the parameters sit in SGPRs.  This replaces gala's table of
// function pointers (potential/potential/src/cpotential.h:10-36) with no
// indirect calls.  Parameter-only subexpressions (G*m, b*b, ...) are folded
// on the host into d[]; the products are the same IEEE values gala forms on
// every call (builtin_potentials.cpp:221-233 etc.), so nothing changes but
// the work.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

#include "gala_amd.h"
#include "gamd_scf.hpp"

namespace gamd {

constexpr int MAXC = GAMD_MAX_COMPONENTS;

struct DevComp {
    int32_t type;
    int32_t shift_rotate;
    int32_t nmax, lmax;
    double p[8];          // raw parameters, p[0] = G (gala's pars layout)
    double d[4];          // host-folded constants, see fold_component()
    double q0[3];
    double R[9];
    const double *coef;   // SCF: device, the table of gamd_scf.hpp
};

struct DevPot {
    int32_t n;
    int32_t has_scf;
    int32_t all_unshifted;
    int32_t layout;       // LAYOUT_* below: selects a straight-line evaluator
    DevComp c[MAXC];
};

// Component layouts with a dedicated straight-line evaluator.  With a runtime
// loop over components each component is its own basic block and the four
// dependent sqrt/divide/log chains run one after the other; written out
// straight, the scheduler interleaves them, which is what a lone lane in the
// tail of a persistent launch needs.
// MW: Hernquist, Hernquist, MN, NFW, unshifted.  SCF: one unshifted SCF
// component of any size; SCF106: the same with nmax = 10, lmax = 6, written out
// whole.
enum { LAYOUT_GENERIC = 0, LAYOUT_MW = 1, LAYOUT_SCF106 = 2, LAYOUT_SCF = 3 };

// ---------------------------------------------------------------------------
// Natural log with a short dependency chain, for finite x > 0.  The library
// log costs ~470 cycles of latency for one lane on gfx950 (a divide ~76, an
// FMA ~6), and a lone lane in the tail of a persistent launch is latency-
// bound.  Method: x = m 2^e with m in [sqrt(1/2), sqrt(2)); log m =
// 2 atanh(s) = 2 s sum_k s^(2k)/(2k+1), s = (m-1)/(m+1), |s| <= 0.1716, so
// twelve terms reach 1e-20; the series is summed by Estrin's scheme (depth
// ~6 FMAs) and e ln2 is added with ln2 split in two (the high part has 21
// trailing zero bits, so e * ln2_hi is exact).  Error ~1-2 ulp.
// argument reduction: x = 2^e (1 + f) with 1 + f in [sqrt(1/2), sqrt(2))
__device__ __forceinline__ void log_reduce(double x, double &f, int &e) {
    const double m = frexp(x, &e);  // m in [0.5, 1)
    const bool low = m < 0.7071067811865476;
    f = fma(m, low ? 2.0 : 1.0, -1.0);  // 2 m - 1 or m - 1, exact before the one rounding
    e -= low ? 1 : 0;
}

// z * k + c with a polynomial's constants k and c in registers that outlive
// it: written as fma the compiler copies c first (it prefers the form that
// accumulates in place), a copy per term of every log
__device__ __forceinline__ double fma_const(double z, double k, double c) {
    double d;
    asm("v_fma_f64 %0, %1, %2, %3" : "=v"(d) : "v"(z), "s"(k), "v"(c));
    return d;
}

// the series' polynomial in z = s^2 (z2 = z^2, ...)
__device__ __forceinline__ double log_poly(double z, double z2, double z4, double z8) {
    const double p01 = fma(z, 0.3333333333333333, 1.0);
    const double p23 = fma_const(z, 0.14285714285714285, 0.2);
    const double p45 = fma_const(z, 0.09090909090909091, 0.1111111111111111);
    const double p67 = fma_const(z, 0.06666666666666667, 0.07692307692307693);
    const double p89 = fma_const(z, 0.05263157894736842, 0.058823529411764705);
    const double pab = fma_const(z, 0.043478260869565216, 0.047619047619047616);
    const double q03 = fma(z2, p23, p01);
    const double q47 = fma(z2, p67, p45);
    const double q8b = fma(z2, pab, p89);
    return fma(z8, q8b, fma(z4, q47, q03));
}

// ln(2^e (1 + f)) from s = f / (2 + f)
template <class Poly>
__device__ __forceinline__ double log_series(double s, int e, const Poly &poly) {
    const double z = s * s;
    const double z2 = z * z, z4 = z2 * z2, z8 = z4 * z4;
    const double P = poly(z, z2, z4, z8);
    const double ed = (double)e;
    const double lm = (s + s) * P;
    return fma(ed, 0.6931471803691238, fma(ed, 1.9082149292705877e-10, lm));
}
__device__ __forceinline__ double log_series(double s, int e) {
    return log_series(s, e, [](double z, double z2, double z4, double z8) {
        return log_poly(z, z2, z4, z8);
    });
}

__device__ __forceinline__ double log_fast(double x) {
    double f;
    int e;
    log_reduce(x, f, e);
    return log_series(f / (2.0 + f), e);
}

// 1/sqrt(x) for finite x > 0: the hardware estimate (v_rsq_f64) refined by
// two Newton steps y <- y + y (1/2 - (x/2) y^2) in FMA form (~1 ulp; a
// correctly rounded sqrt is ~110 cycles of latency on gfx950, this ~60).
__device__ __forceinline__ double rsqrt_nr(double x) {
    double y = __builtin_amdgcn_rsq(x);
    const double hx = 0.5 * x;
    double r = fma(-hx * y, y, 0.5);
    y = fma(y, r, y);
    r = fma(-hx * y, y, 0.5);
    return fma(y, r, y);
}

// 1/d for finite nonzero d: v_rcp_f64 refined by two Newton steps (~1 ulp).
__device__ __forceinline__ double rcp_nr(double d) {
    double y = __builtin_amdgcn_rcp(d);
    double e = fma(-d, y, 1.0);
    y = fma(y, e, y);
    e = fma(-d, y, 1.0);
    return fma(y, e, y);
}

// ---------------------------------------------------------------------------
// analytic components: accumulate the gradient (gala's *_gradient_single
// semantics, grad += ...).  r is |q| when the caller already has it (a
// composite shares one sqrt across its unshifted spherical components).

// Hernquist, builtin_potentials.cpp:221-233.  d = [G m, c]
__device__ __forceinline__ void hernquist_grad(const DevComp &c, double x, double y, double z,
                                               double r, double &gx, double &gy, double &gz) {
    const double rc = r + c.d[1];
    const double fac = c.d[0] / (rc * rc * r);
    gx += fac * x;
    gy += fac * y;
    gz += fac * z;
}

// Plummer, builtin_potentials.cpp:302-314.  d = [G m, b^2]
__device__ __forceinline__ void plummer_grad(const DevComp &c, double x, double y, double z,
                                             double r2, double &gx, double &gy, double &gz) {
    const double R2b = r2 + c.d[1];
    const double fac = c.d[0] / sqrt(R2b) / R2b;
    gx += fac * x;
    gy += fac * y;
    gz += fac * z;
}

// Miyamoto-Nagai, builtin_potentials.cpp:1298-1312.  d = [G m, a, b^2]
// pow(D, -1.5) is formed as 1/(D sqrt(D)) (a sqrt and a divide instead of a
// log/exp pair; within 2 ulp of gala's pow).
__device__ __forceinline__ void mn_grad(const DevComp &c, double x, double y, double z,
                                        double &gx, double &gy, double &gz) {
    const double sqrtz = sqrt(z * z + c.d[2]);
    const double zd = c.d[1] + sqrtz;
    const double D = x * x + y * y + zd * zd;
    const double fac = c.d[0] / (D * sqrt(D));
    gx += fac * x;
    gy += fac * y;
    gz += fac * z * (1.0 + c.d[1] / sqrtz);
}

// Spherical NFW, builtin_potentials.cpp:835-850.  d = [G m / r_s, r_s, r_s^2]
// NaN at r = 0 exactly as there (0/0).
__device__ __forceinline__ void nfw_grad(const DevComp &c, double x, double y, double z, double r,
                                         double &gx, double &gy, double &gz) {
    const double u = r / c.d[1];
    const double fac = c.d[0] / (u * u * u) / c.d[2] * (log(1.0 + u) - u / (1.0 + u));
    gx += fac * x;
    gy += fac * y;
    gz += fac * z;
}

__device__ __forceinline__ double comp_value_analytic(const DevComp &c, double x, double y,
                                                      double z) {
    const double *p = c.p;
    switch (c.type) {
    case GAMD_HERNQUIST: {  // :211-219
        const double r = sqrt(x * x + y * y + z * z);
        return -p[0] * p[1] / (r + p[2]);
    }
    case GAMD_PLUMMER: {  // :292-300
        const double r2 = x * x + y * y + z * z;
        return -p[0] * p[1] / sqrt(r2 + p[2] * p[2]);
    }
    case GAMD_MIYAMOTONAGAI: {  // :1287-1296
        const double zd = p[2] + sqrt(z * z + p[3] * p[3]);
        return -p[0] * p[1] / sqrt(x * x + y * y + zd * zd);
    }
    case GAMD_NFW: {  // :819-833
        const double v_h2 = -p[0] * p[1] / p[2];
        const double u = sqrt(x * x + y * y + z * z) / p[2];
        if (u == 0.0) return v_h2;
        return v_h2 * log(1.0 + u) / u;
    }
    default:
        return 0.0;
    }
}

__device__ __forceinline__ double comp_density_analytic(const DevComp &c, double x, double y,
                                                        double z) {
    const double *p = c.p;
    const double PI = 3.141592653589793;
    switch (c.type) {
    case GAMD_HERNQUIST: {  // :235-244
        const double r = sqrt(x * x + y * y + z * z);
        const double rho0 = p[1] / (2.0 * PI * p[2] * p[2] * p[2]);
        const double w = 1.0 + r / p[2];
        return rho0 / ((r / p[2]) * (w * w * w));
    }
    case GAMD_PLUMMER: {  // :316-324
        const double r2 = x * x + y * y + z * z;
        const double w = 1.0 + r2 / (p[2] * p[2]);
        return 3.0 * p[1] / (4.0 * PI * p[2] * p[2] * p[2]) / (w * w * sqrt(w));
    }
    case GAMD_MIYAMOTONAGAI: {  // :1314-1331
        const double M = p[1], a = p[2], b = p[3];
        const double R2 = x * x + y * y;
        const double sz = sqrt(z * z + b * b);
        const double numer = (b * b * M / (4.0 * PI)) * (a * R2 + (a + 3.0 * sz) * (a + sz) * (a + sz));
        const double D = R2 + (a + sz) * (a + sz);
        const double denom = D * D * sqrt(D) * sz * sz * sz;
        return numer / denom;
    }
    case GAMD_NFW: {  // :852-863
        const double r = sqrt(x * x + y * y + z * z);
        const double rho0 = p[1] / (4.0 * PI * p[2] * p[2] * p[2]);
        const double w = 1.0 + r / p[2];
        return rho0 / ((r / p[2]) * (w * w));
    }
    default:
        return 0.0;
    }
}

// Hessians (row-major 3x3, accumulated): the second derivatives of the same
// potentials, H = f(r) I + (f'(r)/r) q q^T for the spherical ones.
__device__ __forceinline__ void comp_hessian_analytic(const DevComp &c, double x, double y,
                                                      double z, double *H) {
    const double *p = c.p;
    const double r2 = x * x + y * y + z * z, r = sqrt(r2);
    double f = 0.0, g = 0.0;
    switch (c.type) {
    case GAMD_HERNQUIST: {
        const double GM = p[0] * p[1], rc = r + p[2];
        f = GM / (r * rc * rc);
        g = -GM * (3.0 * r + p[2]) / (r2 * r * rc * rc * rc);
        break;
    }
    case GAMD_PLUMMER: {
        const double GM = p[0] * p[1], D = r2 + p[2] * p[2];
        const double Dm32 = 1.0 / (D * sqrt(D));
        f = GM * Dm32;
        g = -3.0 * GM * Dm32 / D;
        break;
    }
    case GAMD_NFW: {
        const double GM = p[0] * p[1], rs = p[2], u = r / rs;
        f = GM / (r2 * r) * (log(1.0 + u) - u / (1.0 + u));
        g = (-3.0 * f / r + GM / (r2 * rs * rs * (1.0 + u) * (1.0 + u))) / r;
        break;
    }
    case GAMD_MIYAMOTONAGAI: {
        const double GM = p[0] * p[1], b = p[3];
        const double s = sqrt(z * z + b * b), zeta = p[2] + s;
        const double D = x * x + y * y + zeta * zeta;
        const double Dm32 = 1.0 / (D * sqrt(D)), Dm52 = Dm32 / D;
        const double w = zeta * z / s;
        H[0] += GM * (Dm32 - 3.0 * x * x * Dm52);
        H[4] += GM * (Dm32 - 3.0 * y * y * Dm52);
        const double hxy = -3.0 * GM * x * y * Dm52;
        const double hxz = -3.0 * GM * x * w * Dm52;
        const double hyz = -3.0 * GM * y * w * Dm52;
        H[1] += hxy;
        H[3] += hxy;
        H[2] += hxz;
        H[6] += hxz;
        H[5] += hyz;
        H[7] += hyz;
        H[8] += GM * ((z * z / (s * s) + zeta * b * b / (s * s * s)) * Dm32 - 3.0 * w * w * Dm52);
        return;
    }
    default:
        return;
    }
    const double q[3] = {x, y, z};
#pragma unroll
    for (int i = 0; i < 3; i++)
#pragma unroll
        for (int j = 0; j < 3; j++) H[3 * i + j] += (i == j ? f : 0.0) + g * q[i] * q[j];
}

// ---------------------------------------------------------------------------
// SCF basis expansion (gamd_scf.hpp): one out-of-line copy per kernel of the
// value and of the gradient.  The sum is long, and inlining it at each of
// DOP853's stage evaluations would multiply code size (and compile time) with
// no gain, since the call overhead is small next to the sum.
// The table and sizes are those of one component of a potential, the same in
// every lane that calls; arguments arrive in vector registers and return to
// scalar ones here.
__device__ __forceinline__ const double *wave_uniform(const double *p) {
    const uint64_t v = reinterpret_cast<uint64_t>(p);
    const uint32_t lo = __builtin_amdgcn_readfirstlane((uint32_t)v);
    const uint32_t hi = __builtin_amdgcn_readfirstlane((uint32_t)(v >> 32));
    return reinterpret_cast<const double *>(((uint64_t)hi << 32) | lo);
}

__device__ __noinline__ double scf_value(const double *__restrict__ table, double G, double M,
                                         double rs, int nmax, int lmax, double x, double y,
                                         double z) {
    table = wave_uniform(table);
    nmax = __builtin_amdgcn_readfirstlane(nmax);
    lmax = __builtin_amdgcn_readfirstlane(lmax);
    double phi, gx, gy, gz;
    if (nmax == 10 && lmax == 6)
        scf_field<10, 6, true, false>(table, G, M, rs, 10, 6, x, y, z, phi, gx, gy, gz);
    else
        scf_field<-1, GAMD_SCF_MAX_LMAX, true, false>(table, G, M, rs, nmax, lmax, x, y, z, phi,
                                                      gx, gy, gz);
    return phi;
}

__device__ __noinline__ double3 scf_grad(const double *__restrict__ table, double G, double M,
                                         double rs, int nmax, int lmax, double x, double y,
                                         double z) {
    table = wave_uniform(table);
    nmax = __builtin_amdgcn_readfirstlane(nmax);
    lmax = __builtin_amdgcn_readfirstlane(lmax);
    double phi, gx, gy, gz;
    if (nmax == 10 && lmax == 6)
        scf_field<10, 6, false, true>(table, G, M, rs, 10, 6, x, y, z, phi, gx, gy, gz);
    else
        scf_field<-1, GAMD_SCF_MAX_LMAX, false, true>(table, G, M, rs, nmax, lmax, x, y, z, phi,
                                                      gx, gy, gz);
    return make_double3(gx, gy, gz);
}

__device__ __forceinline__ void scf_add_grad(const DevComp &c, double x, double y, double z,
                                             double &gx, double &gy, double &gz) {
    const double3 g = scf_grad(c.coef, c.p[0], c.p[1], c.p[2], c.nmax, c.lmax, x, y, z);
    gx += g.x;
    gy += g.y;
    gz += g.z;
}

// SCF density (bfe.cpp:20-59): rho_nl = K_nl/(2 pi) sqrt(4 pi) s^l / (s (1+s)^(2l+3)) C_n(xi)
__device__ inline double scf_density(const DevComp &c, double x, double y, double z) {
    const int nmax = c.nmax, lmax = c.lmax;
    const double FOURPI_SQRT = 3.544907701811031, PI = 3.141592653589793;
    const double M = c.p[1], rs = c.p[2];
    const double R2 = x * x + y * y, r = sqrt(R2 + z * z), Rc = sqrt(R2);
    const double s = r / rs, X = z / r, sinth = Rc / r;
    double cphi = 1.0, sphi = 0.0;
    if (Rc > 0.0) {
        cphi = x / Rc;
        sphi = y / Rc;
    }
    const double xi = (s - 1.0) / (s + 1.0), ops = 1.0 + s;
    double cm[GAMD_SCF_MAX_LMAX + 1], sm[GAMD_SCF_MAX_LMAX + 1];
    double y1[GAMD_SCF_MAX_LMAX + 1], y2[GAMD_SCF_MAX_LMAX + 1];
    cm[0] = 1.0;
    sm[0] = 0.0;
    for (int m = 1; m <= lmax; m++) {
        cm[m] = cm[m - 1] * cphi - sm[m - 1] * sphi;
        sm[m] = sm[m - 1] * cphi + cm[m - 1] * sphi;
    }
    for (int m = 0; m <= lmax; m++) y1[m] = y2[m] = 0.0;
    double ymm = 1.0 / FOURPI_SQRT, rho = 0.0;
    const double *table = c.coef;  // the block of l
    double pre = FOURPI_SQRT / (2.0 * PI) / (s * ops * ops * ops);  // s^l/(s (1+s)^(2l+3)) at l=0
    for (int l = 0; l <= lmax; l++) {
        const double a = 2.0 * l + 1.5;
        for (int m = 0; m <= l; m++) {
            double v;
            if (m == l) v = ymm;
            else if (m == l - 1) v = sqrt(2.0 * m + 3.0) * X * y1[m];
            else {
                const double l2 = (double)l * l, m2 = (double)m * m;
                v = sqrt((4.0 * l2 - 1.0) / (l2 - m2)) *
                    (X * y1[m] - sqrt(((l - 1.0) * (l - 1.0) - m2) / (4.0 * (l - 1.0) * (l - 1.0) - 1.0)) * y2[m]);
            }
            double c0 = 1.0, c1 = 0.0, A = 0.0, B = 0.0;
            for (int n = 0; n <= nmax; n++) {
                double Cn = n == 0 ? 1.0 : (n == 1 ? 2.0 * a * xi : (2.0 * xi * (n + a - 1.0) * c0 - (n + 2.0 * a - 2.0) * c1) / n);
                c1 = c0;
                c0 = Cn;
                const double Knl = 0.5 * n * (n + 4 * l + 3) + (l + 1) * (2 * l + 1);
                const double rnl = Knl * pre * Cn;
                const double *st = table + n * scf_row(l) + SCF_ROW_HEAD;
                A += rnl * st[m == 0 ? 0 : 2 * m - 1];
                B += rnl * (m == 0 ? 0.0 : st[2 * m]);  // sin(0 phi) = 0
            }
            rho += v * (A * cm[m] + B * sm[m]);
            y2[m] = y1[m];
            y1[m] = v;
        }
        ymm = -sqrt((2.0 * l + 3.0) / (2.0 * l + 2.0)) * sinth * ymm;
        pre = pre * s / (ops * ops);
        table += (nmax + 1) * scf_row(l) + 1 + 3 * l;
    }
    return rho * M / (rs * rs * rs);
}

// ---------------------------------------------------------------------------
// composite evaluation (cpotential.cpp:170-287).  Components run in table
// order; a shifted/rotated component is evaluated at R (q - q0) and its
// gradient rotated back with R^T.

template <bool WITH_SCF>
__device__ __forceinline__ void comp_grad(const DevComp &c, double x, double y, double z,
                                          double &gx, double &gy, double &gz) {
    switch (c.type) {
    case GAMD_HERNQUIST:
        hernquist_grad(c, x, y, z, sqrt(x * x + y * y + z * z), gx, gy, gz);
        break;
    case GAMD_PLUMMER:
        plummer_grad(c, x, y, z, x * x + y * y + z * z, gx, gy, gz);
        break;
    case GAMD_MIYAMOTONAGAI:
        mn_grad(c, x, y, z, gx, gy, gz);
        break;
    case GAMD_NFW:
        nfw_grad(c, x, y, z, sqrt(x * x + y * y + z * z), gx, gy, gz);
        break;
    case GAMD_SCF:
        if (WITH_SCF) scf_add_grad(c, x, y, z, gx, gy, gz);
        break;
    default:
        break;
    }
}

__device__ __forceinline__ void shift_rotate(const DevComp &c, double x, double y, double z,
                                             double &xt, double &yt, double &zt) {
    const double tx = x - c.q0[0], ty = y - c.q0[1], tz = z - c.q0[2];
    xt = c.R[0] * tx + c.R[1] * ty + c.R[2] * tz;
    yt = c.R[3] * tx + c.R[4] * ty + c.R[5] * tz;
    zt = c.R[6] * tx + c.R[7] * ty + c.R[8] * tz;
}

// grad Phi at (x, y, z): overwritten (c_gradient zeroes first).
template <bool WITH_SCF>
__device__ __forceinline__ void pot_grad(const DevPot &P, double x, double y, double z,
                                         double &gx, double &gy, double &gz) {
    gx = 0.0;
    gy = 0.0;
    gz = 0.0;
    if (P.all_unshifted) {
        // one |q| shared by every unshifted spherical component
        const double r2 = x * x + y * y + z * z;
        const double r = sqrt(r2);
        for (int i = 0; i < P.n; i++) {
            const DevComp &c = P.c[i];
            switch (c.type) {
            case GAMD_HERNQUIST: hernquist_grad(c, x, y, z, r, gx, gy, gz); break;
            case GAMD_PLUMMER: plummer_grad(c, x, y, z, r2, gx, gy, gz); break;
            case GAMD_MIYAMOTONAGAI: mn_grad(c, x, y, z, gx, gy, gz); break;
            case GAMD_NFW: nfw_grad(c, x, y, z, r, gx, gy, gz); break;
            case GAMD_SCF:
                if (WITH_SCF) scf_add_grad(c, x, y, z, gx, gy, gz);
                break;
            default: break;
            }
        }
        return;
    }
    for (int i = 0; i < P.n; i++) {
        const DevComp &c = P.c[i];
        if (!c.shift_rotate) {
            comp_grad<WITH_SCF>(c, x, y, z, gx, gy, gz);
        } else {
            double xt, yt, zt, tx = 0.0, ty = 0.0, tz = 0.0;
            shift_rotate(c, x, y, z, xt, yt, zt);
            comp_grad<WITH_SCF>(c, xt, yt, zt, tx, ty, tz);
            gx += c.R[0] * tx + c.R[3] * ty + c.R[6] * tz;
            gy += c.R[1] * tx + c.R[4] * ty + c.R[7] * tz;
            gz += c.R[2] * tx + c.R[5] * ty + c.R[8] * tz;
        }
    }
}

// Gradient of a body's potential PP at q, centred on the body's position xp:
// c_gradient of the potential with every component's origin set to xp
// (c_nbody_acceleration / c_nbody_gradient_symplectic force do_shift_rotate
// = 1, cpotential.cpp:389-442): q' = R (q - xp), gradient rotated back with
// R^T, summed over components into a zeroed f2 that the caller adds.
template <bool WITH_SCF>
__device__ __forceinline__ void body_grad(const DevPot &PP, double x, double y, double z,
                                          double px, double py, double pz, double &fx,
                                          double &fy, double &fz) {
    fx = 0.0;
    fy = 0.0;
    fz = 0.0;
    for (int i = 0; i < PP.n; i++) {
        const DevComp &c = PP.c[i];
        const double tx = x - px, ty = y - py, tz = z - pz;
        const double xt = c.R[0] * tx + c.R[1] * ty + c.R[2] * tz;
        const double yt = c.R[3] * tx + c.R[4] * ty + c.R[5] * tz;
        const double zt = c.R[6] * tx + c.R[7] * ty + c.R[8] * tz;
        double ux = 0.0, uy = 0.0, uz = 0.0;
        comp_grad<WITH_SCF>(c, xt, yt, zt, ux, uy, uz);
        fx += c.R[0] * ux + c.R[3] * uy + c.R[6] * uz;
        fy += c.R[1] * ux + c.R[4] * uy + c.R[7] * uz;
        fz += c.R[2] * ux + c.R[5] * uy + c.R[8] * uz;
    }
}

// The Milky-Way layout (nucleus and bulge Hernquist, Miyamoto-Nagai disk, NFW
// halo, gala's MilkyWayPotential order): the same formulas as the per-
// component functions above, one shared |q|, contributions accumulated in
// table order.

// its gradient where the shared reciprocal of mw_grad under- or overflows
// (extreme radii, r = 0, NaN): the per-component forms
__device__ __forceinline__ void mw_grad_extreme(const DevPot &P, double x, double y, double z,
                                                double &gx, double &gy, double &gz) {
    const DevComp &h1 = P.c[0], &h2 = P.c[1], &mn = P.c[2], &nf = P.c[3];
    // opaque: nothing of the ordinary evaluation is kept for this one
    asm("" : "+v"(x), "+v"(y), "+v"(z));
    const double R2 = x * x + y * y;
    const double r2 = R2 + z * z;
    const double ir = rsqrt_nr(r2);
    const double r = r2 * ir;
    const double s2 = z * z + mn.d[2];
    const double isz = rsqrt_nr(s2);
    const double sqrtz = s2 * isz;
    const double zd = mn.d[1] + sqrtz;
    const double D = R2 + zd * zd;
    const double iD = rsqrt_nr(D);
    const double f3 = mn.d[0] * (iD * iD * iD);
    const double f3z = 1.0 + mn.d[1] * isz;
    const double u = r * nf.d[3];
    const double opu = 1.0 + u;
    double lf;
    int le;
    log_reduce(opu, lf, le);
    const double rc1 = r + h1.d[1];
    const double rc2 = r + h2.d[1];
    const double d1 = rc1 * rc1 * r, d2 = rc2 * rc2 * r;
    const double f1 = h1.d[0] / d1, f2 = h2.d[0] / d2;
    const double lg = log_series(lf / (2.0 + lf), le);
    const double f4 = nf.d[0] / (u * u * u) / nf.d[2] * (lg - u / opu);
    gx = 0.0;
    gy = 0.0;
    gz = 0.0;
    gx += f1 * x;
    gy += f1 * y;
    gz += f1 * z;
    gx += f2 * x;
    gy += f2 * y;
    gz += f2 * z;
    gx += f3 * x;
    gy += f3 * y;
    gz += f3 * z * f3z;
    gx += f4 * x;
    gy += f4 * y;
    gz += f4 * z;
}

// A lone wave (a few orbits, the longest orbits of an uneven launch, a stream's
// progenitor) pays the latency of this chain at every step, so all of it up to
// the gradient is one basic block: the disk's two roots fill the waits of the
// r -> log -> reciprocal chain, and the only branch, out of it, is the rare one
// at the end.  With a branch around the shared reciprocal the compiler moved
// the disk behind it, and a step ran ~20 instructions more: 1,024 Leapfrog
// orbits x 10,000 steps, all saved, 3.73 -> 3.23 ms; 1,048,576 x 1,000 (FP64
// issue, 96 % busy) 3.98 -> 3.76 ms; the uneven DOP853 launch over 1,048,576
// orbits, its longest orbit's 23,800 attempts in a row, 129 -> 115 ms.  The same
// operations on the same values, so the same results bit for bit.
struct MwFactors {
    double f1, f2, f3, f3z, f4;  // of q: nucleus, bulge, disk (and its z), halo
    bool extreme;                // they are not to be used
};
struct MwConstants {
    double m1, c1, m2, c2;    // nucleus and bulge: G m, c
    double m3, a3, b3sq;      // disk: G m, a, b^2
    double m4, irs4;          // halo: G m, 1 / r_s
    __device__ __forceinline__ explicit MwConstants(const DevPot &P)
        : m1(P.c[0].d[0]), c1(P.c[0].d[1]), m2(P.c[1].d[0]), c2(P.c[1].d[1]), m3(P.c[2].d[0]),
          a3(P.c[2].d[1]), b3sq(P.c[2].d[2]), m4(P.c[3].d[0] * P.c[3].d[1]), irs4(P.c[3].d[3]) {}
};
// how a lane evaluates them: all of it alone
struct MwAlone {
    __device__ __forceinline__ static void rsqrt_pair(double a, double b, double &ra, double &rb) {
        ra = rsqrt_nr(a);
        rb = rsqrt_nr(b);
    }
    __device__ __forceinline__ double operator()(double z, double z2, double z4, double z8) const {
        return log_poly(z, z2, z4, z8);
    }
};
template <class Lanes>
__device__ __forceinline__ MwFactors mw_factors(const MwConstants &m, const Lanes &lanes, double x,
                                                double y, double z) {
    const double R2 = x * x + y * y;
    const double r2 = R2 + z * z;
    // |q|, 1/|q|^3, sqrt(z^2 + b^2), its inverse and D^(-3/2) from three
    // reciprocal square roots instead of three correctly rounded roots and
    // their divides
    const double s2 = z * z + m.b3sq;
    double ir, isz;
    lanes.rsqrt_pair(r2, s2, ir, isz);
    const double r = r2 * ir;
    const double ir3 = ir * ir * ir;
    const double sqrtz = s2 * isz;
    const double zd = m.a3 + sqrtz;
    const double D = R2 + zd * zd;
    const double iD = rsqrt_nr(D);
    const double f3 = m.m3 * (iD * iD * iD);
    const double f3z = 1.0 + m.a3 * isz;
    // NFW in the equivalent form G m / r^3 (log(1+u) - u/(1+u)), u = r / r_s
    // (v_h2 / u^3 / r_s^2 = G m / r^3)
    const double u = r * m.irs4;
    const double opu = 1.0 + u;
    double lf;
    int le;
    log_reduce(opu, lf, le);
    const double tf = 2.0 + lf;
    // The remaining denominators -- the two Hernquist ones, 1 + u and the
    // log's 2 + f -- share one reciprocal (batched inversion: invert the
    // product, peel the factors off with multiplies).
    const double rc1 = r + m.c1;
    const double rc2 = r + m.c2;
    const double d1 = rc1 * rc1 * r, d2 = rc2 * rc2 * r;
    const double p12 = d1 * d2;
    const double p3 = p12 * opu;
    const double p = p3 * tf;
    const double inv = rcp_nr(p);
    const double slog = lf * (inv * p3);
    const double inv3 = inv * tf;
    const double inv2 = inv3 * opu;
    const double i4 = inv3 * p12;
    const double f1 = m.m1 * (inv2 * d2);
    const double f2 = m.m2 * (inv2 * d1);
    const double lg = log_series(slog, le, lanes);
    const double f4 = m.m4 * (lg - u * i4) * ir3;
    // p's high word outside [1e-280's, 1e280's): one compare of integers
    constexpr unsigned lo = 0x05CD0B15u, hi = 0x7A11A0FCu;
    return {f1, f2, f3, f3z, f4, (unsigned)__double2hiint(p) - lo >= hi - lo};
}

__device__ __forceinline__ void mw_grad(const DevPot &P, double x, double y, double z,
                                        double &gx, double &gy, double &gz) {
    const MwFactors m = mw_factors(MwConstants(P), MwAlone{}, x, y, z);
    gx = 0.0;
    gy = 0.0;
    gz = 0.0;
    gx += m.f1 * x;
    gy += m.f1 * y;
    gz += m.f1 * z;
    gx += m.f2 * x;
    gy += m.f2 * y;
    gz += m.f2 * z;
    gx += m.f3 * x;
    gy += m.f3 * y;
    gz += m.f3 * z * m.f3z;
    gx += m.f4 * x;
    gy += m.f4 * y;
    gz += m.f4 * z;
    if (__builtin_expect(__any(m.extreme), 0))
        if (m.extreme) mw_grad_extreme(P, x, y, z, gx, gy, gz);
}

// mw_grad along one axis (0, 1, 2), q being the position along it: for lanes
// that hold one component each
template <class Lanes>
__device__ __forceinline__ double mw_grad_along(const DevPot &P, const MwConstants &mc,
                                                const Lanes &lanes, double x, double y, double z,
                                                int axis, double q) {
    const MwFactors m = mw_factors(mc, lanes, x, y, z);
    double g = 0.0;
    g += m.f1 * q;
    g += m.f2 * q;
    double gr = g, gz = g;
    gr += m.f3 * q;
    gz += m.f3 * q * m.f3z;
    g = axis == 2 ? gz : gr;
    g += m.f4 * q;
    if (__builtin_expect(__any(m.extreme), 0)) {
        double ex, ey, ez;
        mw_grad_extreme(P, x, y, z, ex, ey, ez);
        if (m.extreme) g = axis == 2 ? ez : (axis == 1 ? ey : ex);
    }
    return g;
}

// grad Phi with the layout chosen at compile time (LAYOUT_GENERIC reads the
// table's runtime layout and falls back to the general loop)
template <bool WITH_SCF, int LAYOUT>
__device__ __forceinline__ void pot_grad_l(const DevPot &P, double x, double y, double z,
                                           double &gx, double &gy, double &gz) {
    if (LAYOUT == LAYOUT_MW) {
        mw_grad(P, x, y, z, gx, gy, gz);
    } else if (LAYOUT == LAYOUT_SCF106) {
        const DevComp &c = P.c[0];
        double phi;
        scf_field<10, 6, false, true>(c.coef, c.p[0], c.p[1], c.p[2], 10, 6, x, y, z, phi, gx, gy,
                                      gz);
    } else if (LAYOUT == LAYOUT_SCF) {
        const DevComp &c = P.c[0];
        double phi;
        scf_field<-1, GAMD_SCF_MAX_LMAX, false, true>(c.coef, c.p[0], c.p[1], c.p[2], c.nmax,
                                                      c.lmax, x, y, z, phi, gx, gy, gz);
    } else {
        pot_grad<WITH_SCF>(P, x, y, z, gx, gy, gz);
    }
}

// waves per SIMD that the registers of an inlined expansion leave room for
// (168 VGPRs written out whole, which is three; 228 with any size)
constexpr int scf_waves(int layout) {
    return layout == LAYOUT_SCF106 || layout == LAYOUT_SCF ? 2 : 1;
}

template <bool WITH_SCF>
__device__ __forceinline__ double comp_value(const DevComp &c, double x, double y, double z) {
    if (WITH_SCF && c.type == GAMD_SCF)
        return scf_value(c.coef, c.p[0], c.p[1], c.p[2], c.nmax, c.lmax, x, y, z);
    return comp_value_analytic(c, x, y, z);
}

template <bool WITH_SCF>
__device__ __forceinline__ double pot_value(const DevPot &P, double x, double y, double z) {
    double v = 0.0;
    for (int i = 0; i < P.n; i++) {
        const DevComp &c = P.c[i];
        if (!c.shift_rotate) {
            v = v + comp_value<WITH_SCF>(c, x, y, z);
        } else {
            double xt, yt, zt;
            shift_rotate(c, x, y, z, xt, yt, zt);
            v = v + comp_value<WITH_SCF>(c, xt, yt, zt);
        }
    }
    return v;
}

// c_d2_dr2, cpotential.cpp:346-371
template <bool WITH_SCF>
__device__ __forceinline__ double pot_d2_dr2(const DevPot &P, double x, double y, double z) {
    const double h = 1e-2;
    const double r = sqrt(x * x + y * y + z * z);
    double d2 = pot_value<WITH_SCF>(P, x + h * x / r, y + h * y / r, z + h * z / r);
    d2 = d2 - 2.0 * pot_value<WITH_SCF>(P, x, y, z);
    d2 = d2 + pot_value<WITH_SCF>(P, x - h * x / r, y - h * y / r, z - h * z / r);
    return d2 / (h * h);
}

}  // namespace gamd
