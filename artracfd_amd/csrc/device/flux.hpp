// flux.hpp - per-face numerical fluxes evaluated on the device.
//
// The convective flux is the characteristic-wise, flux-vector-split WENO
// reconstruction of the solver (convective_flux.c:48-124 with the state
// algebra of cfd_commons.c:79-246 and weno5.c:35-62 / weno3.c:35-55); the
// viscous flux is its second-order central face flux (diffusive_flux.c:58-312).
// Every expression keeps the reference's operand order and the translation
// units are compiled with -ffp-contract=off, so a face flux is bit-identical
// to the CPU evaluation (up to the sign of an exact zero).
#pragma once

#include <hip/hip_runtime.h>

namespace artra {

constexpr int kComp = 5;

struct FluxModel {
    double gamma;
    double cv;
    double refMu;   // nondimensional viscosity scale (> 0 enables viscous flux)
    double refT;
    int roe;        // 1: Roe average, 0: arithmetic mean
    int sw;         // 1: Steger-Warming split, 0: local Lax-Friedrichs
};

__host__ __device__ __forceinline__ double sq(double x) { return x * x; }

// Jiang-Shu fifth-order WENO of one characteristic component from the
// five upwind-ordered values f0..f4 (value sought at the face after f2).
__host__ __device__ __forceinline__ double weno5(double f0, double f1, double f2, double f3, double f4)
{
    const double eps = 1.0e-6;
    const double IS0 = (13.0 / 12.0) * sq(f0 - 2.0 * f1 + f2) + (1.0 / 4.0) * sq(f0 - 4.0 * f1 + 3.0 * f2);
    const double IS1 = (13.0 / 12.0) * sq(f1 - 2.0 * f2 + f3) + (1.0 / 4.0) * sq(f1 - f3);
    const double IS2 = (13.0 / 12.0) * sq(f2 - 2.0 * f3 + f4) + (1.0 / 4.0) * sq(3.0 * f2 - 4.0 * f3 + f4);
    const double a0 = (1.0 / 10.0) / sq(eps + IS0);
    const double a1 = (6.0 / 10.0) / sq(eps + IS1);
    const double a2 = (3.0 / 10.0) / sq(eps + IS2);
    const double w0 = a0 / (a0 + a1 + a2);
    const double w1 = a1 / (a0 + a1 + a2);
    const double w2 = a2 / (a0 + a1 + a2);
    const double q0 = (1.0 / 6.0) * (2.0 * f0 - 7.0 * f1 + 11.0 * f2);
    const double q1 = (1.0 / 6.0) * (-f1 + 5.0 * f2 + 2.0 * f3);
    const double q2 = (1.0 / 6.0) * (2.0 * f2 + 5.0 * f3 - f4);
    return w0 * q0 + w1 * q1 + w2 * q2;
}

// Third-order WENO from f0..f2 (value sought at the face after f1).
__host__ __device__ __forceinline__ double weno3(double f0, double f1, double f2)
{
    const double eps = 1.0e-6;
    const double IS0 = sq(f1 - f0);
    const double IS1 = sq(f2 - f1);
    const double a0 = (1.0 / 3.0) / sq(eps + IS0);
    const double a1 = (2.0 / 3.0) / sq(eps + IS1);
    const double w0 = a0 / (a0 + a1);
    const double w1 = a1 / (a0 + a1);
    const double q0 = (1.0 / 2.0) * (-f0 + 3.0 * f1);
    const double q1 = (1.0 / 2.0) * (f1 + f2);
    return w0 * q0 + w1 * q1;
}

// Left eigenvector matrix of the Euler flux Jacobian along S at the face
// state (u, v, w, c); rows are characteristic fields (acoustic -, entropy /
// shear x3 in axis order, acoustic +).
template <int S>
__host__ __device__ __forceinline__ void left_vectors(double gamma, double u, double v, double w, double c, double L[5][5])
{
    const double q = 0.5 * (u * u + v * v + w * w);
    const double b = (gamma - 1.0) / (2.0 * c * c);
    const double d = 1.0 / (2.0 * c);
    if (S == 0) {
        L[0][0] = b * q + d * u;         L[0][1] = -b * u - d;            L[0][2] = -b * v;
        L[0][3] = -b * w;                L[0][4] = b;
        L[1][0] = -2.0 * b * q + 1.0;    L[1][1] = 2.0 * b * u;           L[1][2] = 2.0 * b * v;
        L[1][3] = 2.0 * b * w;           L[1][4] = -2.0 * b;
        L[2][0] = -2.0 * b * q * v;      L[2][1] = 2.0 * b * v * u;       L[2][2] = 2.0 * b * v * v + 1.0;
        L[2][3] = 2.0 * b * w * v;       L[2][4] = -2.0 * b * v;
        L[3][0] = -2.0 * b * q * w;      L[3][1] = 2.0 * b * w * u;       L[3][2] = 2.0 * b * w * v;
        L[3][3] = 2.0 * b * w * w + 1.0; L[3][4] = -2.0 * b * w;
        L[4][0] = b * q - d * u;         L[4][1] = -b * u + d;            L[4][2] = -b * v;
        L[4][3] = -b * w;                L[4][4] = b;
    } else if (S == 1) {
        L[0][0] = b * q + d * v;         L[0][1] = -b * u;                L[0][2] = -b * v - d;
        L[0][3] = -b * w;                L[0][4] = b;
        L[1][0] = -2.0 * b * q * u;      L[1][1] = 2.0 * b * u * u + 1.0; L[1][2] = 2.0 * b * v * u;
        L[1][3] = 2.0 * b * w * u;       L[1][4] = -2.0 * b * u;
        L[2][0] = -2.0 * b * q + 1.0;    L[2][1] = 2.0 * b * u;           L[2][2] = 2.0 * b * v;
        L[2][3] = 2.0 * b * w;           L[2][4] = -2.0 * b;
        L[3][0] = -2.0 * b * q * w;      L[3][1] = 2.0 * b * w * u;       L[3][2] = 2.0 * b * w * v;
        L[3][3] = 2.0 * b * w * w + 1.0; L[3][4] = -2.0 * b * w;
        L[4][0] = b * q - d * v;         L[4][1] = -b * u;                L[4][2] = -b * v + d;
        L[4][3] = -b * w;                L[4][4] = b;
    } else {
        L[0][0] = b * q + d * w;         L[0][1] = -b * u;                L[0][2] = -b * v;
        L[0][3] = -b * w - d;            L[0][4] = b;
        L[1][0] = -2.0 * b * q * u;      L[1][1] = 2.0 * b * u * u + 1.0; L[1][2] = 2.0 * b * v * u;
        L[1][3] = 2.0 * b * w * u;       L[1][4] = -2.0 * b * u;
        L[2][0] = -2.0 * b * q * v;      L[2][1] = 2.0 * b * v * u;       L[2][2] = 2.0 * b * v * v + 1.0;
        L[2][3] = 2.0 * b * w * v;       L[2][4] = -2.0 * b * v;
        L[3][0] = -2.0 * b * q + 1.0;    L[3][1] = 2.0 * b * u;           L[3][2] = 2.0 * b * v;
        L[3][3] = 2.0 * b * w;           L[3][4] = -2.0 * b;
        L[4][0] = b * q - d * w;         L[4][1] = -b * u;                L[4][2] = -b * v;
        L[4][3] = -b * w + d;            L[4][4] = b;
    }
}

// F = R (hp + hn) with R the right eigenvectors along S.  The reference
// accumulates all 25 products from 0.0; the structural zeros and ones of R
// contribute exact no-ops, so only the nonzero products are formed, in the
// same column order, starting from 0.0.
template <int S>
__host__ __device__ __forceinline__ void inverse_project(double u, double v, double w, double hT, double c, const double h[5],
                                                double F[5])
{
    const double q = 0.5 * (u * u + v * v + w * w);
    const double vel[3] = {u, v, w};
    const double un = vel[S];
    // row 0: columns 0, 1+S, 4 are 1
    F[0] = ((0.0 + h[0]) + h[1 + S]) + h[4];
    // rows 1..3 (momentum m)
#pragma unroll
    for (int m = 0; m < 3; ++m) {
        const double r0 = (m == S) ? vel[m] - c : vel[m];
        const double r4 = (m == S) ? vel[m] + c : vel[m];
        double acc = 0.0 + r0 * h[0];
        // column 1+t: entropy column (t == S) carries vel[m] only when m == S; shear column t carries 1 at m == t
#pragma unroll
        for (int t = 0; t < 3; ++t) {
            if (t == S) {
                if (m == S) acc = acc + vel[m] * h[1 + t];
            } else if (t == m) {
                acc = acc + h[1 + t];
            }
        }
        F[1 + m] = acc + r4 * h[4];
    }
    // row 4
    {
        double acc = 0.0 + (hT - un * c) * h[0];
#pragma unroll
        for (int t = 0; t < 3; ++t) {
            const double r = (t == S) ? vel[S] * vel[S] - q : vel[t];
            acc = acc + r * h[1 + t];
        }
        F[4] = acc + (hT + un * c) * h[4];
    }
}

// Convective numerical flux at the face between stencil nodes K0 and K0+1,
// from the conservative states st[0..NS-1] (nodes i-2..i+3 for WENO5,
// i-1..i+2 for WENO3; NS = 6 or 4).
template <int S, int NS>
__host__ __device__ __forceinline__ void convective_flux(const FluxModel &mdl, const double st[NS][5], double F[5])
{
    constexpr int K0 = (NS == 6) ? 2 : 1;
    const double gamma = mdl.gamma;
    // face average (cfd_commons.c:79-112)
    const double *UL = st[K0];
    const double *UR = st[K0 + 1];
    const double rhoL = UL[0];
    const double uL = UL[1] / UL[0], vL = UL[2] / UL[0], wL = UL[3] / UL[0];
    const double hTL = (UL[4] / UL[0]) * gamma - 0.5 * (uL * uL + vL * vL + wL * wL) * (gamma - 1.0);
    const double rhoR = UR[0];
    const double uR = UR[1] / UR[0], vR = UR[2] / UR[0], wR = UR[3] / UR[0];
    const double hTR = (UR[4] / UR[0]) * gamma - 0.5 * (uR * uR + vR * vR + wR * wR) * (gamma - 1.0);
    double u, v, w, hT;
    if (mdl.roe) {
        const double D = sqrt(rhoR / rhoL);
        u = (uL + D * uR) / (1.0 + D);
        v = (vL + D * vR) / (1.0 + D);
        w = (wL + D * wR) / (1.0 + D);
        hT = (hTL + D * hTR) / (1.0 + D);
    } else {
        u = 0.5 * (uL + uR);
        v = 0.5 * (vL + vR);
        w = 0.5 * (wL + wR);
        hT = 0.5 * (hTL + hTR);
    }
    const double c = sqrt((gamma - 1.0) * (hT - 0.5 * (u * u + v * v + w * w)));
    const double vel[3] = {u, v, w};
    const double un = vel[S];
    // split eigenvalues (cfd_commons.c:113-148)
    const double lam[5] = {un - c, un, un, un, un + c};
    double lp[5], ln[5];
    if (mdl.sw) {
        const double eps = 1.0e-3;
#pragma unroll
        for (int r = 0; r < 5; ++r) {
            lp[r] = 0.5 * (lam[r] + sqrt(lam[r] * lam[r] + eps * eps));
            ln[r] = 0.5 * (lam[r] - sqrt(lam[r] * lam[r] + eps * eps));
        }
    } else {
        const double star = fabs(lam[2]) + lam[4] - lam[2];
#pragma unroll
        for (int r = 0; r < 5; ++r) {
            lp[r] = 0.5 * (lam[r] + star);
            ln[r] = 0.5 * (lam[r] - star);
        }
    }
    double L[5][5];
    left_vectors<S>(gamma, u, v, w, c, L);
    // characteristic variables of the stencil, then WENO per field
    double hsum[5];
#pragma unroll
    for (int r = 0; r < 5; ++r) {
        double W[NS];
#pragma unroll
        for (int m = 0; m < NS; ++m) {
            double acc = 0.0;
#pragma unroll
            for (int cc = 0; cc < 5; ++cc) acc = acc + L[r][cc] * st[m][cc];
            W[m] = acc;
        }
        double hp, hn;
        if (NS == 6) {
            hp = weno5(lp[r] * W[0], lp[r] * W[1], lp[r] * W[2], lp[r] * W[3], lp[r] * W[4]);
            hn = weno5(ln[r] * W[5], ln[r] * W[4], ln[r] * W[3], ln[r] * W[2], ln[r] * W[1]);
        } else {
            hp = weno3(lp[r] * W[0], lp[r] * W[1], lp[r] * W[2]);
            hn = weno3(ln[r] * W[3], ln[r] * W[2], ln[r] * W[1]);
        }
        hsum[r] = hp + hn;
    }
    inverse_project<S>(u, v, w, hT, c, hsum, F);
}

// Viscous numerical flux at the face between node P and its +S neighbour E.
// g[a] are the states at P -/+ the first tangential axis, g[b] along the
// second, and the same for E: nb[0]=P-a, nb[1]=P+a, nb[2]=P-b, nb[3]=P+b,
// nb[4]=E-a, nb[5]=E+a, nb[6]=E-b, nb[7]=E+b.  Tangential axes: X face
// (y, z), Y face (x, z), Z face (x, y).
template <int S>
__host__ __device__ __forceinline__ void viscous_flux(const FluxModel &mdl, const double dd[3], const double P[5],
                                             const double E[5], const double nb[8][5], double F[5])
{
    constexpr int TA = (S == 0) ? 1 : 0;
    constexpr int TB = (S == 2) ? 1 : 2;
    const double cv = mdl.cv;
    const double velP[3] = {P[1] / P[0], P[2] / P[0], P[3] / P[0]};
    const double velE[3] = {E[1] / E[0], E[2] / E[0], E[3] / E[0]};
    const double TP = (P[4] - 0.5 * (P[1] * P[1] + P[2] * P[2] + P[3] * P[3]) / P[0]) / (P[0] * cv);
    const double TE = (E[4] - 0.5 * (E[1] * E[1] + E[2] * E[2] + E[3] * E[3]) / E[0]) / (E[0] * cv);
    // g[m][n] = d vel_m / d x_n
    double g[3][3];
#pragma unroll
    for (int m = 0; m < 3; ++m) {
        g[m][S] = (velE[m] - velP[m]) * dd[S];
        g[m][TA] = 0.25 * (nb[1][1 + m] / nb[1][0] + nb[5][1 + m] / nb[5][0] - nb[0][1 + m] / nb[0][0] -
                           nb[4][1 + m] / nb[4][0]) * dd[TA];
        g[m][TB] = 0.25 * (nb[3][1 + m] / nb[3][0] + nb[7][1 + m] / nb[7][0] - nb[2][1 + m] / nb[2][0] -
                           nb[6][1 + m] / nb[6][0]) * dd[TB];
    }
    const double dT = (TE - TP) * dd[S];
    const double uh = 0.5 * (velP[0] + velE[0]);
    const double vh = 0.5 * (velP[1] + velE[1]);
    const double wh = 0.5 * (velP[2] + velE[2]);
    const double Ts = 0.5 * (TP + TE) * mdl.refT;
    const double mu = mdl.refMu * (1.458e-6 * pow(Ts, 1.5) / (Ts + 110.4));
    const double heatK = mdl.gamma * mdl.cv * mu / 0.71;
    const double divV = g[0][0] + g[1][1] + g[2][2];
    F[0] = 0.0;
    if (S == 0) {
        F[1] = mu * (g[0][0] + g[0][0] - (2.0 / 3.0) * divV);
        F[2] = mu * (g[0][1] + g[1][0]);
        F[3] = mu * (g[0][2] + g[2][0]);
    } else if (S == 1) {
        F[1] = mu * (g[1][0] + g[0][1]);
        F[2] = mu * (g[1][1] + g[1][1] - (2.0 / 3.0) * divV);
        F[3] = mu * (g[1][2] + g[2][1]);
    } else {
        F[1] = mu * (g[2][0] + g[0][2]);
        F[2] = mu * (g[2][1] + g[1][2]);
        F[3] = mu * (g[2][2] + g[2][2] - (2.0 / 3.0) * divV);
    }
    F[4] = heatK * dT + F[1] * uh + F[2] * vh + F[3] * wh;
}

}  // namespace artra

// ---------------------------------------------------------------------------
// Fast variant.  Same numerical flux, evaluated with fewer FP64 instructions;
// results agree with the reference order to rounding level (checked against
// the 1e-10 relative-L2 contract on every golden case):
//  * one reciprocal per density instead of one division per velocity, shared
//    by the two nodes of a face;
//  * the characteristic projection uses the structure of the left
//    eigenvectors: with K = q U0 - vel.mom + U4 and M = un U0 - U_{1+S},
//    W = (bK + dM, U0 - 2bK [entropy] / U_{1+t} - 2b vel_t K [shear], bK - dM);
//  * WENO weights without their own divisions (weno5_field);
//  * reciprocals and square roots by Newton steps on the hardware estimates
//    (within an ulp), without the scaling and fix-up of the IEEE sequences:
//    densities, sound speeds and weight sums are far from the ends of the
//    exponent range;
//  * fused multiply-adds throughout.
// The sweeps are bound by FP64 issue, so instructions are what counts: the
// WENO5 sweep kernel holds 622 FP64 instructions with the arrangement below
// and 787 with expanded smoothness indicators, IEEE divisions and roots
// (six steps at 255^3 and the field's read-back: 57.5 against 62.6 ms).
namespace artra {
namespace fast {

// 1 / x: the hardware estimate (about 2^-26) refined twice.  Zero,
// infinity and subnormal x are outside its domain.
__host__ __device__ __forceinline__ double reciprocal(double x)
{
#ifdef __HIP_DEVICE_COMPILE__
    double y = __builtin_amdgcn_rcp(x);
    y = fma(fma(-x, y, 1.0), y, y);
    return fma(fma(-x, y, 1.0), y, y);
#else
    return 1.0 / x;
#endif
}

// sqrt(x) and 1 / sqrt(x) of a positive normal x: the hardware reciprocal
// root refined by two coupled Goldschmidt steps, the root then corrected by
// its residual.
__host__ __device__ __forceinline__ void root_pair(double x, double &root, double &inverse)
{
#ifdef __HIP_DEVICE_COMPILE__
    const double y = __builtin_amdgcn_rsq(x);
    double g = x * y, h = 0.5 * y;
    double r = fma(-h, g, 0.5);
    g = fma(g, r, g);
    h = fma(h, r, h);
    r = fma(-h, g, 0.5);
    h = fma(h, r, h);
    g = fma(fma(-g, g, x), h, g);
    root = g;
    inverse = h + h;
#else
    root = sqrt(x);
    inverse = 1.0 / root;
#endif
}

__host__ __device__ __forceinline__ double root(double x)
{
    double g, h;
    root_pair(x, g, h);
    return g;
}

// a b + c for a constant c, with c read from scalar registers: left to
// itself the compiler copies c to vector registers first and accumulates
// into the copy, one instruction more.
__host__ __device__ __forceinline__ double fma_constant(double a, double b, double c)
{
#ifdef __HIP_DEVICE_COMPILE__
    double d;
    asm("v_fma_f64 %0, %1, %2, %3" : "=v"(d) : "v"(a), "v"(b), "s"(c));
    return d;
#else
    return fma(a, b, c);
#endif
}

// One characteristic field of the split WENO5 flux, h = WENO5(lp W0..lp W4)
// + WENO5(ln W5..ln W1), from the field's six stencil values W0..W5 and its
// split eigenvalues, as h = base + num / den: Jiang-Shu WENO5 (weno5 above)
// of the scaled values lp W and ln W, arranged for fewer operations and one
// division per field (the two sides over a common denominator).
//  * The smoothness indicators are quadratic forms of the differences
//    d_i = W_{i+1} - W_i, so they are formed once on W and scaled by lp^2 or
//    ln^2.  Completed squares leave three shared terms c d_i^2, c = 39/64:
//    13 a^2 + 3 b^2 = 16 ((d0 - 11/8 d1)^2 + c d1^2) for the outer
//    sub-stencils, 16 ((d1 - 5/8 d2)^2 + c d2^2) for the middle one: sums of
//    squares, no cancellation.
//  * 3/4 (eps + IS) replaces eps + IS: the common factor cancels in the
//    weights t_k = 10 C_k prod_{j != k} (eps + IS_j)^2.
//  * The candidate values are the central node plus differences,
//    q_k = W2 + R_k / 6 (W3 - R_k / 6 on the mirrored side), so each side is
//    its central value plus N / (6 D), N = sum t_k R_k, D = sum t_k.
// den >= (7.5e-7)^8: no underflow; the product of two dens (divide pairs
// below) overflows only for smoothness indicators beyond about 1e19.
__host__ __device__ __forceinline__ void weno5_field(const double W[6], double lp, double ln, double &num, double &den,
                                                     double &base)
{
    const double eps34 = 0.75e-6, c = 39.0 / 64.0;
    const double d0 = W[1] - W[0], d1 = W[2] - W[1], d2 = W[3] - W[2], d3 = W[4] - W[3], d4 = W[5] - W[4];
    const double s1 = (c * d1) * d1, s2 = (c * d2) * d2, s3 = (c * d3) * d3;
    // plus side (W0..W4), minus side (W5..W1)
    const double xp0 = fma(-1.375, d1, d0), xp1 = fma(-0.625, d2, d1), xp2 = fma(-1.375, d2, d3);
    const double xm0 = fma(-1.375, d3, d4), xm1 = fma(-0.625, d2, d3), xm2 = fma(-1.375, d2, d1);
    const double lp2 = lp * lp, ln2 = ln * ln;
    const double ep0 = fma_constant(lp2, fma(xp0, xp0, s1), eps34);
    const double ep1 = fma_constant(lp2, fma(xp1, xp1, s2), eps34);
    const double ep2 = fma_constant(lp2, fma(xp2, xp2, s2), eps34);
    const double em0 = fma_constant(ln2, fma(xm0, xm0, s3), eps34);
    const double em1 = fma_constant(ln2, fma(xm1, xm1, s2), eps34);
    const double em2 = fma_constant(ln2, fma(xm2, xm2, s2), eps34);
    const double gp0 = ep0 * ep0, gp1 = ep1 * ep1, gp2 = ep2 * ep2;
    const double gm0 = em0 * em0, gm1 = em1 * em1, gm2 = em2 * em2;
    // D = g1 g2 + 3 g0 (2 g2 + g1), N / 2 = g1 g2 (R0 / 2) + 3 g0 (g2 R1 + g1 R2 / 2)
    const double pp = gp1 * gp2, hp = 3.0 * gp0, pm = gm1 * gm2, hm = 3.0 * gm0;
    const double Dp = fma(hp, fma(2.0, gp2, gp1), pp), Dm = fma(hm, fma(2.0, gm2, gm1), pm);
    const double dd2 = d2 + d2;
    const double Np = fma(hp, fma(gp2, d1 + dd2, gp1 * fma(-0.5, d3, dd2)), pp * fma(2.5, d1, -d0));
    const double Nm = fma(hm, fma(gm2, d3 + dd2, gm1 * fma(-0.5, d1, dd2)), pm * fma(2.5, d3, -d4));
    const double third = 1.0 / 3.0;
    base = fma(ln, W[3], lp * W[2]);
    den = Dp * Dm;
    num = fma((third * lp) * Np, Dm, -(((third * ln) * Nm) * Dp));
}

// Two quotients from one division: a/b and c/d as a (d q) and c (b q), q = 1/(b d).
__host__ __device__ __forceinline__ void divide_pair(double a, double b, double c, double d, double &x, double &y)
{
    const double q = reciprocal(b * d);
    x = a * (d * q);
    y = c * (b * q);
}

// x + a/b and y + c/d from one division.
__host__ __device__ __forceinline__ void add_quotients(double x, double a, double b, double y, double c, double d,
                                                       double &u, double &v)
{
    const double q = reciprocal(b * d);
    u = fma(a, d * q, x);
    v = fma(c, b * q, y);
}

__host__ __device__ __forceinline__ double weno3(double f0, double f1, double f2)
{
    const double eps = 1.0e-6;
    const double e0 = eps + (f1 - f0) * (f1 - f0), e1 = eps + (f2 - f1) * (f2 - f1);
    const double t0 = (1.0 / 3.0) * (e1 * e1), t1 = (2.0 / 3.0) * (e0 * e0);
    const double Q0 = fma(3.0, f1, -f0), Q1 = f1 + f2;
    return fma(t0, Q0, t1 * Q1) * reciprocal(2.0 * (t0 + t1));
}

}  // namespace fast

// Average state and split eigenvalues of a face (fast arithmetic).
struct FaceState {
    double u, v, w, hT, c, q, b, d, un, g1;
    double lp[5], ln[5];
};

// Velocities and total enthalpy of one node from its conserved state and
// the reciprocal of its density.
__host__ __device__ __forceinline__ void velocity_enthalpy(double gamma, const double U[5], double r, double nv[4])
{
    nv[0] = U[1] * r;
    nv[1] = U[2] * r;
    nv[2] = U[3] * r;
    nv[3] = fma(-0.5 * (gamma - 1.0), fma(nv[2], nv[2], fma(nv[1], nv[1], nv[0] * nv[0])), gamma * (U[4] * r));
}

template <int S>
__host__ __device__ __forceinline__ void face_state(const FluxModel &mdl, const double UL[5], const double UR[5],
                                                    FaceState &fs)
{
    double rL, rR, nL[4], nR[4];
    fast::divide_pair(1.0, UL[0], 1.0, UR[0], rL, rR);
    velocity_enthalpy(mdl.gamma, UL, rL, nL);
    velocity_enthalpy(mdl.gamma, UR, rR, nR);
    if (mdl.roe) {
        const double D = fast::root(UR[0] * rL);
        const double inv = fast::reciprocal(1.0 + D);
        fs.u = fma(D, nR[0], nL[0]) * inv;
        fs.v = fma(D, nR[1], nL[1]) * inv;
        fs.w = fma(D, nR[2], nL[2]) * inv;
        fs.hT = fma(D, nR[3], nL[3]) * inv;
    } else {
        fs.u = 0.5 * (nL[0] + nR[0]);
        fs.v = 0.5 * (nL[1] + nR[1]);
        fs.w = 0.5 * (nL[2] + nR[2]);
        fs.hT = 0.5 * (nL[3] + nR[3]);
    }
    fs.q = 0.5 * fma(fs.u, fs.u, fma(fs.v, fs.v, fs.w * fs.w));
    fs.g1 = mdl.gamma - 1.0;
    // b = (gamma - 1) / (2 c^2) and d = 1 / (2 c) of the eigenvectors
    double rc;
    fast::root_pair(fs.g1 * (fs.hT - fs.q), fs.c, rc);
    fs.d = 0.5 * rc;
    fs.b = (0.5 * fs.g1) * (rc * rc);
    fs.un = (S == 0) ? fs.u : (S == 1) ? fs.v : fs.w;
    const double lam[5] = {fs.un - fs.c, fs.un, fs.un, fs.un, fs.un + fs.c};
    if (mdl.sw) {
#pragma unroll
        for (int r = 0; r < 5; ++r) {
            const double size = fast::root(fma(lam[r], lam[r], 1.0e-6));
            fs.lp[r] = 0.5 * (lam[r] + size);
            fs.ln[r] = 0.5 * (lam[r] - size);
        }
    } else {
        const double star = fabs(fs.un) + fs.c;
#pragma unroll
        for (int r = 0; r < 5; ++r) {
            fs.lp[r] = 0.5 * (lam[r] + star);
            fs.ln[r] = 0.5 * (lam[r] - star);
        }
    }
}

// F = R h (right eigenvectors along S).
template <int S>
__host__ __device__ __forceinline__ void project_back(const FaceState &fs, const double h[5], double F[5])
{
    const double vel[3] = {fs.u, fs.v, fs.w};
    const double ha = h[0] + h[4], chd = fs.c * (h[4] - h[0]);
    F[0] = ha + h[1 + S];
#pragma unroll
    for (int m = 0; m < 3; ++m) F[1 + m] = (m == S) ? fma(vel[m], F[0], chd) : fma(vel[m], ha, h[1 + m]);
    double e = fma(fs.un, chd, fs.hT * ha);
#pragma unroll
    for (int t = 0; t < 3; ++t) e = fma((t == S) ? fma(fs.un, fs.un, -fs.q) : vel[t], h[1 + t], e);
    F[4] = e;
}

// The fast WENO5 flux at the face between stencil nodes 2 and 3, at(m, c)
// giving component c of node m = 0..5.  The fields are formed one after the
// other from the per-node projections K and M (acoustic fields 0 and 4
// first, then the entropy and shear fields, whose node components are read
// again), so that only one field's stencil values are live.  The one
// definition every sweep uses: a face's flux does not depend on the kernel
// that computes it.
template <int S, class At>
__host__ __device__ __forceinline__ void weno5_flux(const FluxModel &mdl, const At &at, double F[5])
{
    FaceState fs;
    {
        double UL[5], UR[5];
#pragma unroll
        for (int c = 0; c < 5; ++c) {
            UL[c] = at(2, c);
            UR[c] = at(3, c);
        }
        face_state<S>(mdl, UL, UR, fs);
    }
    double K[6], M[6];                              // b K and M
#pragma unroll
    for (int m = 0; m < 6; ++m) {
        const double U0 = at(m, 0), U1 = at(m, 1), U2 = at(m, 2), U3 = at(m, 3), U4 = at(m, 4);
        K[m] = fs.b * fma(-fs.v, U2, fma(-fs.u, U1, fma(-fs.w, U3, fma(fs.q, U0, U4))));
        M[m] = fma(fs.un, U0, -((S == 0) ? U1 : (S == 1) ? U2 : U3));
    }
    double h[5];
    {
        double W[6], num[2], den[2], base[2];
#pragma unroll
        for (int m = 0; m < 6; ++m) W[m] = fma(fs.d, M[m], K[m]);
        fast::weno5_field(W, fs.lp[0], fs.ln[0], num[0], den[0], base[0]);
#pragma unroll
        for (int m = 0; m < 6; ++m) W[m] = fma(-fs.d, M[m], K[m]);
        fast::weno5_field(W, fs.lp[4], fs.ln[4], num[1], den[1], base[1]);
        fast::add_quotients(base[0], num[0], den[0], base[1], num[1], den[1], h[0], h[4]);
    }
    const double vel[3] = {fs.u, fs.v, fs.w};
    double num[3], den[3], base[3];
#pragma unroll
    for (int t = 0; t < 3; ++t) {
        const double k = (t == S) ? -2.0 : -2.0 * vel[t];
        double W[6];
#pragma unroll
        for (int m = 0; m < 6; ++m) W[m] = fma(k, K[m], at(m, (t == S) ? 0 : 1 + t));
        fast::weno5_field(W, fs.lp[1 + t], fs.ln[1 + t], num[t], den[t], base[t]);
    }
    fast::add_quotients(base[0], num[0], den[0], base[1], num[1], den[1], h[1], h[2]);
    h[3] = fma(num[2], fast::reciprocal(den[2]), base[2]);
    project_back<S>(fs, h, F);
}

namespace fast {

template <int S, int NS>
__host__ __device__ __forceinline__ void convective_flux(const FluxModel &mdl, const double st[NS][5], double F[5])
{
    if (NS == 6) {
        weno5_flux<S>(mdl, [&](int m, int c) { return st[m][c]; }, F);
        return;
    }
    constexpr int K0 = (NS == 6) ? 2 : 1;
    FaceState fs;
    face_state<S>(mdl, st[K0], st[K0 + 1], fs);
    const double vel[3] = {fs.u, fs.v, fs.w};
    double W[5][NS];
#pragma unroll
    for (int m = 0; m < NS; ++m) {
        const double *U = st[m];
        const double K = fs.b * fma(-fs.u, U[1], fma(-fs.v, U[2], fma(-fs.w, U[3], fma(fs.q, U[0], U[4]))));
        const double M = fma(fs.un, U[0], -U[1 + S]);
        W[0][m] = fma(fs.d, M, K);
        W[4][m] = fma(-fs.d, M, K);
#pragma unroll
        for (int t = 0; t < 3; ++t)
            W[1 + t][m] = (t == S) ? fma(-2.0, K, U[0]) : fma(-2.0 * vel[t], K, U[1 + t]);
    }
    double h[5];
#pragma unroll
    for (int r = 0; r < 5; ++r) {
        const double hp = weno3(fs.lp[r] * W[r][0], fs.lp[r] * W[r][1], fs.lp[r] * W[r][2]);
        const double hn = weno3(fs.ln[r] * W[r][3], fs.ln[r] * W[r][2], fs.ln[r] * W[r][1]);
        h[r] = hp + hn;
    }
    project_back<S>(fs, h, F);
}

// Differences across a node along the transverse axis T: velocity
// components S and T of its +T neighbour R less those of its -T neighbour L
// (a face along S needs no other transverse gradient).
template <int S, int T>
__host__ __device__ __forceinline__ void transverse_difference(const double L[5], const double R[5], double out[2])
{
    double rL, rR;
    divide_pair(1.0, L[0], 1.0, R[0], rL, rR);
    out[0] = fma(R[1 + S], rR, -(L[1 + S] * rL));
    out[1] = fma(R[1 + T], rR, -(L[1 + T] * rL));
}

// Viscous flux at the face between P and its +S neighbour E from their
// states and transverse differences (tP, tE: [0..1] along the first
// tangential axis, [2..3] along the second).
template <int S>
__host__ __device__ __forceinline__ void viscous_flux(const FluxModel &mdl, const double dd[3], const double P[5],
                                                      const double E[5], const double tP[4], const double tE[4],
                                                      double F[5])
{
    constexpr int TA = (S == 0) ? 1 : 0;
    constexpr int TB = (S == 2) ? 1 : 2;
    double rP, rE;
    divide_pair(1.0, P[0], 1.0, E[0], rP, rE);
    const double velP[3] = {P[1] * rP, P[2] * rP, P[3] * rP};
    const double velE[3] = {E[1] * rE, E[2] * rE, E[3] * rE};
    const double rcv = 1.0 / mdl.cv;
    const double TP = (P[4] * rP - 0.5 * fma(velP[0], velP[0], fma(velP[1], velP[1], velP[2] * velP[2]))) * rcv;
    const double TE = (E[4] * rE - 0.5 * fma(velE[0], velE[0], fma(velE[1], velE[1], velE[2] * velE[2]))) * rcv;
    const double qa = 0.25 * dd[TA], qb = 0.25 * dd[TB];
    const double gSA = qa * (tP[0] + tE[0]), gAA = qa * (tP[1] + tE[1]);       // d u_S / d a, d u_a / d a
    const double gSB = qb * (tP[2] + tE[2]), gBB = qb * (tP[3] + tE[3]);
    const double gSS = (velE[S] - velP[S]) * dd[S];
    const double gAS = (velE[TA] - velP[TA]) * dd[S], gBS = (velE[TB] - velP[TB]) * dd[S];
    const double Ts = 0.5 * (TP + TE) * mdl.refT;
    // (root(0) is not a number: a face between nodes without pressure has no viscosity)
    const double rTs = (Ts == 0.0) ? 0.0 : root(Ts);
    const double mu = (mdl.refMu * 1.458e-6) * (Ts * rTs) * reciprocal(Ts + 110.4);
    const double heatK = mdl.gamma * mdl.cv * (1.0 / 0.71) * mu;
    const double divV = gSS + gAA + gBB;
    F[0] = 0.0;
    F[1 + S] = mu * fma(2.0, gSS, (-2.0 / 3.0) * divV);
    F[1 + TA] = mu * (gAS + gSA);
    F[1 + TB] = mu * (gBS + gSB);
    const double uh = 0.5 * (velP[0] + velE[0]);
    const double vh = 0.5 * (velP[1] + velE[1]);
    const double wh = 0.5 * (velP[2] + velE[2]);
    F[4] = fma(heatK, (TE - TP) * dd[S], fma(F[1], uh, fma(F[2], vh, F[3] * wh)));
}

// The same from the eight neighbours nb of the exact form above.
template <int S>
__host__ __device__ __forceinline__ void viscous_flux(const FluxModel &mdl, const double dd[3], const double P[5],
                                                      const double E[5], const double nb[8][5], double F[5])
{
    constexpr int TA = (S == 0) ? 1 : 0;
    constexpr int TB = (S == 2) ? 1 : 2;
    double tP[4], tE[4];
    transverse_difference<S, TA>(nb[0], nb[1], tP);
    transverse_difference<S, TB>(nb[2], nb[3], tP + 2);
    transverse_difference<S, TA>(nb[4], nb[5], tE);
    transverse_difference<S, TB>(nb[6], nb[7], tE + 2);
    viscous_flux<S>(mdl, dd, P, E, tP, tE, F);
}

}  // namespace fast
}  // namespace artra
