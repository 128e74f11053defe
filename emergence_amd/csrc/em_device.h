// Device-side physics of the Euler system (ideal / NASG gas) for the
// gfx950 kernels.  Each function restates the reference formula it cites
// (paths relative to the reference repository root) in the same evaluation
// order, so that a build without FMA contraction reproduces the reference
// CPU arithmetic bit for bit; the contracted build differs by rounding only.
//
// Every function is generic over the real type R (double, or float for the
// FP32 variant, as the reference's `Real` trait, compressible-cuda/src/
// lib.rs:26-48): constants are written R(c), so a float instantiation
// computes in float throughout and the double one is the original
// arithmetic.
//
// Characteristic matrices are used in their sparse form (8 non-zeros in L,
// 9 in R): skipping the exact-zero products of the reference's dense 5x5
// loops changes at most the sign of a zero.
#pragma once
#include <hip/hip_runtime.h>

#include <cmath>
#include <cstdint>

#include "em_div.h"

namespace em {

template <class R>
struct EosT {
    R gamma, p_inf, b, q;
    // 1 / (gamma - 1), correctly rounded, for div_by; NaN where the mid-range
    // forms cannot vouch for their ranges (gamma near or below one, negative
    // p_inf or q), which sends every operand the general way
    R rg = gamma - R(1) >= R(1e-3) && gamma <= R(1e3) && p_inf >= R(0) && q >= R(0) ? R(1) / (gamma - R(1)) : R(NAN);
};
using Eos = EosT<double>;

// EOS parameters in another real type (the reference's R::from_f64)
template <class R>
__host__ __device__ inline EosT<R> eos_as(const Eos& e) {
    return EosT<R>{R(e.gamma), R(e.p_inf), R(e.b), R(e.q)};
}

// fluid/crates/compressible/src/eos.rs:36-40
template <class R>
__device__ __forceinline__ R eos_pressure(const EosT<R>& e, R rho, R en) {
    R v = R(1.0) / rho;
    return (e.gamma - R(1.0)) * (en - e.q) / (v - e.b) - e.gamma * e.p_inf;
}
// eos.rs:43-53 (rho_e = rho * energy)
template <class R>
__device__ __forceinline__ R eos_rho_e(const EosT<R>& e, R rho, R p) {
    R v = R(1.0) / rho;
    return rho * ((p + e.gamma * e.p_inf) * (v - e.b) / (e.gamma - R(1.0)) + e.q);
}
// eos.rs:55-59 and system.rs:219-222 (sqrt(max(c^2, 0)))
template <class R>
__device__ __forceinline__ R sound_speed(const EosT<R>& e, R rho, R p) {
    R v = R(1.0) / rho;
    R c2 = e.gamma * (p + e.p_inf) * v * v / (v - e.b);
    return sqrt(fmax(c2, R(0.0)));
}
// system.rs:404-407 with eos.rs:76-79
template <class R>
__device__ __forceinline__ bool admissible(const EosT<R>& e, R rho, R p) {
    return isfinite(rho) && isfinite(p) && rho > R(0.0) && R(1.0) / rho > e.b && p + e.p_inf > R(0.0);
}

// system.rs:197-203
template <class R>
__device__ __forceinline__ void to_prim(const EosT<R>& e, const R u[5], R w[5]) {
    R rho = u[0];
    R vx = u[1] / rho, vy = u[2] / rho, vz = u[3] / rho;
    R en = u[4] / rho - R(0.5) * (vx * vx + vy * vy + vz * vz);
    w[0] = rho;
    w[1] = vx;
    w[2] = vy;
    w[3] = vz;
    w[4] = eos_pressure(e, rho, en);
}
// system.rs:210-217
template <class R>
__device__ __forceinline__ void to_cons(const EosT<R>& e, const R w[5], R u[5]) {
    R rho = w[0];
    R ke = R(0.5) * rho * (w[1] * w[1] + w[2] * w[2] + w[3] * w[3]);
    u[0] = rho;
    u[1] = rho * w[1];
    u[2] = rho * w[2];
    u[3] = rho * w[3];
    u[4] = eos_rho_e(e, rho, w[4]) + ke;
}
// to_cons with the cell's rho_e = eos_rho_e(e, w[0], w[4]) already at hand
// (the same expressions, system.rs:210-217): a cell's rho_e is computed once
// per tile and reused by every face that needs its conserved state.
template <class R>
__device__ __forceinline__ void to_cons_re(const R w[5], R re, R u[5]) {
    R rho = w[0];
    R ke = R(0.5) * rho * (w[1] * w[1] + w[2] * w[2] + w[3] * w[3]);
    u[0] = rho;
    u[1] = rho * w[1];
    u[2] = rho * w[2];
    u[3] = rho * w[3];
    u[4] = re + ke;
}
// Physical flux from (w, q = to_cons(w)): system.rs:336-348 and the closure
// of riemann_flux (system.rs:268-279) compute the same expressions.
template <int D, class R>
__device__ __forceinline__ void phys_flux(const R w[5], const R q[5], R f[5]) {
    constexpr int un = 1 + D;
    R u = w[un];
    f[0] = q[0] * u;
    f[1] = q[1] * u;
    f[2] = q[2] * u;
    f[3] = q[3] * u;
    f[un] += w[4];
    f[4] = (q[4] + w[4]) * u;
}

// to_prim, its divisions by rho through one reciprocal; v = 1 / rho.  (The
// float variant keeps the plain forms throughout: its results on flat
// sub-stencils hang on the contracted expressions' last bits.)
template <class R>
__device__ __forceinline__ void to_prim_v(const EosT<R>& e, const R u[5], R w[5], R& v) {
    const R rho = u[0];
    if constexpr (sizeof(R) == 4) {
        to_prim(e, u, w);
        v = R(1.0) / rho;
    } else {
        const R r = rcp_mid(rho);
        v = inv_by(rho, r);
        const R vx = div_by_pos(u[1], rho, r), vy = div_by_pos(u[2], rho, r), vz = div_by_pos(u[3], rho, r);
        const R en = div_by_pos(u[4], rho, r) - R(0.5) * (vx * vx + vy * vy + vz * vz);
        w[0] = rho;
        w[1] = vx;
        w[2] = vy;
        w[3] = vz;
        const R a = (e.gamma - R(1.0)) * (en - e.q), vb = v - e.b;
        w[4] = div_by_pos(a, vb, rcp_volume(e, rho, vb)) - e.gamma * e.p_inf;
        // an overflowing quotient leaves p infinite or NaN
        if (!in_mid(rho) || !in_mid(vb) || too_small(u[1]) || too_small(u[2]) || too_small(u[3]) || too_small(u[4]) ||
            too_small(a) || !(fabs(w[4]) <= Mid<R>::huge)) {
            to_prim(e, u, w);
            v = R(1.0) / rho;
        }
    }
}
// eos_rho_e with v = 1 / rho given and the division by the constant
// gamma - 1 through its reciprocal.
template <class R>
__device__ __forceinline__ R eos_rho_e_v(const EosT<R>& e, R rho, R p, R v) {
    if constexpr (sizeof(R) == 4) {
        return eos_rho_e(e, rho, p);
    } else {
        const R a = (p + e.gamma * e.p_inf) * (v - e.b);
        R x = div_by_pos(a, e.gamma - R(1.0), e.rg);
        if (too_small(a) || !(fabs(x) <= Mid<R>::huge)) x = a / (e.gamma - R(1.0));
        return rho * (x + e.q);
    }
}

// rcp_mid(vb) of vb = v - b, v = RN(1 / rho): without a covolume rho itself
// is the reciprocal to an ulp and one Newton step finishes it
__device__ __forceinline__ double rcp_volume(const Eos& e, double rho, double vb) {
    return e.b == 0.0 ? rcp_step(vb, rho) : rcp_mid(vb);
}

// True where the conserved state q is admissible with so much room that the
// rounded evaluation (to_prim, then admissible) cannot decide otherwise, and
// is finite; no division.  With d = (E - |m|^2 / 2 rho - rho q - p_inf (1 -
// rho b)) rho = rho^2 (v - b) (p + p_inf) / (gamma - 1), the test asks for
// d > margin times the sum of the terms' magnitudes; the rounding of either
// evaluation is below 1e-5 of that slack in double and a tenth of it in float.
template <class R>
__device__ __forceinline__ bool clearly_admissible(const EosT<R>& e, const R q[5]) {
    const R rho = q[0];
    const R a = rho * q[4], k = R(0.5) * (q[1] * q[1] + q[2] * q[2] + q[3] * q[3]);
    const R rb = rho * e.b;
    const R y = rho * (rho * e.q), z = rho * e.p_inf * (R(1.0) - rb);
    const R d = a - k - y - z;
    const R size = fabs(a) + k + fabs(y) + fabs(z);
    return in_mid(rho) && fabs(rb) <= R(0.5) && d > Mid<R>::margin * size && d > Mid<R>::lo * Mid<R>::lo &&
           size < Mid<R>::hi * Mid<R>::hi && e.gamma - R(1.0) > R(0.01);
}

// The flux and the selected star state of HLLC once the two sound speeds
// and conserved states are known (system.rs:268-312).  MID: densities, sound
// speeds and velocities are in the middle of the exponent range, il and ir
// their densities' reciprocals (rcp_mid).
template <int D, bool MID = false, class R>
__device__ __forceinline__ void hllc_flux(const R wl[5], const R wr[5], const R ql[5], const R qr[5], R cl, R cr,
                                          R il, R ir, R f[5]) {
    constexpr int un = 1 + D;
    R ul = wl[un], ur = wr[un];
    R sl = fmin(ul - cl, ur - cr);
    R sr = fmax(ul + cl, ur + cr);
    if (sl >= R(0.0)) {
        phys_flux<D>(wl, ql, f);
        return;
    }
    if (sr <= R(0.0)) {
        phys_flux<D>(wr, qr, f);
        return;
    }
    R rl = wl[0], rr = wr[0], pl = wl[4], pr = wr[4];
    R ss = (pr - pl + rl * ul * (sl - ul) - rr * ur * (sr - ur)) / (rl * (sl - ul) - rr * (sr - ur));
    // one side is selected by the contact speed; its star state and flux
    // (value selects keep both register arrays out of scratch memory)
    const bool left = ss >= R(0.0);
    R w[5], q[5];
#pragma unroll
    for (int k = 0; k < 5; ++k) {
        w[k] = left ? wl[k] : wr[k];
        q[k] = left ? ql[k] : qr[k];
    }
    R s = left ? sl : sr;
    R rho = w[0], u = w[un];
    const R h = rho * (s - u);
    R fac = h / (s - ss);
    R en;
    if constexpr (MID)
        en = div_by(q[4], rho, left ? il : ir);
    else
        en = q[4] / rho;
    R qs[5];
    qs[0] = fac;
    qs[1] = fac * w[1];
    qs[2] = fac * w[2];
    qs[3] = fac * w[3];
    qs[un] = fac * ss;
    qs[4] = fac * (en + (ss - u) * (ss + w[4] / h));
    R fw[5];
    phys_flux<D>(w, q, fw);
#pragma unroll
    for (int k = 0; k < 5; ++k) f[k] = fw[k] + s * (qs[k] - q[k]);
}

// HLLC with Davis wave-speed bounds: system.rs:260-312.  Returns the flux.
template <int D, class R>
__device__ __forceinline__ void hllc(const EosT<R>& e, const R wl[5], const R wr[5], R f[5]) {
    const R cl = sound_speed(e, wl[0], wl[4]), cr = sound_speed(e, wr[0], wr[4]);
    R ql[5], qr[5];
    to_cons(e, wl, ql);
    to_cons(e, wr, qr);
    hllc_flux<D>(wl, wr, ql, qr, cl, cr, cl, cr, f);
}

// KEEP-PE two-point flux: system.rs:317-334
template <int D, class R>
__device__ __forceinline__ void split_flux(const EosT<R>& e, const R a[5], const R b[5], R f[5]) {
    constexpr int un = 1 + D;
    R rho = R(0.5) * (a[0] + b[0]);
    R u = R(0.5) * (a[un] + b[un]);
    R c = rho * u;
    f[0] = c;
    f[1] = c * R(0.5) * (a[1] + b[1]);
    f[2] = c * R(0.5) * (a[2] + b[2]);
    f[3] = c * R(0.5) * (a[3] + b[3]);
    f[un] += R(0.5) * (a[4] + b[4]);
    R kin = c * R(0.5) * (a[1] * b[1] + a[2] * b[2] + a[3] * b[3]);
    R rhoe = R(0.5) * (eos_rho_e(e, a[0], a[4]) + eos_rho_e(e, b[0], b[4]));
    R pw = R(0.5) * (a[un] * b[4] + b[un] * a[4]);
    f[4] = kin + u * rhoe + pw;
}

// split_flux with the two cells' rho_e given (each computed once per tile)
template <int D, class R>
__device__ __forceinline__ void split_flux_re(const R a[5], const R b[5], R rea, R reb,
                                              R f[5]) {
    constexpr int un = 1 + D;
    R rho = R(0.5) * (a[0] + b[0]);
    R u = R(0.5) * (a[un] + b[un]);
    R c = rho * u;
    f[0] = c;
    f[1] = c * R(0.5) * (a[1] + b[1]);
    f[2] = c * R(0.5) * (a[2] + b[2]);
    f[3] = c * R(0.5) * (a[3] + b[3]);
    f[un] += R(0.5) * (a[4] + b[4]);
    R kin = c * R(0.5) * (a[1] * b[1] + a[2] * b[2] + a[3] * b[3]);
    R rhoe = R(0.5) * (rea + reb);
    R pw = R(0.5) * (a[un] * b[4] + b[un] * a[4]);
    f[4] = kin + u * rhoe + pw;
}

// WENO5-Z interpolation of point values to the midpoint x_{2+1/2}:
// scheme.rs:69-86 (EPS = 1e-40, scheme.rs:55).  Division by 8 is an exact
// power-of-two scaling, written as a multiplication.  In FP32 the epsilon is
// 1e-30, as in the reference's f32 kernels (compressible-cuda/src/
// kernels.cu:263): with 1e-40 (a float denormal), a stencil with one exactly
// flat sub-stencil squares tau / 1e-40 past FLT_MAX, and the midpoint falls
// back to first order.
template <class R>
__device__ __forceinline__ R weno5z_interp(R v0, R v1, R v2, R v3, R v4) {
    R q0 = (R(3.0) * v0 - R(10.0) * v1 + R(15.0) * v2) * R(0.125);
    R q1 = (-v1 + R(6.0) * v2 + R(3.0) * v3) * R(0.125);
    R q2 = (R(3.0) * v2 + R(6.0) * v3 - v4) * R(0.125);
    R t0 = v0 - R(2.0) * v1 + v2, s0 = v0 - R(4.0) * v1 + R(3.0) * v2;
    R t1 = v1 - R(2.0) * v2 + v3, s1 = v1 - v3;
    R t2 = v2 - R(2.0) * v3 + v4, s2 = R(3.0) * v2 - R(4.0) * v3 + v4;
    const R c13 = R(13.0) / R(12.0);
    R b0 = c13 * (t0 * t0) + R(0.25) * (s0 * s0);
    R b1 = c13 * (t1 * t1) + R(0.25) * (s1 * s1);
    R b2 = c13 * (t2 * t2) + R(0.25) * (s2 * s2);
    R tau = fabs(b0 - b2);
    const R eps = sizeof(R) == 4 ? R(1e-30) : R(1e-40);
    R r0 = tau / (b0 + eps), r1 = tau / (b1 + eps), r2 = tau / (b2 + eps);
    R a0 = R(0.0625) * (R(1.0) + r0 * r0);
    R a1 = R(0.625) * (R(1.0) + r1 * r1);
    R a2 = R(0.3125) * (R(1.0) + r2 * r2);
    return (a0 * q0 + a1 * q1 + a2 * q2) / (a0 + a1 + a2);
}

// WCNS midpoint flux: characteristic WENO5-Z interpolation of the six
// primitive states w_{j-2..j+3}, component k of cell j read through ld(j, k),
// to the midpoint j+1/2, first-order fallback on an inadmissible state, HLLC
// there.  scheme.rs:286-333, with the eigenvectors of system.rs:232-258
// applied in sparse form.  Returns true on the first-order fallback.
// FIELDS: the characteristic fields in a loop of one body (for FP64, where
// midpoint_flux_mid takes almost every midpoint and this is cold code that
// only fills the instruction cache), else unrolled.
template <int D, bool FIELDS, class R, class LD>
__device__ __forceinline__ bool midpoint_flux(const EosT<R>& e, LD&& ld, R f[5]) {
    constexpr int un = 1 + D;
    constexpr int t1 = 1 + (D + 1) % 3;
    constexpr int t2 = 1 + (D + 2) % 3;
    R rho = R(0.5) * (ld(2, 0) + ld(3, 0));
    R avp = R(0.5) * (ld(2, 4) + ld(3, 4));
    R c = sound_speed(e, rho, avp);
    // L rows (waves u-c, entropy, shear t1, shear t2, u+c)
    R l0un = -rho / (R(2.0) * c);
    R l04 = R(1.0) / (R(2.0) * c * c);
    R l14 = -R(1.0) / (c * c);
    R l4un = rho / (R(2.0) * c);
    R l44 = R(1.0) / (R(2.0) * c * c);
    // R columns: r[0][0]=r[0][1]=r[0][4]=1, r[un][0]=-c/rho, r[un][4]=c/rho,
    // r[t1][2]=r[t2][3]=1, r[4][0]=r[4][4]=c*c
    R run0 = -c / rho, run4 = c / rho, r40 = c * c;
    R wl[5], wr[5];
#pragma unroll
    for (int k = 0; k < 5; ++k) wl[k] = wr[k] = R(0.0);
    auto field = [&](int a) {
        R ch[6];
        if (a == 0) {
#pragma unroll
            for (int j = 0; j < 6; ++j) ch[j] = l0un * ld(j, un) + l04 * ld(j, 4);
        } else if (a == 1) {
#pragma unroll
            for (int j = 0; j < 6; ++j) ch[j] = ld(j, 0) + l14 * ld(j, 4);
        } else if (a == 4) {
#pragma unroll
            for (int j = 0; j < 6; ++j) ch[j] = l4un * ld(j, un) + l44 * ld(j, 4);
        } else if (a == 2) {
#pragma unroll
            for (int j = 0; j < 6; ++j) ch[j] = ld(j, t1);
        } else {
#pragma unroll
            for (int j = 0; j < 6; ++j) ch[j] = ld(j, t2);
        }
        const R cl = weno5z_interp(ch[0], ch[1], ch[2], ch[3], ch[4]);
        const R cr = weno5z_interp(ch[5], ch[4], ch[3], ch[2], ch[1]);
        if (a == 0) {
            wl[0] = cl;
            wr[0] = cr;
            wl[un] = run0 * cl;
            wr[un] = run0 * cr;
            wl[4] = r40 * cl;
            wr[4] = r40 * cr;
        } else if (a == 1) {
            wl[0] = wl[0] + cl;
            wr[0] = wr[0] + cr;
        } else if (a == 2) {
            wl[t1] = cl;
            wr[t1] = cr;
        } else if (a == 3) {
            wl[t2] = cl;
            wr[t2] = cr;
        } else {
            wl[0] = wl[0] + cl;
            wr[0] = wr[0] + cr;
            wl[un] = wl[un] + run4 * cl;
            wr[un] = wr[un] + run4 * cr;
            wl[4] = wl[4] + r40 * cl;
            wr[4] = wr[4] + r40 * cr;
        }
    };
    if constexpr (FIELDS) {
#pragma unroll 1
        for (int a = 0; a < 5; ++a) field(a);
    } else {
#pragma unroll
        for (int a = 0; a < 5; ++a) field(a);
    }
    bool fb = false;
    if (!admissible(e, wl[0], wl[4]) || !admissible(e, wr[0], wr[4])) {
        fb = true;
#pragma unroll
        for (int k = 0; k < 5; ++k) {
            wl[k] = ld(2, k);
            wr[k] = ld(3, k);
        }
    }
    hllc<D>(e, wl, wr, f);
    return fb;
}

// weno5z_interp where every |v| < 2^-200: beta + eps is eps and 1 + r^2 is 1,
// which leaves the linear weights, whose sum is 1.
__device__ __forceinline__ double weno5_linear(double v0, double v1, double v2, double v3, double v4) {
    const double q0 = (3.0 * v0 - 10.0 * v1 + 15.0 * v2) * 0.125;
    const double q1 = (-v1 + 6.0 * v2 + 3.0 * v3) * 0.125;
    const double q2 = (3.0 * v2 + 6.0 * v3 - v4) * 0.125;
    return 0.0625 * q0 + 0.625 * q1 + 0.3125 * q2;
}

// Both WENO5-Z interpolations of a midpoint's six point values, left (v0..v4)
// and right (v5, v4, .., v1): the values weno5z_interp gives, with fewer
// operations and no range scaling.
//   * 2x, 4x and x/4 are exact, so a sum with them is one fma with the same
//     rounding; 6x = 2 (3x) and 10x = 2 (5x) share their products.  The
//     contracted build (EM_CONTRACT) keeps weno5z_interp's expressions, whose
//     fused rounding residues keep beta above zero on flat stencils.
//   * The factor 1/8 of the candidates and 1/16 of the linear weights
//     (1, 10, 5)/16 are powers of two: the weighted sum is formed without
//     them and scaled once.
//   * tau / (beta + eps): the reciprocals of the three (rcp3_mid), and of the
//     two weight sums (rcp2_mid), are taken jointly.  A tau too small for the
//     core leaves 1 + r^2 = 1 either way.
// left and right are 8 times the interpolated values.  top is raised to the
// high word of the product of the three beta + eps, ok cleared where the last
// quotient needs the general division: the caller falls back to
// weno5z_interp unless ok, top below beta_max and both values finite.  The
// weight sums reach 2^1002 there (flat sub-stencils beside a jump of 2^183);
// where the product of the two overflows (from a jump of about 2^62 on) or a
// weighted sum does, the values come out infinite.  TINY: zero fields and
// fields below 2^-200 are taken here as well (ahead of a front in gas at rest
// the velocities fall off to denormals over many cells: a tenth of all cells
// in a shock-bubble run).  91 issue slots a side (a reciprocal counts
// four) against about 125.
template <bool TINY>
__device__ __forceinline__ void weno5z_pair(const double v[6], double& left, double& right, unsigned& top, bool& ok) {
#ifndef EM_CONTRACT
    const double m0 = 3.0 * v[0], m2 = 3.0 * v[2], m3 = 3.0 * v[3], m5 = 3.0 * v[5];
    const double f1 = 5.0 * v[1], f4 = 5.0 * v[4];
#endif
    const double c13 = 13.0 / 12.0;
    double N[2], S[2];
#pragma unroll
    for (int s = 0; s < 2; ++s) {
        const double a = s ? v[5] : v[0], b = s ? v[4] : v[1], c = s ? v[3] : v[2], d = s ? v[2] : v[3], g = s ? v[1] : v[4];
#ifndef EM_CONTRACT
        const double ma = s ? m5 : m0, mc = s ? m3 : m2, md = s ? m2 : m3, fb = s ? f4 : f1;
        const double q0 = __builtin_fma(-2.0, fb, ma) + 15.0 * c;
        const double q1 = __builtin_fma(2.0, mc, -b) + md;
        const double q2 = __builtin_fma(2.0, md, mc) - g;
        const double t0 = __builtin_fma(-2.0, b, a) + c, s0 = __builtin_fma(-4.0, b, a) + mc;
        const double t1 = __builtin_fma(-2.0, c, b) + d, s1 = b - d;
        const double t2 = __builtin_fma(-2.0, d, c) + g, s2 = __builtin_fma(-4.0, d, mc) + g;
        const double b0 = __builtin_fma(0.25, s0 * s0, c13 * (t0 * t0));
        const double b1 = __builtin_fma(0.25, s1 * s1, c13 * (t1 * t1));
        const double b2 = __builtin_fma(0.25, s2 * s2, c13 * (t2 * t2));
#else
        const double q0 = 3.0 * a - 10.0 * b + 15.0 * c;
        const double q1 = -b + 6.0 * c + 3.0 * d;
        const double q2 = 3.0 * c + 6.0 * d - g;
        const double t0 = a - 2.0 * b + c, s0 = a - 4.0 * b + 3.0 * c;
        const double t1 = b - 2.0 * c + d, s1 = b - d;
        const double t2 = c - 2.0 * d + g, s2 = 3.0 * c - 4.0 * d + g;
        const double b0 = c13 * (t0 * t0) + 0.25 * (s0 * s0);
        const double b1 = c13 * (t1 * t1) + 0.25 * (s1 * s1);
        const double b2 = c13 * (t2 * t2) + 0.25 * (s2 * s2);
#endif
        const double tau = fabs(b0 - b2);
        const double d0 = b0 + 1e-40, d1 = b1 + 1e-40, d2 = b2 + 1e-40;
        double i0, i1, i2;
        top = max(top, top_word(rcp3_mid(d0, d1, d2, i0, i1, i2)));
        const double r0 = div_by(tau, d0, i0), r1 = div_by(tau, d1, i1), r2 = div_by(tau, d2, i2);
        const double a0 = 1.0 + r0 * r0;
        const double a1 = 10.0 * (1.0 + r1 * r1);
        const double a2 = 5.0 * (1.0 + r2 * r2);
        N[s] = a0 * q0 + a1 * q1 + a2 * q2;
        S[s] = a0 + a1 + a2;
    }
    double il, ir;
    rcp2_mid(S[0], S[1], il, ir);
    left = div_by_fix(N[0], S[0], il);
    right = div_by_fix(N[1], S[1], ir);
    bool fine = fabs(left) >= Mid<double>::tiny && fabs(right) >= Mid<double>::tiny;
    if (TINY && !fine) {
        fine = (fabs(left) >= Mid<double>::tiny || N[0] == 0.0) && (fabs(right) >= Mid<double>::tiny || N[1] == 0.0);
        const double m = fmax(fmax(fmax(fabs(v[0]), fabs(v[1])), fmax(fabs(v[2]), fabs(v[3]))), fmax(fabs(v[4]), fabs(v[5])));
        if (!fine && m < 0x1p-200) {
            fine = true;
            left = 8.0 * weno5_linear(v[0], v[1], v[2], v[3], v[4]);
            right = 8.0 * weno5_linear(v[5], v[4], v[3], v[2], v[1]);
        }
    }
    ok = ok && fine;
}

// midpoint_flux for operands in the middle of the exponent range, stencil
// value k of cell j read through ld(j, k): the same flux, or false (and no
// flux) where some operand is outside, or a reconstruction inadmissible: the
// caller then evaluates midpoint_flux.  The pass is bound by its FP64
// instruction count (VALU 86% busy), much of it divisions: 61 per midpoint,
// here 3 in the general form (hllc_flux) and the rest through shared
// reciprocals.  With the load phase's and the limiter's divisions (to_prim_v,
// clearly_admissible) the 256^3 Weno x pass went from 2,544 to 2,033 VALU
// instructions per cell in the same tiles, the three passes from 4.29 to 3.56
// ms (1,857 and 3.11 ms in segments, em_pass.hip).
//   * l4un = -l0un and l44 = l04 = -l14 / 2 exactly (powers of two and signs),
//     so the fields 0, 1 and 4 need two products per cell.
//   * zero1, zero2: the axes of the transverse velocities t1, t2 are
//     inactive (uniform); where such a component is +0 on the whole wave its
//     reconstructions are +0 and are not evaluated.
template <int D, class LD>
__device__ __forceinline__ bool midpoint_flux_mid(const Eos& e, bool zero1, bool zero2, LD&& ld, double f[5]) {
    constexpr int un = 1 + D;
    constexpr int t1 = 1 + (D + 1) % 3;
    constexpr int t2 = 1 + (D + 2) % 3;
    const double rho = 0.5 * (ld(2, 0) + ld(3, 0));
    const double avp = 0.5 * (ld(2, 4) + ld(3, 4));
    const double irho = rcp_mid(rho);
    const double v = inv_by(rho, irho);
    const double vb = v - e.b;
    const double c2 = div_by(e.gamma * (avp + e.p_inf) * v * v, vb, rcp_volume(e, rho, vb));
    double ic;
    const double c = sqrt_mid(c2, ic);
    const double cc = c * c;
    const double lu = 0.5 * div_by(rho, c, ic);                  // rho / (2 c)
    const double lp = 0.5 * inv_by(cc, rcp_step(cc, ic * ic));   // 1 / (2 c^2)
    const double ru = 0.125 * div_by(c, rho, irho);              // c / rho, of the sums times 8
    const double cc8 = 0.125 * cc;
    bool ok = e.rg > 0.0;
    unsigned top = 0;
    double wl[5], wr[5];
    {
        double ch[6], l0, r0, l1, r1, l4, r4;
#pragma unroll
        for (int j = 0; j < 6; ++j) ch[j] = lp * ld(j, 4) - lu * ld(j, un);
        weno5z_pair<false>(ch, l0, r0, top, ok);
#pragma unroll
        for (int j = 0; j < 6; ++j) ch[j] = lp * ld(j, 4) + lu * ld(j, un);
        weno5z_pair<false>(ch, l4, r4, top, ok);
#pragma unroll
        for (int j = 0; j < 6; ++j)
#ifndef EM_CONTRACT
            ch[j] = __builtin_fma(-2.0, lp * ld(j, 4), ld(j, 0));
#else
            ch[j] = ld(j, 0) - 2.0 * lp * ld(j, 4);
#endif
        weno5z_pair<false>(ch, l1, r1, top, ok);
        wl[0] = 0.125 * (l0 + l1 + l4);
        wr[0] = 0.125 * (r0 + r1 + r4);
        wl[un] = ru * l4 - ru * l0;
        wr[un] = ru * r4 - ru * r0;
        wl[4] = cc8 * l0 + cc8 * l4;
        wr[4] = cc8 * r0 + cc8 * r4;
    }
#pragma unroll
    for (int s = 0; s < 2; ++s) {
        const int t = s ? t2 : t1;
        double ch[6];
#pragma unroll
        for (int j = 0; j < 6; ++j) ch[j] = ld(j, t);
        wl[t] = wr[t] = 0.0;
        if (!(s ? zero2 : zero1) || __any(any_bits(ch[0], ch[1], ch[2]) | any_bits(ch[3], ch[4], ch[5])))
            weno5z_pair<true>(ch, wl[t], wr[t], top, ok);
        wl[t] *= 0.125;
        wr[t] *= 0.125;
    }
    // both states admissible, with sound speeds in range
    const double il = rcp_mid(wl[0]), ir = rcp_mid(wr[0]);
    const double vl = inv_by(wl[0], il), vr = inv_by(wr[0], ir);
    const double vbl = vl - e.b, vbr = vr - e.b;
    const double c2l = div_by(e.gamma * (wl[4] + e.p_inf) * vl * vl, vbl, rcp_volume(e, wl[0], vbl));
    const double c2r = div_by(e.gamma * (wr[4] + e.p_inf) * vr * vr, vbr, rcp_volume(e, wr[0], vbr));
    // all of [lo, hi]: high words order like positive values, a negative one
    // or NaN is above them all
    const unsigned mn = min(min(min(top_word(rho), top_word(vb)), min(top_word(c2), top_word(wl[0]))),
                            min(min(min(top_word(wr[0]), top_word(vbl)), top_word(vbr)), min(top_word(c2l), top_word(c2r))));
    const unsigned mx = max(max(max(top_word(rho), top_word(vb)), max(top_word(c2), top_word(wl[0]))),
                            max(max(max(top_word(wr[0]), top_word(vbl)), top_word(vbr)), max(top_word(c2l), top_word(c2r))));
    ok = ok && top < top_word(Mid<double>::beta_max) && mn >= top_word(Mid<double>::lo) && mx < top_word(Mid<double>::hi);
    double ql[5], qr[5];
#pragma unroll
    for (int s = 0; s < 2; ++s) {
        const double* w = s ? wr : wl;
        double* q = s ? qr : ql;
        const double ke = 0.5 * w[0] * (w[1] * w[1] + w[2] * w[2] + w[3] * w[3]);
        q[0] = w[0];
        q[1] = w[0] * w[1];
        q[2] = w[0] * w[2];
        q[3] = w[0] * w[3];
        const double a = (w[4] + e.gamma * e.p_inf) * (s ? vbr : vbl);
        q[4] = w[0] * (div_by(a, e.gamma - 1.0, e.rg) + e.q) + ke;
    }
    // both energies are positive; below the bound the velocities are in range
    // and no reconstruction is infinite
    if (!(ok && ql[4] + qr[4] < Mid<double>::energy_max)) return false;
    double x;
    hllc_flux<D, true>(wl, wr, ql, qr, sqrt_mid(c2l, x), sqrt_mid(c2r, x), il, ir, f);
    return true;
}

// Flux-form weights of the 6th-order midpoint-to-node difference:
// scheme.rs:92
__device__ constexpr double S6_0 = 75.0 / 64.0 - 25.0 / 384.0 + 3.0 / 640.0;
__device__ constexpr double S6_1 = -25.0 / 384.0 + 3.0 / 640.0;
__device__ constexpr double S6_2 = 3.0 / 640.0;
// 6th-order split-form coefficients: scheme.rs:89
__device__ constexpr double A6_0 = 0.75;
__device__ constexpr double A6_1 = -0.15;
__device__ constexpr double A6_2 = 1.0 / 60.0;

// Fourth difference of a 5-value window: scheme.rs:97-99
template <class R>
__device__ __forceinline__ R d4(R q0, R q1, R q2, R q3, R q4) {
    return fabs(q0 - R(4.0) * q1 + R(6.0) * q2 - R(4.0) * q3 + q4);
}

// Conserved ghost state of the characteristic (non-reflecting) boundary:
// boundary.rs:57-95, for side (0 low, 1 high), boundary cell u_b, its
// interior neighbour u_b1, far-field u_far, layer depth m.
template <int D, class R>
__device__ __forceinline__ void characteristic_ghost(const EosT<R>& e, const R ub[5], const R ub1[5],
                                                     const R uf[5], int side, R m, R out[5]) {
    constexpr int un = 1 + D;
    constexpr int t1 = 1 + (D + 1) % 3;
    constexpr int t2 = 1 + (D + 2) % 3;
    R wi[5], wf[5], w1[5];
    to_prim(e, ub, wi);
    to_prim(e, uf, wf);
    to_prim(e, ub1, w1);
    R rho = wi[0], c = sound_speed(e, wi[0], wi[4]);
    R L[5][5], Rm[5][5];
#pragma unroll
    for (int a = 0; a < 5; ++a)
#pragma unroll
        for (int k = 0; k < 5; ++k) {
            L[a][k] = R(0.0);
            Rm[a][k] = R(0.0);
        }
    L[0][un] = -rho / (R(2.0) * c);
    L[0][4] = R(1.0) / (R(2.0) * c * c);
    L[1][0] = R(1.0);
    L[1][4] = -R(1.0) / (c * c);
    L[2][t1] = R(1.0);
    L[3][t2] = R(1.0);
    L[4][un] = rho / (R(2.0) * c);
    L[4][4] = R(1.0) / (R(2.0) * c * c);
    Rm[0][0] = R(1.0);
    Rm[un][0] = -c / rho;
    Rm[4][0] = c * c;
    Rm[0][1] = R(1.0);
    Rm[t1][2] = R(1.0);
    Rm[t2][3] = R(1.0);
    Rm[0][4] = R(1.0);
    Rm[un][4] = c / rho;
    Rm[4][4] = c * c;
    R u = wi[un];
    R lam[5] = {u - c, u, u, u, u + c};
    R outward = side == 1 ? R(1.0) : -R(1.0);
    R dw[5];
#pragma unroll
    for (int k = 0; k < 5; ++k) dw[k] = wi[k] - wf[k] + m * (wi[k] - w1[k]);
    R wg[5];
#pragma unroll
    for (int k = 0; k < 5; ++k) wg[k] = wf[k];
#pragma unroll
    for (int kf = 0; kf < 5; ++kf) {
        if (lam[kf] * outward > R(0.0)) {
            R amp = -R(0.0);
#pragma unroll
            for (int q = 0; q < 5; ++q) amp += L[kf][q] * dw[q];
#pragma unroll
            for (int q = 0; q < 5; ++q) wg[q] += Rm[q][kf] * amp;
        }
    }
    to_cons(e, wg, out);
}

// Conserved state of the ghost cell at pencil coordinate g (outside [0, n))
// of a pencil whose interior cell x is read by ld(x, out).  Follows
// Solver::fill_ghosts (solver.rs:278-348) and reflected_ghost
// (boundary.rs:102-145): periodic wraps (also around axes shorter than the
// ghost depth), outflow copies the boundary cell, Dirichlet gives the fixed
// state, characteristic extrapolates outgoing waves, reflect mirrors with the
// normal momentum negated (and resolves deep images through the opposite
// side's condition).  Every ghost depends only on its own pencil, so the
// value is the same as after the reference's axis-ordered sweeps.
// Kinds: 0 periodic, 1 outflow, 2 reflect, 3 Dirichlet, 4 characteristic.
template <int D, class R, class LD>
__device__ __forceinline__ void bc_ghost(const EosT<R>& e, int n, int g, const int kind[2], const R (*state)[5],
                                         LD ld, R u[5]) {
    int x = g;
    bool flip = false;
    for (int it = 0; it < 64; ++it) {
        if (x >= 0 && x < n) {
            ld(x, u);
            break;
        }
        const int side = x >= n ? 1 : 0;
        const int k = side ? kind[1] : kind[0];
        if (k == 2) {
            x = side == 0 ? -1 - x : 2 * n - 1 - x;
            flip = !flip;
            continue;
        }
        if (k == 0) {
            ld(((x % n) + n) % n, u);
        } else if (k == 1) {
            ld(side == 0 ? 0 : n - 1, u);
        } else if (k == 3) {
#pragma unroll
            for (int q = 0; q < 5; ++q) u[q] = side ? state[1][q] : state[0][q];
        } else {
            R ub[5], ub1[5];
            ld(side == 0 ? 0 : n - 1, ub);
            ld(side == 0 ? 1 : n - 2, ub1);
            R uf[5];
#pragma unroll
            for (int q = 0; q < 5; ++q) uf[q] = side ? state[1][q] : state[0][q];
            characteristic_ghost<D>(e, ub, ub1, uf, side, side == 0 ? R(-x) : R(x - n + 1), u);
        }
        break;
    }
    if (flip) u[1 + D] *= -R(1.0);
}

}  // namespace em
