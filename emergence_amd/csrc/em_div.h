// Division and square root for operands known to lie in the middle of the
// exponent range, and the range tests that establish it.
//
// The compiler's IEEE division scales both operands (v_div_scale x2), takes
// v_rcp, two Newton steps, the quotient, one correction, and undoes the
// scaling (v_div_fmas, v_div_fixup): 11 instructions, of which the
// reciprocal counts four, in a chain through VCC.  Far from overflow and
// underflow the scaling is the identity, so the steps between give the same
// correctly rounded quotient, and the reciprocal can be shared by every
// quotient of one divisor (and, through products, by several divisors).
// div_by is that core: with r = 1/b to within about half an ulp,
//   q = RN(a r),  rem = a - b q (exact),  RN(q + rem r) = RN(a / b).
// It needs |b|, |a| and |a/b| within 2^+-900 (or a = +0; div_by_pos and
// div_by_fix also keep the sign of -0).  The callers test their operands (Mid)
// and hand everything else to the general expressions.
#pragma once
#include <hip/hip_runtime.h>

namespace em {

template <class R>
struct Mid;
template <>
struct Mid<double> {
    static constexpr double lo = 0x1p-100, hi = 0x1p+100;  // densities, squared sound speeds
    static constexpr double tiny = 0x1p-900;               // quotients and dividends below go the general way
    static constexpr double huge = 0x1p+800;
    static constexpr double beta_max = 0x1p+100;  // product of three WENO smoothness indicators
    static constexpr double energy_max = 0x1p+300;  // total energies of a midpoint's two states
    static constexpr double margin = 1e-9;        // relative slack of clearly_admissible (rounding: about 1e-15)
};
template <>
struct Mid<float> {  // clearly_admissible only
    static constexpr float lo = 0x1p-40f, hi = 0x1p+40f;
    static constexpr float margin = 1e-3f;  // (rounding: up to 1e-4 as gamma nears 1.01)
};

// x within [lo, hi] (false for NaN)
template <class R>
__device__ __forceinline__ bool in_mid(R x) {
    return x >= Mid<R>::lo && x <= Mid<R>::hi;
}
// x is neither zero nor large enough for the core (true for NaN): the
// quotient or dividend needs the general division
template <class R>
__device__ __forceinline__ bool too_small(R x) {
    return !(fabs(x) >= Mid<R>::tiny) && x != R(0.0);
}

__device__ __forceinline__ double rcp_step(double b, double r) { return __builtin_fma(__builtin_fma(-b, r, 1.0), r, r); }
// 1/b to about half an ulp
__device__ __forceinline__ double rcp_mid(double b) {
    return rcp_step(b, rcp_step(b, __builtin_amdgcn_rcp(b)));
}

// a / b from r = rcp_mid(b)
__device__ __forceinline__ double div_by(double a, double b, double r) {
    const double q = a * r;
    return __builtin_fma(__builtin_fma(-b, q, a), r, q);
}
// the same with the sign of a zero dividend and infinite or NaN dividends
// as IEEE division gives them
__device__ __forceinline__ double div_by_fix(double a, double b, double r) {
    return __builtin_amdgcn_div_fixup(div_by(a, b, r), b, a);
}
// a / b, b > 0: div_by with the sign of a zero dividend (div_by turns -0 into
// +0; a reflecting wall makes -0 of every zero momentum)
__device__ __forceinline__ double div_by_pos(double a, double b, double r) { return copysign(div_by(a, b, r), a); }
// 1 / b from r = rcp_mid(b)
__device__ __forceinline__ double inv_by(double b, double r) { return rcp_step(b, r); }

// sqrt(x), x within [lo, hi]: v_rsq and the coupled Newton iteration of
// sqrt and 1 / (2 sqrt) with two residual corrections (Goldschmidt; Markstein
// 2000), correctly rounded; inv = rcp_mid of the root, from the iteration's
// own 1 / (2 sqrt).
__device__ __forceinline__ double sqrt_mid(double x, double& inv) {
    const double y = __builtin_amdgcn_rsq(x);
    double g = x * y, h = 0.5 * y;
    const double r = __builtin_fma(-h, g, 0.5);
    g = __builtin_fma(g, r, g);
    h = __builtin_fma(h, r, h);
    g = __builtin_fma(__builtin_fma(-g, g, x), h, g);
    g = __builtin_fma(__builtin_fma(-g, g, x), h, g);
    inv = rcp_step(g, h + h);
    return g;
}

// 1/d0, 1/d1, 1/d2 through one reciprocal of the product, which is returned
// (doubles of at least 2^-133 with a product up to 2^100); each gets its own
// last Newton step.  Singly 8 issue slots each, jointly 18 for the three.
__device__ __forceinline__ double rcp3_mid(double d0, double d1, double d2, double& r0, double& r1, double& r2) {
    const double p = d0 * d1, pp = p * d2;
    const double r = rcp_step(pp, __builtin_amdgcn_rcp(pp));
    const double r01 = r * d2;
    r0 = rcp_step(d0, r01 * d1);
    r1 = rcp_step(d1, r01 * d0);
    r2 = rcp_step(d2, r * p);
    return pp;
}
// the same for two doubles of at least 2^-1 (NaN where their product overflows;
// div_by_fix then makes the quotients infinite)
__device__ __forceinline__ void rcp2_mid(double d0, double d1, double& r0, double& r1) {
    const double p = d0 * d1;
    const double r = rcp_step(p, __builtin_amdgcn_rcp(p));
    r0 = rcp_step(d0, r * d1);
    r1 = rcp_step(d1, r * d0);
}

// High word of a non-negative value, which orders like the value (NaN above
// all): a running bound at one instruction per two values.
__device__ __forceinline__ unsigned top_word(double x) { return (unsigned)__double2hiint(x); }

// a value equal on all lanes, kept in scalar registers
__device__ __forceinline__ double wave_uniform(double x) {
    return __hiloint2double(__builtin_amdgcn_readfirstlane(__double2hiint(x)),
                            __builtin_amdgcn_readfirstlane(__double2loint(x)));
}

// Scalar-cache copy of *p, the same for the whole wave, from memory that no
// kernel running meanwhile writes.  Through an ordinary pointer a kernel that
// also stores reads such arguments with vector loads into vector registers.
template <class T>
__device__ __forceinline__ T scalar_copy(const T* p) {
    static_assert(sizeof(T) % 4 == 0, "whole words");
    const __attribute__((address_space(4))) unsigned* s =
        (const __attribute__((address_space(4))) unsigned*)(unsigned long long)p;
    unsigned t[sizeof(T) / 4];
#pragma unroll
    for (int i = 0; i < (int)(sizeof(T) / 4); ++i) t[i] = s[i];
    T r;
    __builtin_memcpy(&r, t, sizeof(T));
    return r;
}

// x, unknown to the optimiser
__device__ __forceinline__ int opaque(int x) {
    asm volatile("" : "+v"(x));
    return x;
}

// some bit of the three set (false only for +0, +0, +0)
__device__ __forceinline__ unsigned any_bits(double a, double b, double c) {
    const unsigned long long m = (unsigned long long)(__double_as_longlong(a) | __double_as_longlong(b) | __double_as_longlong(c));
    return (unsigned)(m >> 32) | (unsigned)m;
}

}  // namespace em
