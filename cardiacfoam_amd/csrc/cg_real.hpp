// Double-precision arithmetic of the FP64 model kernels: `real` is a double whose division
// and tanh are written for gfx950; every other operation is the built-in one.
//
// What it is for: the FP64 ionic kernels are bound by VALU issue, and a quarter to a third
// of their instructions were divisions (ORd: 273 of them, 11 instructions and a wait each,
// 3000 of 7229).
//   a / c, c known at compile time: a times the rounded 1/c and one residual correction
//     (3 instructions; correctly rounded but for rare ties, as the correction's error is
//     ~2^-105 of the quotient);
//   a / b: v_rcp_f64, one Newton step, a times that and one residual correction, then
//     v_div_fixup_f64 for zeros, infinities and NaN (7 instructions).  v_rcp_f64 starts at
//     ~2^-27, so the step leaves 2^-53 and the corrected quotient is within 0.5000001 ulp.
//     No scaling: quotients whose divisor lies beyond 2^1022, or that underflow, lose bits
//     of a value that is zero for every model here.
//   tanh(x) = 1 - 2 / (exp(2x) + 1): absolute error 2e-16 in place of a relative one of
//     1 ulp.  Every use in the models is 1 + tanh(x), whose own rounding is as large.
#pragma once
#include "cg_common.hpp"

namespace cg {

struct real {
    double v;
    real() = default;
    CG_HD constexpr real(double x) : v(x) {}
    CG_HD constexpr explicit operator double() const { return v; }
    CG_HD real& operator+=(real o) { v += o.v; return *this; }
    CG_HD real& operator-=(real o) { v -= o.v; return *this; }
    CG_HD real& operator*=(real o) { v *= o.v; return *this; }
};

CG_HD double real_quot(double a, double b)
{
#if defined(__HIP_DEVICE_COMPILE__)
    if (__builtin_constant_p(b)) {
        const double y = 1.0 / b, q = a * y;
        return __builtin_fma(__builtin_fma(-q, b, a), y, q);
    }
    const double y0 = __builtin_amdgcn_rcp(b);
    const double y = __builtin_fma(__builtin_fma(-b, y0, 1.0), y0, y0);
    const double q = a * y;
    return __builtin_amdgcn_div_fixup(__builtin_fma(__builtin_fma(-b, q, a), y, q), b, a);
#else
    return a / b;
#endif
}

CG_HD real operator+(real a, real b) { return a.v + b.v; }
CG_HD real operator-(real a, real b) { return a.v - b.v; }
CG_HD real operator*(real a, real b) { return a.v * b.v; }
CG_HD real operator/(real a, real b) { return real_quot(a.v, b.v); }
CG_HD real operator-(real a) { return -a.v; }
CG_HD bool operator<(real a, real b) { return a.v < b.v; }
CG_HD bool operator>(real a, real b) { return a.v > b.v; }
CG_HD bool operator<=(real a, real b) { return a.v <= b.v; }
CG_HD bool operator>=(real a, real b) { return a.v >= b.v; }
CG_HD bool operator==(real a, real b) { return a.v == b.v; }
CG_HD bool operator!=(real a, real b) { return a.v != b.v; }

CG_HD real cexp(real x) { return exp(x.v); }
CG_HD real clog(real x) { return log(x.v); }
CG_HD real csqrt(real x) { return sqrt(x.v); }
CG_HD real cpow(real x, real y) { return pow(x.v, y.v); }
CG_HD real fabs(real x) { return __builtin_fabs(x.v); }
CG_HD real ctanh(real x) { return 1.0 - real_quot(2.0, exp(2.0 * x.v) + 1.0); }
CG_HD real ghk_quot(real v, real, real ekv) { return v / (ekv - 1.0); }

} // namespace cg
