// The FP64 arithmetic type of the model kernels: a double whose division is arranged for
// the shape the ionic models have, everything else the plain operator.
//
// The compiler expands a/b into 11 FP64 instructions (two operand scalings, a reciprocal at
// a quarter of the rate, four refinements, quotient, remainder, scaled correction, special
// cases) and the wait states between them; ORd has 273 divisions in a cell step, 40 % of
// its instructions.  Written out here without the scalings:
//   by a constant c      q = a RN(1/c); q + (a - c q) RN(1/c); special cases   (4)
//   by a power of two    a (1/c)                                               (1)
//   1/b                  reciprocal, two refinements, special cases            (6)
//   a/b                  reciprocal, one refinement, quotient and its exact
//                        remainder's correction, special cases                 (7)
// Error: the hardware's reciprocal is within 2^-24 (2^29 ulp), one refinement brings it
// to 2^-48, two to rounding.  q is then within 2^-48 of a/b, its remainder is formed in one
// fma and correct to 2^-53, and the correction (the remainder times the reciprocal) to
// 2^-48: a relative 2^-96 before the last rounding, so the quotient is within 0.5 + 2^-42 ulp,
// the correctly rounded one unless a/b lies that close to the middle of two doubles (the
// order of operations is that of Markstein, IBM J. Res. Dev. 34, 1990, whose theorem asks
// for a rounded reciprocal).  Below 2^-969 the remainder rounds as a subnormal does.
// Infinite, zero and NaN operands and overflowing quotients give IEEE results through
// v_div_fixup (measured).  A divisor below 2^-1024 with a finite quotient gives an infinite
// one: a gate's dt/tau, Grandi's and ToRORd's at 1.39 V, where exp(-dt/tau) is 0 either way.
// In 6e8 random quotients (a/b, 1/b, by 3, 0.7 and 26.7137; exponents to +-480) none differed
// from the compiler's division.
// Measured: 30 implicit FP64 ORd steps of 2.1M cells 34.4 -> 29.3 ms (ionic kernel 732 ->
// 592 us), 200 explicit BuenoOrovio steps of 147k cells 2.10 -> 1.70 ms.
#pragma once
#include <hip/hip_runtime.h>
#include <cstdint>
#include <cmath>

namespace cg {

__host__ __device__ constexpr bool pow2_double(double b)
{
    return (__builtin_bit_cast(uint64_t, b) & 0xfffffffffffffull) == 0;
}

__device__ __forceinline__ double div_f64(double a, double b)
{
    // known after inlining: a constant divisor of ordinary size
    if (__builtin_constant_p(b) && __builtin_fabs(b) > 1e-290 && __builtin_fabs(b) < 1e290) {
        const double rb = 1.0 / b;
        if (pow2_double(b)) return a * rb;
        const double q = a * rb;
        const double r = __builtin_fma(-b, q, a);
        return __builtin_amdgcn_div_fixup(__builtin_fma(r, rb, q), b, a);
    }
    double r = __builtin_amdgcn_rcp(b);
    r = __builtin_fma(__builtin_fma(-b, r, 1.0), r, r);
    if (__builtin_constant_p(a) && a == 1.0)
        return __builtin_amdgcn_div_fixup(__builtin_fma(__builtin_fma(-b, r, 1.0), r, r), b, a);
    const double q = a * r;
    return __builtin_amdgcn_div_fixup(__builtin_fma(__builtin_fma(-b, q, a), r, q), b, a);
}

struct F64 {
    double v;
    F64() = default;
    __host__ __device__ __forceinline__ constexpr F64(double x) : v(x) {}
    __host__ __device__ __forceinline__ explicit operator double() const { return v; }
    __host__ __device__ __forceinline__ explicit operator float() const { return float(v); }

    friend __device__ __forceinline__ F64 operator+(F64 a, F64 b) { return a.v + b.v; }
    friend __device__ __forceinline__ F64 operator-(F64 a, F64 b) { return a.v - b.v; }
    friend __device__ __forceinline__ F64 operator*(F64 a, F64 b) { return a.v * b.v; }
    friend __device__ __forceinline__ F64 operator/(F64 a, F64 b) { return div_f64(a.v, b.v); }
    friend __device__ __forceinline__ F64 operator-(F64 a) { return -a.v; }
    __device__ __forceinline__ F64& operator+=(F64 b) { v += b.v; return *this; }
    __device__ __forceinline__ F64& operator-=(F64 b) { v -= b.v; return *this; }
    __device__ __forceinline__ F64& operator*=(F64 b) { v *= b.v; return *this; }
    friend __device__ __forceinline__ bool operator<(F64 a, F64 b) { return a.v < b.v; }
    friend __device__ __forceinline__ bool operator>(F64 a, F64 b) { return a.v > b.v; }
    friend __device__ __forceinline__ bool operator<=(F64 a, F64 b) { return a.v <= b.v; }
    friend __device__ __forceinline__ bool operator>=(F64 a, F64 b) { return a.v >= b.v; }
    friend __device__ __forceinline__ bool operator==(F64 a, F64 b) { return a.v == b.v; }
    friend __device__ __forceinline__ bool operator!=(F64 a, F64 b) { return a.v != b.v; }
    friend __device__ __forceinline__ F64 fabs(F64 a) { return __builtin_fabs(a.v); }
};
static_assert(sizeof(F64) == 8, "states of an FP64 handle are plain doubles");

// (one name for both sides of HD templates; the kernels run on the device)
__device__ __forceinline__ F64 cexp(F64 x) { return ::exp(x.v); }
__device__ __forceinline__ F64 clog(F64 x) { return ::log(x.v); }
__device__ __forceinline__ F64 ctanh(F64 x) { return ::tanh(x.v); }
__device__ __forceinline__ F64 csqrt(F64 x) { return ::sqrt(x.v); }
__device__ __forceinline__ F64 cpow(F64 x, F64 y) { return ::pow(x.v, y.v); }
__device__ __forceinline__ F64 ghk_quot(F64 v, F64, F64 ekv) { return v / (ekv - 1.0); }

} // namespace cg
