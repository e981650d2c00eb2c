// Division by a constant of the launch (a cell width) with the result of the
// division itself, bit for bit, at a fifth of its instructions.
//
// Markstein's theorem (IBM J. Res. Dev. 34, 1990; Muller et al., Handbook of
// Floating-Point Arithmetic): with y = RN(1/b) and q within one ulp of a/b,
// r = RN(a - b q) is exact and RN(q + r y) is the correctly rounded quotient.
// q = RN(a y) may be up to two ulps off, so one such step makes it faithful
// and the second one rounds it correctly: one product and four fused
// multiply-adds instead of the ~25 instructions (scaling, reciprocal
// estimate, refinement, fix-up) of a general FP64 division.  The theorem
// needs quotient and residual clear of under- and overflow: the exponent of
// a has to lie in [2^-512, 2^512), tested on the high word, and that of b in
// [2^-128, 2^128] and positive, tested on the host (span = 0 otherwise).  Anything else
// (infinities, NaN, extreme values; zeros are exact) takes the division.
#pragma once
#include <cmath>
#include <cstdint>
#include <cstring>

#if defined(__HIPCC__)
#include <hip/hip_runtime.h>
#define XDIV_FN __host__ __device__ inline
#else
#define XDIV_FN inline
#endif

struct exact_div {
    double   b, y;      // divisor and its correctly rounded reciprocal
    uint32_t span;      // width of the accepted exponent range of a (high word), 0: none
};

#define XDIV_LO   ((uint32_t)(1023 - 512) << 20)
#define XDIV_SPAN ((uint32_t)1024 << 20)

static inline exact_div make_exact_div(double b) {
    return exact_div{b, 1.0 / b, (b >= 0x1p-128 && b <= 0x1p128) ? XDIV_SPAN : 0u};
}

XDIV_FN uint32_t xdiv_hi(double a) {
#if defined(__HIP_DEVICE_COMPILE__)
    return (uint32_t)__double2hiint(a);
#else
    uint64_t u;
    std::memcpy(&u, &a, 8);
    return (uint32_t)(u >> 32);
#endif
}

// The steps alone: RN(a / d.b) for a in the accepted range or +-0 (the
// residuals are formed as b q - a, which keeps the sign of a zero).
XDIV_FN double xdiv_core(double a, const exact_div &d) {
    const double q0 = a * d.y;
    const double q1 = fma(-fma(d.b, q0, -a), d.y, q0);
    return fma(-fma(d.b, q1, -a), d.y, q1);
}
// Whether xdiv_core's result is the quotient.
XDIV_FN bool xdiv_takes(double a, const exact_div &d) {
    return (xdiv_hi(a) & 0x7fffffffu) - XDIV_LO < d.span || (a == 0.0 && d.span != 0u);
}

// RN(a / d.b)
XDIV_FN double xdiv(double a, const exact_div &d) {
    double q = xdiv_core(a, d);
    if (__builtin_expect(!xdiv_takes(a, d), 0)) q = a / d.b;
    return q;
}
