// Scalar functions of the generated Taylor steps, placed before every step prelude.
// Each does one step's use of a library function in the few instructions that this use
// needs; all code forms of a system call the same ones, so they round alike (no implicit
// fusion of a product into an add in here, for the same reason). Outside the device
// compiler (the CPU tests of the generated code) the hardware's approximations come from the C library.
//
// Why: at one wavefront per SIMD, which the register and group forms run at, every
// instruction takes 4 to 5 cycles to issue, whatever it is, and pow() is about 150
// of them (logarithm and exponential in extended precision, every special case). Measured when
// they came in, with pow() and with these functions: four pendulums to t = 100 1.09 -> 0.80 ms,
// 65,536 six-body systems to t = 10 56.2 -> 52.6 ms. VALU instructions of hyx_step_k, with pow() and
// now: pendulum 1,086 and 784, planar CR3BP in the quad form 1,797 and 1,555.

template <int R>
__device__ __forceinline__ double hyx_ipow(double y)
{
    if constexpr (R == 1)
        return y;
    else if constexpr (R % 2 == 0) {
        const double t = hyx_ipow<R / 2>(y);
        return t * t;
    } else
        return hyx_ipow<R - 1>(y) * y;
}

// (num / den)^(1/R) of the step-size rule, rnum = 1 / num: with q = den / num, Newton's
// iteration for q y^R = 1, y <- y + y (1 - q y^R) / R, which needs no division. It starts from
// a single-precision exp2(-log2(q) / R), whose error is below 1e-5 / R (the logarithm's absolute
// one, at most 4e-5, over R), and the error of an iteration is (R + 1) / 2 times the square of
// the last, so two reach double precision; the rounding of q y^R enters y divided by R. q is scaled by
// 2^(-R e) and y by 2^e, so that no power of y leaves the exponent range, whatever q.
// den = 0 gives inf and den = inf gives 0, as pow() does; num / den beyond the largest double
// (q below 2^-1024) gives inf too, as the division in pow(num / den, 1 / R) does.
template <int R>
__device__ __forceinline__ double hyx_root(double rnum, double den)
{
#pragma STDC FP_CONTRACT OFF
    const double q = den * rnum;
#ifdef __AMDGCN__
    const double m = __builtin_amdgcn_frexp_mant(q);
    const float l = __builtin_amdgcn_logf((float)m), ef = (float)__builtin_amdgcn_frexp_exp(q);
#else
    int ex = 0;
    const double m = frexp(q, &ex);
    const float l = log2f((float)m), ef = (q - q == 0.0) ? (float)ex : 0.0f;
#endif
    const float e = __builtin_rintf(ef * (1.0f / R));
    const float t = ((float)R * e - ef - l) * (1.0f / R);
#ifdef __AMDGCN__
    const float y0 = __builtin_amdgcn_exp2f(t);
#else
    const float y0 = exp2f(t);
#endif
    const int ei = (int)e;
    const double qs = ldexp(q, -R * ei);
    double y = (double)y0;
    y = __builtin_fma(y * (1.0 / R), __builtin_fma(-qs, hyx_ipow<R>(y), 1.0), y);
    y = __builtin_fma(y * (1.0 / R), __builtin_fma(-qs, hyx_ipow<R>(y), 1.0), y);
    // Beyond the largest double: a scale that overflows. (One select of an integer: flushing q to
    // zero first takes a step of 200 CR3BP orbits 2.5 % longer, and a return at the end, which becomes
    // a branch around the iterations, one of four pendulums 5 %.)
    const double r = ldexp(y, q <= 0x1p-1024 ? 4096 : -ei);
    // q = 0 or inf: the start is the value.
    return (q == 0.0 || q == __builtin_inf()) ? (double)y0 : r;
}

// s ~ x^(-1/2) to about one ulp, and its correction: p + pl = s^2 exactly, and
// e = 1 - x s^2 to double precision of its own, so x^(-1/2) = s (1 + e/2 + O(e^2)), e^2 < 2^-100.
__device__ __forceinline__ void hyx_rsqrt_parts(double x, double &s, double &p, double &pl, double &e)
{
#pragma STDC FP_CONTRACT OFF
#ifdef __AMDGCN__
    const double s0 = __builtin_amdgcn_rsq(x); // at least 20 bits
#else
    const double s0 = 1.0 / sqrt(x) * (1.0 + 0x1p-21);
#endif
    const double e0 = __builtin_fma(-(x * s0), s0, 1.0);
    s = __builtin_fma(s0 * e0, __builtin_fma(e0, 0.375, 0.5), s0);
    p = s * s;
    pl = __builtin_fma(s, s, -p);
    e = __builtin_fma(-x, pl, __builtin_fma(-x, p, 1.0));
}

// Arguments whose powers stay far from the ends of the exponent range (false for NaN).
__device__ __forceinline__ bool hyx_mid_range(double x) { return x > 0x1p-300 && x < 0x1p+300; }

// x^(-3/2) and rx = 1 / x, both rounded once from a result with about 100 bits.
__device__ __forceinline__ double hyx_pow_m3_2(double x, double &rx)
{
#pragma STDC FP_CONTRACT OFF
    if (!hyx_mid_range(x)) {
        rx = 1.0 / x;
        return pow(x, -1.5);
    }
    double s, p, pl, e;
    hyx_rsqrt_parts(x, s, p, pl, e);
    rx = p + __builtin_fma(p, e, pl);
    const double c = s * p;
    const double cl = __builtin_fma(s, pl, __builtin_fma(s, p, -c));
    return c + __builtin_fma(c * 1.5, e, cl);
}

// x^(-1/2) and rx = 1 / x.
__device__ __forceinline__ double hyx_pow_m1_2(double x, double &rx)
{
#pragma STDC FP_CONTRACT OFF
    if (!hyx_mid_range(x)) {
        rx = 1.0 / x;
        return pow(x, -0.5);
    }
    double s, p, pl, e;
    hyx_rsqrt_parts(x, s, p, pl, e);
    rx = p + __builtin_fma(p, e, pl);
    return __builtin_fma(s * 0.5, e, s);
}

