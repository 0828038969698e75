// Transcendental functions of the point-wise and G-space kernels, by
// precision.  FP64 has the library's logarithm, exponential and general power;
// its roots and quotients are those at the end of this file, whose largest
// errors are stated there (the library's division and square root: half an
// ulp; 1 / sqrt 1.5).  FP32 (the
// FP32-bulk pipeline, whose accuracy is set by single-precision storage and
// FFTs anyway) uses the hardware approximations v_sqrt_f32, v_rsq_f32,
// v_rcp_f32, v_log_f32 (log2) and v_exp_f32 (exp2), each within about 1 ulp,
// instead of the library's range-reduced forms of 10 to 40 instructions.
#pragma once
#include <hip/hip_runtime.h>

#include <cmath>

namespace ofdft {
namespace fm {

template <typename T> __device__ __forceinline__ T sqrt(T x) { return ::sqrt(x); }
template <> __device__ __forceinline__ float sqrt<float>(float x) { return __builtin_amdgcn_sqrtf(x); }

// FP32 square root of x > 0 from the hardware reciprocal root, corrected to
// within about half an ulp (the vW term multiplies its rounding by G^2)
__device__ __forceinline__ float sqrt_c(float x) {
    const float y = __builtin_amdgcn_rsqf(x), g = x * y;
    // denormals and infinity keep the plain hardware root
    return x > 1e-37f && x < (float)INFINITY ? __builtin_fmaf(__builtin_fmaf(-g, g, x), 0.5f * y, g)
                                             : __builtin_amdgcn_sqrtf(x);
}

template <typename T> __device__ __forceinline__ T rcp(T x) { return (T)1 / x; }
template <> __device__ __forceinline__ float rcp<float>(float x) { return __builtin_amdgcn_rcpf(x); }

template <typename T> __device__ __forceinline__ T rsq(T x) { return (T)1 / ::sqrt(x); }
template <> __device__ __forceinline__ float rsq<float>(float x) { return __builtin_amdgcn_rsqf(x); }

// a / b
template <typename T> __device__ __forceinline__ T div(T a, T b) { return a / b; }
template <> __device__ __forceinline__ float div<float>(float a, float b) { return a * __builtin_amdgcn_rcpf(b); }

// natural logarithm for arguments away from 1 (absolute error of log2 about
// 1 ulp of its result's scale)
template <typename T> __device__ __forceinline__ T log(T x) { return ::log(x); }
template <> __device__ __forceinline__ float log<float>(float x) {
    return __builtin_amdgcn_logf(x) * 0.693147180559945309f;
}

// x^y for x > 0
template <typename T> __device__ __forceinline__ T pow(T x, T y) { return ::pow(x, y); }
template <> __device__ __forceinline__ float pow<float>(float x, float y) {
    return __builtin_amdgcn_exp2f(y * __builtin_amdgcn_logf(x));
}

// cube root for x >= 0: exp2(log2(x) / 3) refined by one Newton step
// y <- y - (y^3 - x) / (3 y^2)
template <typename T> __device__ __forceinline__ T cbrt(T x) { return ::cbrt(x); }
template <> __device__ __forceinline__ float cbrt<float>(float x) {
    const float y = __builtin_amdgcn_exp2f(__builtin_amdgcn_logf(x) * (1.0f / 3.0f));
    const float r = __builtin_amdgcn_rcpf(y * y);
    const float z = y - (y - x * r) * (1.0f / 3.0f);
    return x > 0.0f ? z : 0.0f;
}

// Roots of one finite a > 0 in FP64, denormals too: a = m 2^(6 q) with m in
// [1/2, 32), and s = m^(-1/6) by one third-order step from the FP32 hardware
// log2 and exp2.  Its powers, each with one correction, give the roots, about
// 20 instructions in all, where the library's cbrt, sqrt and division take ten
// times that.  Largest errors in ulps: a^(-1/6) 0.9, square root 0.5,
// reciprocal square root 1.0, cube root 0.75.
struct SixthRoot {
    double m, s;
    int q;
    __device__ __forceinline__ explicit SixthRoot(double a) {
        const int e = __builtin_amdgcn_frexp_exp(a);
        q = (e + 1536) / 6 - 256;  // floor(e / 6)
        m = __builtin_amdgcn_ldexp(__builtin_amdgcn_frexp_mant(a), e - 6 * q);
        s = (double)__builtin_amdgcn_exp2f(__builtin_amdgcn_logf((float)m) * (-1.0f / 6.0f));
        const double s3 = s * s * s;
        const double h = __builtin_fma(-m, s3 * s3, 1.0);
        s = __builtin_fma(s * h, __builtin_fma(h, 7.0 / 72.0, 1.0 / 6.0), s);
    }
    __device__ __forceinline__ double inv_sixth() const { return __builtin_amdgcn_ldexp(s, -q); }
    __device__ __forceinline__ double sqrt() const {
        const double s3 = s * s * s, y = m * s3;
        return __builtin_amdgcn_ldexp(__builtin_fma(__builtin_fma(-y, y, m), 0.5 * s3, y), 3 * q);
    }
    __device__ __forceinline__ double rsq() const {
        const double y = s * s * s;
        return __builtin_amdgcn_ldexp(__builtin_fma(__builtin_fma(-m * y, y, 1.0), 0.5 * y, y), -3 * q);
    }
    __device__ __forceinline__ double cbrt() const {
        const double s2 = s * s, s4 = s2 * s2, y = m * s4;
        return __builtin_amdgcn_ldexp(__builtin_fma(__builtin_fma(-y * y, y, m), s4 * (1.0 / 3.0), y), 2 * q);
    }
};
// square root in FP64 of normal numbers, zeros, infinity and NaN (negative:
// NaN), within half an ulp: a Goldschmidt step on the hardware reciprocal root
// and a correction
__device__ __forceinline__ double sqrt_n(double x) {
    const double y = __builtin_amdgcn_rsq(x);
    double g = x * y, h = 0.5 * y;
    const double r = __builtin_fma(-h, g, 0.5);
    g = __builtin_fma(g, r, g);
    h = __builtin_fma(h, r, h);
    g = __builtin_fma(__builtin_fma(-g, g, x), h, g);
    return x == 0.0 || x == (double)INFINITY ? x : g;
}
__device__ __forceinline__ float sqrt_n(float x) { return sqrt(x); }
// a / b in FP64 within half an ulp for |b| and the quotient within 2^+-1000,
// zeros, infinities and NaN as the division: two Newton steps on the hardware
// reciprocal and a correction of the quotient
__device__ __forceinline__ double div_n(double a, double b) {
    double r = __builtin_amdgcn_rcp(b);
    r = __builtin_fma(__builtin_fma(-b, r, 1.0), r, r);
    r = __builtin_fma(__builtin_fma(-b, r, 1.0), r, r);
    const double q = a * r;
    return __builtin_amdgcn_div_fixup(__builtin_fma(__builtin_fma(-b, q, a), r, q), b, a);
}

}  // namespace fm
}  // namespace ofdft
