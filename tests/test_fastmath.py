"""The FP64 roots and quotients of csrc/fastmath.h on the CPU, compiled with
stand-ins for the hardware approximations whose errors are at the
instructions' bounds (2^-22 for the FP64 reciprocal and reciprocal root, an
ulp for the FP32 log2 and exp2), against 64-bit mantissas."""
import json
import os
import subprocess

import pytest

from conftest import ROOT

SRC = r"""
#include <cmath>
#include <cstdint>
#include <cstdio>
#include <random>
static std::mt19937_64 rng(1);
static double uni() { return (double)(rng() >> 11) * 0x1p-53; }
static double off(int bits) { return 1.0 + std::ldexp(2.0 * uni() - 1.0, -bits); }
#define BUILTIN(T, name, ...) static T __builtin_amdgcn_##name(__VA_ARGS__)
BUILTIN(double, rcp, double x) { return 1.0 / x * off(22); }
BUILTIN(double, rsq, double x) { return 1.0 / std::sqrt(x) * off(22); }
BUILTIN(float, rcpf, float x) { return 1.0f / x; }
BUILTIN(float, rsqf, float x) { return 1.0f / std::sqrt(x); }
BUILTIN(float, sqrtf, float x) { return std::sqrt(x); }
BUILTIN(float, logf, float x) { return (float)(std::log2((double)x) * off(23)); }
BUILTIN(float, exp2f, float x) { return (float)(std::exp2((double)x) * off(23)); }
BUILTIN(int, frexp_exp, double x) { int e = 0; if (std::isfinite(x)) std::frexp(x, &e); return e; }
BUILTIN(double, frexp_mant, double x) { int e; return std::isfinite(x) ? std::frexp(x, &e) : x; }
BUILTIN(double, ldexp, double x, int e) { return std::ldexp(x, e); }
// quotient q of a / b: the special values of the division
BUILTIN(double, div_fixup, double q, double b, double a) {
    const bool special = a == 0 || b == 0 || !std::isfinite(a) || !std::isfinite(b);
    return special ? a / b : q;
}
#include "fastmath.h"
using namespace ofdft::fm;
static double ulps(double v, long double exact) {
    int e;
    std::frexp((double)exact, &e);
    return (double)std::fabs(((long double)v - exact) / std::ldexp(1.0L, (e < -1021 ? -1021 : e) - 53));
}
static double number(int lo, int hi) { return std::ldexp(0.5 + 0.5 * uni(), lo + (int)(rng() % (uint64_t)(hi - lo + 1))); }
int main() {
    double sixth = 0, sq = 0, rs = 0, cb = 0, sn = 0, dv = 0;
    for (int i = 0; i < 1000000; ++i) {
        const double a = i % 4 ? number(-120, 40) : number(-1073, 1024);  // densities, and every exponent
        const long double x = a, r = std::sqrt(x);
        const SixthRoot w(a);
        sixth = std::fmax(sixth, ulps(w.inv_sixth(), 1.0L / std::cbrt(r)));
        sq = std::fmax(sq, ulps(w.sqrt(), r));
        rs = std::fmax(rs, ulps(w.rsq(), 1.0L / r));
        cb = std::fmax(cb, ulps(w.cbrt(), std::cbrt(x)));
        const double n = number(-960, 1000), b = number(-990, 990), c = number(-9, 9) * b;
        sn = std::fmax(sn, ulps(sqrt_n(n), std::sqrt((long double)n)));
        dv = std::fmax(dv, std::fmax(ulps(div_n(1.0, b), 1.0L / b), ulps(div_n(c, b), (long double)c / b)));
    }
    const double inf = INFINITY;
    const bool special = div_n(1.0, inf) == 0.0 && div_n(1.0, 0.0) == inf && div_n(-1.0, 0.0) == -inf &&
                         div_n(0.0, 2.0) == 0.0 && div_n(inf, 2.0) == inf && std::isnan(div_n(NAN, 1.0)) &&
                         std::isnan(div_n(0.0, 0.0)) && sqrt_n(0.0) == 0.0 && sqrt_n(inf) == inf &&
                         std::isnan(sqrt_n(-1.0)) && std::isnan(sqrt_n(NAN));
    std::printf("{\"sixth\": %.4f, \"sqrt\": %.4f, \"rsq\": %.4f, \"cbrt\": %.4f, \"sqrt_n\": %.4f, \"div_n\": %.4f, "
                "\"special\": %d}\n", sixth, sq, rs, cb, sn, dv, (int)special);
}
"""


@pytest.fixture(scope="module")
def errors(tmp_path_factory):
    d = tmp_path_factory.mktemp("fastmath")
    src, exe = str(d / "t.cpp"), str(d / "t")
    with open(src, "w") as f:
        f.write(SRC)
    subprocess.run(["g++", "-O2", "-std=c++17", "-ffp-contract=off", "-D__HIP_PLATFORM_AMD__", "-I/opt/rocm/include",
                    "-I" + os.path.join(ROOT, "dftpy_amd", "csrc"), src, "-o", exe], check=True, capture_output=True)
    return json.loads(subprocess.run([exe], check=True, capture_output=True, text=True).stdout)


# ulps: the final correction's rounding (1/2), for the cube root and the
# reciprocal root also that of the product it corrects by (1/3 and 1/2 of an
# ulp of it), for the inverse sixth root the last step's (0.9)
@pytest.mark.parametrize("name,most", [("sixth", 0.95), ("sqrt", 0.51), ("rsq", 1.01), ("cbrt", 0.84), ("sqrt_n", 0.51),
                                       ("div_n", 0.51)])
def test_largest_error(errors, name, most):
    assert 0.0 < errors[name] <= most


def test_special_values(errors):
    assert errors["special"] == 1
