"""The FP64 functions of mdg_math64.h on the CPU: the header compiled for the host,
the hardware's estimates stood in for by values up to 2^-23 off, against 113-bit
results."""
import os
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

PRELUDE = r"""
#include <cmath>
#include <cstdint>
#include <cstdio>
#include <cstring>
#include <quadmath.h>
typedef __float128 quad;
static uint64_t g_seed = 88172645463325252ull;
static uint64_t rnd() { g_seed ^= g_seed << 13; g_seed ^= g_seed >> 7; return g_seed ^= g_seed << 17; }
static double uni() { return (double)(rnd() >> 11) / 9007199254740992.0; }
// an estimate: relative error up to 2^-23 either way
static double off(double v) { return v * (1.0 + (2.0 * uni() - 1.0) / 8388608.0); }
#define __device__
#define __forceinline__ inline
#define __builtin_amdgcn_rcp(x) off(1.0 / (x))
#define __builtin_amdgcn_rsq(x) off(1.0 / std::sqrt(x))
#include "mdg_math64.h"
static double ulp(double v) { int e; std::frexp(v, &e); return std::ldexp(1.0, e - 53); }
"""


@pytest.fixture(scope="module")
def run(tmp_path_factory):
    d = tmp_path_factory.mktemp("math64")
    (d / "hip").mkdir()
    (d / "hip" / "hip_runtime.h").write_text("")

    def go(name, body):
        src, exe = d / (name + ".cpp"), d / name
        src.write_text(PRELUDE + "int main()\n{\n" + body + "\n}\n")
        subprocess.run(["g++", "-std=gnu++17", "-O2", "-mfma", "-ffp-contract=off", "-I" + str(d),
                        "-I" + os.path.join(ROOT, "mdbas_amd", "csrc"), "-o", str(exe), str(src),
                        "-lquadmath"], check=True)
        out = subprocess.run([str(exe)], check=True, capture_output=True, text=True, timeout=100)
        return [float(v) for v in out.stdout.split()]

    return go


def test_erfc_coefficients(run):
    """The table against its definition (1 + 2x) exp(x^2) erfc(x), over x in [0, 6]
    and on to where erfc leaves the doubles: truncation of 8e-17 and the rounding of
    the coefficients, of which the largest alone gives 1.1e-16 of 1 or less."""
    worst, = run("coef", r"""
    quad w = 0;
    for (int i = 0; i <= 26000; i++) {
        const quad x = (quad)i / 1000, y = (x - 3.75Q) / (x + 3.75Q);
        quad p = mdg_erfcx_c[MDG_ERFCX_N - 1];
        for (int k = MDG_ERFCX_N - 2; k >= 0; k--) p = p * y + mdg_erfcx_c[k];
        const quad f = (1 + 2 * x) * expq(x * x) * erfcq(x);
        const quad e = fabsq(p / f - 1);
        if (e > w) w = e;
    }
    printf("%.4g\n", (double)w);""")
    print("table", worst)
    assert worst < 2e-16


def test_erfc_and_gaussian(run):
    """mdg_erfc64 over x in [0, 6], as its comment states: within 4.2e-16 (rms
    1.1e-16), the Gaussian within 2.2e-16."""
    e, rms, z = run("erfc", r"""
    quad we = 0, wz = 0;
    double s = 0;
    const int n = 600000;
    for (int i = 0; i <= n; i++) {
        const double x = 6.0 * (i + (i < n ? uni() : 0.0)) / n;
        double ez;
        const double g = mdg_erfc64(x, ez);
        const quad f = erfcq(x), h = expq(-(quad)x * x);
        const quad e = fabsq((g - f) / f), z = fabsq((ez - h) / h);
        if (e > we) we = e;
        if (z > wz) wz = z;
        s += (double)(e * e);
    }
    printf("%.4g %.4g %.4g\n", (double)we, sqrt(s / n), (double)wz);""")
    print("erfc", e, "rms", rms, "gaussian", z)
    assert e < 4.3e-16 and rms < 1.2e-16 and z < 2.3e-16


def test_reciprocal_and_root(run):
    """mdg_rcp64 within 0.51 ulp, mdg_rsqrt64 within an ulp, its square root within
    0.51 ulp (all in units of the result's last place)."""
    a, b, c = run("rcp", r"""
    quad w[3] = {0, 0, 0};
    for (int i = 0; i < 2000000; i++) {
        const double x = std::ldexp(1.0 + uni(), (int)(rnd() % 200) - 100);
        double r;
        const double v[3] = {mdg_rcp64(x), mdg_rsqrt64(x, r), 0};
        const quad f[3] = {1 / (quad)x, 1 / sqrtq(x), sqrtq(x)};
        for (int k = 0; k < 3; k++) {
            const quad e = fabsq((k == 2 ? r : v[k]) - f[k]) / ulp((double)f[k]);
            if (e > w[k]) w[k] = e;
        }
    }
    printf("%.4g %.4g %.4g\n", (double)w[0], (double)w[1], (double)w[2]);""")
    print("ulps: rcp", a, "rsqrt", b, "sqrt", c)
    assert a < 0.51 and b < 1.0 and c < 0.51


def test_division(run):
    """mdg_div64 is IEEE division for random operands, and where the quotient lies
    next to a midpoint of two doubles (a rounding of the dividend off it) never more
    than one double from it."""
    bad, near, far = run("div", r"""
    int bad = 0, near = 0, far = 0;
    for (int i = 0; i < 4000000; i++) {
        const double a = std::ldexp(1.0 + uni(), (int)(rnd() % 60) - 30) * (rnd() & 1 ? 1 : -1);
        const double b = std::ldexp(1.0 + uni(), (int)(rnd() % 60) - 30) * (rnd() & 1 ? 1 : -1);
        bad += mdg_div64(a, b) != a / b;
    }
    for (int i = 0; i < 1000000; i++) {
        // a: the double nearest to a midpoint (54 bits, the last one set) times b
        const double b = 1.0 + uni();
        const quad m = 1 + ((quad)(rnd() >> 12) + 0.5Q) / 4503599627370496.0Q;
        const double a = (double)(m * (quad)b);
        const double q = mdg_div64(a, b), t = a / b;
        near += q != t;
        far += std::fabs(q - t) > ulp(t);
    }
    printf("%d %d %d\n", bad, near, far);""")
    print("division: random", bad, "next to a midpoint", near, "further off", far)
    assert bad == 0 and far == 0
