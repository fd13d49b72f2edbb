"""exact_div.hpp (the transforms' normalisation and the RK3 stage's thirds)
against the division, bit for bit, on the host."""
import os
import subprocess

from spectral2d_amd import build

PROGRAM = r"""
#include "exact_div.hpp"
#include <cmath>
#include <cstdint>
#include <cstdio>
#include <cstring>
#include <limits>
#include <vector>

template <typename T, typename U>
static bool same(T a, T b)
{
    U x, y;
    std::memcpy(&x, &a, sizeof a);
    std::memcpy(&y, &b, sizeof b);
    return x == y || (a != a && b != b);
}

static uint64_t rng = 88172645463325252ull;
static uint64_t next() { return rng ^= rng << 13, rng ^= rng >> 7, rng ^= rng << 17; }

template <typename T>
static std::vector<T> values(int emin, int emax)
{
    using L = std::numeric_limits<T>;
    std::vector<T> v = {0, 1, 2, 3, (T)(1.0 / 3), L::denorm_min(), 3 * L::denorm_min(), L::min(),
                        L::max(), L::infinity(), L::quiet_NaN(), (T)1e-37, (T)1e37};
    if (sizeof(T) == 8) for (double x : {1e-281, 1e-280, 1e-279, 1e299, 1e300, 1e301}) v.push_back((T)x);
    for (int k = 0; k < 200000; ++k)
        v.push_back((T)std::ldexp(1.0 + (double)(next() >> 12) / 4503599627370496.0,
                                  emin + (int)(next() % (uint64_t)(emax - emin))));
    for (size_t k = 0, n = v.size(); k < n; ++k) v.push_back(-v[k]);
    return v;
}

int main()
{
    int bad = 0;
    auto check = [&](const char *what, double x, double d, bool ok) {
        if (!ok && ++bad < 20) std::printf("%s(%a, %g)\n", what, x, d);
    };
    const double side[] = {48, 72, 96, 144, 288, 576, 1152, 1536, 2304, 3072};
    std::vector<double> v = values<double>(-1074, 1023);
    for (double nx : side)
        for (double ny : side) {
            const double d = nx * ny, r = 1.0 / d;
            for (size_t k = 0; k < v.size(); k += nx == ny ? 1 : 7) {
                bool odd = false;
                double y = s2d::div_by(v[k], d, r, &odd);
                if (odd) y = v[k] / d;
                check("div_by", v[k], d, same<double, uint64_t>(y, v[k] / d));
            }
        }
    for (double x : v) check("div3_any", x, 3, same<double, uint64_t>(s2d::div3_any(x), x / 3.0));
    for (float x : values<float>(-149, 127))
        check("div3_any float", x, 3, same<float, uint32_t>(s2d::div3_any(x), x / 3.0f));
    std::printf("%d wrong\n", bad);
    return bad != 0;
}
"""


def test_equals_division(tmp_path):
    src, exe = tmp_path / "exact_div.hip", tmp_path / "exact_div"
    src.write_text(PROGRAM)
    flags = [f for f in build.HIPCC_FLAGS if f not in ("-shared", "-fPIC")]
    r = subprocess.run([build.hipcc(), *flags, str(src), "-o", str(exe)], capture_output=True,
                       text=True)
    assert r.returncode == 0, r.stdout + r.stderr
    env = dict(os.environ, LD_LIBRARY_PATH="")
    r = subprocess.run([str(exe)], capture_output=True, text=True, env=env)
    assert r.returncode == 0, r.stdout
