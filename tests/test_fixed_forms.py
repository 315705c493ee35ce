"""The device forms of the Fixed products and quotient (ft_device.h) against
their 64-bit statements, on the host: whole-number results, so equality."""
import os
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

SRC = r'''
#include <cstdio>
#include <cstdlib>
#include "ft_device.h"
using namespace ft;
static uint64_t s = SEED;
static uint64_t rnd() { s += 0x9E3779B97F4A7C15ull; uint64_t z = s; z = (z ^ (z >> 30)) * 0xBF58476D1CE4E5B9ull;
                        z = (z ^ (z >> 27)) * 0x94D049BB133111EBull; return z ^ (z >> 31); }
static int32_t any() {  // all magnitudes, and the ends
    const int k = (int)(rnd() % 34);
    if (k == 32) return (int32_t)0x80000000;
    if (k == 33) return 0x7FFFFFFF;
    const int32_t v = (int32_t)((uint32_t)rnd() >> k);
    return rnd() & 1 ? v : (int32_t)(0u - (uint32_t)v);
}
static int32_t unit() { const uint64_t r = rnd(); return r % 8 == 0 ? FX_ONE : (r % 8 == 1 ? 0 : (int32_t)((r >> 8) % (FX_ONE + 1))); }
static int bad(const char *w, long a, long b, long got, long want) { printf("%s(%ld, %ld) = %ld, not %ld\n", w, a, b, got, want); return 1; }
int main() {
    for (int i = 0; i < 3000000; ++i) {
        const int32_t a = any(), u = unit(), v = unit();
        if (fx_mul_frac(a, u) != fx_mul(a, u)) return bad("fx_mul_frac", a, u, fx_mul_frac(a, u), fx_mul(a, u));
        if (fx_mul_unit(u, v) != fx_mul(u, v)) return bad("fx_mul_unit", u, v, fx_mul_unit(u, v), fx_mul(u, v));
        int32_t d = any();
        if (!d) d = 1;
        if (i % 5 == 0 && a != INT32_MIN) {  // quotients next to a whole number
            const int64_t q = (int64_t)a * 65536 / d;
            if (q) d = (int32_t)((int64_t)a * 65536 / q);
            if (!d) d = 1;
        }
        const double n = fabs((double)a) * 65536.0, dd = fabs((double)d);
        const double rel[5] = {0.0, 0x1p-49, -0x1p-49, 0x1p-52, -0x1p-52};  // the reciprocal's error bound, both ways
        for (double e : rel) {
            const int32_t got = fx_div_from(n, dd, (1.0 / dd) * (1.0 + e), (a < 0) != (d < 0));
            if (got != fx_div(a, d)) return bad("fx_div_from", a, d, got, fx_div(a, d));
        }
    }
    return 0;
}
'''


@pytest.mark.parametrize("seed", [1, 2])
def test_fixed_forms(tmp_path, seed):
    src, exe = tmp_path / "f.cpp", tmp_path / "f"
    src.write_text(SRC)
    subprocess.run(["g++", "-O2", "-std=c++17", "-ffp-contract=off", "-march=native", f"-DSEED={seed}ull",
                    f"-I{os.path.join(ROOT, 'footile_amd', 'csrc')}", "-o", str(exe), str(src)], check=True)
    r = subprocess.run([str(exe)], stdout=subprocess.PIPE, text=True)
    assert r.returncode == 0, r.stdout
