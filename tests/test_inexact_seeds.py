"""The k-th roots from FP32 seeds (jellyfysh_amd/csrc/ecmc_math.h) with seeds as far off as the kernels'
hardware seeds may be, 2^-20 of max(|log2 x|, 1), 2^-20 of 2^y and 2^-46 of 1/x with every combination of
signs: the error still stays below what the rounding tests assume, to the ends of the range."""
import os
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

PROGRAM = r"""
#define ECMC_HOST_BUILD 1
#define ECMC_HOST_SEEDS 1
#include <math.h>
#include <stdio.h>
#include <stdlib.h>
#include <quadmath.h>
namespace ecmc {
static double off[3];
static float seed_log2(double x) { double l = log2(x); return (float)(l + off[0] * 0x1p-20 * fmax(fabs(l), 1.0)); }
static float seed_exp2(float y) { return (float)(exp2((double)y) * (1.0 + off[1] * 0x1p-20)); }
static double seed_rcp(double x) { return (1.0 / x) * (1.0 + off[2] * 0x1p-46); }
}
#include "ecmc_math.h"
using namespace ecmc;
static unsigned long long st = 88172645463325252ull;
static double unif() {
    st ^= st << 13; st ^= st >> 7; st ^= st << 17;
    return (double)(st >> 11) * 0x1p-53;
}
int main(int argc, char **argv) {
    const int p = atoi(argv[1]);
    const double range = atof(argv[2]), y = 2.0 / p;
    const int num = (p & 1) ? 2 : 1, den = (p & 1) ? p : p / 2;
    __float128 worst = 0;
    for (int signs = 0; signs < 8; signs++) {
        for (int k = 0; k < 3; k++) off[k] = (signs >> k) & 1 ? 1.0 : -1.0;
        for (long i = 0; i < 30000; i++) {
            double x = exp2((2 * unif() - 1) * range);
            if (i < 200) x = exp2((i & 1 ? 1 : -1) * (range - 1e-3 * i));
            double lo, hi = (p == 6 || p == 12) ? root36_seeded(x, p == 12, lo) : rational_pow_seeded(x, y, num, den, lo);
            __float128 t = powq((__float128)x, (__float128)y), e = fabsq(((__float128)hi + lo - t) / t);
            if (e > worst) worst = e;
        }
    }
    printf("%.3f\n", (double)log2q(worst));
    return 0;
}
"""


@pytest.mark.parametrize("power,reach,assumed", [(6, 100, 68), (12, 100, 68), (3, 60, 66), (5, 60, 66), (9, 60, 66), (31, 60, 66)])
def test_roots_from_inexact_seeds(tmp_path, power, reach, assumed):
    gxx = shutil.which("g++")
    if gxx is None:
        pytest.skip("needs g++")
    src, exe = tmp_path / "seeds.cpp", tmp_path / "seeds"
    src.write_text(PROGRAM)
    subprocess.run([gxx, "-O2", "-std=c++17", "-ffp-contract=off", "-I", os.path.join(ROOT, "jellyfysh_amd", "csrc"),
                    str(src), "-o", str(exe), "-lquadmath"], check=True, capture_output=True)
    worst = float(subprocess.run([str(exe), str(power), str(reach)], capture_output=True, text=True, check=True).stdout)
    print(worst)
    assert worst < -assumed
