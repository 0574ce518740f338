"""The exponential of the attention softmax (zl_exp.h, the same arithmetic on host and device) against the 64-bit mantissa
exponential of the C library."""
import os
import shutil
import subprocess

import pytest

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "zerollm_amd", "csrc")

PROGRAM = r"""
#include <cstdio>
#include <cstdint>
#include <cstring>
#include <limits>
#include "zl_exp.h"
int main() {
  double worst = 0, sub = 0;  // in ulps of the exact value, normal and subnormal results
  uint64_t z = 1;
  for (int i = 0; i < 4000000; i++) {
    z = z * 6364136223846793005ull + 1442695040888963407ull;
    const double u = (double)(z >> 11) * 0x1p-53;
    // differences of float32 scores: small ones, ordinary ones, down to underflow; and next to multiples of ln 2
    double x = i % 4 == 0 ? -u : i % 4 == 1 ? -20 * u : i % 4 == 2 ? -745 * u : -0.6931471805599453 * (double)(int)(700 * u) - 1e-9 * u;
    if (i % 8 == 0) x = (double)(float)x;
    const long double want = expl((long double)x);
    const double got = zl::exp_neg(x), w = (double)want;
    const bool normal = w >= std::numeric_limits<double>::min();
    const long double ulp = normal ? (long double)(nextafter(w, 2 * w) - w) : 0x1p-1074L;
    const double e = (double)(fabsl((long double)got - want) / ulp);
    double &m = normal ? worst : sub;
    if (!(e <= m)) m = e;
  }
  const double nan = std::numeric_limits<double>::quiet_NaN(), inf = std::numeric_limits<double>::infinity();
  const bool special = zl::exp_neg(0.0) == 1.0 && zl::exp_neg(-0.0) == 1.0 && zl::exp_neg(-inf) == 0.0 && zl::exp_neg(-1e300) == 0.0 &&
                       zl::exp_neg(-746.0) == 0.0 && zl::exp_neg(nan) != zl::exp_neg(nan);
  printf("%.4f %.4f %d\n", worst, sub, special);
}
"""


@pytest.mark.skipif(shutil.which("g++") is None, reason="needs a host compiler")
def test_within_an_ulp_of_the_exact_value(tmp_path):
    src, exe = tmp_path / "e.cpp", tmp_path / "e"
    src.write_text(PROGRAM)
    subprocess.run(["g++", "-O2", "-std=c++17", "-ffp-contract=off", "-I", CSRC, str(src), "-o", str(exe)], check=True)
    worst, sub, special = subprocess.run([str(exe)], check=True, capture_output=True, text=True).stdout.split()
    print(f"largest error {worst} ulp, of subnormal results {sub}")
    # the polynomial's last step rounds once (half an ulp), its steps before and the two roundings of r add less than that
    assert float(worst) < 1.0 and float(sub) <= 1.0 and special == "1"
