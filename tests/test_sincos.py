"""The f64 sine and cosine of the Helmholtz pair kernel (fmm_amd/csrc/sincos.hpp), compiled for
the host, against long double: within 0.85 ulp and 0.295 ulp rms over the phases k r of leaf
pairs, as precise as a good math library's (two roundings: 0.5 ulp for the last sum and what the
reduced argument and the polynomial's terms leave; rms 0.289 is the last rounding alone)."""
import os
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

SOURCE = r"""
#include <algorithm>
#include <cmath>
#include <cstdio>
#include <random>
#include "sincos.hpp"
int main() {
  std::mt19937_64 gen(7);
  for (double top : {0.7, 6.0, 60.0, 600.0, 1.0e6}) {
    std::uniform_real_distribution<double> u(-top, top);
    double most = 0.0, sum = 0.0;
    const int n = 400000;
    for (int i = 0; i < n; ++i) {
      const double x = u(gen);
      double v[2];
      fmmh::dev::sincos_f64(x, &v[0], &v[1]);
      const long double want[2] = {sinl(x), cosl(x)};
      for (int k = 0; k < 2; ++k) {
        int e;
        std::frexp(double(want[k]), &e);
        const double err = double(fabsl(v[k] - want[k]) / ldexpl(1.0L, e - 53));
        most = std::max(most, err);
        sum += err * err;
      }
    }
    double s, c;
    fmmh::dev::sincos_f64(0.0, &s, &c);
    std::printf("%g %.4f %.4f %d\n", top, most, std::sqrt(sum / (2 * n)), s == 0.0 && c == 1.0);
  }
}
"""


def test_sine_and_cosine_of_the_pair_kernel(tmp_path):
    if shutil.which("g++") is None:
        pytest.skip("no g++")
    src = tmp_path / "t.cpp"
    src.write_text(SOURCE)
    exe = tmp_path / "t"
    subprocess.run(["g++", "-std=c++17", "-O2", "-ffp-contract=off", "-D__HIP_PLATFORM_AMD__",
                    "-I" + os.path.join(ROOT, "fmm_amd", "csrc"), "-isystem/opt/rocm/include", str(src), "-o",
                    str(exe)], check=True)
    rows = [line.split() for line in subprocess.run([str(exe)], capture_output=True, text=True,
                                                    check=True).stdout.splitlines()]
    assert len(rows) == 5
    for top, most, rms, zero in rows:
        print(f"|x| < {top}: {most} ulp, rms {rms}")
        assert float(most) < 0.85 and float(rms) < 0.295 and zero == "1"
