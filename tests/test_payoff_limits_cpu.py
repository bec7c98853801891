"""The FP64 Romano-Touzi payoff (rb_math64.h, compiled for the host) where its fields leave the range of double:
the limit of S' Phi(d1) - K Phi(d2) for integrals as a caller's Gaussians can make them."""
import os
import subprocess

import pytest

from test_math64_cpu import CSRC, _hipcc

SRC = r"""
#include <cmath>
#include <cstdio>
#include "rb_math64.h"
using namespace rb;
int main() {
    const double rho = -0.5;
    // ln S' = -Iv / 8 - Is / 2
    const double cases[][2] = {{0.04, -1400.0}, {0.04, -1419.6}, {0.04, -2000.0}, {900.0, -2000.0}, {0.0, -2000.0}, {1e6, -1e6},
                               {0.04, -INFINITY}, {0.04, INFINITY}, {0.04, 2000.0}, {1e5, 0.0}, {0.04, NAN}};
    for (const auto& c : cases) {
        const PathRt64 q = path_rt64(c[0], c[1], rho);
        for (double K : {0.5, 1.0, 2.0}) std::printf("%.17g ", rt_payoff64(EXP2_TAB, q, K, log(K)));
    }
    return 0;
}
"""


def test_limits_of_the_payoff(tmp_path):
    hipcc = _hipcc()
    if hipcc is None:
        pytest.skip("hipcc not available")
    (tmp_path / "limits.cpp").write_text(SRC)
    exe = str(tmp_path / "limits")
    r = subprocess.run([hipcc, "-O1", "-std=c++17", "-ffp-contract=off", "-x", "hip", "--cuda-host-only", "-I" + CSRC,
                        str(tmp_path / "limits.cpp"), "-o", exe], capture_output=True, text=True, timeout=600)
    assert r.returncode == 0, r.stderr[-3000:]
    v = [float(x) for x in subprocess.run([exe], capture_output=True, text=True, timeout=60).stdout.split()]
    got = [v[i:i + 3] for i in range(0, len(v), 3)]
    inf = float("inf")
    import math
    for row, lnS in zip(got[:2], (699.995, 709.795)):
        # exp(709.795) is above the largest double
        want = math.exp(lnS) if lnS < 709.78 else inf
        assert all(x == want or abs(x / want - 1) < 1e-12 for x in row), row
    for row in got[2:5]:
        assert row == [inf] * 3, row
    # deep in the variance: S' = exp(-1.25e5 + 5e5) is infinite with d1 = ln S' / sig + sig / 2
    assert got[5] == [inf] * 3
    assert got[6] == [inf] * 3
    for row in got[7:9]:
        assert row == [0.0] * 3, row
    assert all(x == 0.0 for x in got[9])  # S' = exp(-12500) = 0
    assert all(math.isnan(x) for x in got[10])
