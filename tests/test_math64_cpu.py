"""CPU check of the FP64 elementary functions of the FP64 kernels (rb_math64.h), compiled for the
host, against long double: 2^(y/32), -2 ln u, and Box-Muller on edge and random words.

Bounds, in units of eps = 2^-52: exp2 rounds a table entry (1/2), a product folded into one FMA
(1/2) and carries a fit error of 0.4, so 1.5 eps bounds it; the logarithm adds a table term and a
polynomial (two roundings of terms not larger than twice the result), 2 eps; the normals relative to
their radius add a square root, a product and a polynomial of one rounding each, 3 eps.  A payoff is a
sum of S', K and two tails, each rounded a few times: 8 eps of S' + K (to first order it does not
depend on the rounding of d1, since S' phi(d1) = K phi(d2)); zero variance gives the intrinsic value,
and NaN at the money as 0 / 0 does."""
import os
import shutil
import subprocess

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
CSRC = os.path.join(HERE, "..", "rbergomi_amd", "csrc")

SRC = r"""
#include <cmath>
#include <cstdio>
#include <random>
#include "rb_math64.h"
using namespace rb;
int main() {
    std::mt19937_64 g(1);
    double2 lg[LOG_N];
    for (int i = 0; i < LOG_N; ++i) lg[i] = make_double2(LOG_TAB[2 * i], LOG_TAB[2 * i + 1]);
    long double e_exp = 0, e_log = 0, e_bm = 0;
    for (int i = 0; i < 500000; ++i) {
        const double y = (double(g() >> 11) * 0x1p-53 - 0.5) * (i & 1 ? 64.0 : 60000.0);
        const long double want = exp2l((long double)y / 32);
        e_exp = fmaxl(e_exp, fabsl(exp2_32(EXP2_TAB, y) - want) / want);
    }
    for (int i = 0; i < 500000; ++i) {
        // both ends of the range, powers of two and their neighbours, random words
        const uint32_t r = uint32_t(g());
        const uint32_t x = i < 5000 ? uint32_t(i) : i < 10000 ? ~uint32_t(i - 5000)
                         : i < 10100 ? (1u << (i % 32)) + uint32_t(i / 32 % 3) - 1u
                         : i < 200000 ? r >> (i % 32) : i < 300000 ? ~(r >> (i % 32)) : r;
        const uint32_t x1 = i < 10100 ? x * 2654435761u : i < 20000 ? uint32_t(i % 8) << 29 : uint32_t(g());
        const long double w = -2 * logl(((long double)x + 0.5L) * 0x1p-32L);
        e_log = fmaxl(e_log, fabsl(neg2_log_u32(lg, x) - w) / w);
        double z0, z1;
        box_muller_f64(lg, x, x1, z0, z1);
        const long double th = 2 * acosl(-1.0L) * (((long double)x1 + 0.5L) * 0x1p-32L), rad = sqrtl(w);
        e_bm = fmaxl(e_bm, fmaxl(fabsl(z0 - rad * cosl(th)), fabsl(z1 - rad * sinl(th))) / rad);
    }
    long double e_pay = 0;
    for (int i = 0; i < 300000; ++i) {
        auto u = [&] { return double(g() >> 11) * 0x1p-53; };
        PathRt64 q;
        q.lnS = (u() - 0.5) * (i & 1 ? 0.6 : 6.0);
        q.sig = i % 3 ? exp(-9.0 * u()) * 1.5 : 0.05 + u();
        q.S = exp(q.lnS);
        q.isig = 1.0 / q.sig;
        const double K = exp((u() - 0.5) * 1.5), lnK = log(K);
        const long double S = expl((long double)q.lnS), d1 = ((long double)q.lnS - logl(K)) / q.sig + q.sig / 2.0L, d2 = d1 - q.sig;
        const long double want = 0.5L * (S * erfcl(-d1 * sqrtl(0.5L)) - K * erfcl(-d2 * sqrtl(0.5L)));
        e_pay = fmaxl(e_pay, fabsl(rt_payoff64(EXP2_TAB, q, K, lnK) - want) / (S + K));
    }
    auto at = [](double lnS, double K) {
        PathRt64 q{lnS, exp(lnS), 0.0, INFINITY};
        return rt_payoff64(EXP2_TAB, q, K, log(K));
    };
    std::printf("%.4Lf %.4Lf %.4Lf %.4Lf\n", e_exp / 0x1p-52L, e_log / 0x1p-52L, e_bm / 0x1p-52L, e_pay / 0x1p-52L);
    std::printf("%.17g %.17g %.17g\n", at(0.0, 0.5), at(0.0, 2.0), at(0.0, 1.0));
    std::printf("%.17g %.17g %.17g %.17g\n", exp2_32(EXP2_TAB, 1e300), exp2_32(EXP2_TAB, -1e300), exp2_32(EXP2_TAB, 0.0),
                exp2_32(EXP2_TAB, 32.0 * 1023));
    return 0;
}
"""


def _hipcc():
    for c in ("/opt/rocm/bin/hipcc", shutil.which("hipcc")):
        if c and os.path.exists(c):
            return c
    return None


def test_elementary_functions(tmp_path):
    hipcc = _hipcc()
    if hipcc is None:
        pytest.skip("hipcc not available")
    src = tmp_path / "math64.cpp"
    src.write_text(SRC)
    exe = str(tmp_path / "math64")
    r = subprocess.run([hipcc, "-O1", "-std=c++17", "-ffp-contract=off", "-x", "hip", "--cuda-host-only", "-I" + CSRC, str(src),
                        "-o", exe], capture_output=True, text=True, timeout=600)
    assert r.returncode == 0, r.stderr[-3000:]
    out = subprocess.run([exe], capture_output=True, text=True, timeout=600)
    assert out.returncode == 0
    first, zero, second = out.stdout.strip().splitlines()
    e_exp, e_log, e_bm, e_pay = (float(x) for x in first.split())
    assert e_exp < 1.5 and e_log < 2.0 and e_bm < 3.0 and e_pay < 8.0, first
    inside, outside, at_money = (float(x) for x in zero.split())
    assert (inside, outside) == (0.5, 0.0) and at_money != at_money
    assert [float(x) for x in second.split()] == [float("inf"), 0.0, 1.0, float(2 ** 1023)]
