"""The device's own forms of the FP64 elementary functions (rb_math64.h refines v_rsq_f64 and v_rcp_f64 where the host
compiles the library's root and division), against long double.

Bounds in eps = 2^-52.  Normals: 3 eps of their radius, as on the host (a logarithm to 2 eps under the root, the
root, a polynomial and two products).  Payoffs of one step (N = 1: Iv = T xi, Is = sqrt(T xi) W1, three roundings each):
8 eps of S' + K for the payoff of given fields, and with |ln S'| and sigma below 1 another 4.5 eps of S' from ln S'
and 1 from sigma: 14 eps."""
import ctypes
import subprocess

import numpy as np
import pytest

pytestmark = pytest.mark.gpu
EPS = 2.0 ** -52


@pytest.fixture(scope="module")
def rb():
    import rbergomi_amd
    return rbergomi_amd


def test_normals(rb, orc):
    seed, np_, N = [2024, 7], 30000, 8
    L = rb.load()
    out = np.zeros((np_, 1, N))
    s = np.array(seed, dtype=np.uint64)
    assert L.rb_probe_normals(s.ctypes.data_as(ctypes.POINTER(ctypes.c_uint64)), 2, 0, np_, 1, N,
                              out.ctypes.data_as(ctypes.POINTER(ctypes.c_double))) == 0
    ctr = np.zeros((np_, N // 4, 4), dtype=np.uint32)
    ctr[..., 0] = np.arange(N // 4)
    ctr[..., 1] = np.arange(np_)[:, None]
    words = np.zeros_like(ctr)
    u32 = ctypes.POINTER(ctypes.c_uint32)
    key = orc.philox_key(seed)
    assert L.rb_probe_philox(np.ascontiguousarray(ctr).ctypes.data_as(u32), key.ctypes.data_as(u32), ctr.size // 4,
                             words.ctypes.data_as(u32)) == 0
    u = (words.astype(np.longdouble) + np.longdouble(0.5)) * np.longdouble(2.0) ** -32
    r, th = np.sqrt(-2 * np.log(u[..., 0::2])), 2 * np.arccos(np.longdouble(-1)) * u[..., 1::2]
    ref = np.stack([r * np.cos(th), r * np.sin(th)], axis=-1).reshape(np_, N)
    rad = np.repeat(r.reshape(np_, N // 2), 2, axis=1)
    assert float(np.max(np.abs(out[:, 0] - ref) / rad)) < 3 * EPS


SRC = r"""
#include <math.h>
extern "C" void payoffs(long n, const double* W, int m, const double* K, double xi, double T, double rho, double* out, double* scale) {
    for (long p = 0; p < n; ++p)
        for (int k = 0; k < m; ++k) {
            const long double Iv = (long double)T * xi, Is = sqrtl(Iv) * W[p];
            const long double r = rho, sig = sqrtl((1 - r * r) * Iv), lnS = -0.5L * r * r * Iv + r * Is, S = expl(lnS);
            const long double d1 = (lnS - logl((long double)K[k])) / sig + 0.5L * sig, d2 = d1 - sig, c = sqrtl(0.5L);
            const long double v = 0.5L * (S * erfcl(-d1 * c) - K[k] * erfcl(-d2 * c));
            out[p * m + k] = fabsl(out[p * m + k] - v);
            scale[p * m + k] = S + K[k];
        }
}
"""


@pytest.mark.parametrize("xi,T,rho", [(0.04, 1.0, -0.7), (0.01, 0.1, -0.95), (0.3, 2.0, 0.3)])
def test_payoffs(rb, tmp_path, xi, T, rho):
    (tmp_path / "p.cpp").write_text(SRC)
    lib = str(tmp_path / "p.so")
    subprocess.check_call(["g++", "-O2", "-shared", "-fPIC", str(tmp_path / "p.cpp"), "-o", lib])
    f = ctypes.CDLL(lib).payoffs
    d, dp = ctypes.c_double, ctypes.POINTER(ctypes.c_double)
    f.argtypes = [ctypes.c_long, dp, ctypes.c_int, dp, d, d, d, dp, dp]
    W = np.random.default_rng(5).standard_normal(20000)
    lim = 0.95 / (abs(rho) * np.sqrt(xi * T))
    W = np.clip(W, -lim, lim)
    K = np.exp(np.linspace(-4.0, 4.0, 33) * np.sqrt(xi * T))
    Z = np.zeros((len(W), 2, 1))
    Z[:, 0, 0] = W
    got, _, _ = rb.payoff_samples_v2(xi, [0.1], [1.0], [rho], np.full(33, T), K, 1, Z)
    got = np.ascontiguousarray(got)
    scale = np.zeros_like(got)
    P = lambda a: a.ctypes.data_as(dp)
    f(len(W), P(W), 33, P(K), xi, T, rho, P(got), P(scale))
    assert np.max(got / scale) < 14 * EPS
