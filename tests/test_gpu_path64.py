"""The single-pass FP64 path kernels (k_path64, k_path64_fft) at the edges of its tiles and dispatch, against the
oracle on the same Gaussians: row blocks of 16 (N = 16 k, 16 k + 1, 16 k + 2), the sub-tile counts
(N <= 17, <= 33, above), tiles with absent paths, groups beyond one job (2, 4, 8 per job), many units
with the paths' second stream kept in LDS or not, and both workgroup sizes; for the transform
kernel (N > 384) both ends of every transform length, an odd number of paths and absent pairs.

Tolerances are the FP64 path's: integrals 1e-10 relative with a floor of 1e-3, prices and standard
errors 1e-12 absolute."""
import ctypes

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def rb():
    import rbergomi_amd
    return rbergomi_amd


@pytest.fixture(scope="module")
def orc():
    from oracle import pyoracle
    return pyoracle


def _params(units, mats, seed):
    rng = np.random.default_rng(seed)
    H = rng.uniform(0.03, 0.45, units)
    return H, rng.uniform(0.5, 2.5, units), rng.uniform(-0.95, -0.2, units), np.linspace(0.1, 1.5, mats), \
        rng.uniform(0.8, 1.2, mats)


EDGES = [(1, 3), (2, 64), (16, 65), (17, 70), (18, 33), (33, 40), (34, 17), (64, 16), (65, 15), (113, 20), (129, 1),
         (241, 18), (257, 16), (304, 17), (384, 33), (385, 9), (512, 8), (513, 5), (1024, 3), (1025, 1), (2048, 3),
         (2049, 2), (4095, 1), (4096, 3)]


@pytest.mark.parametrize("N,M", EDGES)
def test_integrals_at_tile_edges(rb, orc, N, M):
    print("path64 integrals N=%d M=%d" % (N, M), flush=True)
    xi, (H, eta, rho, T, K) = 0.05, _params(2, 3, N)
    Z = np.random.default_rng(N + 1).standard_normal((M, 2, N))
    dp = ctypes.POINTER(ctypes.c_double)
    a = [np.ascontiguousarray(v) for v in (H, eta, rho, T, K)]
    P = [v.ctypes.data_as(dp) for v in a]
    out = np.zeros((M, 6, 2))
    L = rb.load()
    rc = L.rb_probe_integrals(xi, P[0], P[1], P[2], 2, P[3], P[4], 3, N, M, Z.ctypes.data_as(dp), None,
                              out.ctypes.data_as(dp))
    assert rc == 0, L.rb_last_error()
    ref = orc.integrals_rt_samples(xi, H, eta, rho, T, K, N, Z)
    assert np.max(np.abs(out - ref) / np.maximum(np.abs(ref), 1e-3)) < 1e-10


# (units, maturities, N): groups per job 2, 4 and 8 with remainders; units with W1perp in LDS
# (N = 100, 200) and drawn again (N = 400); 512 threads with and without it
SHAPES = [(1, 1, 100), (1, 3, 300), (1, 5, 100), (1, 9, 260), (1, 17, 64), (3, 2, 100), (5, 1, 200), (4, 3, 400),
          (2, 9, 30), (70, 1, 48),
          (1, 1, 500), (3, 2, 385), (1, 9, 1000), (2, 2, 1500), (5, 1, 4000)]


@pytest.mark.parametrize("method", [0, 1])
@pytest.mark.parametrize("units,mats,N", SHAPES)
def test_seeded_prices_match_oracle(rb, orc, units, mats, N, method):
    print("path64 prices units=%d maturities=%d N=%d method=%d" % (units, mats, N, method), flush=True)
    xi, M, seed = 0.04, 333, [N, units]
    H, eta, rho, T, K = _params(units, mats, 7 * N + units)
    price, iv, stat = rb.price_v2(xi, H, eta, rho, T, K, N, M, seed, method=method)
    Z = orc.normals_philox(seed, 0, M, 3 if method else 2, N)
    fn = orc.payoff_mc_samples if method else orc.payoff_rt_samples
    pr, st = orc.price_stat(fn(xi, H, eta, rho, T, K, N, Z))
    assert np.max(np.abs(price - pr)) < 1e-12
    assert np.max(np.abs(stat - st)) < 1e-12


# payoff sums of one, two and four paths per thread, each with a ragged last block, on 33 options (two
# jobs); the oracle prices the same paths
@pytest.mark.parametrize("M", [1000, (1 << 19) + 257, (1 << 20) + 1031])
@pytest.mark.parametrize("method", [0, 1])
def test_payoff_sums_of_several_paths_per_thread(rb, orc, M, method):
    print("payoff sums M=%d method=%d" % (M, method), flush=True)
    xi, N, seed = 0.04, 3, [M]
    K = np.exp(np.linspace(-0.4, 0.3, 33))
    price, _, stat = rb.price_v2(xi, [0.1], [1.9], [-0.7], np.full(33, 0.7), K, N, M, seed, method=method)
    fn = orc.payoff_mc_samples if method else orc.payoff_rt_samples
    pay = fn(xi, [0.1], [1.9], [-0.7], np.full(33, 0.7), K, N, orc.normals_philox(seed, 0, M, 3 if method else 2, N))
    pr, st = orc.price_stat(pay)
    assert np.max(np.abs(price - pr)) < 1e-12
    assert np.max(np.abs(stat - st)) < 1e-12


def test_extreme_coefficients_stay_finite_where_the_model_is(rb):
    """eta = 0 (the integrand is exactly xi past the last step's pad), and an eta whose exponents
    underflow: prices of the first are Black-Scholes on xi, none is NaN"""
    K = np.array([0.9, 1.0, 1.1])
    price, iv, _ = rb.price_v2(0.04, [0.1], [0.0], [0.0], np.ones(3), K, 37, 50, [1])
    assert np.max(np.abs(iv - 0.2)) < 1e-10
    price, _, _ = rb.price_v2(0.04, [0.1], [400.0], [-0.5], np.ones(3), K, 37, 50, [1])
    assert np.all(np.isfinite(price))


# either side of the choice between products and transforms, which depends on units and groups: transforms of
# length 512 (N <= 256), products and transforms up to N = 384
@pytest.mark.parametrize("units,mats,N", [(1, 1, 231), (1, 1, 256), (2, 2, 224), (3, 1, 193), (4, 1, 255), (1, 5, 256),
                                          (1, 1, 336), (1, 1, 368), (1, 8, 384), (3, 3, 340)])
def test_choice_of_kernel(rb, orc, units, mats, N):
    xi, (H, eta, rho, T, K) = 0.04, _params(units, mats, N)
    for method in (0, 1):
        M = 131
        print("path64 choice N=%d units=%d mats=%d method=%d" % (N, units, mats, method), flush=True)
        Z = orc.normals_philox([11, N], 0, M, 2 + method, N)
        fn = orc.payoff_mc_samples if method else orc.payoff_rt_samples
        price, stat = orc.price_stat(fn(xi, H, eta, rho, T, K, N, Z))
        p, _, s = rb.price_v2(xi, H, eta, rho, T, K, N, M, [11, N], precision=rb.PREC_FP64, method=method)
        assert np.max(np.abs(p - price)) < 1e-12 and np.max(np.abs(s - stat)) < 1e-12
