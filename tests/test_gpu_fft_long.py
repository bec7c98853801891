"""The FFT path kernel (k_fused_fft) against the FP64 path on the same Philox counters: both ends of
every transform length with an absent second path, requests whose integrals take several launches
(more than 4 MiB), and units split over workgroups.

Tolerance: the FP32 transform and sums leave the integrals within 2e-6 relative, which moves a price
of a unit spot by less than 2e-6, and FP32 payoffs are within 1e-6: 5e-6 together."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def rb():
    import rbergomi_amd
    return rbergomi_amd


CASES = [(1, 3, 1, 1), (2, 7, 5, 2), (257, 9, 1, 3), (512, 5, 2, 2), (513, 3, 1, 1), (1024, 4, 3, 1), (2047, 3, 1, 2),
         (2048, 4, 7, 1), (2050, 5, 2, 2), (4095, 3, 5, 1), (4096, 2, 1, 4), (4098, 3, 2, 1), (8191, 2, 1, 2),
         (300, 60001, 3, 3), (1030, 45001, 2, 4)]


@pytest.mark.parametrize("method", [0, 1])
@pytest.mark.parametrize("N,M,units,mats", CASES)
def test_prices_match_fp64(rb, N, M, units, mats, method):
    print("fft kernel N=%d M=%d units=%d mats=%d method=%d" % (N, M, units, mats, method), flush=True)
    rng = np.random.default_rng(N + M)
    H = rng.uniform(0.03, 0.45, units)
    eta, rho = rng.uniform(0.5, 2.0, units), rng.uniform(-0.9, 0.3, units)
    T = np.repeat(np.linspace(0.1, 1.0, mats), 2)
    K = rng.uniform(0.85, 1.15, 2 * mats)
    a = rb.price_v2(0.04, H, eta, rho, T, K, N, M, [5, N], precision=rb.PREC_FP64, method=method)
    b = rb.price_v2(0.04, H, eta, rho, T, K, N, M, [5, N], precision=rb.PREC_FP32_FFT, method=method)
    assert np.max(np.abs(np.asarray(b[0]) - np.asarray(a[0]))) <= 5e-6
    assert np.max(np.abs(np.asarray(b[2]) - np.asarray(a[2]))) <= 5e-6
