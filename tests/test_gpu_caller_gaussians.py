"""Caller's Gaussians that are not finite, or no Gaussians at all, on the FP64 path: what they do stays with
their path, against the oracle on the same values.  N on both sides of the kernels' dispatch (products to N = 200,
transforms of every length above), two H so that a workgroup has more than one convolution, and both estimators.

Tolerance of finite payoffs: the FP64 path's 1e-12."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def rb():
    import rbergomi_amd
    return rbergomi_amd


@pytest.mark.parametrize("method", [0, 1])
@pytest.mark.parametrize("N", [20, 100, 200, 385, 512, 1000, 2048, 4096])
def test_other_paths_and_unused_steps_are_not_touched(rb, orc, N, method):
    print("caller's values N=%d method=%d" % (N, method), flush=True)
    xi, H, eta, rho, T, K = 0.05, [0.08, 0.3], [1.5, 0.8], [-0.8, -0.4], [0.6], [1.02]
    clean = np.random.default_rng(N).standard_normal((19, 2 + method, N))
    k = N // 2
    Z = clean.copy()
    Z[2, 0, k] = np.inf          # W1: the path is lost, its pair (3) and its tile (all) are not
    Z[5, 0, 0] = np.nan
    Z[8, 0, N - 2] = -np.inf
    Z[11, 0, k] = 1e30
    Z[12, 1, k] = -np.inf        # W1perp of one step: that step has no variance
    Z[14, 1, N - 1] = np.nan     # W1perp of the last step is not used
    Z[17, 1, N - 1] = np.inf
    Z[18, 0, 0] = -1e7           # S' beyond the largest double: an infinite payoff
    fn = orc.payoff_mc_samples if method else orc.payoff_rt_samples
    got, _, _ = rb.payoff_samples_v2(xi, H, eta, rho, T, K, N, Z, method=method)
    ref = fn(xi, H, eta, rho, T, K, N, Z)
    assert np.all(ref[18] == np.inf) and np.all(got[18] == np.inf)
    lost = [2, 5, 8, 11, 18]
    kept = [p for p in range(len(Z)) if p not in lost]
    assert np.all(np.isfinite(ref[kept]))
    assert np.max(np.abs(got[kept] - ref[kept])) < 1e-12
    if method == 0:
        assert not np.any(np.isfinite(got[[2, 5, 11]]))
    # the same values as without the lost paths' (the transform of a clean pair is not the direct sum: 1e-12)
    calm, _, _ = rb.payoff_samples_v2(xi, H, eta, rho, T, K, N, clean, method=method)
    same = [p for p in kept if p not in (12, 14, 17)]
    assert np.max(np.abs(got[same] - calm[same])) < 1e-12
