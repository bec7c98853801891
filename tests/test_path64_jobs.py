"""Workgroups of the FP64 path kernels that price several jobs one after another (a job: one H and up to eight
of its groups), against the oracle on the same Gaussians.  A tile's jobs are spread over as many workgroups as bring four
to every compute unit, so this needs tiles enough: the first test, without a device, asserts that every case has
workgroups of several jobs, in the kernel, with the threads and with W1perp kept or not as named, so that
no case degrades unnoticed when the rules of the launch change.

Tolerance: the FP64 path's 1e-12 absolute of prices and standard errors."""
import numpy as np
import pytest

import recording

# kernel, threads, W1perp kept in LDS; units, maturities, N, M
CASES = [
    ("k_path64I", 256, 1, 5, 1, 100, 8200),    # another H every job
    ("k_path64I", 256, 1, 1, 17, 64, 9600),    # the same H: Gamma stays in LDS
    ("k_path64I", 512, 1, 1, 17, 200, 8200),
    ("k_path64I", 512, 0, 1, 17, 340, 8200),   # W1perp drawn again by every job
    ("k_path64I", 512, 0, 1, 17, 376, 8200),
    ("k_path64_fftI", 256, 0, 5, 1, 256, 8200),  # two pairs a wave
    ("k_path64_fftI", 256, 0, 4, 1, 500, 4203),  # a wave a pair
    ("k_path64_fftI", 256, 0, 1, 17, 500, 4203),
    ("k_path64_fftI", 256, 0, 3, 1, 1000, 2101),  # two, four and eight waves a pair
    ("k_path64_fftI", 256, 0, 3, 1, 1500, 1051),
    ("k_path64_fftI", 512, 0, 3, 1, 2100, 1051),
]


def _inputs(units, mats, N):
    rng = np.random.default_rng(7 * N + units)
    H = rng.uniform(0.03, 0.45, units)
    return (0.04, H, rng.uniform(0.5, 2.5, units), rng.uniform(-0.95, -0.2, units), np.linspace(0.1, 1.5, mats),
            rng.uniform(0.8, 1.2, mats))


@pytest.mark.parametrize("method", [0, 1])
def test_cases_have_workgroups_of_several_jobs(tmp_path, method):
    lib = recording.build(tmp_path)
    out = recording.run(lib, """
for k, t, perp, units, mats, N, M in %r:
    rb.price_v2(0.04, np.linspace(0.05, 0.4, units), [1.9] * units, [-0.7] * units, np.linspace(0.1, 1.5, mats), [1.0] * mats, N, M, [1], method=%d)
    (name, f), = [x for x in launches("k_path64") if "np" in x[1]]
    print(k in name and f["block"] == t and f["perp"] == perp and 2 * f["nsplit"] <= f["njobs"] + 1 and f["nsplit"] < f["njobs"], name, f)
""" % (CASES, method))
    lines = out.splitlines()
    assert len(lines) == len(CASES) and all(x.startswith("True") for x in lines), out


@pytest.mark.gpu
@pytest.mark.parametrize("method", [0, 1])
@pytest.mark.parametrize("kernel,threads,perp,units,mats,N,M", CASES)
def test_prices_match_the_oracle(orc, kernel, threads, perp, units, mats, N, M, method):
    import rbergomi_amd as rb
    print("jobs %s units=%d maturities=%d N=%d M=%d method=%d" % (kernel, units, mats, N, M, method), flush=True)
    args, seed = _inputs(units, mats, N), [N, units]
    price, _, stat = rb.price_v2(*args, N, M, seed, method=method)
    Z = orc.normals_philox(seed, 0, M, 2 + method, N)
    fn = orc.payoff_mc_samples if method else orc.payoff_rt_samples
    pr, st = orc.price_stat(fn(*args, N, Z))
    assert np.max(np.abs(price - pr)) < 1e-12
    assert np.max(np.abs(stat - st)) < 1e-12
    if N == 500:  # the same paths as a caller's Gaussians
        _, pr2, st2 = rb.payoff_samples_v2(*args, N, Z, method=method)
        assert np.max(np.abs(pr2 - pr)) < 1e-12 and np.max(np.abs(st2 - st)) < 1e-12


# the long-path mixed-precision kernel's loop over units: transforms of 2^10 to 2^14 points (at the FFT precision below
# N = 1025), threads of a pair 64 to 512
UNITS = [(500, 9000), (1000, 4300), (1500, 2100), (3000, 1300), (6000, 1300)]
H3, ETA3, RHO3 = [0.07, 0.21, 0.4], [1.9, 1.1, 0.7], [-0.9, -0.6, -0.3]


def test_unit_cases_have_workgroups_of_several_units(tmp_path):
    lib = recording.build(tmp_path)
    out = recording.run(lib, """
for N, M in %r:
    rb.price_v2(0.04, %r, %r, %r, [1.0], [1.0], N, M, [1], precision=rb.PREC_FP32_FFT)
    (name, f), = launches("k_fused_fft")
    print(f["grid_y"] < 3, name, f)
""" % (UNITS, H3, ETA3, RHO3))
    assert [x.split()[0] for x in out.splitlines()] == ["True"] * len(UNITS), out


@pytest.mark.gpu
@pytest.mark.parametrize("method", [0, 1])
@pytest.mark.parametrize("N,M", UNITS)
def test_units_of_one_workgroup_price_as_alone(N, M, method):
    """The paths of a call do not depend on its parameter sets, so every set's prices are the same bits alone."""
    import rbergomi_amd as rb
    T, K = np.array([0.4, 1.1]), np.array([0.95, 1.05])
    kw = dict(precision=rb.PREC_FP32_FFT, method=method)
    print("units N=%d M=%d method=%d" % (N, M, method), flush=True)
    price, _, stat = rb.price_v2(0.04, H3, ETA3, RHO3, T, K, N, M, [3, N], **kw)
    for h in range(3):
        p, _, s = rb.price_v2(0.04, H3[h:h + 1], ETA3[h:h + 1], RHO3[h:h + 1], T, K, N, M, [3, N], **kw)
        assert np.array_equal(p, price[2 * h:2 * h + 2]) and np.array_equal(s, stat[2 * h:2 * h + 2])


@pytest.mark.gpu
def test_spectra_above_the_pinned_size_price_as_alone():
    """Beyond N = 4096 the spectra are formed on the host: 40 of them are copied from pageable memory, one is not."""
    import rbergomi_amd as rb
    n, N, M = 40, 5000, 700
    H, eta, rho = np.linspace(0.05, 0.44, n), np.full(n, 1.2), np.full(n, -0.6)
    kw = dict(precision=rb.PREC_SPLIT_FP16)
    print("pageable spectra", flush=True)
    price, _, stat = rb.price_v2(0.04, H, eta, rho, [1.0], [1.0], N, M, [3], **kw)
    for h in (0, 17, n - 1):
        p, _, s = rb.price_v2(0.04, H[h:h + 1], eta[:1], rho[:1], [1.0], [1.0], N, M, [3], **kw)
        assert p[0] == price[h] and s[0] == stat[h]
