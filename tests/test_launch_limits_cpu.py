"""Launches of the FP64 path at path counts that one grid does not hold, planned by the built library on the
recording runtime (recording.py), which refuses a grid as HIP does (gridDim * blockDim of 2^32 or more): every
path is launched once, in chunks whose payoff blocks are whole."""
import pytest

import recording


@pytest.fixture(scope="module")
def lib(tmp_path_factory):
    return recording.build(tmp_path_factory.mktemp("recording"))


CODE = """
for method in (rb.METHOD_RT, rb.METHOD_MC):
    for N in (1, 17, 33, 64, 128, 200, 256, 300, 360, 384, 385, 512, 513, 1024, 1025, 2048, 2049, 4096):
        for M in ((1 << 24) + 1, 1000000007):
            p = rb.Plan(0.04, [0.1], [1.9], [-0.7], [1.0], [1.0], N, M, [1], method=method)
            p.run()
            p.close()
            at = 0
            for name, f in launches("k_path64"):
                if "np" not in f:
                    continue
                assert f["p0"] == at and f["grid"] * f["block"] < 2 ** 32, (N, M, name, f)
                at += f["np"]
                assert at == M or f["np"] % 1024 == 0, (N, M, name, f)
            assert at == M, (N, M, at)
# the mirrored paths of the turbo-charged estimator, with its pilot paths in a launch of their own
for N in (200, 4096):
    M, pilot = 300000000, 50000
    rb.price_rows_turbo([0.04], [0.1], [1.9], [-0.7], [1.0], [1.0], N, M, [1], m_control=pilot)
    assert sum(f["np"] for _, f in launches("k_path64") if "np" in f) == M + pilot
print("ok")
"""


def test_every_path_is_launched_within_the_grid(lib):
    assert recording.run(lib, CODE).strip().endswith("ok")


# requests whose partial sums, 16 bytes per option and work item, fill a bounded memory
BOUNDED = """
from rbergomi_amd.serving import Request, Server
opts = np.linspace(0.05, 1.0, 5), np.linspace(0.8, 1.2, 100)
T, K = np.repeat(opts[0], 100), np.tile(opts[1], 5)
H, eta, rho = np.linspace(0.05, 0.4, 10), np.full(10, 1.9), np.full(10, -0.7)
# 5000 options: 20 MB of sums in 256 items, 80 MB in 1024, of 64 MiB
rb.price_noalloc(0.04, H, eta, rho, T, K, 64, 1 << 18, [1])
# the same items, so the same sums, in a call that allocates
noalloc = [f["items"] for _, f in launches("k_fusedI")]
rb.price_v2(0.04, H, eta, rho, T, K, 64, 1 << 18, [1], precision=rb.PREC_SPLIT_FP16)
assert [f["items"] for _, f in launches("k_fusedI")] == noalloc == [256]
# the same request in a server of 32 MiB
s = Server(max_device_bytes=32 << 20)
s.wait(s.submit(Request(0.04, H, eta, rho, T, K, 64, 1 << 18, [1])))
for M in (1 << 30, 1 << 24):  # 4096 items and more
    try:
        rb.price_noalloc(0.04, H, eta, rho, T, K, 64, M, [1])
        assert False
    except rb.RbError as e:
        assert e.code == 5
    try:
        s.submit(Request(0.04, H, eta, rho, T, K, 64, M, [1]))
        assert False
    except rb.RbError as e:
        assert e.code == 5
s.close()
print("ok")
"""


def test_partial_sums_fit_bounded_memory(lib):
    assert recording.run(lib, BOUNDED).strip().endswith("ok")


PILOTS = """
row = [0.04], [0.1], [1.9], [-0.7], [1.0], [1.0]
for N in (64, 256, 1024, 4096):
    fit = int(6e9 / (24 * N + 32)) // 256 * 256
    rb.price_rows_turbo(*row, N, 1000, [1], m_control=fit)
    try:
        rb.price_rows_turbo(*row, N, 1000, [1], m_control=fit + 1)
        assert False
    except rb.RbError as e:
        assert e.code == 5
print("ok")
"""


def test_pilot_paths_of_the_turbo_estimator_are_limited(lib):
    """rb_price_rows_turbo's m_control: 6 GB of two streams, one process and two pairs of integrals a path."""
    assert recording.run(lib, PILOTS).strip().endswith("ok")


OPTIONS = """
from rbergomi_amd.serving import Request, Server
s = Server()
for N, L in ((1025, 4096), (4096, 8192), (8192, 16384)):
    most = (160 * 1024 - 1536 - 8 * (L + L // 32) - 64) // 16
    for n in (most, most + 1):
        one = 0.04, [0.1], [1.9], [-0.7], np.full(n, 1.0), np.linspace(0.5, 1.5, n), N, 1000, [1]
        for call in (lambda: rb.price_v2(*one, precision=rb.PREC_SPLIT_FP16), lambda: s.wait(s.submit(Request(*one)))):
            try:
                call()
                assert n == most
            except rb.RbError as e:
                assert n == most + 1 and e.code == 5 and "LDS" not in str(e) and str(n) in str(e), e
s.close()
print("ok")
"""


def test_options_of_a_long_path_request_are_limited(lib):
    """A limit of the interface, and the message says so."""
    assert recording.run(lib, OPTIONS).strip().endswith("ok")
