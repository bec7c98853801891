"""k_fused with two and with three workgroups per CU: a request that takes three alone takes two in a
batch with one whose tile leaves no room for a third, and in a batch of another number of groups
per pass.  Both forms execute the same operations in the same order, so results are equal bit for bit."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def rb():
    import rbergomi_amd
    rbergomi_amd.load()
    return rbergomi_amd


@pytest.mark.parametrize("method", [0, 1])
@pytest.mark.parametrize("prec,N", [("PREC_SPLIT_FP16", 60), ("PREC_SPLIT_FP16", 200), ("PREC_SPLIT_FP16", 300),
                                    ("PREC_SPLIT_FP16", 512), ("PREC_SPLIT_BF16", 250), ("PREC_SPLIT_BF16", 290),
                                    ("PREC_FP32_GEMM", 270)])
def test_alone_and_beside_a_large_request(rb, prec, N, method):
    from rbergomi_amd.serving import Request, price_batch
    code = getattr(rb, prec)
    T8 = np.repeat(np.linspace(0.2, 1.6, 8), 40)
    big = Request(0.05, [0.2], [1.2], [-0.5], T8, np.tile(np.linspace(0.7, 1.3, 40), 8), 512, 700, [9])
    for mats in (1, 2, 3, 4, 5, 6, 8):
        print("fused waves %s N=%d method=%d mats=%d" % (prec, N, method, mats), flush=True)
        T = np.repeat(np.linspace(0.1, 1.0, mats), 3)
        K = np.tile([0.85, 1.0, 1.2], mats)
        r = [Request(0.04, [0.07], [1.9], [-0.8], T, K, N, 5001, [3, N]) for _ in range(2)]
        price_batch([r[0]], precision=code, method=method)
        price_batch([r[1], big], precision=code, method=method)
        for what in ("price", "iv", "stat"):
            assert np.array_equal(getattr(r[0], what), getattr(r[1], what), equal_nan=True)
