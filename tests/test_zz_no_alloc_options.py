"""rb_price_noalloc with as many options as its scratch holds the sums of: the same items, and so the same bits, as
rb_price_v2 (test_launch_limits_cpu.py counts the items)."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def test_many_options_price_as_price_v2():
    import rbergomi_amd as rb
    T, K = np.repeat(np.linspace(0.05, 1.0, 5), 100), np.tile(np.linspace(0.8, 1.2, 100), 5)
    args = (0.04, np.linspace(0.05, 0.4, 10), np.full(10, 1.9), np.full(10, -0.7), T, K, 64, 1 << 17, [5])
    print("noalloc options=5000", flush=True)
    got = rb.price_noalloc(*args)
    ref = rb.price_v2(*args, precision=rb.PREC_SPLIT_FP16)
    for a, b in zip(got, ref):
        assert np.array_equal(a, b, equal_nan=True)
