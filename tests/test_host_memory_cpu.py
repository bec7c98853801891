"""The pinned host memory of plans, batches and the server, read from the built library's calls on the recording
runtime (recording.py)."""
import pytest

import recording


@pytest.fixture(scope="module")
def lib(tmp_path_factory):
    return recording.build(tmp_path_factory.mktemp("recording"))


# one call of every kind whose results a kernel writes to host memory: FP64, FP64 rows, the fused kernel, the
# long-path kernel, a batch and the server
CALLS = """
from rbergomi_amd.serving import Request, Server, price_batch
one = (0.04, [0.1], [1.9], [-0.7], [1.0], [1.0])
def calls():
    rb.price_v2(*one, 64, 1000, [1])
    rb.price_rows([0.04], [0.1], [1.9], [-0.7], [1.0], [1.0], 64, 1000, [1])
    rb.price_v2(*one, 64, 1000, [1], precision=rb.PREC_SPLIT_FP16)
    rb.price_v2(*one, 2048, 1000, [1], precision=rb.PREC_SPLIT_FP16)
    price_batch([Request(*one, 64, 1000, [1]), Request(*one, 1500, 1000, [1])])
    s = Server()
    s.wait(s.submit(Request(*one, 64, 1000, [1])))
    s.wait(s.submit(Request(*one, 1500, 1000, [1])))
    s.close()
"""


def test_results_go_to_coherent_memory(lib):
    """Without the flag coherence is the environment's (HIP_HOST_COHERENT), and a host that reads after
    hipEventQuery may see old values."""
    out = recording.run(lib, CALLS + "calls(); print(rec.rec_pinned_most() > 0, rec.rec_pinned_flags())")
    some, flags = out.split()
    assert some == "True"
    assert int(flags) & 0x40000000  # hipHostMallocCoherent
    assert int(flags) & 0x1         # hipHostMallocPortable


# the results of every kind of call, whether pinned memory can be had or not
RESULTS = """
from rbergomi_amd.serving import Request, Server, price_batch
one = (0.04, [0.123], [1.9], [-0.7], [0.5, 1.0, 1.5], [0.9, 1.0, 1.1])
def check(r):
    price, iv, stat = r
    assert np.array_equal(price, [1, 2, 3]) and np.array_equal(stat, [1001, 1002, 1003]) and np.array_equal(iv, [2001, 2002, 2003]), r
def plan(N, **kw):
    p = rb.Plan(*one, N, 1000, [1], **kw)
    p.run()
    check(p.results())
    p.close()
def served(*sizes):
    s = Server()
    for r in [s.submit(Request(*one, N, 1000, [1])) for N in sizes]:
        s.wait(r)
        check((r.price, r.iv, r.stat))
    s.close()
def calls():
    plan(64)
    assert [v["mH0"] for _, v in launches("k_path64I")] == [123000]
    plan(500)
    assert [v["mH0"] for _, v in launches("k_path64_fftI")] == [123000]
    plan(6000)
    check(rb.price_v2(*one, 64, 1000, [1], precision=rb.PREC_FP32))
    for N in (64, 2048, 6000):
        plan(N, precision=rb.PREC_SPLIT_FP16)
    for r in price_batch([Request(*one, 1500, 1000, [1])]):
        check((r.price, r.iv, r.stat))
    served(64, 1500)
"""


def test_results_without_pinned_memory(lib):
    """Pinned memory only saves copies: a call is priced without it too, tables and results then
    through pageable memory."""
    recording.run(lib, RESULTS + "calls()")
    recording.run(lib, RESULTS + "rec.rec_fail_pinned_from(0); calls(); assert rec.rec_pinned_most() == 0")


def test_large_tables_are_not_pinned(lib):
    """The exact sampler's factors (16 N^2 bytes per H) and the long-path spectra formed on the host (N > 4096)
    go up from pageable memory."""
    out = recording.run(lib, """
H = [0.1, 0.2, 0.3]
p = rb.Plan(0.04, H, [1.9] * 3, [-0.7] * 3, [1.0], [1.0], 400, 1000, [1], scheme=rb.SCHEME_CHOLESKY)
p.run()
q = rb.Plan(0.04, np.linspace(0.05, 0.4, 50), [1.9] * 50, [-0.7] * 50, [1.0], [1.0], 5000, 1000, [1], precision=rb.PREC_SPLIT_FP16)
q.run()
print(rec.rec_pinned_most())
""")
    assert int(out) <= 1 << 20
