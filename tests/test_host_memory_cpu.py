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
