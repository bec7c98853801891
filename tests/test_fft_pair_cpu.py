"""CPU check of the transforms that the long-path kernel runs (fft_pair_emulation.cpp): first pass, tables by pass,
spectrum order and padding of rb_fft_lds.h, compiled for the host, against a direct FP64 convolution."""
import os
import subprocess

import pytest

from test_fft_lds_cpu import CSRC, HERE, _hipcc


def test_long_path_transforms_match_direct_convolution(tmp_path):
    hipcc = _hipcc()
    if hipcc is None:
        pytest.skip("hipcc not available")
    exe = str(tmp_path / "fft_pair_emulation")
    r = subprocess.run([hipcc, "-O1", "-std=c++17", "-x", "hip", "--cuda-host-only", "-I" + CSRC,
                        os.path.join(HERE, "fft_pair_emulation.cpp"), "-o", exe], capture_output=True, text=True, timeout=600)
    assert r.returncode == 0, r.stderr[-3000:]
    out = subprocess.run([exe], capture_output=True, text=True, timeout=300)
    print(out.stdout)
    assert out.returncode == 0, out.stdout
    assert out.stdout.strip().endswith("OK")
