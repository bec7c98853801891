"""The exponent's conversion to an integer (rb_math64.h) out of the integer's range, where every step past a path's last
one takes it: the host's values, and no conversion in the device code that the compiler may take for undefined (LLVM's
fptosi gives poison there)."""
import subprocess

import pytest

from test_math64_cpu import CSRC, _hipcc

HOST = r"""
#include <cmath>
#include <cstdio>
#include "rb_math64.h"
int main() {
    for (double n : {0.0, -7.0, 2147483646.0, 2147483647.0, 2147483648.0, 1e300, (double)INFINITY, -2147483648.0, -2147483649.0,
                     -1e300, (double)-INFINITY, (double)NAN})
        std::printf("%d ", rb::whole_i32(n));
    for (double y : {-1e10, -1e290, 1e10}) std::printf("%g ", rb::exp2_32(rb::EXP2_TAB, y));
    return 0;
}
"""

DEVICE = r"""
#include <hip/hip_runtime.h>
#include "rb_math64.h"
__global__ void k(const double* t, double* x) { x[threadIdx.x] = rb::exp2_32(t, x[threadIdx.x]); }
"""


def test_host_values(tmp_path):
    hipcc = _hipcc()
    if hipcc is None:
        pytest.skip("hipcc not available")
    (tmp_path / "h.cpp").write_text(HOST)
    exe = str(tmp_path / "h")
    r = subprocess.run([hipcc, "-O1", "-std=c++17", "-x", "hip", "--cuda-host-only",
                        "-Xarch_host", "-fsanitize=float-cast-overflow", "-Xarch_host", "-fno-sanitize-recover=all", "-I" + CSRC,
                        str(tmp_path / "h.cpp"), "-o", exe], capture_output=True, text=True, timeout=600)
    assert r.returncode == 0, r.stderr[-3000:]
    out = subprocess.run([exe], capture_output=True, text=True, timeout=60)
    assert out.returncode == 0, out.stderr
    top, bottom = 2 ** 31 - 1, -2 ** 31
    assert out.stdout.split() == [str(x) for x in (0, -7, top - 1, top, top, top, top, bottom, bottom, bottom, bottom, 0)] + \
        ["0", "0", "inf"]


def test_device_code_converts_by_the_saturating_instruction(tmp_path):
    hipcc = _hipcc()
    if hipcc is None:
        pytest.skip("hipcc not available")
    (tmp_path / "d.hip").write_text(DEVICE)
    r = subprocess.run([hipcc, "-O3", "-std=c++17", "--offload-arch=gfx950", "--cuda-device-only", "-S", "-emit-llvm", "-I" + CSRC,
                        str(tmp_path / "d.hip"), "-o", str(tmp_path / "d.ll")], capture_output=True, text=True, timeout=600)
    assert r.returncode == 0, r.stderr[-3000:]
    ir = (tmp_path / "d.ll").read_text()
    assert "v_cvt_i32_f64" in ir and "fptosi" not in ir
