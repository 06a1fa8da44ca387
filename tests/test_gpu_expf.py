"""The exponential's two forms (csrc/waam_math.h): the device's scales with one instruction where the
host's multiplies twice. Bit equality of the kernels with the oracle rests on their agreeing, so every
one of the 2^32 float words goes through both."""

from __future__ import annotations

import ctypes
import shutil
import subprocess
from pathlib import Path

import pytest
import torch

from waam_solver_amd._lib import lib

pytestmark = pytest.mark.gpu

CSRC = Path(__file__).resolve().parents[1] / "waam_solver_amd" / "csrc"
CHECK = """
#include <stdint.h>
#include <string.h>
#include "waam_math.h"
/* words first .. first + n - 1: how many differ from y, and the first that does */
long check(const uint32_t *y, uint32_t first, long n, uint32_t *at)
{
    long bad = 0;
#pragma omp parallel for reduction(+ : bad)
    for (long e = 0; e < n; ++e) {
        uint32_t w = first + (uint32_t)e, u;
        float x, v;
        memcpy(&x, &w, 4);
        v = waam_expf(x);
        memcpy(&u, &v, 4);
        int nan_u = (u & 0x7fffffffu) > 0x7f800000u, nan_y = (y[e] & 0x7fffffffu) > 0x7f800000u;
        if (nan_u ? !nan_y : u != y[e]) {
#pragma omp critical
            { if (bad == 0) *at = w; }
            ++bad;
        }
    }
    return bad;
}
"""


def test_every_word_equals_the_host_form(hip_device, tmp_path):
    cc = shutil.which("gcc")
    if cc is None:
        pytest.skip("no C compiler")
    (tmp_path / "c.c").write_text(CHECK)
    subprocess.run([cc, "-O2", "-fopenmp", "-ffp-contract=off", "-shared", "-fPIC", f"-I{CSRC}",
                    str(tmp_path / "c.c"), "-o", str(tmp_path / "c.so")], check=True)
    host = ctypes.CDLL(str(tmp_path / "c.so"))
    host.check.restype = ctypes.c_long
    host.check.argtypes = [ctypes.c_void_p, ctypes.c_uint32, ctypes.c_long, ctypes.c_void_p]
    n = 1 << 27
    base = torch.arange(n, dtype=torch.int32, device=hip_device)
    y = torch.empty(n, dtype=torch.float32, device=hip_device)
    out = torch.empty(n, dtype=torch.float32, pin_memory=True)
    st = torch.cuda.current_stream().cuda_stream
    for c in range((1 << 32) // n):
        first = c * n
        x = base + (first - (1 << 32) if first >= 1 << 31 else first)  # the words as int32
        lib().call("waam_expf_array", x.data_ptr(), y.data_ptr(), n, st)
        out.copy_(y)
        at = ctypes.c_uint32()
        bad = host.check(out.data_ptr(), first, n, ctypes.addressof(at))
        print(f"[expf] words from {first:#010x}: {bad} differ", flush=True)
        assert bad == 0, f"{bad} words differ, the first {at.value:#010x}"
