"""The phase timings say so where the kernel that ran holds no stamps (here: the shipped library, which has none at all)."""
import io

import pytest
import torch

import mm_amx_amd as mx

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dt,tile", [("bf16", ""), ("w8", ""), ("i8", "128x64")])
def test_a_kernel_without_stamps(monkeypatch, dt, tile):
    mx.init(0)
    monkeypatch.setenv("MMX_LIB_PATH", mx.lib_path())  # (the module points the binding at the instrumented build otherwise)
    from mm_amx_amd import phase_stamps as ps
    ws = torch.zeros(ps.COUNTER_BYTES + ps.STAMP_OFFSET + ps.STAMP_BYTES, dtype=torch.uint8, device="cuda")
    out = io.StringIO()
    ps.run(ws, dt, 64, 1024, 256, tile, 0, out=out)
    assert mx.last_kernel() in out.getvalue() and "no stamps" in out.getvalue()
