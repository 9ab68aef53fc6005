"""The module with the native host side of calls (_host_call): the library works without it, and it is used only by the Python
and the torch that it was built for."""
import os
import subprocess
import sys
import sysconfig

import pytest

from mm_amx_amd import build as B

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


@pytest.mark.parametrize("module", ["None", "other", "types.ModuleType('mm_amx_amd._host_call')"])
def test_the_library_works_without_the_module(module):
    """Not there, built for another torch, or built before it said for which: one warning, and the Python form takes every call."""
    r = subprocess.run([sys.executable, "-c", f"""
import sys, types, warnings
other = types.ModuleType('mm_amx_amd._host_call')
other.torch_version = '1.0'
sys.modules['mm_amx_amd._host_call'] = {module}
import mm_amx_amd as mx
from mm_amx_amd import _lib as L
with warnings.catch_warnings(record=True) as seen:
    warnings.simplefilter('always')
    assert mx.packed_b_bytes(mx.BF16, 64, 32) == 64 * 32 * 2
    mx.lib()
assert L._native is None
assert [str(w.message) for w in seen if 'native host side' in str(w.message)].__len__() == 1, seen
"""], cwd=ROOT, capture_output=True, text=True, timeout=300)
    assert r.returncode == 0, r.stderr


def test_the_module_is_of_this_python_and_torch():
    import torch
    from mm_amx_amd import _host_call
    assert B.HOST_CALL.endswith(sysconfig.get_config_var("EXT_SUFFIX")) and _host_call.__file__ == B.HOST_CALL
    assert _host_call.torch_version == str(torch.__version__)
