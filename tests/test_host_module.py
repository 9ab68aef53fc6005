"""The module with the native host side of calls (_host_call): the library works without it, and it is used only by the Python
and the torch that it was built for; and what its build leaves behind."""
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


@pytest.fixture
def scratch_build(tmp_path, monkeypatch):
    """build() in a folder of its own, with compilers that are scripts there; returns a function that writes them."""
    for name, at in (("CSRC", tmp_path), ("LIB", tmp_path / "lib.so"), ("HOST_CALL", tmp_path / "host.so")):
        monkeypatch.setattr(B, name, str(at))
    monkeypatch.setenv("PATH", str(tmp_path), prepend=os.pathsep)

    def compiler(name, body):
        (tmp_path / name).write_text("#!/bin/sh\n" + body)
        (tmp_path / name).chmod(0o755)
    return compiler


OUTPUT = 'while [ "$1" != -o ]; do shift; done; echo made > "$2"'


def test_a_failed_build_leaves_no_compiler_running(scratch_build, tmp_path):
    scratch_build("hipcc", "exit 1")
    scratch_build("g++", f"sleep 2; {OUTPUT}")
    with pytest.raises(RuntimeError, match="hipcc"):
        B.build()
    assert (tmp_path / "host.so").exists()  # (it was waited for)


def test_a_failed_module_is_an_error_and_the_library_is_there(scratch_build, tmp_path):
    scratch_build("hipcc", OUTPUT)
    scratch_build("g++", "exit 1")
    with pytest.raises(RuntimeError, match="g\\+\\+"):
        B.build()
    assert (tmp_path / "lib.so").exists()


def test_the_library_builds_with_hipcc_alone(scratch_build, tmp_path, monkeypatch):
    """No torch, no headers of Python, or no g++: the library is for C and C++ callers too."""
    scratch_build("hipcc", OUTPUT)
    for hide in (lambda m: m.setitem(sys.modules, "torch", None), lambda m: m.setattr(B.sysconfig, "get_paths", lambda: {"include": str(tmp_path)}),
                 lambda m: m.setattr(B.shutil, "which", lambda name: None)):
        with monkeypatch.context() as m:
            hide(m)
            assert B.build() == str(tmp_path / "lib.so") and (tmp_path / "lib.so").exists()
        (tmp_path / "lib.so").unlink()
        assert not (tmp_path / "host.so").exists()
