"""The disk cache of compiled kernels (csrc/hb_runtime.cpp) beside another
HIP: a process that has loaded PyTorch first compiles with the hiprtc PyTorch
brings, and neither takes that compiler's code for the library's own nor the
other way round."""
import os
import subprocess
import sys

import pytest

import herbert_hip as hb

CODE = """
import sys, ctypes
if %d: import torch
sys.path.insert(0, %r)
import herbert_hip as hb
v = ctypes.c_int()
assert hb.lib.hipRuntimeGetVersion(ctypes.byref(v)) == 0
d = hb.Desc(kind=hb.Kind.ROUND_PROBE)
hb.check(hb.lib.hb_kernel_precompile(ctypes.byref(d)))
print("hip", v.value)
"""


def compile_in(cache, torch_first):
    """Precompiles one kernel in a process of its own: its HIP's version."""
    env = dict(os.environ, HB_CACHE_DIR=str(cache))
    code = CODE % (torch_first, os.path.dirname(hb.LIB_PATH))
    r = subprocess.run([sys.executable, "-c", code], capture_output=True, text=True, env=env)
    assert r.returncode == 0, r.stderr
    return int(r.stdout.split()[-1])


def test_entries_of_two_compilers(tmp_path):
    if compile_in(tmp_path / "a", True) == compile_in(tmp_path / "b", False):
        pytest.skip("PyTorch and the library use one HIP")
    own = set(os.listdir(tmp_path / "b"))
    theirs = set(os.listdir(tmp_path / "a"))
    assert len(own) == len(theirs) == 1
    # Their code first: the library's own compiler still writes its own.
    compile_in(tmp_path / "a", False)
    assert set(os.listdir(tmp_path / "a")) == own | theirs and not own & theirs
    # The library's own first: the other process loads it, and marks it used.
    entry = tmp_path / "b" / own.pop()
    os.utime(entry, (1, 1))
    compile_in(tmp_path / "b", True)
    assert os.listdir(tmp_path / "b") == [entry.name] and entry.stat().st_mtime > 1
