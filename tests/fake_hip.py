"""Runs code in a child process on a HIP runtime without a device
(fake_hip.c): the library's host code with kernels that are recorded and not
run, allocations and copies that fail where a test says so, and time counted in
kernels.  The code sees `pa` (the binding), `wd` (its decks), `fake` (the
runtime: fail_malloc, fail_bytes, fail_copy, fail_wait, error, launches, queued,
live, copied, max_threads),
`slow(name)`, which makes kernels of that name take 100 times as long, and
`clear()` and `names()`, the kernels run since."""
import subprocess
import sys
from pathlib import Path

import pytest

HERE = Path(__file__).resolve().parent
ROOT = HERE.parent

PROLOGUE = """
import ctypes, sys
sys.path[:0] = [{pkg!r}, {here!r}]
_f = ctypes.CDLL({so!r}, mode=ctypes.RTLD_GLOBAL)
_f.fake_names.restype = ctypes.c_char_p
class _Fake:
    def __getattr__(self, k): return ctypes.c_int64.in_dll(_f, "fake_" + k).value
    def __setattr__(self, k, v): ctypes.c_int64.in_dll(_f, "fake_" + k).value = v
fake = _Fake()
clear = _f.fake_clear
def slow(name): (ctypes.c_char * 64).in_dll(_f, "fake_slow").value = name.encode()
def names(): return _f.fake_names().decode().split()
import pennant_amd as pa
from pennant_amd import decks as wd
"""


@pytest.fixture(scope="session")
def run_fake(tmp_path_factory):
    so = tmp_path_factory.mktemp("fake_hip") / "libfake_hip.so"
    subprocess.run(["gcc", "-O1", "-shared", "-fPIC", "-o", str(so), str(HERE / "fake_hip.c")], check=True)
    head = PROLOGUE.format(pkg=str(ROOT / "pennant-legion_amd"), here=str(HERE), so=str(so))

    def run(code):
        r = subprocess.run([sys.executable, "-c", head + code], capture_output=True, text=True, timeout=120)
        assert r.returncode == 0, r.stdout + r.stderr
        return r.stdout
    return run
