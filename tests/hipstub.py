"""Runs a piece of Python in a process of its own whose HIP runtime is
tests/hip_stub.cpp: `stub` and `h` (the library, rc_amd._lib.lib()) are
defined in it."""
import os
import subprocess
import sys
from pathlib import Path

HERE = Path(__file__).resolve().parent

PRELUDE = """
import ctypes as C, sys
stub = C.CDLL(sys.argv[1], mode=C.RTLD_GLOBAL)
stub.stub_live.restype = stub.stub_frees.restype = C.c_size_t
stub.stub_launches.restype = C.c_long
stub.stub_limit.argtypes = [C.c_size_t]
sys.path.insert(0, sys.argv[2])
from rc_amd import _lib
h = _lib.lib()
"""


def run(tmp_path, code: str) -> str:
    so = tmp_path / "libhipstub.so"
    if not so.exists():
        subprocess.run(["g++", "-std=c++17", "-O1", "-shared", "-fPIC",
                        str(HERE / "hip_stub.cpp"), "-o", str(so), "-lpthread"], check=True)
    p = subprocess.run([sys.executable, "-c", PRELUDE + code, str(so), str(HERE.parent)],
                       capture_output=True, text=True, timeout=120,
                       env={**os.environ, "PYTHONPATH": str(HERE)})
    assert p.returncode == 0, p.stdout + p.stderr
    return p.stdout
