"""A launch that fails is the call's error, whichever way a mixture takes (the runtime's launch stands aside for one that fails; nothing reaches a device)."""
import subprocess
import sys

import pytest

from nano_vllm_x_amd import _lib

STUB = """
static int last;
int hipLaunchKernel(void) { last = 98; return 98; }
int hipGetLastError(void) { int e = last; last = 0; return e; }
int __hipPushCallConfiguration(void) { return 0; }
int __hipPopCallConfiguration(void) { return 0; }
"""
CALL = """
import ctypes, sys
ctypes.CDLL(sys.argv[1], mode=ctypes.RTLD_GLOBAL)
lib, i64, f = ctypes.CDLL(sys.argv[2]), ctypes.c_int64, ctypes.c_float
at = ctypes.c_void_p(1 << 20)      # (nothing reads it)
tokens, width, ff = map(int, sys.argv[3:])
end = (at, at, i64(1), at, i64(1), f(1e-5), at, None)
print(lib.nvx_internal_moe_postnorm(at, i64(width), 0, at, at, i64(2), at, at, i64(4), f(1), f(1), f(0), 1, at, at, i64(tokens), i64(width), i64(ff), 1, *end))
"""


@pytest.fixture(scope="module")
def stub(tmp_path_factory):
    d = tmp_path_factory.mktemp("launch")
    (d / "stub.c").write_text(STUB)
    subprocess.run(["gcc", "-shared", "-fPIC", "-o", str(d / "stub.so"), str(d / "stub.c")], check=True)
    return str(d / "stub.so")


@pytest.mark.parametrize("tokens,width,ff,what", [(16, 128, 64, "tiles"), (16, 130, 66, "rows"), (5000, 128, 64, "grouped"), (16, 8192, 64, "tiles, the norm by itself")])
def test_a_failed_launch_is_reported(stub, tokens, width, ff, what):
    got = subprocess.run([sys.executable, "-c", CALL, stub, _lib.LIB_PATH, str(tokens), str(width), str(ff)], capture_output=True, text=True, timeout=120)
    assert got.returncode == 0, got.stderr
    assert int(got.stdout.split()[-1]) != 0, what
