"""A launch whose set-up fails says so on every call, not on the first alone.

The library is loaded over a stand-in for the runtime's calls in question, in a
process of its own (no GPU, nothing is launched)."""
import subprocess
import sys

import pytest

import _dip_hip as K

SHIM = r"""
#include <stdio.h>
#include <stdlib.h>
static int last = 0, launches = 0, device = 0, refused = 1, asked = 0;
void shim_device(int d) { device = d; }
void shim_refuse(int r) { refused = r; }
int shim_launches(void) { return launches; }
int shim_asked(void) { return asked; }
int hipGetDevice(int* d) { *d = device; return 0; }
int hipDeviceGetAttribute(int* v, int a, int d) { *v = 256; return 0; }
int hipGetLastError(void) { int e = last; last = 0; return e; }
int hipFuncSetAttribute(const void* f, int a, int v) { ++asked; return refused ? (last = 1) : 0; }
int __hipPushCallConfiguration() { return 0; }
int __hipPopCallConfiguration() { return 0; }
int hipLaunchKernel(const void* f) { ++launches; return 0; }
"""

CALLS = r"""
import ctypes, sys
shim = ctypes.CDLL(sys.argv[1], mode=ctypes.RTLD_GLOBAL)
lib = ctypes.CDLL(sys.argv[2])
buf = (ctypes.c_uint8 * 65536)()
p = ctypes.c_void_p(ctypes.addressof(buf) + (-ctypes.addressof(buf)) % 64)
n = ctypes.c_int64
calls = {
    "split": lambda: lib.dip_int4_gemm(p, p, p, p, n(4), n(64), n(256), None),
    "split gate and up": lambda: lib.dip_int4_gemm_swiglu(p, p, p, p, p, p, n(4), n(64), n(256), None),
    "tiled": lambda: lib.dip_int4_gemm(p, p, p, p, n(64), n(40960), n(128), None),
    "transposed": lambda: lib.dip_int4_gemm_t(p, p, p, p, n(4), n(128), n(8), None, n(0), None),
    "top-k": lambda: lib.dip_topk_select(p, p, n(100), n(5), p, n(4096), None),
}
"""


def _run(tmp_path, body):
    src, so = tmp_path / "shim.c", tmp_path / "shim.so"
    src.write_text(SHIM)
    subprocess.run(["gcc", "-shared", "-fPIC", "-o", str(so), str(src)], check=True)
    r = subprocess.run([sys.executable, "-c", CALLS + body, str(so), str(K.LIB_PATH)],
                       capture_output=True, text=True, timeout=120)
    assert r.returncode == 0, r.stdout + r.stderr
    return r.stdout


@pytest.mark.parametrize("call", ["split", "split gate and up", "tiled", "transposed", "top-k"])
def test_failed_setup_is_reported_every_time(tmp_path, call):
    out = _run(tmp_path, f"print([calls[{call!r}]() for _ in range(3)], shim.shim_launches())")
    assert out.split() == ["[1,", "1,", "1]", "0"], out


@pytest.mark.parametrize("call", ["split", "transposed", "top-k"])
def test_setup_runs_once_per_device(tmp_path, call):
    out = _run(tmp_path, f"""
f = calls[{call!r}]
assert f() != 0 and shim.shim_launches() == 0  # refused
shim.shim_refuse(0)
assert f() == 0 and shim.shim_launches() > 0  # asked again, and granted
seen = shim.shim_asked()
assert f() == 0 and shim.shim_asked() == seen
shim.shim_device(1)      # another device of the same process
assert f() == 0 and shim.shim_asked() > seen
seen = shim.shim_asked()
assert f() == 0 and shim.shim_asked() == seen
print("ok")
""")
    assert out.strip() == "ok"
