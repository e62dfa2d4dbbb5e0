"""The cases of the prompt GEMMs' GPU tests reach every kernel the library holds
for them, whatever the lines of the dispatch are.

The library is loaded over a stand-in for the runtime that notes which kernels
it registers and launches, in a process of its own (no GPU, nothing runs).  The
stand-in reports 256 compute units."""
import json
import subprocess
import sys

import _dip_hip as K
from test_gpu_gate_up import CASES as GATE_UP
from test_gpu_gemm_t_tiles import CASES as TRANSPOSED
from test_gpu_gemm_tiles import CASES as PLAIN

SHIM = r"""
#include <string.h>
static const void* fn[4096];
static const char* name[4096];
static int n = 0, hit[4096];
int __hipRegisterFunction(void** m, const void* f, char* d, const char* s) {
  if (n < 4096) { fn[n] = f; name[n++] = strdup(s); }
  return 0;
}
int shim_count(void) { return n; }
const char* shim_name(int i) { return name[i]; }
int shim_hit(int i) { return hit[i]; }
int __hipPushCallConfiguration() { return 0; }
int __hipPopCallConfiguration() { return 0; }
int hipLaunchKernel(const void* f) {
  for (int i = 0; i < n; ++i) if (fn[i] == f) hit[i] = 1;
  return 0;
}
int hipGetDevice(int* d) { *d = 0; return 0; }
int hipDeviceGetAttribute(int* v, int a, int d) { *v = 256; return 0; }
int hipGetLastError(void) { return 0; }
int hipFuncSetAttribute(const void* f, int a, int v) { return 0; }
"""

CALLS = r"""
import ctypes, json, sys
shim = ctypes.CDLL(sys.argv[1], mode=ctypes.RTLD_GLOBAL)
lib = ctypes.CDLL(sys.argv[2])
shim.shim_name.restype = ctypes.c_char_p
lib.dip_int4_gemm_t_workspace_size.restype = ctypes.c_size_t
cases = json.loads(sys.argv[3])
N, P = ctypes.c_int64, ctypes.c_void_p
p, odd = P(1 << 20), P((1 << 20) + 2)  # never dereferenced
st = []
for m, n, k in cases["plain"]:
    st += [lib.dip_int4_gemm(p, s, p, p, N(m), N(n), N(k), None) for s in (p, odd)]
for m, n, k in cases["gate_up"]:
    st += [lib.dip_int4_gemm_swiglu(p, p, p, s, p, p, N(m), N(n), N(k), None) for s in (p, odd)]
for m, k, n in cases["transposed"]:
    ws = ctypes.c_size_t(lib.dip_int4_gemm_t_workspace_size(N(m), N(n), N(k)))
    st.append(lib.dip_int4_gemm_t(p, p, p, p, N(m), N(n), N(k), p, ws, None))
assert not any(st), st
names = {shim.shim_name(i).decode(): shim.shim_hit(i) for i in range(shim.shim_count())}
print(json.dumps({n: h for n, h in names.items() if "int4_gemm" in n}))
"""


def test_cases_reach_every_prompt_gemm(tmp_path):
    src, so = tmp_path / "shim.c", tmp_path / "shim.so"
    src.write_text(SHIM)
    subprocess.run(["gcc", "-shared", "-fPIC", "-o", str(so), str(src)], check=True)
    cases = json.dumps({"plain": PLAIN, "gate_up": GATE_UP, "transposed": TRANSPOSED})
    r = subprocess.run([sys.executable, "-c", CALLS, str(so), str(K.LIB_PATH), cases],
                       capture_output=True, text=True, timeout=120)
    assert r.returncode == 0, r.stdout + r.stderr
    kernels = json.loads(r.stdout)
    assert len(kernels) > 30
    assert not [n for n, hit in kernels.items() if not hit]
