"""What the library's launchers leave behind when the HIP runtime refuses a
kernel's LDS size: the call takes another path or returns FP4X_NOT_TAKEN, and
the launch that then runs is not reported as failed by the refusal's error.
The runtime calls are a stand-in (preloaded, no GPU): hipFuncSetAttribute
fails and records its error, hipGetLastError returns and clears it, launches
succeed and do nothing."""
import os
import shutil
import subprocess
import sys

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
PKG = os.path.join(ROOT, "qwen3.8-flash-next-fp4-local-spark_amd")

RUNTIME = r"""
#include <cstddef>
struct dim3_ { unsigned x, y, z; };
static int last = 0;
static int launches = 0;
extern "C" {
int hipGetDevice(int* d) { *d = 0; return 0; }
int hipDeviceGetAttribute(int* v, int, int) { *v = 256; return 0; }
int hipFuncSetAttribute(const void*, int, int) { return last = 1; }
int hipGetLastError(void) { int e = last; last = 0; return e; }
int hipPeekAtLastError(void) { return last; }
const char* hipGetErrorString(int) { return "stand-in"; }
int __hipPushCallConfiguration(dim3_, dim3_, size_t, void*) { return 0; }
int __hipPopCallConfiguration(dim3_* g, dim3_* b, size_t* s, void** st) {
  *g = *b = dim3_{1, 1, 1}; *s = 0; *st = nullptr; return 0;
}
int hipLaunchKernel(const void*, dim3_, dim3_, void**, size_t, void*) { ++launches; return 0; }
int fp4x_test_launches(void) { return launches; }
}
"""

CALLS = r"""
import ctypes, os, sys
import _fp4x
L = _fp4x.lib()
run = ctypes.CDLL(os.environ["FP4X_TEST_RUNTIME"])
P = ctypes.c_void_p(1 << 40)                       # never read: nothing runs


def rows(fmt, M, N, K, w1=None):
    return L.fp4x_linear_rows(fmt, P, K, P, w1, P, 1.0, P, 0, M, N, K, None)


refused = 0
for fmt in (_fp4x.FMT_MX8, _fp4x.FMT_W8_F32, _fp4x.FMT_W8_F16, _fp4x.FMT_W6, _fp4x.FMT_NV4, _fp4x.FMT_BF16):
    w1 = P if fmt == _fp4x.FMT_W6 else None
    for M, N, K in ((24, 16384, 2560), (39, 2560, 6144), (256, 16384, 2560), (256, 1280, 2560), (17, 512, 2560)):
        before = run.fp4x_test_launches()
        rc = rows(fmt, M, N, K, w1)
        assert rc in (_fp4x.OK, _fp4x.NOT_TAKEN), (fmt, M, N, K, rc, L.fp4x_last_error())
        assert (run.fp4x_test_launches() > before) == (rc == _fp4x.OK)
        refused += rc == _fp4x.NOT_TAKEN
        assert run.hipPeekAtLastError() == 0, ("error left set", fmt, M, N, K)
assert refused, "no call asked for more than 64 KB of LDS"
print("refused", refused)
"""


def test_refused_lds_size_leaves_no_error(tmp_path):
    gxx = shutil.which("g++")
    if gxx is None or not os.path.exists(os.path.join(PKG, "libfp4x.so")):
        pytest.skip("no g++ or no library")
    src, so = tmp_path / "runtime.cpp", tmp_path / "runtime.so"
    src.write_text(RUNTIME)
    r = subprocess.run([gxx, "-O1", "-shared", "-fPIC", str(src), "-o", str(so)], capture_output=True, text=True)
    assert r.returncode == 0, r.stderr[-2000:]
    env = {**os.environ, "PYTHONPATH": PKG, "FP4X_TEST_RUNTIME": str(so)}
    env["LD_PRELOAD"] = " ".join(filter(None, [str(so), os.environ.get("LD_PRELOAD")]))
    r = subprocess.run([sys.executable, "-c", CALLS], capture_output=True, text=True, env=env, timeout=300)
    assert r.returncode == 0, r.stdout[-1000:] + r.stderr[-3000:]
