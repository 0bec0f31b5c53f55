"""A stand-in for the HIP runtime calls that the library's launchers make
(preloaded into a Python process of its own, no GPU): launches do nothing and
are recorded by kernel name, so that a CPU test can tell which kernel a call
takes.  256 CUs of 160 KB LDS.  With FP4X_TEST_REFUSE=1 hipFuncSetAttribute
fails and leaves its error for hipGetLastError, as the runtime does."""
import os
import shutil
import subprocess
import sys

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
PKG = os.path.join(ROOT, "qwen3.8-flash-next-fp4-local-spark_amd")

RUNTIME = r"""
#include <cstddef>
#include <cstdlib>
#include <map>
#include <string>
struct dim3_ { unsigned x, y, z; };
static std::map<const void*, std::string>& names() { static auto* m = new std::map<const void*, std::string>; return *m; }
static std::string& log_() { static auto* s = new std::string; return *s; }
static int last = 0;
static dim3_ cfg_grid, cfg_block;
extern "C" {
void** __hipRegisterFatBinary(const void*) { static void* h; return &h; }
void __hipUnregisterFatBinary(void**) {}
void __hipRegisterFunction(void**, const void* host, char*, const char* name, unsigned, void*, void*, void*, void*, int*) {
  names()[host] = name;
}
void __hipRegisterVar(void**, void*, char*, const char*, int, size_t, int, int) {}
int hipGetDevice(int* d) { *d = 0; return 0; }
int hipDeviceGetAttribute(int* v, int, int) { *v = 256; return 0; }
int hipFuncSetAttribute(const void*, int, int) {
  const char* e = getenv("FP4X_TEST_REFUSE");
  return e && e[0] == '1' ? (last = 1) : 0;
}
int hipOccupancyMaxActiveBlocksPerMultiprocessor(int* n, const void*, int, size_t) { *n = 4; return 0; }
int hipGetLastError(void) { int e = last; last = 0; return e; }
int hipPeekAtLastError(void) { return last; }
const char* hipGetErrorString(int) { return "stand-in"; }
int __hipPushCallConfiguration(dim3_ g, dim3_ b, size_t, void*) { cfg_grid = g; cfg_block = b; return 0; }
int __hipPopCallConfiguration(dim3_* g, dim3_* b, size_t* s, void** st) {
  *g = cfg_grid; *b = cfg_block; *s = 0; *st = nullptr; return 0;
}
int hipLaunchKernel(const void* fn, dim3_, dim3_, void**, size_t, void*) {
  log_() += names()[fn] + "\n";
  return 0;
}
const char* fp4x_test_log(void) { return log_().c_str(); }
void fp4x_test_clear(void) { log_().clear(); }
}
"""

PRELUDE = r"""
import ctypes, json, os, sys
import _fp4x as B
L = B.lib()
rt = ctypes.CDLL(os.environ["FP4X_TEST_RUNTIME"])
rt.fp4x_test_log.restype = ctypes.c_char_p
P = ctypes.c_void_p(1 << 40)                       # planes, never read: nothing runs
FMT = {"mx8": B.FMT_MX8, "w8": B.FMT_W8_F32, "w8_f16": B.FMT_W8_F16, "w6": B.FMT_W6, "nv4": B.FMT_NV4,
       "bf16": B.FMT_BF16}


def launched(fn, *args):
    # (status, names of the kernels that one call launches)
    rt.fp4x_test_clear()
    rc = fn(*args)
    return rc, rt.fp4x_test_log().decode().split()


def linear(fmt, M, N, K, ks=1, scales=P, out=B.DT_F32):
    # the linear of up to 16 rows
    part, tick = (P, P) if ks > 1 else (None, None)
    tail = (P, out, M, N, K, ks, part, tick, None)
    if fmt == "mx8":
        return launched(L.fp4x_mx8_linear, P, K, P, scales, *tail)
    if fmt == "bf16":
        return launched(L.fp4x_bf16_linear, P, K, P, *tail)
    if fmt == "w6":
        return launched(L.fp4x_w6_linear, P, K, P, P, scales, *tail)
    if fmt == "nv4":
        return launched(L.fp4x_nv4_linear, P, K, P, scales, 1.0, *tail)
    return launched(L.fp4x_w8_linear, P, K, P, scales, B.DT_F16 if fmt == "w8_f16" else B.DT_F32, *tail)


def rows(fmt, M, N, K, scales=P, out=B.DT_F32):
    # the linear of any number of rows
    return launched(L.fp4x_linear_rows, FMT[fmt], P, K, P, P if fmt == "w6" else None,
                    None if fmt == "bf16" else scales, 1.0, P, out, M, N, K, None)


def switches(**env):
    for k, v in env.items():
        os.environ.pop(k, None)
        if v is not None:
            os.environ[k] = v
    B.reload_env()
"""


def available():
    return shutil.which("g++") is not None and os.path.exists(os.path.join(PKG, "libfp4x.so"))


def build(folder):
    src, so = os.path.join(folder, "runtime.cpp"), os.path.join(folder, "runtime.so")
    with open(src, "w") as f:
        f.write(RUNTIME)
    r = subprocess.run(["g++", "-O1", "-shared", "-fPIC", src, "-o", so], capture_output=True, text=True)
    assert r.returncode == 0, r.stderr[-2000:]
    return so


def run(so, code, **env):
    """Runs PRELUDE and code with the stand-in; the output of its prints."""
    full = {**{k: v for k, v in os.environ.items() if not k.startswith("FP4X_")}, "PYTHONPATH": PKG,
            "FP4X_TEST_RUNTIME": so, **env}
    full["LD_PRELOAD"] = " ".join(filter(None, [so, os.environ.get("LD_PRELOAD")]))
    r = subprocess.run([sys.executable, "-c", PRELUDE + code], capture_output=True, text=True, env=full, timeout=300)
    assert r.returncode == 0, r.stdout[-1500:] + r.stderr[-3000:]
    return r.stdout
