"""Where the blocked GEMM's scale loads read (GemmScales of csrc/fp4x_gemm.h,
compiled for the host): every dword that the kernel asks for lies within the
scale plane and holds the bytes that the unit's lanes take from it, for every
row-byte count a format has (2 to 8 per 64 or 128 K values), every N around
the strips' edges, and every strip base the tile shapes make, among them the
last row, which the columns past N are clamped to."""
import os
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
CSRC = os.path.join(ROOT, "qwen3.8-flash-next-fp4-local-spark_amd", "csrc")

PROGRAM = r"""
#include "fp4x_gemm.h"
#include <cstdio>
using namespace fp4x;

static long bad = 0, seen = 0;

// one strip of 16 rows based at ns, its row r at ns + (r >> 2) * 4 nt + (r & 3)
static void strip(int64_t ns, int64_t N, int K, int ub, int nt) {
  const uint8_t* plane = reinterpret_cast<const uint8_t*>(uintptr_t(1) << 40);
  const int rb = ub * K / kGemmKB, units = (K + kGemmKB - 1) / kGemmKB;
  const int64_t bytes = N * rb, left = N - 1 - ns;
  const int lim = left < 16 * nt ? (int)left : 16 * nt;
  for (int r = 0; r < 16; ++r) {
    const int rm = (r >> 2) * 4 * nt + (r & 3), row = rm < lim ? rm : lim;
    GemmScales g;
    g.set(plane, ns, row, rb, N);
    for (int ku = 0; ku < units; ++ku) {
      const int64_t want = (ns + row) * rb + ku * ub;      // the unit's first scale byte
      const int need = ku * kGemmKB + kGemmKB <= K ? ub : ub / 2;
      for (int d = 0; d < 2; ++d) {
        const int64_t a = g.at(ku, ub, d) - plane;
        ++seen;
        bool ok = a >= 0 && a + 4 <= bytes && a % 4 == 0;
        // the dword that holds wanted bytes is that one, unless it runs past
        // the plane (the last two bytes of an odd plane are read apart)
        const int64_t own = want / 4 * 4 + 4 * d;
        if (own < want + need && own + 4 <= bytes) ok &= a == own;
        if (!ok && bad++ < 5)
          printf("K=%d N=%lld ub=%d nt=%d strip %lld row %d unit %d dword %d: byte %lld of %lld\n", K, (long long)N, ub,
                 nt, (long long)ns, row, ku, d, (long long)a, (long long)bytes);
      }
    }
  }
}

int main() {
  for (int ub : {4, 8})                                    // MXFP8, W8 fp16: 4 bytes per 128 values; the others 8
    for (int K = 64; K <= 1088; K += 64)
      for (int64_t N = 1; N <= 140; ++N) {
        if (N * ub * K / kGemmKB < 4) continue;            // not taken
        for (int nt = 1; nt <= 2; ++nt)
          for (int64_t n0 = 0; n0 < (N + 127) / 128 * 128; n0 += 16 * nt)   // also the waves past N
            for (int t = 0; t < nt; ++t) strip(n0 + 4 * t < N ? n0 + 4 * t : N - 1, N, K, ub, nt);
      }
  printf("%ld loads, %ld out of place\n", seen, bad);
  return bad != 0;
}
"""


def test_scale_loads_stay_in_the_plane(tmp_path):
    rocm = os.environ.get("ROCM_PATH", "/opt/rocm")
    hipcc = os.path.join(rocm, "bin", "hipcc")
    hipcc = hipcc if os.path.exists(hipcc) else shutil.which("hipcc")
    if hipcc is None:
        pytest.skip("no hipcc")
    src, exe = tmp_path / "scales.hip", tmp_path / "scales"
    src.write_text(PROGRAM)
    r = subprocess.run([hipcc, "--offload-host-only", "-O2", "-std=c++17", "-I", CSRC, str(src), "-o", str(exe)],
                       capture_output=True, text=True)
    assert r.returncode == 0, r.stderr[-3000:]
    r = subprocess.run([str(exe)], capture_output=True, text=True)
    assert r.returncode == 0, r.stdout[-3000:]
