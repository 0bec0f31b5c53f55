"""Which kernel a dense linear launches, without a GPU (tests/standin.py, 256
CUs): the path switches, the mixer's up projection, the lines between the
few-rows kernels and the blocked GEMM, and the tile shapes that the GEMM's GPU
tests mean to run."""
import pytest

import standin
from test_gpu_gemm import TILES, UP_TO_16


@pytest.fixture(scope="module")
def route(tmp_path_factory):
    if not standin.available():
        pytest.skip("no g++ or no library")
    so = standin.build(tmp_path_factory.mktemp("standin"))
    return lambda code, **env: standin.run(so, code, **env)


def test_switches_that_force_the_core(route):
    """FP4X_ROWS=0 and a format's stream switch send its calls to the MFMA core
    also where the blocked GEMM would take them, for any number of rows."""
    route(r"""
STREAM = {"mx8": "FP4X_MX8_STREAM", "w8": "FP4X_W8_STREAM", "w8_f16": "FP4X_W8_STREAM", "w6": "FP4X_W6_STREAM",
          "nv4": "FP4X_NV4_STREAM"}
for fmt in FMT:
    for M, N, K in ((16, 8300, 1984), (6, 5000, 1920), (13, 1600, 1088), (24, 512, 2560), (256, 16384, 2560)):
        call = linear if M <= 16 else rows
        rc, names = call(fmt, M, N, K)
        assert rc == B.OK and "gemm_kernel" in names[0], (fmt, M, N, K, names)
        for env in ("FP4X_GEMM", "FP4X_ROWS", STREAM.get(fmt)):
            if env is None:
                continue
            switches(**{env: "0"})
            rc, names = call(fmt, M, N, K)
            switches(**{env: None})
            if M > 16:
                assert rc == B.NOT_TAKEN and not names, (fmt, M, N, K, env, names)
            else:
                assert rc == B.OK and "gemv_mfma_kernel" in names[0], (fmt, M, N, K, env, names)
""")


def test_mixer_up_projection_stays_on_the_core(route):
    """[4 H x lr] through w8_linear at 5 to 16 rows, which streams only where lr
    is a multiple of 512: on the MFMA core, whose sums hc_up reproduces, over
    hidden widths and ranks as far apart as H = 1.6 lr."""
    route(r"""
for h in range(1024, 2817, 64):
    for lr in range(192, 641, 64):
        for M in (5, 16):
            for fmt in ("w8", "w8_f16"):
                rc, names = linear(fmt, M, 4 * h, lr)
                assert rc == B.OK and "gemm_kernel" not in names[0], (h, lr, M, fmt, names)
                assert "gemv_mfma_kernel" in names[0] or lr % 512 == 0, (h, lr, M, fmt, names)
""")


def test_few_rows_lines(route):
    """Matrices of few rows at 9 to 16 activation rows, on either side of the
    lines between the few-rows kernels and the blocked GEMM (measured beside
    gemm_before_rows); over 4 rows per CU, and rows too long for the few-rows
    kernels, the GEMM takes all of them."""
    route(r"""
def gemm(fmt, M, N, K, ks=1):
    rc, names = linear(fmt, M, N, K, ks)
    assert rc == B.OK and len(names) == 1, (fmt, M, N, K, names)
    assert "gemm_kernel" in names[0] or "rows_mfma_kernel" in names[0], (fmt, M, N, K, names)
    return "gemm_kernel" in names[0]


for N in (1, 96, 512, 1024):
    for M in range(5, 17):
        for K in (512, 1088, 1984, 2048, 2560, 4032, 4096, 6144):
            for fmt in FMT:
                above = {"nv4": (12, 8, 10), "mx8": (16, 10, 14)}.get(fmt, (12, 10, 14))[(K >= 2048) + (K >= 4096)]
                assert gemm(fmt, M, N, K) == (M > above), (fmt, M, N, K, above)
for fmt in FMT:
    assert gemm(fmt, 13, 1025, 2112) and gemm(fmt, 9, 2000, 1088) and gemm(fmt, 13, 512, 10304)
    if not fmt.startswith("w8"):
        assert gemm(fmt, 13, 1025, 2112, 2)
""")


def test_gpu_gemm_sizes_take_their_tiles(route):
    """The sizes of test_gpu_gemm.py take the tile shapes and kernels that it
    says, in every format."""
    route(f"TILES, UP_TO_16 = {TILES!r}, {UP_TO_16!r}" + r"""
import re


def tile(names):
    return tuple(int(v) for v in re.findall(r"Li(\d+)E", re.search(r"gemm_kernel\S*?((?:Li\d+E){5})", names[0]).group(1)))


for want, sizes in TILES.items():
    for M, N, K in sizes:
        for fmt in FMT:
            rc, names = rows(fmt, M, N, K)
            assert rc == B.OK and tile(names) == want, (fmt, M, N, K, names, want)
some = {(9, 512, 2560): ("nv4",), (13, 96, 1088): ("w8", "w8_f16", "w6", "nv4", "bf16")}
for size in UP_TO_16:
    for fmt in FMT:
        rc, names = linear(fmt, *size)
        assert rc == B.OK and ("gemm_kernel" in names[0]) == (fmt in some.get(size, FMT)), (fmt, size, names)
# exponent 255 of MXFP8 with K parts in 8, 2 and no other waves
assert [tile(rows("mx8", *s)[1])[3] for s in ((20, 3001, 1088), (33, 8193, 704), (50, 16385, 704))] == [8, 2, 1]
""")
