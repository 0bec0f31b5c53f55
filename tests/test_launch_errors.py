"""What the blocked GEMM's launcher leaves behind when the HIP runtime refuses
a kernel's LDS size (tests/standin.py): the call returns FP4X_NOT_TAKEN with no
error set, so the launch that runs instead is not reported as failed."""
import pytest

import standin

CALLS = r"""
refused = 0
for fmt in FMT:
    for M, N, K in ((24, 16384, 2560), (39, 2560, 6144), (256, 16384, 2560), (256, 1280, 2560), (17, 512, 2560)):
        rc, names = rows(fmt, M, N, K)
        assert rc in (B.OK, B.NOT_TAKEN), (fmt, M, N, K, rc, L.fp4x_last_error())
        assert (len(names) == 1) == (rc == B.OK)
        refused += rc == B.NOT_TAKEN
        assert rt.hipPeekAtLastError() == 0, ("error left set", fmt, M, N, K)
assert refused, "no call asked for more than 64 KB of LDS"
"""


def test_refused_lds_size_leaves_no_error(tmp_path):
    if not standin.available():
        pytest.skip("no g++ or no library")
    standin.run(standin.build(tmp_path), CALLS, FP4X_TEST_REFUSE="1")
