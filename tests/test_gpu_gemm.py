"""GPU parity of the blocked GEMM (csrc/fp4x_gemm.h): more than 16 rows, and
the shapes of up to 16 rows that fall to it.

fp32 outputs lie within the MFMA accumulation bound of the exact (float64)
sum (oracle.ordered.mfma_bound; a K split over up to 10 waves adds as many
additions as a K split over 10 slices) and bf16 outputs are the same sums
rounded.  Every tile shape runs in every format (TILES; test_routes.py checks
on the CPU that these sizes take them), off the edges of its row tile (16 ..
128), column tile (16 .. 128) and 128-value K units, with odd N, with fewer
units than waves and with enough for the ring to wrap; other sizes sit at
exact tiles and at the smallest ones.
"""
import numpy as np
import pytest
import torch

from oracle import formats as fm
from oracle import gemv as og
from oracle import ordered

from gpu_helpers import act, bf16_bits, bf16_dev, path_switch, to_f32
from test_gpu_gemv import prep, run

pytestmark = pytest.mark.gpu

FMTS = ["mx8", "w8", "w8_f16", "w6", "nv4", "bf16"]

# tile shape (MT, NT, WN, WK, D): sizes M, N, K that the launcher takes it for
# in every format on 256 CUs (the 16-bit tails of an odd scale plane are at
# K % 128 == 64 and N odd)
TILES = {
    (1, 1, 1, 8, 1): [(17, 33, 192), (31, 33, 1984)],
    (1, 1, 1, 10, 2): [(17, 33, 1088), (31, 33, 3136)],
    (1, 2, 1, 8, 1): [(33, 2049, 320), (33, 2049, 1984)],
    (2, 1, 1, 8, 1): [(81, 1345, 320), (145, 801, 960)],
    (2, 1, 4, 2, 3): [(17, 2049, 192), (17, 8193, 704)],
    (2, 2, 1, 8, 1): [(17, 4097, 576), (17, 4097, 1984)],
    (3, 1, 2, 4, 2): [(17, 4097, 320), (33, 4097, 1344)],
    (3, 1, 4, 2, 2): [(33, 8193, 192), (33, 8193, 704)],
    (4, 1, 4, 2, 2): [(50, 8193, 192), (50, 8193, 704)],
    (4, 1, 8, 1, 2): [(50, 16385, 192), (50, 16385, 704)],
    (8, 1, 8, 1, 2): [(65, 16385, 192), (100, 16385, 704)],
}
UP_TO_16 = [(3, 7001, 1920), (5, 1280, 2560), (9, 512, 2560), (13, 96, 1088), (16, 2560, 6144), (16, 2560, 640),
            (16, 5000, 1984)]


@pytest.fixture(scope="module")
def F():
    import fp4x_kernels
    return fp4x_kernels


def planes_of(fmt, rng, n, k):
    planes, w_op, gs = prep("w8" if fmt == "w8_f16" else fmt, rng, n, k)
    if fmt == "w8_f16":
        planes = (planes[0], planes[1].half())
        w_op = og.operand("w8", planes[0].cpu().numpy(), planes[1].float().cpu().numpy())
    return planes, w_op, gs


def took(fmt, planes, gs, xd, N):
    """fp4x_linear_rows's own result, or None where it leaves the call to the
    16-row launches (a scale plane of under 4 bytes)."""
    import _fp4x as B
    code = {"mx8": B.FMT_MX8, "w8": B.FMT_W8_F32, "w8_f16": B.FMT_W8_F16, "w6": B.FMT_W6, "nv4": B.FMT_NV4,
            "bf16": B.FMT_BF16}[fmt]
    M, K = xd.shape
    w1, s = (planes[1], planes[2]) if fmt == "w6" else (None, None if fmt == "bf16" else planes[1])
    y = torch.empty((M, N), dtype=torch.float32, device=xd.device)
    rc = B.lib().fp4x_linear_rows(code, B.ptr(xd), xd.stride(0), B.ptr(planes[0]), B.ptr(w1), B.ptr(s), gs, B.ptr(y),
                                  B.DT_F32, M, N, K, B.stream_of(xd))
    small = s is not None and s.numel() * s.element_size() < 4
    assert rc == (B.NOT_TAKEN if small else B.OK), rc
    return None if small else to_f32(y)


def check(F, fmt, planes, w_op, gs, x, xd):
    base = "w8" if fmt == "w8_f16" else fmt
    y = to_f32(run(F, base, xd, planes, 1, torch.float32))
    exact = ordered.exact_sum(x, w_op) * gs
    bound = ordered.mfma_bound(x, w_op, 10) * abs(gs)
    assert np.all(np.abs(y - exact) <= bound), (np.abs(y - exact) / bound).max()
    assert np.array_equal(bf16_bits(run(F, base, xd, planes, 1)), fm.bf16_bits(y))
    if x.shape[0] > 16:
        own = took(fmt, planes, gs, xd, y.shape[1])
        assert own is None or np.array_equal(own.view(np.uint32), y.view(np.uint32)), "the blocked GEMM did not run"
    return y


@pytest.mark.parametrize("fmt", FMTS)
@pytest.mark.parametrize("M,N,K", [size for sizes in TILES.values() for size in sizes])
def test_gemm_every_tile_shape(gpu, F, fmt, M, N, K):
    rng = np.random.default_rng(M + N + K)
    planes, w_op, gs = planes_of(fmt, rng, N, K)
    x, _ = act(rng, M, K)
    check(F, fmt, planes, w_op, gs, x, bf16_dev(x))


@pytest.mark.parametrize("fmt", FMTS)
@pytest.mark.parametrize("M,N,K", [(17, 1, 64), (17, 33, 192), (24, 640, 640), (31, 1000, 1088), (40, 130, 2560),
                                   (48, 4100, 576), (65, 97, 1344), (100, 513, 320), (129, 301, 128), (200, 8200, 256),
                                   (256, 1025, 704)])
def test_gemm_rows(gpu, F, fmt, M, N, K):
    rng = np.random.default_rng(M + N + K)
    planes, w_op, gs = planes_of(fmt, rng, N, K)
    x, _ = act(rng, M, K)
    y = check(F, fmt, planes, w_op, gs, x, bf16_dev(x))
    # rows of x further apart than K, in the middle of another tensor
    wide = torch.full((M + 2, K + 24), float("nan"), dtype=torch.bfloat16, device="cuda")
    wide[1:-1, 8:K + 8] = bf16_dev(x)
    y2 = to_f32(run(F, "w8" if fmt == "w8_f16" else fmt, wide[1:-1, 8:K + 8], planes, 1, torch.float32))
    assert np.array_equal(y.view(np.uint32), y2.view(np.uint32))


@pytest.mark.parametrize("fmt", FMTS)
@pytest.mark.parametrize("M,N,K", UP_TO_16)
def test_gemm_up_to_16_rows(gpu, F, fmt, M, N, K, monkeypatch):
    """Shapes of up to 16 rows that fall to it (two of them in some formats only:
    test_routes.py), against the exact sums; FP4X_GEMM=0 (the MFMA core or the few-rows kernel) stays within the same
    bound."""
    rng = np.random.default_rng(M + N + K)
    planes, w_op, gs = planes_of(fmt, rng, N, K)
    x, _ = act(rng, M, K)
    check(F, fmt, planes, w_op, gs, x, bf16_dev(x))
    with path_switch(monkeypatch, "FP4X_GEMM"):
        check(F, fmt, planes, w_op, gs, x, bf16_dev(x))


@pytest.mark.parametrize("fmt", FMTS)
@pytest.mark.parametrize("M,N", [(17, 17), (40, 33), (130, 4099), (33, 2)])
def test_gemm_one_unit_rows(gpu, F, fmt, M, N):
    """K = 64: rows of half a unit and, for MXFP8 and fp16 W8 scales, of two
    scale bytes, so that with N odd the last row begins past the scale plane's
    last whole dword (where the loads go is checked in test_gemm_scales.py)."""
    rng = np.random.default_rng(M + N)
    planes, w_op, gs = planes_of(fmt, rng, N, 64)
    x, _ = act(rng, M, 64)
    check(F, fmt, planes, w_op, gs, x, bf16_dev(x))


@pytest.mark.parametrize("M,N", [(20, 260), (20, 261), (50, 16385)])
def test_gemm_fp16_output(gpu, F, M, N):
    """fp16 outputs are the fp32 ones rounded."""
    rng = np.random.default_rng(N)
    planes, _, _ = planes_of("w8", rng, N, 320)
    xd = bf16_dev(act(rng, M, 320)[0])
    y = run(F, "w8", xd, planes, 1, torch.float32)
    assert torch.equal(run(F, "w8", xd, planes, 1, torch.float16), y.half())


def test_gemm_bf16_short_tail(gpu, F):
    """K a multiple of 16 only (bf16)."""
    rng = np.random.default_rng(5)
    planes, w_op, gs = planes_of("bf16", rng, 75, 208)
    x, _ = act(rng, 37, 208)
    xd = bf16_dev(x)
    y = to_f32(F.bf16_linear(xd, *planes, (32, 16, 1, 4), torch.float32))
    assert np.all(np.abs(y - ordered.exact_sum(x, w_op)) <= ordered.mfma_bound(x, w_op, 10))


@pytest.mark.parametrize("M,N,K", [(3, 3001, 1088), (20, 3001, 1088), (70, 3001, 1088), (33, 8193, 704),
                                   (50, 16385, 704)])
def test_gemm_special_values(gpu, F, M, N, K):
    """MXFP8 exponent 255 (scale +inf) gives +-inf or NaN in its own columns
    only, NaN and inf activations reach their own rows only, as one launch per
    16 rows gives them; K not a multiple of 128, N odd; K parts in 8, 2 and no
    other waves."""
    rng = np.random.default_rng(M)
    (w, s), _, _ = prep("mx8", rng, N, K)
    s = s.clone()
    s[7, 3] = 255
    s[N - 1, K // 32 - 1] = 255
    x = torch.from_numpy(rng.standard_normal((M, K)).astype(np.float32)).to("cuda").to(torch.bfloat16)
    x[1, 40] = float("inf")
    x[2, K - 1] = float("nan")
    got = F.mx8_linear(x, w, s, (32, 64, 1, 4), torch.float32)
    want = torch.cat([x[m:m + 1].double() @ F.dequant_operand("mx8", w, None, s, K=K).double().T for m in range(M)])
    assert torch.equal(torch.isnan(got), torch.isnan(want))
    assert torch.equal(torch.isinf(got), torch.isinf(want))
    inf = torch.isinf(want)
    assert torch.equal(got[inf].double(), want[inf])
    assert not torch.isfinite(got[:, 7]).any() and torch.isfinite(got[0, 8:N - 1]).all()


def test_gemm_unaligned_falls_back(gpu, F):
    """Scales that are only 2-byte aligned take the 16-row launches, with the
    same results as an aligned copy within the bound."""
    rng = np.random.default_rng(9)
    (P, S, gs), w_op, _ = prep("nv4", rng, 260, 640)
    buf = torch.zeros(S.numel() + 2, dtype=torch.uint8, device="cuda")
    buf[2:] = S.view(torch.uint8).view(-1)
    S2 = buf[2:].view(S.shape).view(torch.float8_e4m3fn)
    assert S2.data_ptr() % 4 == 2
    x, _ = act(rng, 21, 640)
    for scales in (S, S2):
        y = to_f32(F.nv4_linear(bf16_dev(x), P, scales, gs, (32, 64, 4), torch.float32))
        assert np.all(np.abs(y - ordered.exact_sum(x, w_op) * gs) <= ordered.mfma_bound(x, w_op, 10) * gs)


def test_gemm_graph(gpu, F):
    """Captured and replayed with the program's own work in between."""
    rng = np.random.default_rng(11)
    planes, _, _ = planes_of("w6", rng, 1000, 1088)
    x = bf16_dev(act(rng, 50, 1088)[0])
    want = run(F, "w6", x, planes, 1)
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g):
        y = run(F, "w6", x, planes, 1)
    for _ in range(3):
        y.zero_()
        g.replay()
        torch.cuda.synchronize()
        assert torch.equal(y, want)
        assert torch.equal(run(F, "w6", x, planes, 1), want)


@pytest.mark.parametrize("fmt", ["mx8", "w8", "w6", "nv4", "bf16"])
@pytest.mark.parametrize("K,bk,ks", [(512, 8, 64), (8320, 64, 130), (8320, 64, 65)])
def test_gemm_refuses_bad_k_splits(gpu, F, fmt, K, bk, ks):
    """K splits that 16 rows refuse (slices that are no whole chunks, or more
    than 64 of them) are refused for more rows too; a good one is accepted."""
    rng = np.random.default_rng(ks)
    planes, _, _ = planes_of(fmt, rng, 32, K)
    x = bf16_dev(act(rng, 20, K)[0])

    def call(m, bk, ks, planes=planes):
        cfg = (32, bk, 4, ks) if fmt == "nv4" else (32, bk, ks, 4)
        fn = {"mx8": F.mx8_linear, "w8": F.w8_linear, "w6": F.w6_linear, "nv4": F.nv4_linear, "bf16": F.bf16_linear}[fmt]
        return fn(x[:m], *planes, cfg)
    for m in (16, 20):
        with pytest.raises(ValueError):
            call(m, bk, ks)
    assert call(20, 32, 2).shape == (20, 32)
    none = [t[:0] if torch.is_tensor(t) else t for t in planes]
    for m in (16, 20):                               # no weight rows
        assert call(m, 32, 2, none).shape == (m, 0)
