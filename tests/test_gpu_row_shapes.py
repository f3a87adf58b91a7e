"""add+RMSNorm, RMSNorm and RMSNorm -> Q8 on both sides of every line where the row kernels change shape (row
lengths at the edges of the threads-per-row and chunks-per-thread steps, leftover 8-float blocks, one row to more
rows than one round of workgroups), bit for bit against the oracle on the first, last and a few other rows."""
from __future__ import annotations

import numpy as np
import pytest

from tests import common as C

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")


@pytest.fixture(scope="module")
def ops():
    if not torch.cuda.is_available():
        pytest.fail("GPU tests need a visible MI355X")
    from v7multiplikator_amd import _lib
    from v7multiplikator_amd import ops as _ops
    _lib.load()
    return _ops


def same(a, b):
    a, b = np.asarray(a), np.asarray(b)
    if a.dtype == np.float32:
        a, b = a.view(np.uint32), b.view(np.uint32)
    return a.shape == b.shape and np.array_equal(a, b)


DIMS = [8, 32, 64, 248, 256, 288, 480, 512, 544, 768, 1000, 1024, 1056, 1984, 2048, 2080, 2336, 3072, 4064, 4096,
        4104, 4128, 5376, 7808, 8160, 8192, 8200, 8224, 9216, 11008, 12288, 12320, 15360, 15392, 16352, 16376, 16384]


@pytest.mark.parametrize("dim", DIMS)
@pytest.mark.parametrize("rows", [1, 256, 257, 513, 1025, 2049])
def test_row_shapes(ops, oracle, dim, rows):
    g = torch.Generator(device="cuda").manual_seed(dim * 31 + rows)
    x = torch.randn(rows, dim, generator=g, device="cuda")
    a = torch.randn(rows, dim, generator=g, device="cuda")
    w = 1 + 0.1 * torch.randn(dim, generator=g, device="cuda")
    pick = sorted({0, rows // 3, rows // 2, rows - 1})
    h = lambda t: t[pick].cpu().numpy()  # noqa: E731
    xh, ah, wh = h(x), h(a), w.cpu().numpy()

    r = x.clone()
    out = ops.fused_add_rmsnorm(r, a, w, eps=1e-6)
    want_o, want_r = oracle.fused_add_rmsnorm(xh, ah, wh, 1e-6)
    assert same(h(out), want_o) and same(h(r), want_r)
    assert torch.equal(r, x + a)  # every residual element, not the picked rows alone
    if dim % 32 == 0:
        assert same(h(ops.rmsnorm(x, w, eps=1e-6)), oracle.rmsnorm(xh, wh, 1e-6))
    for gs in (32, 64):
        if dim % gs == 0:
            q, s = ops.rmsnorm_quantize(x, w, eps=1e-6, gs=gs)
            wq, ws = oracle.rmsnorm_quantize(xh, wh, 1e-6, gs)
            assert same(h(q), wq) and same(h(s), ws)
            r = x.clone()
            q, s = ops.add_rmsnorm_quantize(r, a, w, eps=1e-6, gs=gs)
            wq, ws = oracle.rmsnorm_quantize(want_r, wh, 1e-6, gs)
            assert same(h(q), wq) and same(h(s), ws) and same(h(r), want_r)


# With these widths and row counts every row kernel that is built runs.
ALL_DIMS = [64, 136, 248, 256, 264, 288, 320, 480, 512, 520, 544, 576, 640, 768, 776, 832, 904, 960, 1000, 1024, 1032,
            1056, 1160, 1280, 1344, 1480, 1536, 1792, 1984, 2048, 2056, 2080, 2112, 2304, 2560, 2600, 2816, 3072, 3080,
            3200, 3584, 3840, 4064, 4096, 4104, 4288, 4608, 4864, 5000, 5120, 5376, 5632, 6008, 6144, 6656, 7168, 7680,
            7808, 8160, 8192, 8200, 8448, 9216, 9992, 10112, 11008, 12008, 12288, 12320, 13312, 13824, 14336, 15360,
            16320, 16376, 16384]
ALL_ROWS = [1, 2, 200, 257, 449, 513, 600, 769, 900, 1025, 1200, 1300, 1537, 1800, 2049, 5001, 6200, 7000, 8192]


@pytest.mark.parametrize("dim", ALL_DIMS)
def test_every_row_kernel(ops, oracle, dim):
    """Every row count at which some width changes its kernel, codes on and 4 bytes off their 16-byte boundary; a row
    of denormals and one with an Inf among the compared ones, and nothing written beside the results."""
    most = max(r for r in ALL_ROWS if r * dim <= 24_000_000)
    g = torch.Generator(device="cuda").manual_seed(dim)
    X = torch.randn(most, dim, generator=g, device="cuda")
    A = torch.randn(most, dim, generator=g, device="cuda")
    w = 1 + 0.1 * torch.randn(dim, generator=g, device="cuda")
    wh = w.cpu().numpy()
    for rows in ALL_ROWS:
        if rows > most:
            break
        x, a = X[:rows].clone(), A[:rows].clone()
        pick = sorted({0, rows // 3, rows // 2, rows - 1})
        x[pick[-1]] *= 2.0 ** -130
        a[pick[-1]] = 0.0
        if rows > 4:
            x[pick[1], dim // 2] = float("inf")
        h = lambda t: t[pick].cpu().numpy()  # noqa: E731
        xh, ah = h(x), h(a)
        r, out = x.clone(), torch.full((rows * dim + 64,), 7.0, device="cuda")
        ops.fused_add_rmsnorm(r, a, w, eps=1e-6, out=out[:rows * dim].view(rows, dim))
        want_o, want_r = oracle.fused_add_rmsnorm(xh, ah, wh, 1e-6)
        assert nan_same(h(out[:rows * dim].view(rows, dim)), want_o) and same(h(r), want_r), rows
        assert torch.all(out[rows * dim:] == 7.0)
        if dim % 32 == 0:
            assert nan_same(h(ops.rmsnorm(x, w, eps=1e-6)), oracle.rmsnorm(xh, wh, 1e-6)), rows
        for gs in (32, 64):
            if dim % gs:
                continue
            for off in (0, 4):
                q = torch.full((rows * dim + 64,), 77, dtype=torch.int8, device="cuda")
                codes = q[off:off + rows * dim].view(rows, dim)
                _, s = ops.rmsnorm_quantize(x, w, eps=1e-6, gs=gs, out_q=codes)
                wq, ws = oracle.rmsnorm_quantize(xh, wh, 1e-6, gs)
                assert same(h(codes), wq) and same(h(s), ws), (rows, gs, off)
                r = x.clone()
                _, s = ops.add_rmsnorm_quantize(r, a, w, eps=1e-6, gs=gs, out_q=codes)
                wq, ws = oracle.rmsnorm_quantize(want_r, wh, 1e-6, gs)
                assert same(h(codes), wq) and same(h(s), ws) and same(h(r), want_r), (rows, gs, off)
                assert torch.all(q[:off] == 77) and torch.all(q[off + rows * dim:] == 77)


def nan_same(a, b):
    """Bits, with any NaN for any NaN."""
    a, b = np.asarray(a), np.asarray(b)
    return np.array_equal(np.isnan(a), np.isnan(b)) and same(np.where(np.isnan(a), 0, a), np.where(np.isnan(b), 0, b))
