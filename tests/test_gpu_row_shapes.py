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
