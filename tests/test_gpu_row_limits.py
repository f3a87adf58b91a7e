"""Row counts at which one workgroup per row would be 2^32 threads and more, which HIP refuses: the same bits as calls
over a few of the rows, at both ends and around the row where the second launch begins."""
from __future__ import annotations

import pytest

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


@pytest.mark.parametrize("rows,dim", [((1 << 24) + 5, 520), ((1 << 22) + 5, 4104)])
def test_add_rmsnorm_rows_past_one_grid(ops, rows, dim):
    torch.cuda.empty_cache()
    free, _ = torch.cuda.mem_get_info()
    if free < 9 * rows * dim:
        pytest.skip("needs 9 bytes of free device memory per element")
    residual, add = torch.rand(rows, dim, device="cuda"), torch.rand(rows, dim, device="cuda")
    weight = torch.rand(dim, device="cuda")
    # both ends, and the rows at which a launch of 1024, 512 or 256 threads a row has to end
    starts = sorted({0, rows - 8, *(min(r - 4, rows - 8) for r in (1 << 22, 1 << 23, (1 << 24) - 1))})
    want = []
    for r0 in starts:
        r = residual[r0:r0 + 8].clone()
        want.append(ops.fused_add_rmsnorm(r, add[r0:r0 + 8], weight))
    ops.fused_add_rmsnorm(residual, add, weight, out=residual)  # in place: the row ends as the result
    for r0, w in zip(starts, want):
        assert torch.equal(residual[r0:r0 + 8], w), r0
