"""The binary16 row pack on both sides of 64 chunks of four per row (256 floats), where its grid changes: rows of one
chunk to a few workgroups, row strides wider than the row, row counts that fill no workgroup; against the F16C
conversion of the oracle, with the bytes between the rows left alone."""
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


@pytest.mark.parametrize("row_len", [4, 8, 12, 60, 64, 128, 192, 248, 252, 256, 260, 512, 1020, 1024, 1028, 2052])
@pytest.mark.parametrize("rows", [1, 3, 65, 257, 70000])
def test_row_lengths(ops, oracle, row_len, rows):
    if rows == 70000 and row_len > 260:
        rows = 4099
    src = C.normal(row_len + rows, (rows, 2 * row_len + 8), 3.0)
    src[0, 0], src[rows - 1, row_len - 1], src[rows // 2, row_len] = np.inf, -1e9, np.nan
    t = torch.from_numpy(src).cuda()
    ks, vs = t[:, :row_len], t[:, row_len:2 * row_len]
    bufs = [torch.full((rows, row_len + pad), 7.0, dtype=torch.float16, device="cuda") for pad in (4, 0, 8)]
    ops.kv_pack_f16(ks, bufs[0][:, :row_len])
    ops.kv_pack_f16_kv(ks, vs, bufs[1], bufs[2][:, :row_len])
    for buf, want in zip(bufs, (src[:, :row_len], src[:, :row_len], src[:, row_len:2 * row_len])):
        got = buf.cpu().numpy()
        bits, ref = got[:, :row_len].view(np.uint16), oracle.kv_pack_f16(np.ascontiguousarray(want))
        nan = np.isnan(want)
        assert np.array_equal(bits[~nan], ref[~nan]) and np.all(np.isnan(got[:, :row_len][nan]))
        assert np.all(got[:, row_len:] == 7.0)
