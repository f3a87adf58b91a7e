"""Q8 quantize and SwiGLU -> Q8 where the group kernel's lanes can go wrong: group sizes on both sides of every
lanes-per-group step, rows that end in a partial group of every length modulo 4, x off its 16-byte boundary and
codes off their 4-byte boundary, NaN and Inf inside full and partial groups; bit for bit against the oracle."""
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


def at_offset(a, off):
    """a on the device, its first element `off` elements past an allocation's start."""
    flat = torch.from_numpy(np.ascontiguousarray(a)).reshape(-1)
    buf = torch.zeros(flat.numel() + off, dtype=flat.dtype, device="cuda")
    buf[off:] = flat.cuda()
    return buf[off:].view(a.shape)


def same(t, want):
    got = t.cpu().numpy()
    if want.dtype == np.float32:
        got, want = got.view(np.uint32), want.view(np.uint32)
    return got.shape == want.shape and np.array_equal(got, want)


GROUPS = [1, 2, 3, 4, 5, 8, 9, 16, 17, 31, 32, 33, 48, 64, 65, 128, 129, 200, 256, 257, 1000, 4096]


@pytest.mark.parametrize("gs", GROUPS)
@pytest.mark.parametrize("row_len,off", [(1, 0), (63, 1), (256, 0), (256, 1), (514, 0), (1025, 3), (4099, 2)])
def test_group_sizes_rows_and_offsets(ops, oracle, gs, row_len, off):
    rows = 5
    rng = C.rng(gs * 7919 + row_len)
    x = C.normal(gs + row_len, (rows, row_len), 2.0)
    u = C.normal(gs + row_len + 1, (rows, row_len), 1.5)
    for r, bad in ((1, np.nan), (2, np.inf), (3, np.nan)):  # row 3: also in its last group
        x[r, rng.integers(0, row_len, 1 + row_len // 200)] = bad
    x[3, row_len - 1] = np.nan
    x[4, row_len // 2] = np.float32(2.0 ** 40)
    q = torch.full((rows * row_len + 3,), 77, dtype=torch.int8, device="cuda")
    codes = q[off:off + rows * row_len].view(rows, row_len)
    wq, ws = oracle.quantize(x, gs)
    _, s = ops.quantize_q8(at_offset(x, off), gs=gs, out_q=codes)
    assert same(codes, wq) and same(s, ws)
    assert torch.all(q[:off] == 77) and torch.all(q[off + rows * row_len:] == 77)  # nothing beside the codes
    wq, ws = oracle.swiglu_q8(x, u, gs)
    _, s = ops.swiglu_q8(at_offset(x, off), at_offset(u, off), gs=gs, out_q=codes)
    assert same(codes, wq) and same(s, ws)


def test_more_lanes_than_32_bits_index(ops):
    """2^31 lanes (a group of 1 per lane) and more take 64-bit indices: the same codes and scales as calls over
    parts of the array, around the 2^31 element boundary and at both ends."""
    rows, row_len = (1 << 31) // 100 + 9, 100
    torch.cuda.empty_cache()
    free, _ = torch.cuda.mem_get_info()
    if free < 40 << 30:
        pytest.skip("needs 40 GB of free device memory")
    x = torch.randn(rows, row_len, device="cuda")
    at = (1 << 31) // row_len
    x[at, 3] = float("nan")
    x[rows - 1, 99] = float("inf")
    q, s = ops.quantize_q8(x, gs=1)
    for r0 in (0, at - 8, rows - 16):
        pq, ps = ops.quantize_q8(x[r0:r0 + 16].contiguous(), gs=1)
        assert torch.equal(q[r0:r0 + 16], pq) and torch.equal(s[r0:r0 + 16], ps)


@pytest.mark.parametrize("gs,row_len,rows", [
    (64, 65, (1 << 26) + 9),   # 16 lanes a group, every second group of one element
    (32, 33, (1 << 27) + 9),   # 8 lanes a group
    (257, 258, (1 << 24) + 9),  # 64 lanes a group that walk it in steps, every second group of one element
    (64, 64, (1 << 28) + 9),   # whole groups, one lane per 4 elements would be 2^32 lanes
])
def test_64_bit_lane_indices_with_partial_groups(ops, gs, row_len, rows):
    """2^31 lanes and more with a 64-bit division of the group index by the groups of a row: the same codes and scales
    as calls over a few rows, at both ends and on both sides of the 2^31st lane and the 2^32nd element."""
    n = rows * row_len
    torch.cuda.empty_cache()
    free, _ = torch.cuda.mem_get_info()
    if free < 7 * n:
        pytest.skip("needs 7 bytes of free device memory per element")
    x = torch.rand(rows, row_len, device="cuda")
    spr = -(-row_len // gs)
    lanes = 64 if gs > 256 else gs // 4
    starts = sorted({0, rows - 16, *(min(max(at - 8, 0), rows - 16) for at in ((1 << 31) // (spr * lanes),
                                                                               (1 << 32) // row_len))})
    for r0 in starts:
        x[r0, row_len - 1] = float("nan")
        x[r0 + 9, 3] = float("inf")
        x[r0 + 10, row_len - 1] = 5.0
    q, s = ops.quantize_q8(x, gs=gs)
    s = s.view(rows, spr)
    for r0 in starts:
        pq, ps = ops.quantize_q8(x[r0:r0 + 16].contiguous(), gs=gs)
        assert torch.equal(q[r0:r0 + 16], pq) and torch.equal(s[r0:r0 + 16], ps.view(16, spr)), r0
