"""RMSNorm -> Q8 where norm_q8_row16_kernel runs: more than 256 rows of 512 to 12288 floats, codes on a 16-byte boundary.
Its compiled widths and the run-time one, its chain at whole and partial register sets, its ordered vmaxps tree for
NaN and Inf in every position of a group, and denormal rows, bit for bit against the oracle; the same codes as the
row kernel that codes off that boundary take."""
from __future__ import annotations

import numpy as np
import pytest

from tests import common as C
from tests.test_gpu_parity import denormal_mix

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")

ROWS = 257  # the fewest that take the kernel


@pytest.fixture(scope="module")
def ops():
    if not torch.cuda.is_available():
        pytest.fail("GPU tests need a visible MI355X")
    from v7multiplikator_amd import _lib
    from v7multiplikator_amd import ops as _ops
    _lib.load()
    return _ops


def dev(a):
    return torch.from_numpy(np.ascontiguousarray(a)).cuda()


def same(t, want):
    got = t.cpu().numpy()
    if want.dtype == np.float32:
        got, want = got.view(np.uint32), want.view(np.uint32)
    return got.shape == want.shape and np.array_equal(got, want)


def check(ops, oracle, x, a, w, gs, eps=1e-6):
    """Both forms against the oracle, and against the row kernel through codes 4 bytes off."""
    rows, dim = x.shape
    assert rows > 256 and 512 <= dim <= 12288
    wq, ws = oracle.rmsnorm_quantize(x, w, eps, gs)
    q, s = ops.rmsnorm_quantize(dev(x), dev(w), eps=eps, gs=gs)
    assert q.data_ptr() % 16 == 0
    assert same(q, wq) and same(s, ws)
    r_new = oracle.add_inplace(x, a)
    wq, ws = oracle.rmsnorm_quantize(r_new, w, eps, gs)
    r = dev(x)
    q, s = ops.add_rmsnorm_quantize(r, dev(a), dev(w), eps=eps, gs=gs)
    assert same(r, r_new) and same(q, wq) and same(s, ws)
    buf = torch.zeros(rows * dim + 16, dtype=torch.int8, device="cuda")
    off = buf[4:4 + rows * dim].view(rows, dim)
    _, s2 = ops.add_rmsnorm_quantize(dev(x), dev(a), dev(w), eps=eps, gs=gs, out_q=off)
    assert torch.equal(off, q) and torch.equal(s2, s)


# The compiled widths (2560, 3584 and 3840 with the three-set chain), and run-time widths with a partial wave (544,
# 1056), an odd number of chain steps (1056, 2080), the narrowest and the widest.
WIDTHS = [512, 544, 1056, 2048, 2080, 2304, 2560, 3072, 3584, 3840, 4096, 5120, 6144, 7168, 8192, 12288]


@pytest.mark.parametrize("gs", [32, 64])
@pytest.mark.parametrize("dim", WIDTHS)
def test_widths(ops, oracle, dim, gs):
    if dim % gs:
        pytest.skip("dim must be a multiple of the group size")
    x, a = C.normal(dim + gs, (ROWS, dim), 2.0), C.normal(dim + gs + 1, (ROWS, dim))
    check(ops, oracle, x, a, C.norm_weight(dim, dim), gs)


@pytest.mark.parametrize("gs", [32, 64])
@pytest.mark.parametrize("dim", [544, 2560, 3840, 4096, 12288])
def test_nan_at_every_group_position(ops, oracle, dim, gs):
    """A NaN weight at each position of a group in turn (group g: position g % gs) beside a weight of 2^20 two
    positions on: the ordered tree keeps the NaN or drops it with its partners
    (src/asm/rmsnorm_quantize_kernel.inc:158-187)."""
    if dim % gs:
        pytest.skip("dim must be a multiple of the group size")
    x, a = C.normal(95 + dim, (ROWS, dim)), C.normal(96 + dim, (ROWS, dim))
    w = C.norm_weight(97 + dim, dim)
    g = np.arange(dim // gs)
    w[g * gs + g % gs] = np.nan
    w[g * gs + (g + 2) % gs] = np.float32(2.0 ** 20)
    check(ops, oracle, x, a, w, gs)


@pytest.mark.parametrize("gs", [32, 64])
@pytest.mark.parametrize("dim", [3584, 4096])
def test_nan_and_inf_rows_beside_finite_ones(ops, oracle, dim, gs):
    """Inf and NaN weights in single groups (the other groups of the wave take the tree's path too), and rows whose
    scale is NaN or zero, between ordinary rows."""
    x, a = C.normal(31 + dim, (ROWS, dim)), C.normal(32 + dim, (ROWS, dim))
    x[5, 7] = np.nan
    x[100, dim - 1] = np.inf
    x[101] = np.float32(3e38)
    x[256, 0] = -np.inf
    w = C.norm_weight(33 + dim, dim)
    w[gs * 3 + gs - 1] = np.nan
    w[gs * 9 + 1] = np.inf
    check(ops, oracle, x, a, w, gs)


@pytest.mark.parametrize("eps", [0.0, 1e-6])
@pytest.mark.parametrize("dim", [544, 2560, 4096])
def test_denormal_rows(ops, oracle, dim, eps):
    """Rows of denormals and tiny values in the reference's FTZ + DAZ arithmetic; eps = 0 lets an all-flushed sum of
    squares give an infinite scale."""
    x, a = denormal_mix(501, (ROWS, dim)), denormal_mix(502, (ROWS, dim))[::-1].copy()
    check(ops, oracle, x, a, C.norm_weight(503, dim), 32, eps)
