"""The native path of ops against the Python bodies it stands in front of: for every op the same results and the
same returned objects on the calls it accepts (results given or allocated, parameters, strided heads, other streams),
and the same exception, type and text, on the calls that the Python checks refuse."""
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
    x = torch.ones(4, 64, device="cuda")
    _ops.add_inplace(x, x.clone())
    assert _ops._fast.__name__ == "_ops_native", "the native module is not in use"
    return _ops


def rnd(*shape, seed=0, dtype=torch.float32):
    g = torch.Generator(device="cuda").manual_seed(seed + sum(shape))
    return torch.randn(shape, generator=g, device="cuda").to(dtype)


def qkv(T=5, nq=4, nkv=2, hd=64):
    rows = rnd(T, (nq + 2 * nkv) * hd, seed=3)
    a, b = nq * hd, (nq + nkv) * hd
    return rows, rows[:, :a].view(T, nq, hd), rows[:, a:b].view(T, nkv, hd), rows[:, b:].view(T, nkv, hd)


def tables(hd=64):
    return rnd(9, hd // 2, seed=5), rnd(9, hd // 2, seed=6)


def calls():
    """(name, function of ops returning what the call returns and every tensor it may write)."""
    pos = lambda: torch.arange(5, dtype=torch.int32, device="cuda")  # noqa: E731
    out = []

    def add(name, f):
        out.append(pytest.param(f, id=name))

    for given in (False, True):
        tag = "given" if given else "allocated"

        def fused(o, given=given):
            r, buf = rnd(3, 5, 64), (rnd(3, 5, 64, seed=9) if given else None)
            w = torch.nn.Parameter(rnd(64))
            got = o.fused_add_rmsnorm(r, rnd(3, 5, 64, seed=1), w.detach() if given else w, eps=1e-5, out=buf)
            return got, r, buf, got is buf

        def one_row(o, given=given):  # a contiguous row whose first stride is no row length
            r = rnd(9, 64).as_strided((1, 64), (99, 1))
            return o.fused_add_rmsnorm(r, rnd(1, 64), rnd(64)), o.rmsnorm(r, rnd(64)), o.swiglu(r, r)

        def norm(o, given=given):
            x = rnd(5, 96)
            buf = x if given else None
            got = o.rmsnorm(x, rnd(96), 1e-5, buf)
            return got, got is buf

        def nq8(o, given=given, gs=64):
            x = rnd(7, 128)
            q = torch.zeros(7 * 128, dtype=torch.int8, device="cuda") if given else None
            s = torch.zeros(14, device="cuda") if given else None
            return (*o.rmsnorm_quantize(x, rnd(128), gs=gs, out_q=q, out_s=s), q, s)

        def anq8(o, given=given):
            x = rnd(7, 128)
            q = torch.zeros(7, 128, dtype=torch.int8, device="cuda") if given else None
            return (*o.add_rmsnorm_quantize(x, rnd(7, 128, seed=2), rnd(128), 1e-6, 32, q), x, q)

        def sw(o, given=given):
            g = rnd(3, 130)
            got = o.swiglu(g, rnd(3, 130, seed=4), out=g if given else None)
            return got, got is g

        def swq(o, given=given):
            s = torch.zeros(3, 3, device="cuda") if given else None
            return (*o.swiglu_q8(rnd(3, 130), rnd(3, 130, seed=4), 64, out_s=s), s)

        def quant(o, given=given):
            q = torch.zeros(2, 3, 70, dtype=torch.int8, device="cuda") if given else None
            return (*o.quantize_q8(rnd(2, 3, 70), gs=32, out_q=q), q)

        def emb(o, given=given):
            ids = torch.tensor([[3, 1], [0, 99]], dtype=torch.int32, device="cuda")
            tq = torch.arange(10 * 64, device="cuda").to(torch.int8).view(10, 64)
            buf = torch.zeros(4, 64, device="cuda") if given else None
            got = o.embedding_gather_q8(ids, tq, rnd(10), out=buf)
            return got, got is buf

        def pack(o, given=given):
            src = rnd(6, 64)[:, 16:48]
            buf = torch.zeros(6, 40, dtype=torch.float16, device="cuda")[:, :32] if given else None
            got = o.kv_pack_f16(src, buf)
            return got, got is buf

        def pack2(o, given=given):
            src = rnd(6, 64)
            buf = torch.zeros(6, 32, dtype=torch.float16, device="cuda") if given else None
            return o.kv_pack_f16_kv(src[:, :32], src[:, 32:], v_out=buf)

        for f in (fused, one_row, norm, nq8, anq8, sw, swq, quant, emb, pack, pack2):
            add(f"{f.__name__}-{tag}", f)

        def heads(o, given=given):
            rows, q, k, v = qkv()
            o.rmsnorm_rope_heads(q, rnd(64), *tables(), positions=pos() if given else None, pos0=2)
            o.rope_only_heads(k, *tables(), positions=pos() if given else None, pos0=1)
            return rows

        def qk(o, given=given):
            rows, q, k, v = qkv()
            kc = torch.zeros(5, 2, 64, dtype=torch.float16, device="cuda") if given else None
            got = o.qk_rmsnorm_rope(q, k, rnd(64), rnd(64, seed=8), *tables(), pos0=1, k_cache=kc)
            return rows, kc, got

        def stage(o, given=given):
            rows, q, k, v = qkv()
            kc = torch.zeros(5, 3, 2, 64, dtype=torch.float16, device="cuda")
            got = o.qkv_rope_stage(q, k, v if given else None, *tables(), positions=pos(), q_norm_weight=rnd(64),
                                   k_norm_weight=None, q_bias=None, k_bias=rnd(128), v_bias=rnd(128, seed=1),
                                   k_cache=kc[:, 0], v_cache=kc[:, 2] if given else None, keep_k_f32=given,
                                   keep_v_f32=not given)
            return rows, kc, got

        for f in (heads, qk, stage):
            add(f"{f.__name__}-{tag}", f)

    # forms that one path or the other refuses, or that are nothing to do
    x, w = (lambda: rnd(4, 64)), (lambda: rnd(64))
    add("empty", lambda o: o.fused_add_rmsnorm(rnd(0, 64), rnd(0, 64), w()))
    add("empty_pack", lambda o: o.kv_pack_f16(rnd(0, 8)))
    add("zero_dim", lambda o: o.rmsnorm(rnd(1)[0], w()))
    add("zero_width", lambda o: o.quantize_q8(rnd(4, 0)))
    add("transposed", lambda o: o.rmsnorm(rnd(64, 4).t(), w()))
    add("double", lambda o: o.add_inplace(x(), x().double()))
    add("host", lambda o: o.add_inplace(x(), x().cpu()))
    add("not_a_tensor", lambda o: o.swiglu(x(), [1.0]))
    add("shape", lambda o: o.swiglu(x(), rnd(5, 64)))
    add("weight_size", lambda o: o.rmsnorm(x(), rnd(32)))
    add("weight_shape", lambda o: o.rmsnorm(x(), rnd(8, 8)))
    add("gs_zero", lambda o: o.quantize_q8(x(), gs=0))
    add("gs_negative", lambda o: o.quantize_q8(x(), gs=-4))
    add("gs_float", lambda o: o.quantize_q8(x(), gs=32.0))
    add("gs_library", lambda o: o.quantize_q8(x(), gs=5000))
    add("eps_text", lambda o: o.rmsnorm(x(), w(), eps="1e-5"))
    add("eps_int", lambda o: o.rmsnorm(x(), w(), eps=1))
    add("out_size", lambda o: o.quantize_q8(x(), out_q=torch.zeros(9, dtype=torch.int8, device="cuda")))
    add("alias", lambda o: (lambda t: o.kv_pack_f16(t, t.view(torch.float16)[:, :64]))(x()))
    add("positions", lambda o: o.rope_only_heads(qkv()[1], *tables(), positions=torch.zeros(4, dtype=torch.int32,
                                                                                          device="cuda")))
    add("heads_dim", lambda o: o.rope_only_heads(x(), *tables()))
    add("heads_apart", lambda o: o.rope_only_heads(qkv()[1].transpose(0, 1), *tables()))
    add("pos0_large", lambda o: o.rope_only_heads(qkv()[1], *tables(), pos0=1 << 40))
    add("keep_int", lambda o: o.qkv_rope_stage(*qkv()[1:], *tables(), keep_k_f32=0))
    add("table_scales", lambda o: o.embedding_gather_q8(torch.zeros(1, dtype=torch.int32, device="cuda"),
                                                        torch.zeros(2, 64, dtype=torch.int8, device="cuda"), rnd(3)))

    class Sub(torch.Tensor):
        pass

    add("subclass", lambda o: torch.Tensor(o.rmsnorm(x().as_subclass(Sub), w()).as_subclass(torch.Tensor)))
    return out


def outcome(f, ops):
    try:
        got = f(ops)
    except Exception as e:  # noqa: BLE001 -- the exception is the outcome
        return type(e), str(e)
    torch.cuda.synchronize()
    return got if isinstance(got, tuple) else (got,)


@pytest.mark.parametrize("f", calls())
def test_native_is_the_python_path(ops, monkeypatch, f):
    native = outcome(f, ops)
    monkeypatch.setattr(ops, "_fast", ops._NoNative())
    python = outcome(f, ops)
    assert len(native) == len(python)
    for a, b in zip(native, python):
        if isinstance(b, torch.Tensor):
            assert type(a) is type(b) and a.shape == b.shape and a.dtype == b.dtype and a.stride() == b.stride()
            assert torch.equal(a.contiguous().view(torch.uint8), b.contiguous().view(torch.uint8))
        else:
            assert a == b


class Recorder:
    """Stands in for the native module and notes what each call answered: True where it made the call (a library error
    counts: the library was asked), False where it declined."""

    def __init__(self, mod):
        self.mod, self.made = mod, []

    def __getattr__(self, name):
        def call(*args):
            try:
                r = getattr(self.mod, name)(*args)
            except Exception:
                self.made.append(True)
                raise
            self.made.append(r is not None)
            return r
        return call


# What is not the plain accepted call: declined, or (qk with a K cache) never asked.
DECLINED = {"qk-given": [], "zero_dim": [False], "zero_width": [False], "transposed": [False], "double": [False],
            "host": [False], "not_a_tensor": [False], "shape": [False], "weight_size": [False], "gs_zero": [False],
            "gs_negative": [False], "gs_float": [False], "eps_text": [False], "out_size": [False],
            "positions": [False], "heads_dim": [False], "heads_apart": [False], "pos0_large": [False],
            "keep_int": [False], "table_scales": [False], "subclass": [False]}
CALLS_PER_FORM = {"one_row": 3, "heads": 2}


@pytest.mark.parametrize("name,f", [pytest.param(p.id, p.values[0], id=p.id) for p in calls()])
def test_native_makes_the_accepted_calls(ops, monkeypatch, name, f):
    """Which forms the native path serves itself: falling through to Python gives the same results, so only this
    shows an entry that has stopped accepting."""
    rec = Recorder(ops._fast)
    monkeypatch.setattr(ops, "_fast", rec)
    outcome(f, ops)
    assert rec.made == DECLINED.get(name, [True] * CALLS_PER_FORM.get(name.split("-")[0], 1))


def test_native_declines_under_torch_modes(ops, monkeypatch):
    """A torch function or dispatch mode must see the Python path's torch calls."""
    from torch.overrides import TorchFunctionMode
    from torch.utils._python_dispatch import TorchDispatchMode

    class Function(TorchFunctionMode):
        def __torch_function__(self, func, types, args=(), kwargs=None):
            return func(*args, **(kwargs or {}))

    class Dispatch(TorchDispatchMode):
        def __torch_dispatch__(self, func, types, args=(), kwargs=None):
            return func(*args, **(kwargs or {}))

    x, w = rnd(4, 64), rnd(64)
    want = ops.rmsnorm(x, w)
    for mode in (Function, Dispatch):
        rec = Recorder(ops._fast)
        with monkeypatch.context() as m, mode():
            m.setattr(ops, "_fast", rec)
            got = ops.rmsnorm(x, w)
        assert rec.made == [False] and torch.equal(got, want)


def test_follows_the_current_stream(ops):
    """Work queued on a side stream is seen by a native call made under that stream, and by no other."""
    from v7multiplikator_amd import _lib

    side = torch.cuda.Stream()
    x = torch.zeros(1 << 22, device="cuda")
    torch.cuda.synchronize()
    with torch.cuda.stream(side):
        for _ in range(20):
            x += 1
        ops.add_inplace(x, torch.ones_like(x))
        assert _lib.load().v7g_get_stream() == side.cuda_stream
    torch.cuda.synchronize()
    assert torch.all(x == 21)
    ops.add_inplace(x, x.clone())
    assert (_lib.load().v7g_get_stream() or 0) == torch.cuda.current_stream().cuda_stream
    torch.cuda.synchronize()


# With an allocator that counts: every op that allocates its results, through the native path.
UNDER_THE_GIL = """
import ctypes, sys
import torch
path = sys.argv[1]
torch.cuda.memory.change_current_allocator(torch.cuda.memory.CUDAPluggableAllocator(path, "gil_alloc", "gil_free"))
from v7multiplikator_amd import _lib, ops
count = ctypes.PyDLL(path)
x, w = torch.ones(8, 64, device="cuda"), torch.ones(64, device="cuda")
ids = torch.zeros(3, dtype=torch.int32, device="cuda")
tq, ts = torch.ones(5, 64, device="cuda").to(torch.int8), torch.ones(5, device="cuda")
ops.add_inplace(x, x.clone())
assert ops._fast.__name__ == "_ops_native"
held, made = count.gil_held(), count.gil_all()
keep = [ops._fast.fused_add_rmsnorm(x, x.clone(), w, 1e-6, None), ops._fast.rmsnorm(x, w, 1e-6, None),
        ops._fast.rmsnorm_quantize(x, w, 1e-6, 64, None, None),
        ops._fast.add_rmsnorm_quantize(x, x.clone(), w, 1e-6, 64, None, None), ops._fast.swiglu(x, x, None),
        ops._fast.swiglu_q8(x, x, 64, None, None), ops._fast.quantize_q8(x, 64, None, None),
        ops._fast.embedding_gather_q8(ids, tq, ts, None), ops._fast.kv_pack_f16(x, None),
        ops._fast.kv_pack_f16_kv(x, x, None, None)]
assert all(k is not None for k in keep)
torch.cuda.synchronize()
print("HELD", count.gil_held() - held, "OF", count.gil_all() - made)
"""


def test_results_are_allocated_without_the_gil():
    """An allocation may reach the driver; torch.empty lets the other threads run meanwhile, and so do the ops."""
    import os
    import subprocess
    import sys

    here = os.path.dirname(os.path.abspath(__file__))
    res = subprocess.run([sys.executable, "-c", UNDER_THE_GIL, os.path.join(here, "libgil_alloc.so")],
                         capture_output=True, text=True, timeout=100, cwd=os.path.dirname(here))
    assert res.returncode == 0, res.stderr
    assert "HELD 0 OF 17" in res.stdout, res.stdout
