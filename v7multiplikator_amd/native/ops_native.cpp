// ops_native.cpp -- the accepted calls of v7multiplikator_amd.ops without the Python between the call and the launch.
//
// Each function takes the arguments of the ops function of the same name, positionally, looks at the tensors as that
// function does and, when every check passes, binds the library to torch's current stream, makes the library call and
// returns the result.  Where any check does not pass, or a tensor is not a plain one (a subclass, a functorch wrapper,
// a tensor without storage, a torch mode in force), it returns None having done nothing, and ops runs its own checks,
// which raise what they always raised.  A library error is raised through _lib.check.
//
// Why: the Python checks cost 4-6 us a call for the one-tensor-per-operand entries and 11-16 us for the Q/K and Q/K/V
// stages, more than most kernels of a decoding step.
#include <Python.h>

#include <ATen/ATen.h>
#include <ATen/PythonTorchFunctionTLS.h>
#include <c10/core/impl/TorchDispatchModeTLS.h>
#include <torch/csrc/autograd/python_variable.h>

#include <cstdint>
#include <initializer_list>
#include <limits>

#include "../../include/v7g_lib.h"

namespace {

// The library's entries, by the addresses that ops hands over from its own handle of libv7g.so.
struct Entries {
  decltype(&v7g_set_stream) set_stream;
  decltype(&v7g_fused_add_rmsnorm) fused_add_rmsnorm;
  decltype(&v7g_rmsnorm) rmsnorm;
  decltype(&v7g_rmsnorm_quantize) rmsnorm_quantize;
  decltype(&v7g_add_rmsnorm_quantize) add_rmsnorm_quantize;
  decltype(&v7g_add_inplace) add_inplace;
  decltype(&v7g_rmsnorm_rope_heads) rmsnorm_rope_heads;
  decltype(&v7g_qk_rmsnorm_rope) qk_rmsnorm_rope;
  decltype(&v7g_swiglu_f32) swiglu_f32;
  decltype(&v7g_swiglu_q8) swiglu_q8;
  decltype(&v7g_quantize_q8) quantize_q8;
  decltype(&v7g_embedding_gather_q8) embedding_gather_q8;
  decltype(&v7g_rope_only_heads) rope_only_heads;
  decltype(&v7g_qkv_rope_stage) qkv_rope_stage;
  decltype(&v7g_kv_pack_f16) kv_pack_f16;
  decltype(&v7g_kv_pack_f16_kv) kv_pack_f16_kv;
} lib;
PyObject *raw_stream = nullptr;      // torch's raw current-stream query (device index -> stream handle)
PyObject *current_device = nullptr;  // torch's raw current-device query
PyObject *check = nullptr;           // _lib.check(rc, what)

// "Not a call for this path": unwinds to the wrapper, which returns None.
struct Decline {};
void need(bool ok) {
  if (!ok) throw Decline{};
}
// A Python exception is set.
struct Raised {};

const at::Tensor &tensor(PyObject *o, at::ScalarType type, int64_t device, bool contiguous) {
  need(THPVariable_CheckExact(o));
  const at::Tensor &t = THPVariable_Unpack(o);
  need(t.defined() && t.is_cuda() && t.layout() == at::kStrided && t.has_storage() && t.scalar_type() == type &&
       t.device().index() == device);
  const auto keys = t.key_set();
  need(!keys.has(c10::DispatchKey::FuncTorchBatched) && !keys.has(c10::DispatchKey::FuncTorchGradWrapper) &&
       !keys.has(c10::DispatchKey::Functionalize) && !keys.has(c10::DispatchKey::Python));
  if (contiguous) need(t.is_contiguous());
  return t;
}

float *f32(const at::Tensor &t) { return static_cast<float *>(t.data_ptr()); }
int8_t *i8(const at::Tensor &t) { return static_cast<int8_t *>(t.data_ptr()); }

// One call: the argument count, the device and the modes that would see the Python path's torch calls.
struct Call {
  PyObject *const *a;
  int64_t device;

  Call(PyObject *const *args, Py_ssize_t n, Py_ssize_t want) : a(args) {
    need(n == want && check != nullptr);
    need(!c10::impl::TorchDispatchModeTLS::any_modes_set() && !at::impl::torch_function_mode_enabled());
    PyObject *d = PyObject_CallNoArgs(current_device);
    if (!d) {
      PyErr_Clear();
      throw Decline{};
    }
    device = PyLong_AsLongLong(d);
    Py_DECREF(d);
    if (device < 0) {
      PyErr_Clear();
      throw Decline{};
    }
  }
  const at::Tensor &t(int i, at::ScalarType type, bool contiguous = true) const {
    return tensor(a[i], type, device, contiguous);
  }
  const at::Tensor &f(int i) const { return t(i, at::kFloat); }
  bool none(int i) const { return a[i] == Py_None; }
  // A float or an int, as float() takes it, rounded to binary32 as ctypes' c_float rounds it.
  float number(int i) const {
    need(PyFloat_CheckExact(a[i]) || PyLong_CheckExact(a[i]));
    const double v = PyFloat_AsDouble(a[i]);
    if (v == -1.0 && PyErr_Occurred()) {
      PyErr_Clear();
      throw Decline{};
    }
    return static_cast<float>(v);
  }
  int integer(int i, long long lo = std::numeric_limits<int>::min()) const {
    need(PyLong_CheckExact(a[i]));
    int over = 0;
    const long long v = PyLong_AsLongLongAndOverflow(a[i], &over);
    need(!over && v >= lo && v <= std::numeric_limits<int>::max());
    return static_cast<int>(v);
  }
  bool flag(int i) const {
    need(PyBool_Check(a[i]));
    return a[i] == Py_True;
  }
  void bind() const {
    PyObject *d = PyLong_FromLongLong(device);
    PyObject *s = d ? PyObject_CallOneArg(raw_stream, d) : nullptr;
    Py_XDECREF(d);
    void *h = s ? PyLong_AsVoidPtr(s) : nullptr;
    Py_XDECREF(s);
    if (PyErr_Occurred()) {
      PyErr_Clear();
      throw Decline{};
    }
    lib.set_stream(h);
  }
};

// Releases the GIL, as ctypes does around a call (a launch may wait for room in the queue) and torch.empty around
// an allocation (which may reach the driver).
struct NoGil {
  PyThreadState *state = PyEval_SaveThread();
  ~NoGil() { PyEval_RestoreThread(state); }
};

template <typename F>
auto without_gil(F call) {
  const NoGil g;
  return call();
}

template <typename F>
void launch(const char *what, F call) {
  const int rc = without_gil(call);
  if (rc == V7G_OK) return;
  PyObject *r = PyObject_CallFunction(check, "is", rc, what);
  Py_XDECREF(r);
  if (!r) throw Raised{};
}

int32_t dim32(int64_t v) {
  need(v >= 0 && v <= std::numeric_limits<int>::max());
  return static_cast<int32_t>(v);
}

// The last dimension and the number of rows in front of it.
struct Rows {
  int rows, dim;
  explicit Rows(const at::Tensor &t) {
    need(t.dim() >= 1);
    dim = dim32(t.size(-1));
    need(dim > 0);
    rows = dim32(t.numel() / dim);
  }
};

at::Tensor out_like(const Call &c, int i, const at::Tensor &like) {
  // contiguous, with like's own strides where a dimension of one element leaves them free, as torch.empty_like
  if (c.none(i))
    return without_gil(
        [&] { return at::empty_strided(like.sizes(), like.strides(), like.options().requires_grad(false)); });
  const at::Tensor &o = c.f(i);
  need(o.sizes() == like.sizes());
  return o;
}

struct Q8Out {
  at::Tensor q, s;
};
Q8Out q8_out(const Call &c, int iq, int is, const at::Tensor &like, const Rows &r, int gs) {
  const int64_t spr = (static_cast<int64_t>(r.dim) + gs - 1) / gs;
  Q8Out o;
  if (!c.none(iq)) {
    o.q = c.t(iq, at::kChar);
    need(o.q.numel() == static_cast<int64_t>(r.rows) * r.dim);
  }
  if (!c.none(is)) {
    o.s = c.t(is, at::kFloat);
    need(o.s.numel() == r.rows * spr);
  }
  if (!o.q.defined() || !o.s.defined()) {
    const NoGil g;
    const auto opt = at::TensorOptions().device(like.device());
    if (!o.q.defined()) o.q = at::empty(like.sizes(), opt.dtype(at::kChar));
    if (!o.s.defined()) o.s = at::empty({static_cast<int64_t>(r.rows), spr}, opt.dtype(at::kFloat));
  }
  return o;
}

// [tokens, heads, head_dim] with a token's heads contiguous, the token stride free.
struct Heads {
  int tokens, heads, hd;
  long long stride;
  explicit Heads(const at::Tensor &t) {
    need(t.dim() == 3 && t.stride(2) == 1 && t.stride(1) == t.size(2));
    tokens = dim32(t.size(0));
    heads = dim32(t.size(1));
    hd = dim32(t.size(2));
    stride = t.stride(0);
  }
  bool same(const Heads &o) const { return tokens == o.tokens && heads == o.heads && hd == o.hd; }
};

struct Tables {
  const float *cos, *sin;
  int rows, width;
  Tables(const Call &c, int ic, int is) {
    const at::Tensor &ct = c.f(ic), &st = c.f(is);
    need(ct.dim() == 2 && st.sizes() == ct.sizes());
    cos = f32(ct);
    sin = f32(st);
    rows = dim32(ct.size(0));
    width = dim32(ct.size(1));
  }
};

const int32_t *positions(const Call &c, int i, int tokens) {
  if (c.none(i)) return nullptr;
  const at::Tensor &p = c.t(i, at::kInt);
  need(p.numel() == tokens);
  return static_cast<const int32_t *>(p.data_ptr());
}

const float *head_weight(const Call &c, int i, int64_t n) {
  const at::Tensor &w = c.f(i);
  need(w.numel() == n);
  return f32(w);
}

PyObject *wrap(const at::Tensor &t) {
  PyObject *o = THPVariable_Wrap(t);
  if (!o) throw Raised{};
  return o;
}
PyObject *wrap2(const at::Tensor &a, const at::Tensor &b) {
  PyObject *x = wrap(a), *y = THPVariable_Wrap(b);
  if (!y) {
    Py_DECREF(x);
    throw Raised{};
  }
  PyObject *r = PyTuple_Pack(2, x, y);
  Py_DECREF(x);
  Py_DECREF(y);
  if (!r) throw Raised{};
  return r;
}
PyObject *same(PyObject *o) {
  Py_INCREF(o);
  return o;
}

// ------------------------------------------------------------------ the ops

PyObject *fused_add_rmsnorm(const Call &c) {  // residual, add, weight, eps, out
  const at::Tensor &r = c.f(0), &a = c.f(1), &w = c.f(2);
  const Rows n(r);
  need(a.sizes() == r.sizes() && w.numel() == n.dim);
  const float eps = c.number(3);
  const at::Tensor o = out_like(c, 4, r);
  c.bind();
  launch("fused_add_rmsnorm", [&] {
    return lib.fused_add_rmsnorm(f32(o), f32(r), f32(a), f32(w), n.rows, n.dim, eps);
  });
  return c.none(4) ? wrap(o) : same(c.a[4]);
}

PyObject *rmsnorm(const Call &c) {  // x, weight, eps, out
  const at::Tensor &x = c.f(0), &w = c.f(1);
  const Rows n(x);
  need(w.numel() == n.dim);
  const float eps = c.number(2);
  const at::Tensor o = out_like(c, 3, x);
  c.bind();
  launch("rmsnorm", [&] {
    return lib.rmsnorm(f32(o), f32(x), f32(w), n.rows, n.dim, eps);
  });
  return c.none(3) ? wrap(o) : same(c.a[3]);
}

PyObject *rmsnorm_quantize(const Call &c) {  // x, weight, eps, gs, out_q, out_s
  const at::Tensor &x = c.f(0), &w = c.f(1);
  const Rows n(x);
  need(w.numel() == n.dim);
  const float eps = c.number(2);
  const int gs = c.integer(3, 1);
  const Q8Out o = q8_out(c, 4, 5, x, n, gs);
  c.bind();
  launch("rmsnorm_quantize", [&] {
    return lib.rmsnorm_quantize(i8(o.q), f32(o.s), f32(x), f32(w), n.rows, n.dim, gs, eps);
  });
  return wrap2(o.q, o.s);
}

PyObject *add_rmsnorm_quantize(const Call &c) {  // residual, add, weight, eps, gs, out_q, out_s
  const at::Tensor &r = c.f(0), &a = c.f(1), &w = c.f(2);
  const Rows n(r);
  need(a.sizes() == r.sizes() && w.numel() == n.dim);
  const float eps = c.number(3);
  const int gs = c.integer(4, 1);
  const Q8Out o = q8_out(c, 5, 6, r, n, gs);
  c.bind();
  launch("add_rmsnorm_quantize", [&] {
    return lib.add_rmsnorm_quantize(i8(o.q), f32(o.s), f32(r), f32(a), f32(w), n.rows, n.dim, gs, eps);
  });
  return wrap2(o.q, o.s);
}

PyObject *add_inplace(const Call &c) {  // x, y
  const at::Tensor &x = c.f(0), &y = c.f(1);
  need(x.sizes() == y.sizes());
  c.bind();
  launch("add_inplace", [&] {
    return lib.add_inplace(f32(x), f32(y), x.numel());
  });
  return same(c.a[0]);
}

PyObject *swiglu(const Call &c) {  // gate, up, out
  const at::Tensor &g = c.f(0), &u = c.f(1);
  need(g.sizes() == u.sizes());
  const at::Tensor o = out_like(c, 2, g);
  c.bind();
  launch("swiglu", [&] {
    return lib.swiglu_f32(f32(o), f32(g), f32(u), g.numel());
  });
  return c.none(2) ? wrap(o) : same(c.a[2]);
}

PyObject *swiglu_q8(const Call &c) {  // gate, up, gs, out_q, out_s
  const at::Tensor &g = c.f(0), &u = c.f(1);
  need(g.sizes() == u.sizes());
  const Rows n(g);
  const int gs = c.integer(2, 1);
  const Q8Out o = q8_out(c, 3, 4, g, n, gs);
  c.bind();
  launch("swiglu_q8", [&] {
    return lib.swiglu_q8(i8(o.q), f32(o.s), f32(g), f32(u), n.rows, n.dim, gs);
  });
  return wrap2(o.q, o.s);
}

PyObject *quantize_q8(const Call &c) {  // x, gs, out_q, out_s
  const at::Tensor &x = c.f(0);
  const Rows n(x);
  const int gs = c.integer(1, 1);
  const Q8Out o = q8_out(c, 2, 3, x, n, gs);
  c.bind();
  launch("quantize_q8", [&] {
    return lib.quantize_q8(i8(o.q), f32(o.s), f32(x), n.rows, n.dim, gs);
  });
  return wrap2(o.q, o.s);
}

PyObject *embedding_gather_q8(const Call &c) {  // ids, table_q, table_s, out
  const at::Tensor &ids = c.t(0, at::kInt), &tq = c.t(1, at::kChar), &ts = c.f(2);
  need(tq.dim() == 2);
  const int vocab = dim32(tq.size(0)), dim = dim32(tq.size(1)), n = dim32(ids.numel());
  need(ts.numel() == static_cast<int64_t>(vocab) * dim / 64);
  at::Tensor o;
  if (c.none(3)) {
    o = without_gil([&] {
      return at::empty({static_cast<int64_t>(n), static_cast<int64_t>(dim)}, ts.options().requires_grad(false));
    });
  } else {
    o = c.f(3);
    need(o.numel() == static_cast<int64_t>(n) * dim);
  }
  c.bind();
  launch("embedding_gather_q8", [&] {
    return lib.embedding_gather_q8(f32(o), static_cast<const int32_t *>(ids.data_ptr()), n,
        i8(tq), f32(ts), dim, vocab);
  });
  return c.none(3) ? wrap(o) : same(c.a[3]);
}

PyObject *rmsnorm_rope_heads(const Call &c) {  // buf, norm_weight, cos, sin, positions, pos0, eps
  const at::Tensor &b = c.t(0, at::kFloat, false);
  const Heads h(b);
  const float *w = head_weight(c, 1, h.hd);
  const Tables t(c, 2, 3);
  const int32_t *pos = positions(c, 4, h.tokens);
  const int pos0 = c.integer(5);
  const float eps = c.number(6);
  c.bind();
  launch("rmsnorm_rope_heads", [&] {
    return lib.rmsnorm_rope_heads(f32(b), h.tokens, h.stride, h.heads, h.hd, w, t.cos, t.sin, pos, pos0, t.width,
                                  t.rows, eps);
  });
  return same(c.a[0]);
}

PyObject *rope_only_heads(const Call &c) {  // buf, cos, sin, positions, pos0
  const at::Tensor &b = c.t(0, at::kFloat, false);
  const Heads h(b);
  const Tables t(c, 1, 2);
  const int32_t *pos = positions(c, 3, h.tokens);
  const int pos0 = c.integer(4);
  c.bind();
  launch("rope_only_heads", [&] {
    return lib.rope_only_heads(f32(b), h.tokens, h.stride, h.heads, h.hd, t.cos, t.sin, pos, pos0, t.width, t.rows);
  });
  return same(c.a[0]);
}

// q, k, q_norm_weight, k_norm_weight, cos, sin, positions, pos0, eps (without a K cache)
PyObject *qk_rmsnorm_rope(const Call &c) {
  const at::Tensor &q = c.t(0, at::kFloat, false), &k = c.t(1, at::kFloat, false);
  const Heads hq(q), hk(k);
  need(hk.tokens == hq.tokens && hk.hd == hq.hd);
  const float *qw = head_weight(c, 2, hq.hd), *kw = head_weight(c, 3, hq.hd);
  const Tables t(c, 4, 5);
  const int32_t *pos = positions(c, 6, hq.tokens);
  const int pos0 = c.integer(7);
  const float eps = c.number(8);
  c.bind();
  launch("qk_rmsnorm_rope", [&] {
    return lib.qk_rmsnorm_rope(f32(q), hq.stride, hq.heads, qw, f32(k), hk.stride, hk.heads, kw, hq.tokens, hq.hd,
                               t.cos, t.sin, pos, pos0, t.width, t.rows, eps);
  });
  return same(Py_True);
}

Heads stage_side(const Call &c, v7g_qkv_side &s, int buf, int norm, int bias, int cache, bool keep) {
  const at::Tensor &b = c.t(buf, at::kFloat, false);
  const Heads h(b);
  s.buf = f32(b);
  s.token_stride = h.stride;
  s.n_heads = h.heads;
  s.keep_f32 = keep;
  if (norm >= 0 && !c.none(norm)) s.norm_weight = head_weight(c, norm, h.hd);
  if (!c.none(bias)) s.bias = head_weight(c, bias, static_cast<int64_t>(h.heads) * h.hd);
  if (cache >= 0 && !c.none(cache)) {
    const at::Tensor &k = c.t(cache, at::kHalf, false);
    const Heads hc(k);
    need(hc.same(h));
    s.cache = static_cast<uint16_t *>(k.data_ptr());
    s.cache_stride = hc.stride;
  }
  return h;
}

// q, k, v, cos, sin, positions, pos0, eps, q_norm_weight, k_norm_weight, q_bias, k_bias, v_bias, k_cache, v_cache,
// keep_k_f32, keep_v_f32
PyObject *qkv_rope_stage(const Call &c) {
  v7g_qkv_stage st = {};
  const Tables t(c, 3, 4);
  const Heads hq = stage_side(c, st.q, 0, 8, 10, -1, true);
  const Heads hk = stage_side(c, st.k, 1, 9, 11, 13, c.flag(15));
  need(hk.tokens == hq.tokens && hk.hd == hq.hd);
  const bool keep_v = c.flag(16);
  if (!c.none(2)) {
    const Heads hv = stage_side(c, st.v, 2, -1, 12, 14, keep_v);
    need(hv.tokens == hq.tokens && hv.hd == hq.hd);
  }
  st.n_tokens = hq.tokens;
  st.head_dim = hq.hd;
  st.cos_table = t.cos;
  st.sin_table = t.sin;
  st.positions = positions(c, 5, hq.tokens);
  st.pos0 = c.integer(6);
  st.rope_max_dim = t.width;
  st.table_rows = t.rows;
  st.eps = c.number(7);
  c.bind();
  launch("qkv_rope_stage", [&] {
    return lib.qkv_rope_stage(&st);
  });
  return same(Py_True);
}

const at::Tensor &rows_view(const Call &c, int i, at::ScalarType type) {
  const at::Tensor &t = c.t(i, type, false);
  need(t.dim() == 2 && t.stride(1) == 1);
  return t;
}
at::Tensor f16_out(const Call &c, int i, const at::Tensor &src) {
  if (c.none(i))
    return without_gil(
        [&] { return at::empty(src.sizes(), at::TensorOptions().device(src.device()).dtype(at::kHalf)); });
  const at::Tensor &o = c.t(i, at::kHalf, false);
  need(o.sizes() == src.sizes() && o.stride(1) == 1);
  return o;
}
uint16_t *f16(const at::Tensor &t) { return static_cast<uint16_t *>(t.data_ptr()); }

PyObject *kv_pack_f16(const Call &c) {  // src, out
  const at::Tensor &s = rows_view(c, 0, at::kFloat);
  const int rows = dim32(s.size(0)), n = dim32(s.size(1));
  const at::Tensor o = f16_out(c, 1, s);
  c.bind();
  launch("kv_pack_f16", [&] {
    return lib.kv_pack_f16(f16(o), o.stride(0), f32(s), s.stride(0), rows, n);
  });
  return c.none(1) ? wrap(o) : same(c.a[1]);
}

PyObject *kv_pack_f16_kv(const Call &c) {  // k_src, v_src, k_out, v_out
  const at::Tensor &k = rows_view(c, 0, at::kFloat), &v = rows_view(c, 1, at::kFloat);
  need(v.sizes() == k.sizes() && v.strides() == k.strides());
  const int rows = dim32(k.size(0)), n = dim32(k.size(1));
  const at::Tensor ko = f16_out(c, 2, k), vo = f16_out(c, 3, k);
  c.bind();
  launch("kv_pack_f16_kv", [&] {
    return lib.kv_pack_f16_kv(f16(ko), ko.stride(0), f16(vo), vo.stride(0), f32(k), f32(v), k.stride(0), rows, n);
  });
  return wrap2(ko, vo);
}

// Python entry: None where the call is not for this path.  No C++ exception leaves it.
template <PyObject *(*F)(const Call &), int N>
PyObject *entry(PyObject *, PyObject *const *args, Py_ssize_t n) {
  try {
    return F(Call(args, n, N));
  } catch (const Raised &) {
    return nullptr;
  } catch (const std::bad_alloc &) {
    return PyErr_NoMemory();
  } catch (...) {  // Decline, or an error of torch's that the Python path meets and reports itself
    PyErr_Clear();
    Py_RETURN_NONE;
  }
}

// bind(addresses by entry name, raw stream query, current device query, _lib.check)
PyObject *bind(PyObject *, PyObject *args) {
  PyObject *d, *s, *cd, *ck;
  if (!PyArg_ParseTuple(args, "O!OOO", &PyDict_Type, &d, &s, &cd, &ck)) return nullptr;
  Entries e;
#define V7G_ENTRY(field, name)                                             \
  {                                                                        \
    PyObject *v = PyDict_GetItemString(d, name);                           \
    void *p = v ? PyLong_AsVoidPtr(v) : nullptr;                           \
    if (!p) {                                                              \
      if (!PyErr_Occurred()) PyErr_SetString(PyExc_KeyError, name);        \
      return nullptr;                                                      \
    }                                                                      \
    e.field = reinterpret_cast<decltype(e.field)>(p);                      \
  }
  V7G_ENTRY(set_stream, "v7g_set_stream")
  V7G_ENTRY(fused_add_rmsnorm, "v7g_fused_add_rmsnorm")
  V7G_ENTRY(rmsnorm, "v7g_rmsnorm")
  V7G_ENTRY(rmsnorm_quantize, "v7g_rmsnorm_quantize")
  V7G_ENTRY(add_rmsnorm_quantize, "v7g_add_rmsnorm_quantize")
  V7G_ENTRY(add_inplace, "v7g_add_inplace")
  V7G_ENTRY(rmsnorm_rope_heads, "v7g_rmsnorm_rope_heads")
  V7G_ENTRY(qk_rmsnorm_rope, "v7g_qk_rmsnorm_rope")
  V7G_ENTRY(swiglu_f32, "v7g_swiglu_f32")
  V7G_ENTRY(swiglu_q8, "v7g_swiglu_q8")
  V7G_ENTRY(quantize_q8, "v7g_quantize_q8")
  V7G_ENTRY(embedding_gather_q8, "v7g_embedding_gather_q8")
  V7G_ENTRY(rope_only_heads, "v7g_rope_only_heads")
  V7G_ENTRY(qkv_rope_stage, "v7g_qkv_rope_stage")
  V7G_ENTRY(kv_pack_f16, "v7g_kv_pack_f16")
  V7G_ENTRY(kv_pack_f16_kv, "v7g_kv_pack_f16_kv")
#undef V7G_ENTRY
  lib = e;
  Py_INCREF(s);
  Py_XSETREF(raw_stream, s);
  Py_INCREF(cd);
  Py_XSETREF(current_device, cd);
  Py_INCREF(ck);
  Py_XSETREF(check, ck);
  Py_RETURN_NONE;
}

#define V7G_OP(name, n) \
  { #name, reinterpret_cast<PyCFunction>(reinterpret_cast<void *>(&entry<name, n>)), METH_FASTCALL, nullptr }
PyMethodDef methods[] = {{"bind", &bind, METH_VARARGS, nullptr},
                         V7G_OP(fused_add_rmsnorm, 5),
                         V7G_OP(rmsnorm, 4),
                         V7G_OP(rmsnorm_quantize, 6),
                         V7G_OP(add_rmsnorm_quantize, 7),
                         V7G_OP(add_inplace, 2),
                         V7G_OP(swiglu, 3),
                         V7G_OP(swiglu_q8, 5),
                         V7G_OP(quantize_q8, 4),
                         V7G_OP(embedding_gather_q8, 4),
                         V7G_OP(rmsnorm_rope_heads, 7),
                         V7G_OP(rope_only_heads, 5),
                         V7G_OP(qk_rmsnorm_rope, 9),
                         V7G_OP(qkv_rope_stage, 17),
                         V7G_OP(kv_pack_f16, 2),
                         V7G_OP(kv_pack_f16_kv, 4),
                         {nullptr, nullptr, 0, nullptr}};
PyModuleDef module = {PyModuleDef_HEAD_INIT, "_ops_native", nullptr, -1, methods, nullptr, nullptr, nullptr, nullptr};

}  // namespace

#if !defined(V7G_HEADER_TAG) || !defined(V7G_TORCH_BUILD)
#error "build.py defines V7G_HEADER_TAG and V7G_TORCH_BUILD"
#endif

// ops uses the module only where both attributes match the library and the torch that are running.
PyMODINIT_FUNC PyInit__ops_native(void) {
  PyObject *m = PyModule_Create(&module);
  if (m && (PyModule_AddStringConstant(m, "header_tag", V7G_HEADER_TAG) < 0 ||
            PyModule_AddStringConstant(m, "torch_build", V7G_TORCH_BUILD) < 0)) {
    Py_DECREF(m);
    return nullptr;
  }
  return m;
}
