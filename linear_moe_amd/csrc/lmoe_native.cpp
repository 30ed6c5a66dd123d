// Launch path of the ops in native code: the argument checks, allocations and the argument block of a call, and the
// call of the library's entry point, for the calls that need nothing in front of it -- plain tensors on the current
// device, in types and strides the kernels take.  For every other call the functions return None and the caller (the
// Python of the op: _host.py, simple_gla.py, gla.py, gated_delta_rule.py, recurrent.py) converts, copies or refuses as it
// always did; results are the same bits either way.  What it is for: a call of three to four small kernels takes the GPU
// 5 to 100 us, and the same steps through Python objects and ctypes took the host 20 us per forward and as much
// per backward (figures in linear_moe_amd/_host.py).
#include <Python.h>
#include <dlfcn.h>

#include <cmath>
#include <initializer_list>

#include <ATen/ATen.h>
#include <c10/core/impl/VirtualGuardImpl.h>
#include <torch/csrc/Exceptions.h>
#include <torch/csrc/autograd/python_variable.h>

#include "../../include/lmoe.h"

namespace {

using at::Tensor;
typedef int (*op_fn)(const lmoe_args*, void*);
typedef int (*rec_fn)(const lmoe_args*, int32_t, void*);
typedef int64_t (*split_fn)(const lmoe_args*, int32_t, int32_t);
struct Library {
  op_fn fwd[3], bwd[3];      // by LMOE_OP_*
  rec_fn recurrent;
  split_fn split_floats;
} lib;

constexpr int OP_SIMPLE = LMOE_OP_SIMPLE_GLA, OP_GLA = LMOE_OP_GLA, OP_GDN = LMOE_OP_GATED_DELTA_RULE;

// Not a call for this path.
struct Elsewhere {};
[[noreturn]] void elsewhere() { throw Elsewhere(); }
inline void need(bool ok) { if (!ok) elsewhere(); }

// A tensor as the kernels may read it: an ordinary one (no subclass, no wrapper of a transform, nothing lazy) on device dev
Tensor plain(PyObject* o, int dev) {
  static const c10::DispatchKeySet ordinary({c10::DispatchKey::CUDA, c10::DispatchKey::ADInplaceOrView, c10::DispatchKey::AutogradCUDA, c10::DispatchKey::AutocastCUDA});
  need(THPVariable_CheckExact(o));
  const Tensor& t = THPVariable_Unpack(o);
  need(t.defined() && (t.key_set().raw_repr() & ~ordinary.raw_repr()) == 0 && t.layout() == at::kStrided && t.get_device() == dev);
  return t;
}
Tensor plain_or_none(PyObject* o, int dev) { return o == Py_None ? Tensor() : plain(o, dev); }
int current_device(PyObject* o) {
  need(THPVariable_CheckExact(o) && THPVariable_Unpack(o).is_cuda());
  static const c10::impl::VirtualGuardImpl guard(c10::DeviceType::CUDA);
  return guard.getDevice().index();
}

bool rows_aligned(const Tensor& x) {
  const auto s = x.strides();
  return s[3] == 1 && (reinterpret_cast<uintptr_t>(x.data_ptr()) & 15) == 0 && (s[0] | s[1] | s[2]) % (16 / x.element_size()) == 0;
}
lmoe_tensor desc(const Tensor& x, bool head_first) {
  if (!x.defined()) return lmoe_tensor{nullptr, 0, 0, 0};
  const auto s = x.strides();
  return head_first ? lmoe_tensor{x.data_ptr(), s[0], s[2], s[1]} : lmoe_tensor{x.data_ptr(), s[0], s[1], s[2]};
}
void* ptr(const Tensor& x) { return x.defined() ? x.data_ptr() : nullptr; }
bool f32(const Tensor& x) { return x.scalar_type() == at::kFloat; }
bool bf16(const Tensor& x) { return x.scalar_type() == at::kBFloat16; }

struct Call {
  int dev;
  bool head_first;
  int64_t B, T, H, K, V, N, NT;
  lmoe_args a = {};
  Tensor q, k, v, g, beta, h0;
  typedef std::initializer_list<int64_t> Tail;
  c10::SmallVector<int64_t, 6> chunked_shape(Tail tail) const {                       // [NT, H, ...]
    c10::SmallVector<int64_t, 6> s = {std::max<int64_t>(NT, 1), H};
    s.append(tail.begin(), tail.end());
    return s;
  }
  Tensor chunked(Tail tail, at::ScalarType t) const { return at::empty(chunked_shape(tail), q.options().dtype(t).requires_grad(false)); }
  Tensor states() const { return at::empty({N, H, K, V}, q.options().dtype(at::kFloat)); }
  c10::SmallVector<int64_t, 3> token_shape() const {
    return head_first ? c10::SmallVector<int64_t, 3>{B, H, T} : c10::SmallVector<int64_t, 3>{B, T, H};
  }

  // q, k, v, the gate, beta, the initial state and, for packed input, the tables (N, NT, cu, chunk_map, seq_chunk0, seq_order,
  // nt_dev): checked, and entered into the block
  Call(int op, PyObject* const* o, PyObject* plan, PyObject* scale, bool hf, bool recurrent = false) : dev(current_device(o[0])), head_first(hf) {
    q = plain(o[0], dev); k = plain(o[1], dev); v = plain(o[2], dev);
    need(q.dim() == 4 && v.dim() == 4 && (bf16(q) || f32(q)) && k.scalar_type() == q.scalar_type() && v.scalar_type() == q.scalar_type());
    need(k.sizes() == q.sizes() && v.sizes().slice(0, 3) == q.sizes().slice(0, 3));
    need(q.numel() > 0 && v.numel() > 0);
    B = q.size(0); T = q.size(hf ? 2 : 1); H = q.size(hf ? 1 : 2); K = q.size(3); V = v.size(3);
    need(((K == 64 || K == 128) && (V == 64 || V == 128)) || (op == OP_GDN && !recurrent && K == 128 && V == 256));
    need(rows_aligned(q) && rows_aligned(k) && rows_aligned(v));
    need(B <= INT32_MAX && T <= INT32_MAX && H <= INT32_MAX);
    a.dtype = bf16(q) ? LMOE_BF16 : LMOE_F32;
    N = B; NT = B * ((T + LMOE_CHUNK - 1) / LMOE_CHUNK);
    if (plan != Py_None) {
      need(PyTuple_Check(plan) && PyTuple_GET_SIZE(plan) == 7 && !hf && B == 1);
      N = PyLong_AsLongLong(PyTuple_GET_ITEM(plan, 0)); NT = PyLong_AsLongLong(PyTuple_GET_ITEM(plan, 1));
      const int32_t* p[5];
      for (int i = 0; i < 5; ++i) p[i] = (const int32_t*)ptr(plain_or_none(PyTuple_GET_ITEM(plan, 2 + i), dev));
      a.cu_seqlens = p[0]; a.chunk_map = p[1]; a.seq_chunk0 = p[2]; a.seq_order = p[3]; a.nt_dev = p[4];
    }
    need(NT <= INT32_MAX);
    a.B = B; a.T = T; a.H = H; a.K = K; a.V = V; a.N = N; a.NT = NT;
    const double sc = scale == Py_None ? std::pow((double)K, -0.5) : PyFloat_AsDouble(scale);
    if (sc == -1.0 && PyErr_Occurred()) { PyErr_Clear(); elsewhere(); }
    a.scale = (float)sc;
    a.q = desc(q, hf); a.k = desc(k, hf); a.v = desc(v, hf);
    g = plain_or_none(o[3], dev);
    a.gate = LMOE_GATE_NONE;
    if (g.defined()) {
      need(f32(g) || bf16(g));
      if (op == OP_GLA) {
        need(g.sizes() == q.sizes() && rows_aligned(g) && (recurrent || bf16(q) || f32(g)));
        a.gate = LMOE_GATE_VECTOR;
      } else {
        need(g.dim() == 3 && g.sizes() == at::IntArrayRef(token_shape()));
        a.gate = LMOE_GATE_SCALAR;
      }
      a.g = desc(g, hf); a.g_dtype = f32(g) ? LMOE_F32 : LMOE_BF16;
    } else {
      need(op != OP_GLA);
    }
    beta = plain_or_none(o[4], dev);
    if (op == OP_GDN) {
      need(beta.defined() && (f32(beta) || bf16(beta)) && beta.dim() == 3 && beta.sizes() == at::IntArrayRef(token_shape()));
      a.beta = desc(beta, hf); a.beta_dtype = f32(beta) ? LMOE_F32 : LMOE_BF16;
    }
    h0 = plain_or_none(o[5], dev);
    if (h0.defined()) need(f32(h0) && h0.is_contiguous() && h0.dim() == 4 && h0.sizes() == at::IntArrayRef({N, H, K, V}));
    a.h0 = (const float*)ptr(h0);
  }
  // the buffers of a call that is cut along T
  Tensor cut(int op) {
    const int64_t n = lib.split_floats(&a, op, 1);
    if (n <= 0) return Tensor();
    Tensor ws = at::empty({n}, q.options().dtype(at::kFloat));
    a.seg_ws = (float*)ws.data_ptr();
    return ws;
  }
};

template <typename F> int launch(F f) {
  int rc;
  Py_BEGIN_ALLOW_THREADS
  rc = f();
  Py_END_ALLOW_THREADS
  return rc;
}
PyObject* wrap(const Tensor& t) {
  if (!t.defined()) Py_RETURN_NONE;
  return THPVariable_Wrap(t);
}
// a tuple of tensors (None where undefined), or the return code of a refused launch
PyObject* result(int rc, std::initializer_list<Tensor> out) {
  if (rc != 0) return PyLong_FromLong(rc);
  PyObject* r = PyTuple_New((Py_ssize_t)out.size());
  if (!r) return nullptr;
  Py_ssize_t i = 0;
  for (const Tensor& t : out) {
    PyObject* x = wrap(t);
    if (!x) { Py_DECREF(r); return nullptr; }
    PyTuple_SET_ITEM(r, i++, x);
  }
  return r;
}
template <typename F> PyObject* guarded(F f) {
  HANDLE_TH_ERRORS
  try {
    return f();
  } catch (const Elsewhere&) {
    Py_RETURN_NONE;
  }
  END_HANDLE_TH_ERRORS
}
bool yes(PyObject* o) { return PyObject_IsTrue(o) == 1; }
void* stream_of(PyObject* o) { return PyLong_AsVoidPtr(o); }

// recurrent(op, q, k, v, g, beta, h0, plan, scale, final_state, head_first, qk_eps, stream) -> (o, ht)
PyObject* recurrent(PyObject*, PyObject* const* o, Py_ssize_t n) {
  return guarded([&]() -> PyObject* {
    need(n == 13);
    const int op = (int)PyLong_AsLong(o[0]);
    Call c(op, o + 1, o[7], o[8], yes(o[10]), true);
    const Tensor out = at::empty_like(c.v.detach());
    const Tensor ht = yes(o[9]) ? c.states() : Tensor();
    c.a.o = desc(out, c.head_first); c.a.ht = (float*)ptr(ht); c.a.qk_eps = (float)PyFloat_AsDouble(o[11]);
    void* st = stream_of(o[12]);
    return result(launch([&] { return lib.recurrent(&c.a, op, st); }), {out, ht});
  });
}

// forward(op, q, k, v, g, beta, h0, plan, scale, final_state, head_first, save, normalize, norm_eps, v_act, stream)
//   -> (o, ht, hs, ...) and per op  simple_gla: den, zs;  gla: amat, qe, ke, gdec;  gated delta rule: tinv, pmat, gcum, vnew, seg_p
PyObject* forward(PyObject*, PyObject* const* o, Py_ssize_t n) {
  return guarded([&]() -> PyObject* {
    need(n == 16);
    const int op = (int)PyLong_AsLong(o[0]);
    const bool save = yes(o[11]), v_act = yes(o[14]);
    const int normalize = (int)PyLong_AsLong(o[12]);
    Call c(op, o + 1, o[7], o[8], yes(o[10]));
    const bool hf = c.head_first, two = bf16(c.q);
    const auto dt = c.q.scalar_type();
    void* st = stream_of(o[15]);
    need(op != OP_GDN || two);               // (the 4-byte delta rule needs w and u as well)
    // (v_act: v is a block of a wider tensor; o is a tensor of its own)
    const Tensor out = v_act ? at::empty(c.v.sizes(), c.v.options()) : at::empty_like(c.v);
    const Tensor ht = yes(o[9]) ? c.states() : Tensor();
    c.a.o = desc(out, hf); c.a.ht = (float*)ptr(ht);
    Tensor hs;
    if (op == OP_SIMPLE) {
      Tensor den, zs;
      if (save) hs = c.chunked({c.K, c.V}, dt);
      c.a.hs = ptr(hs);
      if (normalize) {
        need(!c.g.defined() && two);
        den = at::empty(c.token_shape(), c.q.options().dtype(at::kFloat));
        if (save) zs = c.chunked({c.K}, at::kFloat);
        c.a.normalize = normalize; c.a.norm_eps = (float)PyFloat_AsDouble(o[13]); c.a.den = desc(den, hf); c.a.zs = (float*)ptr(zs);
      }
      const Tensor ws = c.cut(op);
      return result(launch([&] { return lib.fwd[op](&c.a, st); }), {out, ht, hs, den, zs});
    }
    if (op == OP_GLA) {
      if (save || !two) hs = c.chunked({c.K, c.V}, dt);
      const Tensor amat = c.chunked({64, 64}, dt), qe = c.chunked({64, c.K}, dt), ke = c.chunked({64, c.K}, dt), gdec = c.chunked({c.K}, at::kFloat);
      c.a.hs = ptr(hs); c.a.amat = ptr(amat); c.a.qe = ptr(qe); c.a.ke = ptr(ke); c.a.gcum = (float*)ptr(gdec);
      const Tensor ws = c.cut(op);
      return result(launch([&] { return lib.fwd[op](&c.a, st); }), {out, ht, hs, amat, qe, ke, gdec});
    }
    Tensor pmat, vnew, seg_p;
    if (save) { hs = c.chunked({c.K, c.V}, dt); pmat = c.chunked({64, 64}, dt); vnew = c.chunked({c.V / 32, 64, 32}, dt); }
    const Tensor tinv = c.chunked({64, 64}, dt), gcum = c.chunked({5, 64}, at::kFloat);
    c.a.hs = ptr(hs); c.a.tinv = ptr(tinv); c.a.pmat = ptr(pmat); c.a.gcum = (float*)ptr(gcum); c.a.vnew.ptr = ptr(vnew);
    c.a.v_act = v_act;
    const Tensor ws = c.cut(op);
    if (ws.defined() && save) {
      seg_p = at::empty({lib.split_floats(&c.a, op, 0)}, c.q.options().dtype(at::kFloat));
      c.a.seg_p = (float*)seg_p.data_ptr();
    }
    return result(launch([&] { return lib.fwd[op](&c.a, st); }), {out, ht, hs, tinv, pmat, gcum, vnew, seg_p});
  });
}

// backward(op, q, k, v, g, beta, h0, plan, scale, do, dht, head_first, saved, extra, stream) -> (dq, dk, dv, dg, dbeta, dh0)
//   saved: what forward returned behind ht;  extra: simple_gla (normalize, norm_eps, o, dden), gated delta rule (v_act, dq, dk,
//   dv, q_raw, k_raw, qk_eps), None where a call has none
PyObject* backward(PyObject*, PyObject* const* o, Py_ssize_t n) {
  return guarded([&]() -> PyObject* {
    need(n == 15);
    const int op = (int)PyLong_AsLong(o[0]);
    Call c(op, o + 1, o[7], o[8], yes(o[11]));
    const bool hf = c.head_first, two = bf16(c.q);
    need(op != OP_GDN || two);
    const Tensor dout = plain(o[9], c.dev);
    need(dout.scalar_type() == c.q.scalar_type() && dout.sizes() == c.v.sizes() && rows_aligned(dout));
    const Tensor dht = plain_or_none(o[10], c.dev);
    if (dht.defined()) need(f32(dht) && dht.is_contiguous() && dht.sizes() == at::IntArrayRef({c.N, c.H, c.K, c.V}));
    c.a.d_o = desc(dout, hf); c.a.dht = (const float*)ptr(dht);
    PyObject* sv = o[12];
    need(PyTuple_Check(sv));
    auto saved = [&](Py_ssize_t i) { need(i < PyTuple_GET_SIZE(sv)); return plain_or_none(PyTuple_GET_ITEM(sv, i), c.dev); };
    // What was saved may have been through a hook, which hands back what it likes; the kernels index the full extent: of the
    // type and size that forward allocated, contiguous and on a 16-byte boundary.  (Anything else: the Python steps convert or
    // refuse it, _host.came_back.)
    auto kept = [&](Py_ssize_t i, at::ScalarType t, Call::Tail tail) {
      const Tensor x = saved(i);
      need(x.defined() && x.is_contiguous() && x.scalar_type() == t && x.sizes() == at::IntArrayRef(c.chunked_shape(tail)));
      need((reinterpret_cast<uintptr_t>(x.data_ptr()) & 15) == 0);
      return x.data_ptr();
    };
    const auto dt = c.q.scalar_type();
    const bool has_extra = o[13] != Py_None;
    auto extra = [&](Py_ssize_t i) { need(PyTuple_Check(o[13]) && i < PyTuple_GET_SIZE(o[13])); return PyTuple_GET_ITEM(o[13], i); };
    auto fresh = [&](const Tensor& x) { return at::empty_like(x.detach()); };
    Tensor dq, dk, dv, dg, dbeta, ws, norm_ws, den, ones;
    const Tensor dh0 = c.h0.defined() ? fresh(c.h0) : Tensor();
    c.a.dh0 = (float*)ptr(dh0);
    c.a.hs = kept(0, dt, {c.K, c.V});
    const Tensor dhs = c.chunked({c.K, c.V}, dt);
    c.a.dhs = ptr(dhs);
    auto gradients = [&] {
      if (!dq.defined()) dq = fresh(c.q);
      if (!dk.defined()) dk = fresh(c.k);
      if (!dv.defined()) dv = fresh(c.v);
      c.a.dq = desc(dq, hf); c.a.dk = desc(dk, hf); c.a.dv = desc(dv, hf);
    };
    if (op == OP_SIMPLE) {
      gradients();
      if (c.g.defined()) { dg = at::empty(c.g.sizes(), c.g.options().dtype(at::kFloat)); c.a.dg = desc(dg, hf); }
      if (has_extra) {
        norm_ws = c.chunked({c.V / 32, 64 + c.K}, at::kFloat);
        c.a.normalize = (int)PyLong_AsLong(extra(0)); c.a.norm_eps = (float)PyFloat_AsDouble(extra(1));
        c.a.zs = (float*)kept(2, at::kFloat, {c.K}); c.a.norm_ws = (float*)norm_ws.data_ptr();
        if (c.a.normalize == 2) {
          den = plain(extra(3), c.dev);
          need(f32(den) && den.is_contiguous() && den.sizes() == at::IntArrayRef(c.token_shape()));
          c.a.dden = desc(den, hf);
        } else {
          ones = plain(extra(2), c.dev);
          den = saved(1);
          need(ones.scalar_type() == dt && ones.sizes() == c.v.sizes() && rows_aligned(ones));
          need(den.defined() && f32(den) && den.is_contiguous() && den.sizes() == at::IntArrayRef(c.token_shape()));
          c.a.o = desc(ones, hf); c.a.den = desc(den, hf);
        }
      }
      ws = c.cut(op);
    } else if (op == OP_GLA) {
      gradients();
      c.a.amat = kept(1, dt, {64, 64}); c.a.qe = kept(2, dt, {64, c.K}); c.a.ke = kept(3, dt, {64, c.K}); c.a.gcum = (float*)kept(4, at::kFloat, {c.K});
      dg = at::empty(c.g.sizes(), c.g.options());             // (in the type of g, by the kernel)
      c.a.dg = desc(dg, hf);
      ws = c.cut(op);
    } else {
      c.a.tinv = kept(1, dt, {64, 64}); c.a.pmat = kept(2, dt, {64, 64}); c.a.gcum = (float*)kept(3, at::kFloat, {5, 64}); c.a.vnew.ptr = kept(4, dt, {c.V / 32, 64, 32});
      const Tensor dvnew = c.chunked({c.V / 32, 64, 32}, dt), seg_p = saved(5);
      c.a.dvnew.ptr = dvnew.data_ptr();
      if (has_extra) {
        c.a.v_act = yes(extra(0));
        const Tensor *like[] = {&c.q, &c.k, &c.v, &c.q, &c.k};
        Tensor given[5];
        for (int i = 0; i < 5; ++i) {
          given[i] = plain_or_none(extra(1 + i), c.dev);
          if (given[i].defined()) need(given[i].sizes() == like[i]->sizes() && given[i].scalar_type() == dt && rows_aligned(given[i]));
        }
        dq = given[0]; dk = given[1]; dv = given[2];
        need(given[3].defined() == given[4].defined());
        if (given[3].defined()) { c.a.q_raw = desc(given[3], hf); c.a.k_raw = desc(given[4], hf); c.a.qk_eps = (float)PyFloat_AsDouble(extra(6)); }
      }
      gradients();
      dg = at::empty(c.beta.sizes(), c.beta.options().dtype(at::kFloat));
      dbeta = at::empty(c.beta.sizes(), c.beta.options());
      c.a.dbeta_bf16 = bf16(dbeta);
      c.a.dg = desc(dg, hf); c.a.dbeta = desc(dbeta, hf);
      if (seg_p.defined()) {
        need(f32(seg_p) && seg_p.is_contiguous() && (reinterpret_cast<uintptr_t>(seg_p.data_ptr()) & 15) == 0);
        ws = c.cut(op);
        need(!ws.defined() || seg_p.numel() == lib.split_floats(&c.a, op, 0));
        if (ws.defined()) c.a.seg_p = (float*)seg_p.data_ptr();
      }
      if (!c.g.defined()) {
        void* st = stream_of(o[14]);
        return result(launch([&] { return lib.bwd[op](&c.a, st); }), {dq, dk, dv, Tensor(), dbeta, dh0});
      }
    }
    void* st = stream_of(o[14]);
    return result(launch([&] { return lib.bwd[op](&c.a, st); }), {dq, dk, dv, dg, dbeta, dh0});
  });
}

// bind(path): the library's entry points
PyObject* bind(PyObject*, PyObject* path) {
  const char* p = PyUnicode_AsUTF8(path);
  if (!p) return nullptr;
  void* h = dlopen(p, RTLD_NOW | RTLD_LOCAL);
  if (!h) return PyErr_Format(PyExc_RuntimeError, "%s", dlerror());
  auto sym = [&](const char* name) { return dlsym(h, name); };
  Library l;
  l.fwd[OP_SIMPLE] = (op_fn)sym("lmoe_chunk_simple_gla_fwd"); l.bwd[OP_SIMPLE] = (op_fn)sym("lmoe_chunk_simple_gla_bwd");
  l.fwd[OP_GLA] = (op_fn)sym("lmoe_chunk_gla_fwd"); l.bwd[OP_GLA] = (op_fn)sym("lmoe_chunk_gla_bwd");
  l.fwd[OP_GDN] = (op_fn)sym("lmoe_chunk_gated_delta_rule_fwd"); l.bwd[OP_GDN] = (op_fn)sym("lmoe_chunk_gated_delta_rule_bwd");
  l.recurrent = (rec_fn)sym("lmoe_fused_recurrent_fwd");
  l.split_floats = (split_fn)sym("lmoe_split_floats");
  for (int i = 0; i < 3; ++i)
    if (!l.fwd[i] || !l.bwd[i]) return PyErr_Format(PyExc_RuntimeError, "%s lacks an entry point", p);
  if (!l.recurrent || !l.split_floats) return PyErr_Format(PyExc_RuntimeError, "%s lacks an entry point", p);
  lib = l;
  return PyLong_FromLong(LMOE_VERSION);
}

PyMethodDef methods[] = {
    {"bind", (PyCFunction)bind, METH_O, nullptr},
    {"recurrent", (PyCFunction)(void (*)(void))recurrent, METH_FASTCALL, nullptr},
    {"forward", (PyCFunction)(void (*)(void))forward, METH_FASTCALL, nullptr},
    {"backward", (PyCFunction)(void (*)(void))backward, METH_FASTCALL, nullptr},
    {nullptr, nullptr, 0, nullptr}};
PyModuleDef module = {PyModuleDef_HEAD_INIT, "_native", nullptr, -1, methods};

}  // namespace

PyMODINIT_FUNC PyInit__native(void) { return PyModule_Create(&module); }
