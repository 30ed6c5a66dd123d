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

// Not a call for this path: the checks return false, and nothing has been allocated or thrown by then (an exception per call cost
// those calls 3 us each: a decoded token with half-precision gates 28 -> 31, so 29).
#define NEED(ok) do { if (!(ok)) return false; } while (0)

// A tensor as the kernels may read it: an ordinary one (no subclass, no wrapper of a transform, nothing lazy) on device dev
bool plain(Tensor& to, PyObject* o, int dev) {
  static const c10::DispatchKeySet ordinary({c10::DispatchKey::CUDA, c10::DispatchKey::ADInplaceOrView, c10::DispatchKey::AutogradCUDA, c10::DispatchKey::AutocastCUDA});
  NEED(THPVariable_CheckExact(o));
  const Tensor& t = THPVariable_Unpack(o);
  NEED(t.defined() && (t.key_set().raw_repr() & ~ordinary.raw_repr()) == 0 && t.layout() == at::kStrided && t.get_device() == dev);
  to = t;
  return true;
}
bool plain_or_none(Tensor& to, PyObject* o, int dev) { return o == Py_None || plain(to, o, dev); }
// the current device; -1 where o is no tensor on a GPU
int current_device(PyObject* o) {
  if (!THPVariable_CheckExact(o) || !THPVariable_Unpack(o).is_cuda()) return -1;
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

bool aligned(const Tensor& x) { return (reinterpret_cast<uintptr_t>(x.data_ptr()) & 15) == 0; }

struct Call {
  int dev;
  bool head_first;
  int64_t B, T, H, K, V, N, NT;
  lmoe_args a = {};
  Tensor q, k, v, g, beta, h0, tables[5];
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
  // a per-token scalar in fp32
  bool token_scalar(const Tensor& x) const { return f32(x) && x.is_contiguous() && x.sizes() == at::IntArrayRef(token_shape()); }
  // a tensor that lies as one of the inputs may
  bool lies_like(const Tensor& x, const Tensor& input) const {
    return x.sizes() == input.sizes() && x.scalar_type() == input.scalar_type() && rows_aligned(x);
  }

  // q, k, v, the gate, beta, the initial state and, for packed input, the tables (N, NT, cu, chunk_map, seq_chunk0, seq_order,
  // nt_dev): checked, and entered into the block
  bool take(int op, PyObject* const* o, PyObject* plan, PyObject* scale, bool hf, bool recurrent = false, bool wu = false) {
    dev = current_device(o[0]); head_first = hf;
    NEED(dev >= 0 && plain(q, o[0], dev) && plain(k, o[1], dev) && plain(v, o[2], dev));
    NEED(q.dim() == 4 && v.dim() == 4 && (bf16(q) || f32(q)) && k.scalar_type() == q.scalar_type() && v.scalar_type() == q.scalar_type());
    NEED(op != OP_GDN || recurrent || wu || bf16(q));         // wu: the 4-byte delta rule too, which needs w and u as well
    NEED(k.sizes() == q.sizes() && v.sizes().slice(0, 3) == q.sizes().slice(0, 3));
    NEED(q.numel() > 0 && v.numel() > 0);
    B = q.size(0); T = q.size(hf ? 2 : 1); H = q.size(hf ? 1 : 2); K = q.size(3); V = v.size(3);
    NEED(((K == 64 || K == 128) && (V == 64 || V == 128)) || (op == OP_GDN && !recurrent && K == 128 && V == 256));
    NEED(rows_aligned(q) && rows_aligned(k) && rows_aligned(v));
    NEED(B <= INT32_MAX && T <= INT32_MAX && H <= INT32_MAX);
    a.dtype = bf16(q) ? LMOE_BF16 : LMOE_F32;
    N = B; NT = B * ((T + LMOE_CHUNK - 1) / LMOE_CHUNK);
    if (plan != Py_None) {
      NEED(PyTuple_Check(plan) && PyTuple_GET_SIZE(plan) == 7 && !hf && B == 1);
      N = PyLong_AsLongLong(PyTuple_GET_ITEM(plan, 0)); NT = PyLong_AsLongLong(PyTuple_GET_ITEM(plan, 1));
      for (int i = 0; i < 5; ++i) NEED(plain_or_none(tables[i], PyTuple_GET_ITEM(plan, 2 + i), dev));
      auto table = [&](int i) { return (const int32_t*)ptr(tables[i]); };
      a.cu_seqlens = table(0); a.chunk_map = table(1); a.seq_chunk0 = table(2); a.seq_order = table(3); a.nt_dev = table(4);
    }
    NEED(NT <= INT32_MAX);
    a.B = B; a.T = T; a.H = H; a.K = K; a.V = V; a.N = N; a.NT = NT;
    const double sc = scale == Py_None ? std::pow((double)K, -0.5) : PyFloat_AsDouble(scale);
    if (sc == -1.0 && PyErr_Occurred()) { PyErr_Clear(); return false; }
    a.scale = (float)sc;
    a.q = desc(q, hf); a.k = desc(k, hf); a.v = desc(v, hf);
    NEED(plain_or_none(g, o[3], dev));
    a.gate = LMOE_GATE_NONE;
    if (g.defined()) {
      NEED(f32(g) || bf16(g));
      if (op == OP_GLA) {
        NEED(g.sizes() == q.sizes() && rows_aligned(g) && (recurrent || bf16(q) || f32(g)));
        a.gate = LMOE_GATE_VECTOR;
      } else {
        NEED(g.dim() == 3 && g.sizes() == at::IntArrayRef(token_shape()));
        a.gate = LMOE_GATE_SCALAR;
      }
      a.g = desc(g, hf); a.g_dtype = f32(g) ? LMOE_F32 : LMOE_BF16;
    } else {
      NEED(op != OP_GLA);
    }
    NEED(plain_or_none(beta, o[4], dev));
    if (op == OP_GDN) {
      NEED(beta.defined() && (f32(beta) || bf16(beta)) && beta.dim() == 3 && beta.sizes() == at::IntArrayRef(token_shape()));
      a.beta = desc(beta, hf); a.beta_dtype = f32(beta) ? LMOE_F32 : LMOE_BF16;
    }
    NEED(plain_or_none(h0, o[5], dev));
    if (h0.defined()) NEED(f32(h0) && h0.is_contiguous() && h0.dim() == 4 && h0.sizes() == at::IntArrayRef({N, H, K, V}));
    a.h0 = (const float*)ptr(h0);
    return true;
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

// Allocations and the launch run without the interpreter's lock, as torch's own allocating functions do: an allocation may wait
// for the device (hipMalloc, or hipFree of cached blocks), and other threads go on meanwhile.
struct Unlocked {
  PyThreadState* const state = PyEval_SaveThread();
  ~Unlocked() { PyEval_RestoreThread(state); }
};
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
bool yes(PyObject* o) { return PyObject_IsTrue(o) == 1; }
// Not a call for this path; what a flag or a number of another kind has raised meanwhile, the Python steps raise in their words.
PyObject* elsewhere() {
  PyErr_Clear();
  Py_RETURN_NONE;
}
void* stream_of(PyObject* o) { return PyLong_AsVoidPtr(o); }

// recurrent(op, q, k, v, g, beta, h0, plan, scale, final_state, head_first, qk_eps, stream) -> (o, ht)
PyObject* recurrent(PyObject*, PyObject* const* o, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  Call c;
  const int op = (int)PyLong_AsLong(o[0]);
  if (n != 13 || !c.take(op, o + 1, o[7], o[8], yes(o[10]), true)) return elsewhere();
  const bool final_state = yes(o[9]);
  c.a.qk_eps = (float)PyFloat_AsDouble(o[11]);
  void* st = stream_of(o[12]);
  if (PyErr_Occurred()) return elsewhere();
  Tensor out, ht;
  int rc;
  {
    const Unlocked unlocked;
    out = at::empty_like(c.v.detach());
    if (final_state) ht = c.states();
    c.a.o = desc(out, c.head_first); c.a.ht = (float*)ptr(ht);
    rc = lib.recurrent(&c.a, op, st);
  }
  return result(rc, {out, ht});
  END_HANDLE_TH_ERRORS
}

// forward(op, q, k, v, g, beta, h0, plan, scale, final_state, head_first, save, normalize, norm_eps, v_act, stream)
//   -> (o, ht, hs, ...) and per op  simple_gla: den, zs;  gla: amat, qe, ke, gdec;  gated delta rule: tinv, pmat, gcum, vnew, seg_p
PyObject* forward(PyObject*, PyObject* const* o, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  Call c;
  const int op = (int)PyLong_AsLong(o[0]);
  if (n != 16 || !c.take(op, o + 1, o[7], o[8], yes(o[10]))) return elsewhere();
  const bool save = yes(o[11]), v_act = yes(o[14]), final_state = yes(o[9]), hf = c.head_first, two = bf16(c.q);
  const int normalize = (int)PyLong_AsLong(o[12]);
  c.a.norm_eps = (float)PyFloat_AsDouble(o[13]);
  void* st = stream_of(o[15]);
  if ((normalize && (c.g.defined() || !two)) || PyErr_Occurred()) return elsewhere();
  const auto dt = c.q.scalar_type();
  Tensor out, ht, hs, den, zs, amat, qe, ke, gcum, tinv, pmat, vnew, seg_p;
  int rc;
  {
    const Unlocked unlocked;
    // (v_act: v is a block of a wider tensor; o is a tensor of its own)
    out = v_act ? at::empty(c.v.sizes(), c.v.options()) : at::empty_like(c.v);
    if (final_state) ht = c.states();
    c.a.o = desc(out, hf); c.a.ht = (float*)ptr(ht);
    if (save || (op == OP_GLA && !two)) hs = c.chunked({c.K, c.V}, dt);
    c.a.hs = ptr(hs);
    if (op == OP_SIMPLE && normalize) {
      den = at::empty(c.token_shape(), c.q.options().dtype(at::kFloat));
      if (save) zs = c.chunked({c.K}, at::kFloat);
      c.a.normalize = normalize; c.a.den = desc(den, hf); c.a.zs = (float*)ptr(zs);
    } else if (op == OP_GLA) {
      amat = c.chunked({64, 64}, dt); qe = c.chunked({64, c.K}, dt); ke = c.chunked({64, c.K}, dt); gcum = c.chunked({c.K}, at::kFloat);
      c.a.amat = ptr(amat); c.a.qe = ptr(qe); c.a.ke = ptr(ke); c.a.gcum = (float*)ptr(gcum);
    } else if (op == OP_GDN) {
      if (save) { pmat = c.chunked({64, 64}, dt); vnew = c.chunked({c.V / 32, 64, 32}, dt); }
      tinv = c.chunked({64, 64}, dt); gcum = c.chunked({5, 64}, at::kFloat);
      c.a.tinv = ptr(tinv); c.a.pmat = ptr(pmat); c.a.gcum = (float*)ptr(gcum); c.a.vnew.ptr = ptr(vnew);
      c.a.v_act = v_act;
    }
    const Tensor ws = c.cut(op);
    if (op == OP_GDN && ws.defined() && save) {
      seg_p = at::empty({lib.split_floats(&c.a, op, 0)}, c.q.options().dtype(at::kFloat));
      c.a.seg_p = (float*)seg_p.data_ptr();
    }
    rc = lib.fwd[op](&c.a, st);
  }
  if (op == OP_SIMPLE) return result(rc, {out, ht, hs, den, zs});
  if (op == OP_GLA) return result(rc, {out, ht, hs, amat, qe, ke, gcum});
  return result(rc, {out, ht, hs, tinv, pmat, gcum, vnew, seg_p});
  END_HANDLE_TH_ERRORS
}

// The arguments of a backward call, checked
struct Backward : Call {
  Tensor dout, dht, saved[6], den, o, given[5];      // given: dq, dk, dv, q_raw, k_raw
  // What was saved may have been through a hook, which hands back what it likes; the kernels index the full extent: of the
  // type and size that forward allocated, contiguous and on a 16-byte boundary.  (Anything else: the Python steps convert or
  // refuse it, _host.came_back.)
  bool kept(int i, at::ScalarType t, Tail tail) const {
    const Tensor& x = saved[i];
    return x.defined() && x.is_contiguous() && x.scalar_type() == t && x.sizes() == at::IntArrayRef(chunked_shape(tail)) && aligned(x);
  }
  bool take_all(int op, PyObject* const* p, bool wu = false) {
    NEED(take(op, p + 1, p[7], p[8], yes(p[11]), false, wu));
    const auto dt = q.scalar_type();
    NEED(plain(dout, p[9], dev) && lies_like(dout, v));
    NEED(plain_or_none(dht, p[10], dev));
    if (dht.defined()) NEED(f32(dht) && dht.is_contiguous() && dht.sizes() == at::IntArrayRef({N, H, K, V}));
    a.d_o = desc(dout, head_first); a.dht = (const float*)ptr(dht);
    const int nsaved = op == OP_SIMPLE ? 3 : op == OP_GLA ? 5 : 6;
    NEED(PyTuple_Check(p[12]) && PyTuple_GET_SIZE(p[12]) == nsaved);
    for (int i = 0; i < nsaved; ++i) NEED(plain_or_none(saved[i], PyTuple_GET_ITEM(p[12], i), dev));
    NEED(kept(0, dt, {K, V}));
    a.hs = ptr(saved[0]);
    PyObject* const extra = p[13];
    const int nextra = op == OP_SIMPLE ? 4 : 7;
    NEED(extra == Py_None || (PyTuple_Check(extra) && PyTuple_GET_SIZE(extra) == nextra));
    if (op == OP_SIMPLE && extra != Py_None) {
      a.normalize = (int)PyLong_AsLong(PyTuple_GET_ITEM(extra, 0)); a.norm_eps = (float)PyFloat_AsDouble(PyTuple_GET_ITEM(extra, 1));
      NEED(kept(2, at::kFloat, {K}));
      a.zs = (float*)ptr(saved[2]);
      if (a.normalize == 2) {
        NEED(plain(den, PyTuple_GET_ITEM(extra, 3), dev) && token_scalar(den));
        a.dden = desc(den, head_first);
      } else {
        NEED(plain(o, PyTuple_GET_ITEM(extra, 2), dev) && lies_like(o, v) && saved[1].defined() && token_scalar(saved[1]));
        a.o = desc(o, head_first); a.den = desc(saved[1], head_first);
      }
    }
    if (op == OP_GLA) {
      NEED(kept(1, dt, {64, 64}) && kept(2, dt, {64, K}) && kept(3, dt, {64, K}) && kept(4, at::kFloat, {K}));
      a.amat = ptr(saved[1]); a.qe = ptr(saved[2]); a.ke = ptr(saved[3]); a.gcum = (float*)ptr(saved[4]);
    }
    if (op == OP_GDN) {
      NEED(kept(1, dt, {64, 64}) && kept(2, dt, {64, 64}) && kept(3, at::kFloat, {5, 64}) && kept(4, dt, {V / 32, 64, 32}));
      a.tinv = ptr(saved[1]); a.pmat = ptr(saved[2]); a.gcum = (float*)ptr(saved[3]); a.vnew.ptr = ptr(saved[4]);
      if (saved[5].defined()) {
        // (as many as the forward call was told: none where the call is not cut)
        const int64_t np = lib.split_floats(&a, op, 0);
        NEED(f32(saved[5]) && saved[5].is_contiguous() && aligned(saved[5]) && (np <= 0 || saved[5].numel() == np));
        if (np > 0) a.seg_p = (float*)ptr(saved[5]);
      }
      if (extra != Py_None) {
        a.v_act = yes(PyTuple_GET_ITEM(extra, 0));
        const Tensor* like[] = {&q, &k, &v, &q, &k};
        for (int i = 0; i < 5; ++i) {
          NEED(plain_or_none(given[i], PyTuple_GET_ITEM(extra, 1 + i), dev));
          if (given[i].defined()) NEED(lies_like(given[i], *like[i]));
        }
        NEED(given[3].defined() == given[4].defined());
        if (given[3].defined()) {
          a.q_raw = desc(given[3], head_first); a.k_raw = desc(given[4], head_first);
          a.qk_eps = (float)PyFloat_AsDouble(PyTuple_GET_ITEM(extra, 6));
        }
      }
    }
    return true;
  }
};

// backward(op, q, k, v, g, beta, h0, plan, scale, do, dht, head_first, saved, extra, stream) -> (dq, dk, dv, dg, dbeta, dh0)
//   saved: what forward returned behind ht;  extra: simple_gla (normalize, norm_eps, o, dden), gated delta rule (v_act, dq, dk,
//   dv, q_raw, k_raw, qk_eps), None where a call has none
PyObject* backward(PyObject*, PyObject* const* o, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  Backward c;
  const int op = (int)PyLong_AsLong(o[0]);
  if (n != 15 || !c.take_all(op, o)) return elsewhere();
  void* st = stream_of(o[14]);
  if (PyErr_Occurred()) return elsewhere();
  const bool hf = c.head_first;
  const auto dt = c.q.scalar_type();
  auto fresh = [&](const Tensor& x) { return at::empty_like(x.detach()); };
  auto or_fresh = [&](const Tensor& x, const Tensor& like) { return x.defined() ? x : fresh(like); };
  Tensor dq, dk, dv, dg, dbeta, dh0;
  int rc;
  {
    const Unlocked unlocked;
    dq = or_fresh(c.given[0], c.q); dk = or_fresh(c.given[1], c.k); dv = or_fresh(c.given[2], c.v);
    if (c.h0.defined()) dh0 = fresh(c.h0);
    const Tensor dhs = c.chunked({c.K, c.V}, dt);
    c.a.dq = desc(dq, hf); c.a.dk = desc(dk, hf); c.a.dv = desc(dv, hf); c.a.dh0 = (float*)ptr(dh0); c.a.dhs = ptr(dhs);
    Tensor dvnew, norm_ws, ws;
    if (op == OP_GLA) {
      dg = at::empty(c.g.sizes(), c.g.options());           // (in the type of g, by the kernel)
    } else if (op == OP_GDN || c.g.defined()) {
      const Tensor& like = op == OP_GDN ? c.beta : c.g;
      dg = at::empty(like.sizes(), like.options().dtype(at::kFloat));
    }
    c.a.dg = desc(dg, hf);
    if (c.a.normalize) {
      norm_ws = c.chunked({c.V / 32, 64 + c.K}, at::kFloat);
      c.a.norm_ws = (float*)norm_ws.data_ptr();
    }
    if (op == OP_GDN) {
      dvnew = c.chunked({c.V / 32, 64, 32}, dt);
      dbeta = at::empty(c.beta.sizes(), c.beta.options());
      c.a.dvnew.ptr = ptr(dvnew); c.a.dbeta_bf16 = bf16(dbeta); c.a.dbeta = desc(dbeta, hf);
    }
    if (op != OP_GDN || c.a.seg_p) ws = c.cut(op);
    rc = lib.bwd[op](&c.a, st);
  }
  return result(rc, {dq, dk, dv, c.g.defined() ? dg : Tensor(), dbeta, dh0});
  END_HANDLE_TH_ERRORS
}

// intact(the arguments of backward) -> (B, T, H, K, V) where backward would take them as they are or, for the 4-byte delta rule,
// where the Python steps may: nothing that was saved has to be converted or refused.  None otherwise.
PyObject* intact(PyObject*, PyObject* const* o, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  Backward c;
  if (n != 15 || !c.take_all((int)PyLong_AsLong(o[0]), o, true) || PyErr_Occurred()) return elsewhere();
  return Py_BuildValue("LLLLL", (long long)c.B, (long long)c.T, (long long)c.H, (long long)c.K, (long long)c.V);
  END_HANDLE_TH_ERRORS
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
    {"intact", (PyCFunction)(void (*)(void))intact, METH_FASTCALL, nullptr},
    {nullptr, nullptr, 0, nullptr}};
PyModuleDef module = {PyModuleDef_HEAD_INIT, "_native", nullptr, -1, methods};

}  // namespace

PyMODINIT_FUNC PyInit__native(void) { return PyModule_Create(&module); }
