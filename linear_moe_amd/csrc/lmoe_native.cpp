// Launch path of the ops in native code: the argument checks, allocations and the argument block of a call, and the
// call of the library's entry point, for the calls that need nothing in front of it -- plain tensors on the current
// device, in types and strides the kernels take.  For every other call the functions return None and the caller (the
// Python of the op: _host.py, simple_gla.py, gla.py, gated_delta_rule.py, recurrent.py) converts, copies or refuses as it
// always did; results are the same bits either way.  What it is for: a call of three to four small kernels takes the GPU
// 5 to 100 us, and the same steps through Python objects and ctypes took the host 20 us per forward and as much
// per backward (figures in linear_moe_amd/_host.py).  The neighbours of the ops (gates, prologue, output gate, routing of a
// mixture of memories: gates.py, layer_io.py, mom.py) take it too: a mixer's step is four autograd nodes and twelve launches.
#include <Python.h>
#include <dlfcn.h>

#include <cmath>
#include <initializer_list>
#include <type_traits>

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
  // the neighbours, in the types of lmoe.h
  decltype(&lmoe_gdn_qkv_prologue_fwd) prologue_fwd;
  decltype(&lmoe_swish_gate_relayout_fwd) swish_fwd;
  decltype(&lmoe_swish_gate_relayout_bwd) swish_bwd;
  decltype(&lmoe_gdn_gates_partials) gates_partials;
  decltype(&lmoe_gdn_gates_fwd) gates_fwd;
  decltype(&lmoe_gdn_gates_bwd) gates_bwd;
  decltype(&lmoe_mom_gather) mom_gather;
  decltype(&lmoe_mom_combine) mom_combine;
  decltype(&lmoe_mom_combine_bwd) mom_combine_bwd;
  decltype(&lmoe_mom_plan_ints) mom_plan_ints;
  decltype(&lmoe_mom_plan) mom_plan;
  decltype(&lmoe_seq_tables) seq_tables;
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
    dev = current_device(o[0]);
    NEED(dev >= 0 && plain(q, o[0], dev) && plain(k, o[1], dev) && plain(v, o[2], dev));
    return take_from(op, o + 3, plan, scale, hf, recurrent, wu);
  }
  // the same with dev, q, k, v set (by plain, or by the caller's own allocation); o: the gate, beta, the initial state
  bool take_from(int op, PyObject* const* o, PyObject* plan, PyObject* scale, bool hf, bool recurrent = false, bool wu = false) {
    head_first = hf;
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
    NEED(plain_or_none(g, o[0], dev));
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
    NEED(plain_or_none(beta, o[1], dev));
    if (op == OP_GDN) {
      NEED(beta.defined() && (f32(beta) || bf16(beta)) && beta.dim() == 3 && beta.sizes() == at::IntArrayRef(token_shape()));
      a.beta = desc(beta, hf); a.beta_dtype = f32(beta) ? LMOE_F32 : LMOE_BF16;
    }
    NEED(plain_or_none(h0, o[2], dev));
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

// What a forward call of an op allocates beside its inputs, and its launch
struct Forward : Call {
  Tensor out, ht, hs, den, zs, amat, qe, ke, gcum, tinv, pmat, vnew, seg_p;
  int launch(int op, bool save, bool final_state, int normalize, bool v_act, void* st) {
    const auto dt = q.scalar_type();
    const bool hf = head_first, two = bf16(q);
    // (v_act: v is a block of a wider tensor; o is a tensor of its own)
    out = v_act ? at::empty(v.sizes(), v.options()) : at::empty_like(v);
    if (final_state) ht = states();
    a.o = desc(out, hf); a.ht = (float*)ptr(ht);
    if (save || (op == OP_GLA && !two)) hs = chunked({K, V}, dt);
    a.hs = ptr(hs);
    if (op == OP_SIMPLE && normalize) {
      den = at::empty(token_shape(), q.options().dtype(at::kFloat));
      if (save) zs = chunked({K}, at::kFloat);
      a.normalize = normalize; a.den = desc(den, hf); a.zs = (float*)ptr(zs);
    } else if (op == OP_GLA) {
      amat = chunked({64, 64}, dt); qe = chunked({64, K}, dt); ke = chunked({64, K}, dt); gcum = chunked({K}, at::kFloat);
      a.amat = ptr(amat); a.qe = ptr(qe); a.ke = ptr(ke); a.gcum = (float*)ptr(gcum);
    } else if (op == OP_GDN) {
      if (save) { pmat = chunked({64, 64}, dt); vnew = chunked({V / 32, 64, 32}, dt); }
      tinv = chunked({64, 64}, dt); gcum = chunked({5, 64}, at::kFloat);
      a.tinv = ptr(tinv); a.pmat = ptr(pmat); a.gcum = (float*)ptr(gcum); a.vnew.ptr = ptr(vnew);
      a.v_act = v_act;
    }
    const Tensor ws = cut(op);
    if (op == OP_GDN && ws.defined() && save) {
      seg_p = at::empty({lib.split_floats(&a, op, 0)}, q.options().dtype(at::kFloat));
      a.seg_p = (float*)seg_p.data_ptr();
    }
    return lib.fwd[op](&a, st);
  }
};

// forward(op, q, k, v, g, beta, h0, plan, scale, final_state, head_first, save, normalize, norm_eps, v_act, stream)
//   -> (o, ht, hs, ...) and per op  simple_gla: den, zs;  gla: amat, qe, ke, gdec;  gated delta rule: tinv, pmat, gcum, vnew, seg_p
PyObject* forward(PyObject*, PyObject* const* o, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  Forward c;
  const int op = (int)PyLong_AsLong(o[0]);
  if (n != 16 || !c.take(op, o + 1, o[7], o[8], yes(o[10]))) return elsewhere();
  const bool save = yes(o[11]), v_act = yes(o[14]), final_state = yes(o[9]);
  const int normalize = (int)PyLong_AsLong(o[12]);
  c.a.norm_eps = (float)PyFloat_AsDouble(o[13]);
  void* st = stream_of(o[15]);
  if ((normalize && (c.g.defined() || !bf16(c.q))) || PyErr_Occurred()) return elsewhere();
  int rc;
  {
    const Unlocked unlocked;
    rc = c.launch(op, save, final_state, normalize, v_act, st);
  }
  if (op == OP_SIMPLE) return result(rc, {c.out, c.ht, c.hs, c.den, c.zs});
  if (op == OP_GLA) return result(rc, {c.out, c.ht, c.hs, c.amat, c.qe, c.ke, c.gcum});
  return result(rc, {c.out, c.ht, c.hs, c.tinv, c.pmat, c.gcum, c.vnew, c.seg_p});
  END_HANDLE_TH_ERRORS
}

// A fused projection [T, B, H 3 D] or [T, B, H, 3 D]; block i of it (q, k, v) as [B, T, H, D]
bool projection(const Tensor& x, int64_t H, int64_t D) {
  return (x.dim() == 3 || x.dim() == 4) && bf16(x) && x.is_contiguous() && aligned(x) && (D == 64 || D == 128) && H > 0 &&
         x.numel() > 0 && x.numel() == x.size(0) * x.size(1) * H * 3 * D;
}
Tensor block_of(const Tensor& x, int64_t H, int64_t D, int i) {
  const int64_t T = x.size(0), B = x.size(1), W = 3 * H * D;
  return at::as_strided(x, {B, T, H, D}, {W, B * W, 3 * D, 1}, x.storage_offset() + i * D);
}

// mixer_forward(qkv, g, beta, H, D, eps, scale, save, stream) -> (o, q, k, v, hs, tinv, pmat, gcum, vnew, seg_p): the prologue on
// the q and k blocks of the projection, and the gated delta rule with SiLU on its v block
PyObject* mixer_forward(PyObject*, PyObject* const* o, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  if (n != 9) return elsewhere();
  Forward c;
  Tensor x;
  c.dev = current_device(o[0]);
  const int64_t H = PyLong_AsLongLong(o[3]), D = PyLong_AsLongLong(o[4]);
  const float eps = (float)PyFloat_AsDouble(o[5]);
  const bool save = yes(o[7]);
  void* st = stream_of(o[8]);
  if (PyErr_Occurred() || c.dev < 0 || !plain(x, o[0], c.dev) || !projection(x, H, D)) return elsewhere();
  {
    const Unlocked unlocked;
    c.q = at::empty({x.size(1), x.size(0), H, D}, x.options()); c.k = at::empty_like(c.q); c.v = block_of(x, H, D, 2);
  }
  PyObject* const rest[] = {o[1], o[2], Py_None};
  if (!c.take_from(OP_GDN, rest, Py_None, o[6], false)) return elsewhere();
  int rc;
  {
    const Unlocked unlocked;
    rc = lib.prologue_fwd(x.data_ptr(), c.q.data_ptr(), c.k.data_ptr(), nullptr, (int32_t)c.T, (int32_t)c.B, (int32_t)H, (int32_t)D, LMOE_BF16, eps, st);
    if (rc == 0) rc = c.launch(OP_GDN, save, false, 0, true, st);
  }
  return result(rc, {c.out, c.q, c.k, c.v, c.hs, c.tinv, c.pmat, c.gcum, c.vnew, c.seg_p});
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

// What a backward call of an op allocates, and its launch
struct Gradients {
  Tensor dq, dk, dv, dg, dbeta, dh0;
  int launch(int op, Backward& c, void* st) {
    const bool hf = c.head_first;
    const auto dt = c.q.scalar_type();
    auto fresh = [&](const Tensor& x) { return at::empty_like(x.detach()); };
    auto or_fresh = [&](const Tensor& x, const Tensor& like) { return x.defined() ? x : fresh(like); };
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
    const int rc = lib.bwd[op](&c.a, st);
    if (!c.g.defined()) dg = Tensor();
    return rc;
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
  Gradients d;
  int rc;
  {
    const Unlocked unlocked;
    rc = d.launch(op, c, st);
  }
  return result(rc, {d.dq, d.dk, d.dv, d.dg, d.dbeta, d.dh0});
  END_HANDLE_TH_ERRORS
}

// mixer_backward(x, eps, the arguments of backward with extra = None) -> (dx, dg, dbeta): q and k were l2norm(silu(.)) of blocks
// of the projection x, v its third block; the op fills the blocks of dx
PyObject* mixer_backward(PyObject*, PyObject* const* o, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  Backward c;
  Tensor x;
  if (n != 17 || PyLong_AsLong(o[2]) != OP_GDN || !c.take_all(OP_GDN, o + 2)) return elsewhere();
  const float eps = (float)PyFloat_AsDouble(o[1]);
  void* st = stream_of(o[16]);
  if (PyErr_Occurred() || !plain(x, o[0], c.dev) || !projection(x, c.H, c.K) || c.V != c.K || x.size(0) != c.T || x.size(1) != c.B || !bf16(c.q))
    return elsewhere();
  Gradients d;
  Tensor dx;
  int rc;
  {
    const Unlocked unlocked;
    dx = at::empty_like(x.detach());
    for (int i = 0; i < 3; ++i) c.given[i] = block_of(dx, c.H, c.K, i);
    c.a.q_raw = desc(block_of(x, c.H, c.K, 0), false); c.a.k_raw = desc(block_of(x, c.H, c.K, 1), false);
    c.a.qk_eps = eps; c.a.v_act = 1;
    rc = d.launch(OP_GDN, c, st);
  }
  return result(rc, {dx, d.dg, d.dbeta});
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

// ---- the neighbours of the ops ----
int dtype_of(const Tensor& x) { return f32(x) ? LMOE_F32 : bf16(x) ? LMOE_BF16 : -1; }
// contiguous, in a type of the library, on a 16-byte boundary
bool dense(const Tensor& x) { return dtype_of(x) >= 0 && x.is_contiguous() && aligned(x) && x.numel() > 0; }
bool fits(int64_t x) { return x >= 0 && x <= INT32_MAX; }

// swish_forward(o, gate, stream) -> (y,)
// swish_backward(o, gate, dy, stream) -> (do, dgate)
struct Swish {
  Tensor o, gate;
  int64_t B, T, W;
  int dev;
  bool take(PyObject* const* p) {
    dev = current_device(p[0]);
    NEED(dev >= 0 && plain(o, p[0], dev) && plain(gate, p[1], dev));
    NEED(o.dim() == 4 && dense(o) && dense(gate) && gate.scalar_type() == o.scalar_type() && gate.numel() == o.numel() && gate.dim() >= 2);
    B = o.size(0); T = o.size(1); W = o.size(2) * o.size(3);
    return gate.size(0) == T && gate.size(1) == B && W % 8 == 0 && fits(B) && fits(T) && fits(W);
  }
};
PyObject* swish_forward(PyObject*, PyObject* const* p, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  Swish c;
  if (n != 3 || !c.take(p)) return elsewhere();
  void* st = stream_of(p[2]);
  if (PyErr_Occurred()) return elsewhere();
  Tensor y;
  int rc;
  {
    const Unlocked unlocked;
    y = at::empty({c.T, c.B, c.W}, c.o.options());
    rc = lib.swish_fwd(c.o.data_ptr(), c.gate.data_ptr(), y.data_ptr(), (int32_t)c.T, (int32_t)c.B, (int32_t)c.W, dtype_of(c.o), st);
  }
  return result(rc, {y});
  END_HANDLE_TH_ERRORS
}
PyObject* swish_backward(PyObject*, PyObject* const* p, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  Swish c;
  Tensor dy;
  if (n != 4 || !c.take(p) || !plain(dy, p[2], c.dev) || !dense(dy) || dy.scalar_type() != c.o.scalar_type() ||
      dy.sizes() != at::IntArrayRef({c.T, c.B, c.W})) return elsewhere();
  void* st = stream_of(p[3]);
  if (PyErr_Occurred()) return elsewhere();
  Tensor d, dgate;
  int rc;
  {
    const Unlocked unlocked;
    d = at::empty_like(c.o.detach()); dgate = at::empty_like(c.gate.detach());
    rc = lib.swish_bwd(c.o.data_ptr(), c.gate.data_ptr(), dy.data_ptr(), d.data_ptr(), dgate.data_ptr(), (int32_t)c.T, (int32_t)c.B, (int32_t)c.W,
                       dtype_of(c.o), st);
  }
  return result(rc, {d, dgate});
  END_HANDLE_TH_ERRORS
}

// gates_forward(a, b, A_log, dt_bias, stream) -> (g, beta)
// gates_backward(a, b, A_log, dt_bias, dg, dbeta, stream) -> (da, db, dA_log, ddt_bias)
struct Gates {
  Tensor a, b, A, bias;
  int64_t H, rows;
  int dev;
  bool take(PyObject* const* p) {
    dev = current_device(p[0]);
    NEED(dev >= 0 && plain(a, p[0], dev) && plain(b, p[1], dev) && plain(A, p[2], dev) && plain(bias, p[3], dev));
    NEED(a.dim() >= 1 && dense(a) && dense(b) && a.sizes() == b.sizes() && a.scalar_type() == b.scalar_type());
    H = a.size(-1); rows = a.numel() / H;
    NEED(fits(H) && f32(A) && f32(bias) && A.is_contiguous() && bias.is_contiguous());
    return A.dim() == 1 && A.size(0) == H && bias.dim() == 1 && bias.size(0) == H;
  }
};
PyObject* gates_forward(PyObject*, PyObject* const* p, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  Gates c;
  if (n != 5 || !c.take(p)) return elsewhere();
  void* st = stream_of(p[4]);
  if (PyErr_Occurred()) return elsewhere();
  Tensor g, beta;
  int rc;
  {
    const Unlocked unlocked;
    g = at::empty(c.a.sizes(), c.a.options().dtype(at::kFloat)); beta = at::empty_like(c.b.detach());
    rc = lib.gates_fwd(c.a.data_ptr(), c.b.data_ptr(), (const float*)c.A.data_ptr(), (const float*)c.bias.data_ptr(), (float*)g.data_ptr(),
                       beta.data_ptr(), c.rows, (int32_t)c.H, dtype_of(c.a), st);
  }
  return result(rc, {g, beta});
  END_HANDLE_TH_ERRORS
}
PyObject* gates_backward(PyObject*, PyObject* const* p, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  Gates c;
  Tensor dg, dbeta;
  if (n != 7 || !c.take(p) || !plain(dg, p[4], c.dev) || !plain(dbeta, p[5], c.dev)) return elsewhere();
  if (!dense(dg) || !f32(dg) || dg.sizes() != c.a.sizes() || !dense(dbeta) || dbeta.scalar_type() != c.b.scalar_type() || dbeta.sizes() != c.b.sizes())
    return elsewhere();
  void* st = stream_of(p[6]);
  if (PyErr_Occurred()) return elsewhere();
  Tensor da, db, dpar, dA, dbias;
  int rc;
  {
    const Unlocked unlocked;
    const int parts = lib.gates_partials(c.rows, (int32_t)c.H);
    rc = parts < 0 ? parts : 0;
    if (rc == 0) {
      const auto f = c.a.options().dtype(at::kFloat);
      da = at::empty_like(c.a.detach()); db = at::empty_like(c.b.detach()); dpar = at::empty({2, c.H}, f);
      const Tensor part = at::empty({parts, 2, c.H}, f);
      rc = lib.gates_bwd(c.a.data_ptr(), c.b.data_ptr(), (const float*)c.A.data_ptr(), (const float*)c.bias.data_ptr(), (const float*)dg.data_ptr(),
                         dbeta.data_ptr(), da.data_ptr(), db.data_ptr(), (float*)part.data_ptr(), (float*)dpar.data_ptr(), c.rows, (int32_t)c.H,
                         dtype_of(c.a), st);
      dA = dpar.select(0, 0); dbias = dpar.select(0, 1);
    }
  }
  return result(rc, {da, db, dA, dbias});
  END_HANDLE_TH_ERRORS
}

// an index table of a routing plan
bool table_of(Tensor& to, PyObject* o, int dev, int64_t numel) {
  NEED(plain(to, o, dev));
  return to.scalar_type() == at::kInt && to.is_contiguous() && to.numel() == numel;
}
// mom_gather(x, rows, src_token, stream) -> (out,): x as `rows` rows, gathered
PyObject* mom_gather(PyObject*, PyObject* const* p, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  if (n != 4) return elsewhere();
  Tensor x, idx;
  const int dev = current_device(p[0]);
  const int64_t rows = PyLong_AsLongLong(p[1]);
  void* st = stream_of(p[3]);
  if (PyErr_Occurred() || dev < 0 || rows <= 0 || !plain(x, p[0], dev) || !dense(x) || x.numel() % rows || !plain(idx, p[2], dev) ||
      !table_of(idx, p[2], dev, idx.numel()) || idx.numel() == 0) return elsewhere();
  const int64_t D = x.numel() / rows;
  if (D % 8 || !fits(D)) return elsewhere();
  Tensor out;
  int rc;
  {
    const Unlocked unlocked;
    out = at::empty({idx.numel(), D}, x.options());
    rc = lib.mom_gather(x.data_ptr(), (const int32_t*)idx.data_ptr(), nullptr, out.data_ptr(), idx.numel(), (int32_t)D, dtype_of(x), st);
  }
  return result(rc, {out});
  END_HANDLE_TH_ERRORS
}
// mom_combine(y, rows, row_of, w or None, tokens, topk, stream) -> (out [tokens, D],): y as `rows` rows
PyObject* mom_combine(PyObject*, PyObject* const* p, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  if (n != 7) return elsewhere();
  Tensor y, row_of, w;
  const int dev = current_device(p[0]);
  const int64_t rows = PyLong_AsLongLong(p[1]), tokens = PyLong_AsLongLong(p[4]), topk = PyLong_AsLongLong(p[5]);
  void* st = stream_of(p[6]);
  if (PyErr_Occurred() || dev < 0 || rows <= 0 || tokens <= 0 || topk <= 0 || !fits(topk) || !plain(y, p[0], dev) || !dense(y) || y.numel() % rows ||
      !table_of(row_of, p[2], dev, tokens * topk) || !plain_or_none(w, p[3], dev)) return elsewhere();
  if (w.defined() && !(w.scalar_type() == y.scalar_type() && w.is_contiguous() && w.numel() == tokens * topk)) return elsewhere();
  const int64_t D = y.numel() / rows;
  if (D % 8 || !fits(D)) return elsewhere();
  Tensor out;
  int rc;
  {
    const Unlocked unlocked;
    out = at::empty({tokens, D}, y.options());
    rc = lib.mom_combine(y.data_ptr(), (const int32_t*)row_of.data_ptr(), ptr(w), out.data_ptr(), tokens, (int32_t)topk, (int32_t)D, dtype_of(y), st);
  }
  return result(rc, {out});
  END_HANDLE_TH_ERRORS
}
// mom_combine_backward(y, rows, row_of, src_choice, w, dout, tokens, topk, stream) -> (dy, dw), as y and w lie
PyObject* mom_combine_backward(PyObject*, PyObject* const* p, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  if (n != 9) return elsewhere();
  Tensor y, row_of, choice, w, g;
  const int dev = current_device(p[0]);
  const int64_t rows = PyLong_AsLongLong(p[1]), tokens = PyLong_AsLongLong(p[6]), topk = PyLong_AsLongLong(p[7]);
  void* st = stream_of(p[8]);
  if (PyErr_Occurred() || dev < 0 || rows <= 0 || tokens <= 0 || topk <= 0 || !fits(topk) || !plain(y, p[0], dev) || !dense(y) || y.numel() % rows ||
      !table_of(row_of, p[2], dev, tokens * topk) || !table_of(choice, p[3], dev, rows) || !plain(w, p[4], dev) || !plain(g, p[5], dev)) return elsewhere();
  const int64_t D = y.numel() / rows;
  if (D % 8 || !fits(D) || w.scalar_type() != y.scalar_type() || !w.is_contiguous() || w.numel() != tokens * topk || !dense(g) ||
      g.scalar_type() != y.scalar_type() || g.numel() != tokens * D) return elsewhere();
  Tensor dy, dw;
  int rc;
  {
    const Unlocked unlocked;
    dy = at::empty_like(y.detach()); dw = at::empty_like(w.detach());
    rc = lib.mom_combine_bwd(y.data_ptr(), (const int32_t*)row_of.data_ptr(), (const int32_t*)choice.data_ptr(), w.data_ptr(), g.data_ptr(),
                             dy.data_ptr(), dw.data_ptr(), tokens, rows, (int32_t)topk, (int32_t)D, dtype_of(y), st);
  }
  return result(rc, {dy, dw});
  END_HANDLE_TH_ERRORS
}
// mom_plan(selected [B, S, topk], memories, cap or -1, stream) -> (cu, max_len, mem_offsets, src_token, src_choice, row_of [B S, topk])
PyObject* mom_plan(PyObject*, PyObject* const* p, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  if (n != 4) return elsewhere();
  Tensor sel;
  const int dev = current_device(p[0]);
  const int64_t E = PyLong_AsLongLong(p[1]), cap = PyLong_AsLongLong(p[2]);
  void* st = stream_of(p[3]);
  if (PyErr_Occurred() || dev < 0 || !plain(sel, p[0], dev) || sel.dim() != 3 || !sel.is_contiguous() ||
      (sel.scalar_type() != at::kInt && sel.scalar_type() != at::kLong)) return elsewhere();
  const int64_t B = sel.size(0), S = sel.size(1), topk = sel.size(2), count = sel.numel();
  if (count == 0 || !fits(count) || !fits(E) || cap < -1 || !fits(cap + 1)) return elsewhere();
  const int64_t ints = lib.mom_plan_ints((int32_t)B, (int32_t)(S * topk), (int32_t)E);
  if (ints <= 0) return elsewhere();
  Tensor wide, cu, token, choice, row_of, longest, offsets;
  int rc;
  {
    const Unlocked unlocked;
    const auto i32 = sel.options().dtype(at::kInt);
    wide = at::empty({E + 2}, sel.options().dtype(at::kLong)); cu = at::empty({E * B + 1}, i32);
    const Tensor counts = at::empty({ints}, i32);
    token = at::empty({count}, i32); choice = at::empty({count}, i32); row_of = at::empty({B * S, topk}, i32);
    longest = wide.select(0, 0); offsets = wide.narrow(0, 1, E + 1);
    rc = lib.mom_plan(sel.data_ptr(), sel.scalar_type() == at::kLong, (int32_t)B, (int32_t)(S * topk), (int32_t)topk, (int32_t)E, (int32_t)cap,
                      (int32_t*)counts.data_ptr(), (int32_t*)cu.data_ptr(), (int64_t*)longest.data_ptr(), (int64_t*)offsets.data_ptr(),
                      (int32_t*)token.data_ptr(), (int32_t*)choice.data_ptr(), (int32_t*)row_of.data_ptr(), st);
  }
  return result(rc, {cu, longest, offsets, token, choice, row_of});
  END_HANDLE_TH_ERRORS
}
// seq_tables(offsets, T, most, stream) -> (cu, chunk_map, seq_chunk0, seq_order or None, nt_dev) of up to `most` sequences
PyObject* seq_tables(PyObject*, PyObject* const* p, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  if (n != 4) return elsewhere();
  Tensor offs;
  const int dev = current_device(p[0]);
  const int64_t T = PyLong_AsLongLong(p[1]), most = PyLong_AsLongLong(p[2]);
  void* st = stream_of(p[3]);
  if (PyErr_Occurred() || dev < 0 || !plain(offs, p[0], dev) || offs.dim() != 1 || !offs.is_contiguous() ||
      (offs.scalar_type() != at::kInt && offs.scalar_type() != at::kLong)) return elsewhere();
  const int64_t N = offs.numel() - 1, nt = (T + LMOE_CHUNK - 1) / LMOE_CHUNK + N;
  if (N < 1 || N > most || T < 0 || !fits(nt)) return elsewhere();
  Tensor cu, map, c0, order, count;
  int rc;
  {
    const Unlocked unlocked;
    const Tensor all = at::empty({2 * nt + 3 * N + 3}, offs.options().dtype(at::kInt));
    map = at::as_strided(all, {nt, 2}, {2, 1}, 0);
    int64_t at = 2 * nt;
    auto part = [&](int64_t k) { const Tensor x = all.narrow(0, at, k); at += k; return x; };
    cu = part(N + 1); c0 = part(N + 1); count = part(1);
    if (N > 1) order = part(N);
    rc = lib.seq_tables(offs.data_ptr(), offs.scalar_type() == at::kLong, (int32_t)N, (int32_t)nt, (int32_t*)cu.data_ptr(), (int32_t*)map.data_ptr(),
                        (int32_t*)c0.data_ptr(), (int32_t*)count.data_ptr(), (int32_t*)ptr(order), st);
  }
  return result(rc, {cu, map, c0, order, count});
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
  bool all = l.recurrent && l.split_floats;
  auto get = [&](auto& f, const char* name) {
    f = (std::remove_reference_t<decltype(f)>)sym(name);
    all = all && f;
  };
  get(l.prologue_fwd, "lmoe_gdn_qkv_prologue_fwd");
  get(l.swish_fwd, "lmoe_swish_gate_relayout_fwd"); get(l.swish_bwd, "lmoe_swish_gate_relayout_bwd");
  get(l.gates_partials, "lmoe_gdn_gates_partials"); get(l.gates_fwd, "lmoe_gdn_gates_fwd"); get(l.gates_bwd, "lmoe_gdn_gates_bwd");
  get(l.mom_gather, "lmoe_mom_gather"); get(l.mom_combine, "lmoe_mom_combine"); get(l.mom_combine_bwd, "lmoe_mom_combine_bwd");
  get(l.mom_plan_ints, "lmoe_mom_plan_ints"); get(l.mom_plan, "lmoe_mom_plan"); get(l.seq_tables, "lmoe_seq_tables");
  if (!all) return PyErr_Format(PyExc_RuntimeError, "%s lacks an entry point", p);
  lib = l;
  return PyLong_FromLong(LMOE_VERSION);
}

PyMethodDef methods[] = {
    {"bind", (PyCFunction)bind, METH_O, nullptr},
    {"recurrent", (PyCFunction)(void (*)(void))recurrent, METH_FASTCALL, nullptr},
    {"forward", (PyCFunction)(void (*)(void))forward, METH_FASTCALL, nullptr},
    {"backward", (PyCFunction)(void (*)(void))backward, METH_FASTCALL, nullptr},
#define LMOE_METHOD(f) {#f, (PyCFunction)(void (*)(void))f, METH_FASTCALL, nullptr}
    LMOE_METHOD(mixer_forward), LMOE_METHOD(mixer_backward), LMOE_METHOD(swish_forward), LMOE_METHOD(swish_backward),
    LMOE_METHOD(gates_forward), LMOE_METHOD(gates_backward), LMOE_METHOD(mom_gather), LMOE_METHOD(mom_combine),
    LMOE_METHOD(mom_combine_backward), LMOE_METHOD(mom_plan), LMOE_METHOD(seq_tables),
#undef LMOE_METHOD
    {"intact", (PyCFunction)(void (*)(void))intact, METH_FASTCALL, nullptr},
    {nullptr, nullptr, 0, nullptr}};
PyModuleDef module = {PyModuleDef_HEAD_INIT, "_native", nullptr, -1, methods};

}  // namespace

PyMODINIT_FUNC PyInit__native(void) { return PyModule_Create(&module); }
