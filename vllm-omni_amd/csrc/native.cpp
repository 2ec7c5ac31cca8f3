// The host path in native code: a CPython module (vllm_omni_amd._native) between the Python layer and the C ABI
// of libomni_dit_hip.so.
//
// Two kinds of functions:
//   * one per kernel wrapper of kernels.py: checks the tensors, takes their addresses and strides, allocates the
//     result and calls the C entry point. A call whose arguments are not of the usual form (or that the C entry
//     point refuses) returns None and enqueues nothing; the Python wrapper then runs its general path, which
//     handles the unusual forms and raises the errors;
//   * one per transformer block: the block's launches one after the other with raw addresses, its intermediate
//     tensors carved out of ONE allocation, weights looked up in the modules' own parameter dictionaries on every
//     call (so replaced or reloaded parameters are seen). A module tree that is not the plain one (a replaced
//     submodule, a hook on one that the Python block would call, a switch set on one) makes the function return None
//     and the Python block runs.
//
// What it is for: a block makes about 14 launches. Through ctypes, with the tensor views and checks in Python, each
// cost 20-35 us of host time, so every problem whose kernels take less than that (up to 512 x 512 pixels, a whole
// block in 250-500 us) ran at the host's pace.
#define PY_SSIZE_T_CLEAN
#include <Python.h>

#include <ATen/ATen.h>
#include <ATen/hip/EmptyTensor.h>
#include <c10/hip/HIPFunctions.h>
#include <c10/hip/HIPGraphsC10Utils.h>
#include <c10/hip/HIPStream.h>
#include <torch/csrc/autograd/python_variable.h>
#include <torch/csrc/jit/frontend/tracer.h>

#include <algorithm>
#include <cstring>
#include <map>
#include <optional>
#include <utility>
#include <vector>

#include "../../include/omni_dit.h"

namespace {

using at::Tensor;

// ---------------------------------------------------------------------------------------------- basics
const Tensor* tensor_of(PyObject* o) { return THPVariable_Check(o) ? &THPVariable_Unpack(o) : nullptr; }

// a tensor or None; false for anything else
bool optional_tensor(PyObject* o, const Tensor** out) {
  *out = nullptr;
  if (o == Py_None) return true;
  *out = tensor_of(o);
  return *out != nullptr;
}

int code_of(const Tensor& t) {
  switch (t.scalar_type()) {
    case at::kBFloat16: return ODIT_BF16;
    case at::kHalf: return ODIT_F16;
    case at::kFloat: return ODIT_F32;
    default: return -1;
  }
}

void* ptr(const Tensor* t) { return t ? t->data_ptr() : nullptr; }
bool aligned16(const void* p) { return (reinterpret_cast<uintptr_t>(p) & 15u) == 0; }

// the stream that work of this call goes to, and its device
struct Where {
  void* stream = nullptr;
  int device = -1;
  Where() {
    static const bool gpu = c10::hip::device_count() > 0;
    if (!gpu) return;  // holds nothing: every call takes the Python path, which refuses CPU tensors
    const auto s = c10::hip::getCurrentHIPStream();
    stream = s.stream();
    device = s.device_index();
  }
  bool holds(const Tensor& t) const { return t.is_cuda() && t.device().index() == device; }
  bool holds(const Tensor* t) const { return t == nullptr || holds(*t); }
};

PyObject* none() { Py_RETURN_NONE; }
PyObject* wrap(Tensor t) { return THPVariable_Wrap(std::move(t)); }
PyObject* wrap2(Tensor a, Tensor b) {
  PyObject* r = PyTuple_New(2);
  PyTuple_SET_ITEM(r, 0, wrap(std::move(a)));
  PyTuple_SET_ITEM(r, 1, wrap(std::move(b)));
  return r;
}

// C++ exceptions (allocation failures) become Python's
#define NATIVE_BEGIN try {
#define NATIVE_END                                        \
  }                                                       \
  catch (const c10::OutOfMemoryError& e) {                \
    PyErr_SetString(PyExc_RuntimeError, e.what_without_backtrace()); \
    return nullptr;                                       \
  }                                                       \
  catch (const std::exception& e) {                       \
    PyErr_SetString(PyExc_RuntimeError, e.what());        \
    return nullptr;                                       \
  }

// Other Python threads run while one of these exists. What allocates, ranks a library's kernels for a new problem or waits
// for room in a full queue (all of it inside the C calls and at::empty) happens under one; nothing under it may touch a
// Python object, and the tensors it works on are held by the caller's arguments or by BlockCall.
class Unlocked {
 public:
  Unlocked() : state_(PyEval_SaveThread()) {}
  ~Unlocked() { PyEval_RestoreThread(state_); }
  Unlocked(const Unlocked&) = delete;
  Unlocked& operator=(const Unlocked&) = delete;

 private:
  PyThreadState* state_;
};
template <typename F> auto unlocked(F f) {
  const Unlocked u;
  return f();
}
// (from the allocator, not through the dispatcher: 0.2 us of a layer's call of 5)
Tensor fresh(at::IntArrayRef sizes, const at::TensorOptions& opts) {
  return unlocked([&] { return Tensor(at::detail::empty_cuda(sizes, c10::typeMetaToScalarType(opts.dtype()), opts.device(), std::nullopt)); });
}

// ------------------------------------------------------------------------------------------- scratch
// Scratch belongs to kernels.py: one buffer per thread, device and stream. (Launches on one stream are ordered, so those of
// one thread can share it. Those of two threads may alternate, and some calls make several launches that hand results to
// each other in it.) What a thread was given is remembered here without a reference of its own and without the interpreter
// lock's help, as the memory is the thread's; kernels.py is asked when there is none, it is gone or too small, and in a
// graph capture, where kernels.py has to keep what the graph will use.
PyObject* g_linear_scratch_fn = nullptr;  // (device index, stream) -> tensor
PyObject* g_attn_scratch_fn = nullptr;    // (device index, stream, bytes) -> tensor

struct Scratch { void* p = nullptr; size_t bytes = 0; };
using ScratchRef = c10::weak_intrusive_ptr<c10::TensorImpl>;
using ScratchPool = std::map<std::pair<int, void*>, ScratchRef>;
constexpr size_t kScratchKept = 64;  // remembered (device, stream) pairs; past that all are forgotten

bool scratch_from(ScratchPool& pool, const Where& w, size_t bytes, Scratch* s, PyObject* (*ask)(const Where&, size_t)) {
  const auto it = pool.find({w.device, w.stream});
  const bool recording = c10::hip::currentStreamCaptureStatusMayInitCtx() != c10::hip::CaptureStatus::None;
  if (it != pool.end() && !recording) {
    if (const auto t = it->second.lock(); t.defined() && static_cast<size_t>(t->numel()) >= bytes) {
      s->p = t->mutable_data();
      s->bytes = static_cast<size_t>(t->numel());
      return true;
    }
  }
  PyObject* got = ask(w, bytes);
  if (got == nullptr) return false;
  const Tensor* t = tensor_of(got);
  if (t == nullptr) { Py_DECREF(got); PyErr_SetString(PyExc_TypeError, "scratch must be a tensor"); return false; }
  if (!recording) {
    if (pool.size() >= kScratchKept) pool.clear();
    pool.insert_or_assign({w.device, w.stream}, ScratchRef(t->getIntrusivePtr()));
  }
  s->p = t->data_ptr();
  s->bytes = static_cast<size_t>(t->numel());
  Py_DECREF(got);  // (kernels.py keeps it)
  return true;
}

bool linear_scratch(const Where& w, Scratch* s) {
  static thread_local ScratchPool pool;
  return scratch_from(pool, w, 1, s, [](const Where& w_, size_t) {
    return PyObject_CallFunction(g_linear_scratch_fn, "in", w_.device, reinterpret_cast<Py_ssize_t>(w_.stream));
  });
}
bool attn_scratch(const Where& w, size_t bytes, Scratch* s) {
  static thread_local ScratchPool pool;
  return scratch_from(pool, w, bytes, s, [](const Where& w_, size_t n) {
    return PyObject_CallFunction(g_attn_scratch_fn, "inn", w_.device, reinterpret_cast<Py_ssize_t>(w_.stream),
                                 static_cast<Py_ssize_t>(n));
  });
}

// ---------------------------------------------------------------------------------------- activations
template <int (*FN)(const void*, void*, int64_t, int, void*)>
PyObject* py_unary(PyObject*, PyObject* const* a, Py_ssize_t n) {  // (x, out or None)
  NATIVE_BEGIN
  const Tensor *x, *o;
  if (n != 2 || !(x = tensor_of(a[0])) || !optional_tensor(a[1], &o)) return none();
  const Where w;
  const int dt = code_of(*x);
  if (dt < 0 || !w.holds(x) || !w.holds(o) || !x->is_contiguous()) return none();
  if (o && (o->sizes() != x->sizes() || o->scalar_type() != x->scalar_type() || !o->is_contiguous())) return none();
  Tensor out = o ? *o : fresh(x->sizes(), x->options());
  if (unlocked([&] { return FN(x->data_ptr(), out.data_ptr(), x->numel(), dt, w.stream); }) != 0) return none();
  if (o) { Py_INCREF(a[1]); return a[1]; }
  return wrap(std::move(out));
  NATIVE_END
}

// ------------------------------------------------------------------------------------------------ adaLN
bool f32_row(const Tensor* t, int64_t C) {
  return t == nullptr || (t->scalar_type() == at::kFloat && t->dim() > 0 && t->numel() == C && t->size(-1) == C && t->stride(-1) == 1);
}

// (x, shift, scale, eps, index, ln_weight, ln_bias, shift_bias, scale_bias, ref_rounding, out)
PyObject* py_adaln(PyObject*, PyObject* const* a, Py_ssize_t n) {
  NATIVE_BEGIN
  const Tensor *x, *sh, *sc, *index, *lw, *lb, *sb, *cb, *o;
  if (n != 11 || !(x = tensor_of(a[0])) || !optional_tensor(a[1], &sh) || !optional_tensor(a[2], &sc) ||
      !optional_tensor(a[4], &index) || !optional_tensor(a[5], &lw) || !optional_tensor(a[6], &lb) ||
      !optional_tensor(a[7], &sb) || !optional_tensor(a[8], &cb) || !optional_tensor(a[10], &o))
    return none();
  const double eps = PyFloat_AsDouble(a[3]);
  if (eps == -1.0 && PyErr_Occurred()) return nullptr;
  const int rr = PyObject_IsTrue(a[9]);
  const Where w;
  const int dt = code_of(*x);
  if (dt < 0 || x->dim() != 3 || x->stride(2) != 1) return none();
  for (const Tensor* t : {x, sh, sc, index, lw, lb, sb, cb, o})
    if (!w.holds(t)) return none();
  const int64_t B = x->size(0), S = x->size(1), C = x->size(2);
  const int64_t need = index ? 2 * B : B;
  const Tensor* first = sh ? sh : sc;
  bool per_token = first && first->dim() == 3;
  if (per_token && index) return none();
  int mod_dt = dt;
  for (const Tensor* t : {sh, sc}) {
    if (!t) continue;
    if (per_token ? (t->dim() != 3 || t->size(0) != B || t->size(1) != S || t->size(2) != C)
                  : (t->dim() != 2 || t->size(1) != C || t->size(0) < need))
      return none();
    if (t->stride(-1) != 1) return none();
    mod_dt = code_of(*t);
  }
  if (sh && sc) {
    if (sh->scalar_type() != sc->scalar_type() || sh->stride(0) != sc->stride(0)) return none();
    if (per_token && sh->stride(1) != sc->stride(1)) return none();
  }
  int64_t ms = 0, mss = 0;
  if (first) {
    ms = first->size(0) > 1 ? first->stride(0) : 0;
    if (per_token) mss = S > 1 ? first->stride(1) : C;
    else if (first->size(0) == 1) ms = first->size(1);
  }
  if (index && (index->dim() != 2 || index->size(0) != B || index->size(1) != S || index->scalar_type() != at::kInt || !index->is_contiguous()))
    return none();
  if (!f32_row(lw, C) || !f32_row(lb, C) || !f32_row(sb, C) || !f32_row(cb, C)) return none();
  if (o && (o->sizes() != x->sizes() || o->scalar_type() != x->scalar_type() || o->stride(2) != 1)) return none();
  Tensor out = o ? *o : fresh({B, S, C}, x->options());
  const int64_t xs[2] = {x->stride(0), x->stride(1)}, os[2] = {out.stride(0), out.stride(1)};
  if (unlocked([&] { return odit_adaln_modulate(x->data_ptr(), out.data_ptr(), ptr(sh), ptr(sc), static_cast<const int32_t*>(ptr(index)),
                          static_cast<const float*>(ptr(lw)), static_cast<const float*>(ptr(lb)),
                          static_cast<const float*>(ptr(sb)), static_cast<const float*>(ptr(cb)), B, S, C, xs, os, ms, mss,
                          static_cast<float>(eps), mod_dt, dt, rr ? ODIT_FLAG_REF_ROUNDING : 0u, w.stream); }) != 0)
    return none();
  if (o) { Py_INCREF(a[10]); return a[10]; }
  return wrap(std::move(out));
  NATIVE_END
}

// AdaLayerNorm.forward_hip without index and affine: (x [B,S,C], mod_params [B,3C] = shift, scale, gate, eps, ref_rounding)
// -> (out, gate [B,1,C])
PyObject* adaln_layer(const Tensor* x, const Tensor* m, double eps, bool rr) {
  const Where w;
  const int dt = code_of(*x), mdt = code_of(*m);
  if (dt < 0 || mdt < 0 || x->dim() != 3 || x->stride(2) != 1 || !w.holds(x) || !w.holds(m) || m->dim() != 2 ||
      m->size(0) != x->size(0) || m->size(1) != 3 * x->size(2) || m->stride(1) != 1)
    return none();
  const int64_t B = x->size(0), S = x->size(1), C = x->size(2);
  Tensor out = fresh({B, S, C}, x->options());
  const int64_t xs[2] = {x->stride(0), x->stride(1)}, os[2] = {S * C, C};
  const char* mp = static_cast<const char*>(m->data_ptr());
  if (unlocked([&] { return odit_adaln_modulate(x->data_ptr(), out.data_ptr(), mp, mp + C * m->element_size(), nullptr, nullptr, nullptr, nullptr, nullptr,
                          B, S, C, xs, os, B > 1 ? m->stride(0) : 0, 0, static_cast<float>(eps), mdt, dt,
                          rr ? ODIT_FLAG_REF_ROUNDING : 0u, w.stream); }) != 0)
    return none();
  return wrap2(std::move(out), m->narrow(1, 2 * C, C).unsqueeze(1));
}
PyObject* py_adaln_layer(PyObject*, PyObject* const* a, Py_ssize_t n) {
  NATIVE_BEGIN
  const Tensor *x, *m;
  if (n != 4 || !(x = tensor_of(a[0])) || !(m = tensor_of(a[1]))) return none();
  const double eps = PyFloat_AsDouble(a[2]);
  const int rr = PyObject_IsTrue(a[3]);
  if (PyErr_Occurred()) return nullptr;
  return adaln_layer(x, m, eps, rr);
  NATIVE_END
}

// (x0, shift0, scale0, x1, shift1, scale1, eps, ref_rounding)
PyObject* py_adaln_pair(PyObject*, PyObject* const* a, Py_ssize_t n) {
  NATIVE_BEGIN
  if (n != 8) return none();
  const Tensor* t[6];
  const Where w;
  for (int i = 0; i < 6; ++i)
    if (!(t[i] = tensor_of(a[i])) || !w.holds(t[i])) return none();
  const double eps = PyFloat_AsDouble(a[6]);
  if (eps == -1.0 && PyErr_Occurred()) return nullptr;
  const int rr = PyObject_IsTrue(a[7]);
  const Tensor &x0 = *t[0], &x1 = *t[3];
  const int dt = code_of(x0), mdt = code_of(*t[1]);
  if (dt < 0 || mdt < 0 || x0.dim() != 3 || x1.dim() != 3 || x1.scalar_type() != x0.scalar_type()) return none();
  const int64_t B = x0.size(0), C = x0.size(2);
  if (x1.size(0) != B || x1.size(2) != C) return none();
  int64_t xs[4], os[4], ms[2];
  int S[2];
  const void *xp[2], *sp[2], *cp[2];
  for (int i = 0; i < 2; ++i) {
    const Tensor &x = *t[3 * i], &sh = *t[3 * i + 1], &sc = *t[3 * i + 2];
    if (x.stride(2) != 1 || sh.dim() != 2 || sc.dim() != 2 || sh.size(0) != B || sc.size(0) != B || sh.size(1) != C ||
        sc.size(1) != C || sh.stride(1) != 1 || sc.stride(1) != 1 || sh.stride(0) != sc.stride(0) ||
        code_of(sh) != mdt || code_of(sc) != mdt)
      return none();
    S[i] = static_cast<int>(x.size(1));
    xs[2 * i] = x.stride(0); xs[2 * i + 1] = x.stride(1);
    os[2 * i] = x.size(1) * C; os[2 * i + 1] = C;
    ms[i] = B > 1 ? sh.stride(0) : 0;
    xp[i] = x.data_ptr(); sp[i] = sh.data_ptr(); cp[i] = sc.data_ptr();
  }
  Tensor o0 = fresh({B, S[0], C}, x0.options()), o1 = fresh({B, S[1], C}, x0.options());
  void* op[2] = {o0.data_ptr(), o1.data_ptr()};
  if (unlocked([&] { return odit_adaln_modulate_pair(xp, op, sp, cp, B, S, C, xs, os, ms, static_cast<float>(eps), mdt, dt,
                               rr ? ODIT_FLAG_REF_ROUNDING : 0u, w.stream); }) != 0)
    return none();
  return wrap2(std::move(o0), std::move(o1));
  NATIVE_END
}

// ------------------------------------------------------------------------------------- QK norm + rotary
struct QkProblem {
  const Tensor *q, *k, *v, *wq, *wk, *cos, *sin;
  int64_t B, S, H, D;
  int rot, w_dtype;
};

// the checks of kernels._qk_problem
bool qk_problem(const Where& w, const Tensor* q, const Tensor* k, const Tensor* v, const Tensor* qo, const Tensor* ko,
                const Tensor* vo, const Tensor* wq, const Tensor* wk, const Tensor* cos, const Tensor* sin, int mode, QkProblem* p) {
  for (const Tensor* t : {q, k, v, qo, ko, vo, wq, wk, cos, sin})
    if (!w.holds(t)) return false;
  if (q->dim() != 4 || code_of(*q) < 0) return false;
  const int64_t B = q->size(0), S = q->size(1), H = q->size(2), D = q->size(3);
  for (const Tensor* t : {q, k, v}) {
    if (!t) continue;
    if (t->sizes() != q->sizes() || t->scalar_type() != q->scalar_type() || t->stride(3) != 1 || t->stride(2) != D ||
        t->stride(0) != q->stride(0) || t->stride(1) != q->stride(1))
      return false;
  }
  const int64_t St = qo->dim() == 4 ? qo->size(1) : -1;
  const Tensor* outs[3] = {qo, ko, vo};
  const Tensor* srcs[3] = {q, k, v};
  for (int i = 0; i < 3; ++i) {
    const Tensor* t = outs[i];
    if ((t == nullptr) != (srcs[i] == nullptr)) return false;
    if (!t) continue;
    if (t->dim() != 4 || t->size(0) != B || t->size(1) != St || t->size(2) != H || t->size(3) != D ||
        t->scalar_type() != q->scalar_type() || !t->is_contiguous())
      return false;
  }
  p->rot = 0;
  if (cos) {
    if (!sin || cos->dim() != 2 || cos->sizes() != sin->sizes() || cos->size(0) != S || cos->scalar_type() != at::kFloat ||
        sin->scalar_type() != at::kFloat || !cos->is_contiguous() || !sin->is_contiguous())
      return false;
    p->rot = static_cast<int>(2 * cos->size(1));
  } else if (sin) {
    return false;
  }
  p->w_dtype = code_of(*q);
  if (mode != ODIT_NORM_NONE) {
    const int64_t want = mode == ODIT_NORM_HEAD ? D : H * D;
    const Tensor* seen = nullptr;
    for (const Tensor* t : {wq, wk}) {
      if (!t) continue;
      if (t->numel() != want || !t->is_contiguous() || code_of(*t) < 0) return false;
      if (seen && seen->scalar_type() != t->scalar_type()) return false;
      seen = t;
    }
    if (seen) p->w_dtype = code_of(*seen);
  }
  p->q = q; p->k = k; p->v = v; p->wq = wq; p->wk = wk; p->cos = cos; p->sin = sin;
  p->B = B; p->S = S; p->H = H; p->D = D;
  return true;
}

// (q, k, v, q_out, k_out, v_out, wq, wk, cos, sin, eps, out_seq_offset, norm_mode, flags) -> True or None
PyObject* py_qknorm_rope(PyObject*, PyObject* const* a, Py_ssize_t n) {
  NATIVE_BEGIN
  if (n != 14) return none();
  const Tensor* t[10];
  for (int i = 0; i < 10; ++i)
    if (!optional_tensor(a[i], &t[i])) return none();
  if (!t[0] || !t[3]) return none();
  const double eps = PyFloat_AsDouble(a[10]);
  const long off = PyLong_AsLong(a[11]), mode = PyLong_AsLong(a[12]), flags = PyLong_AsLong(a[13]);
  if (PyErr_Occurred()) return nullptr;
  const Where w;
  QkProblem p;
  if (!qk_problem(w, t[0], t[1], t[2], t[3], t[4], t[5], t[6], t[7], t[8], t[9], mode, &p)) return none();
  const int64_t st[2] = {p.q->stride(0), p.q->stride(1)};
  if (unlocked([&] { return odit_qknorm_rope(ptr(p.q), ptr(p.k), ptr(p.v), t[3]->data_ptr(), ptr(t[4]), ptr(t[5]), ptr(p.wq), ptr(p.wk),
                       static_cast<const float*>(ptr(p.cos)), static_cast<const float*>(ptr(p.sin)), p.B, p.S, p.H, p.D, p.rot,
                       st, off, t[3]->size(1), static_cast<float>(eps), mode, p.w_dtype, code_of(*p.q), flags, w.stream); }) != 0)
    return none();
  Py_RETURN_TRUE;
  NATIVE_END
}

// (q0, k0, v0, wq0, wk0, cos0, sin0, off0,  q1, ..., off1,  q_out, k_out, v_out, eps, norm_mode, flags) -> True or None
PyObject* py_qknorm_rope_pair(PyObject*, PyObject* const* a, Py_ssize_t n) {
  NATIVE_BEGIN
  if (n != 22) return none();
  const Tensor *qo, *ko, *vo;
  if (!(qo = tensor_of(a[16])) || !optional_tensor(a[17], &ko) || !optional_tensor(a[18], &vo)) return none();
  const double eps = PyFloat_AsDouble(a[19]);
  const long mode = PyLong_AsLong(a[20]), flags = PyLong_AsLong(a[21]);
  if (PyErr_Occurred()) return nullptr;
  const Where w;
  QkProblem p[2];
  int off[2], S[2];
  const void *q[2], *k[2], *v[2], *wq[2], *wk[2];
  const float *cs[2], *sn[2];
  int64_t st[4];
  for (int i = 0; i < 2; ++i) {
    const Tensor* t[7];
    for (int j = 0; j < 7; ++j)
      if (!optional_tensor(a[8 * i + j], &t[j])) return none();
    if (!t[0]) return none();
    const long o = PyLong_AsLong(a[8 * i + 7]);
    if (PyErr_Occurred()) return nullptr;
    if (!qk_problem(w, t[0], t[1], t[2], qo, t[1] ? ko : nullptr, t[2] ? vo : nullptr, t[3], t[4], t[5], t[6], mode, &p[i])) return none();
    off[i] = static_cast<int>(o);
    S[i] = static_cast<int>(p[i].S);
    q[i] = ptr(t[0]); k[i] = ptr(t[1]); v[i] = ptr(t[2]); wq[i] = ptr(t[3]); wk[i] = ptr(t[4]);
    cs[i] = static_cast<const float*>(ptr(t[5])); sn[i] = static_cast<const float*>(ptr(t[6]));
    st[2 * i] = t[0]->stride(0); st[2 * i + 1] = t[0]->stride(1);
  }
  if (p[0].B != p[1].B || p[0].H != p[1].H || p[0].D != p[1].D || p[0].rot != p[1].rot || p[0].w_dtype != p[1].w_dtype ||
      p[0].q->scalar_type() != p[1].q->scalar_type() || (k[0] == nullptr) != (k[1] == nullptr) ||
      (v[0] == nullptr) != (v[1] == nullptr) || (cs[0] == nullptr) != (cs[1] == nullptr))
    return none();
  if (unlocked([&] { return odit_qknorm_rope_pair(q, k, v, qo->data_ptr(), k[0] ? ptr(ko) : nullptr, v[0] ? ptr(vo) : nullptr, wq, wk, cs, sn, p[0].B, S, p[0].H, p[0].D,
                            p[0].rot, st, off, qo->size(1), static_cast<float>(eps), mode, p[0].w_dtype,
                            code_of(*p[0].q), flags, w.stream); }) != 0)
    return none();
  Py_RETURN_TRUE;
  NATIVE_END
}

// ----------------------------------------------------------------------------------------------- layers
// RMSNorm.forward_hip: (x, weight, eps): every row of the last axis on its own
PyObject* rmsnorm(const Tensor* x, const Tensor* wt, double eps) {
  const int dt = code_of(*x);
  if (dt < 0 || x->dim() < 1 || !x->is_contiguous() || wt->scalar_type() != x->scalar_type() || !wt->is_contiguous()) return none();
  const Where w;
  if (!w.holds(x) || !w.holds(wt)) return none();
  const int64_t width = x->size(-1);
  if (wt->numel() != width || width == 0) return none();
  const int64_t rows = x->numel() / width;
  if (rows >= (1ll << 31)) return none();
  const int epv = dt == ODIT_F32 ? 4 : 8;
  const int64_t lanes = width / epv;
  int64_t hd = width;
  int mode = ODIT_NORM_HEAD;
  if (width % epv != 0 || lanes > 64 || (lanes & (lanes - 1)) != 0) {
    mode = ODIT_NORM_ROW;
    hd = 0;
    for (int64_t d : {128, 64, 32, 16, 8})
      if (width % d == 0) { hd = d; break; }
    if (hd == 0) return none();
  }
  Tensor out = fresh(x->sizes(), x->options());
  const int64_t st[2] = {rows * width, width};
  if (unlocked([&] { return odit_qknorm_rope(x->data_ptr(), nullptr, nullptr, out.data_ptr(), nullptr, nullptr, wt->data_ptr(), nullptr, nullptr,
                       nullptr, 1, static_cast<int>(rows), static_cast<int>(width / hd), static_cast<int>(hd), 0, st, 0,
                       static_cast<int>(rows), static_cast<float>(eps), mode, dt, dt, 0u, w.stream); }) != 0)
    return none();
  return wrap(std::move(out));
}
PyObject* py_rmsnorm(PyObject*, PyObject* const* a, Py_ssize_t n) {
  NATIVE_BEGIN
  const Tensor *x, *wt;
  if (n != 3 || !(x = tensor_of(a[0])) || !(wt = tensor_of(a[1]))) return none();
  const double eps = PyFloat_AsDouble(a[2]);
  if (PyErr_Occurred()) return nullptr;
  return rmsnorm(x, wt, eps);
  NATIVE_END
}

// RotaryEmbedding.forward_hip: (x [B,S,H,D], cos, sin float32 [S, rot/2], flags)
PyObject* rotary(const Tensor* x, const Tensor* cs, const Tensor* sn, unsigned flags) {
  // (what the layer's call and then its method ask for in vain is found out before anything is allocated)
  if (x->dim() != 4 || code_of(*x) < 0 || x->stride(3) != 1 || x->stride(2) != x->size(3) || cs->dim() != 2 || cs->scalar_type() != at::kFloat ||
      sn->scalar_type() != at::kFloat)
    return none();
  const Where w;
  if (!w.holds(x)) return none();
  Tensor out = fresh(x->sizes(), x->options());
  QkProblem p;
  if (!qk_problem(w, x, nullptr, nullptr, &out, nullptr, nullptr, nullptr, nullptr, cs, sn, ODIT_NORM_NONE, &p)) return none();
  const int64_t st[2] = {x->stride(0), x->stride(1)};
  if (unlocked([&] { return odit_qknorm_rope(x->data_ptr(), nullptr, nullptr, out.data_ptr(), nullptr, nullptr, nullptr, nullptr,
                       static_cast<const float*>(ptr(cs)), static_cast<const float*>(ptr(sn)), p.B, p.S, p.H, p.D, p.rot, st, 0,
                       p.S, 1e-6f, ODIT_NORM_NONE, code_of(*x), code_of(*x), flags, w.stream); }) != 0)
    return none();
  return wrap(std::move(out));
}
PyObject* py_rotary(PyObject*, PyObject* const* a, Py_ssize_t n) {
  NATIVE_BEGIN
  const Tensor *x, *cs, *sn;
  if (n != 4 || !(x = tensor_of(a[0])) || !(cs = tensor_of(a[1])) || !(sn = tensor_of(a[2]))) return none();
  const long flags = PyLong_AsLong(a[3]);
  if (PyErr_Occurred()) return nullptr;
  return rotary(x, cs, sn, static_cast<unsigned>(flags));
  NATIVE_END
}

// -------------------------------------------------------------------------------------------- attention
bool attn_operand(const Tensor& t) {
  return t.dim() == 4 && t.stride(3) == 1 && t.stride(0) % 8 == 0 && t.stride(1) % 8 == 0 && t.stride(2) % 8 == 0 && aligned16(t.data_ptr());
}

// (q, k, v, v_tail, scale, key_mask, return_lse, split (-1: none), use_workspace)
PyObject* py_attn(PyObject*, PyObject* const* a, Py_ssize_t n) {
  NATIVE_BEGIN
  const Tensor *q, *k, *v, *vt, *mask;
  if (n != 9 || !(q = tensor_of(a[0])) || !(k = tensor_of(a[1])) || !(v = tensor_of(a[2])) || !optional_tensor(a[3], &vt) ||
      !optional_tensor(a[5], &mask))
    return none();
  const double scale = PyFloat_AsDouble(a[4]);
  const int want_lse = PyObject_IsTrue(a[6]), use_ws = PyObject_IsTrue(a[8]);
  const long split = PyLong_AsLong(a[7]);
  if (PyErr_Occurred()) return nullptr;
  const Where w;
  for (const Tensor* t : {q, k, v, vt, mask})
    if (!w.holds(t)) return none();
  if (!attn_operand(*q) || !attn_operand(*k) || !attn_operand(*v) || (vt && !attn_operand(*vt))) return none();
  const int dt = code_of(*q);
  if ((dt != ODIT_BF16 && dt != ODIT_F16) || k->scalar_type() != q->scalar_type() || v->scalar_type() != q->scalar_type() ||
      (vt && vt->scalar_type() != q->scalar_type()))
    return none();
  const int64_t B = q->size(0), Sq = q->size(1), H = q->size(2), D = q->size(3), Sk = k->size(1), Hkv = k->size(2);
  if (k->size(0) != B || k->size(3) != D || v->size(0) != B || v->size(2) != Hkv || v->size(3) != D) return none();
  int k_split = 0;
  if (vt) {
    k_split = static_cast<int>(v->size(1));
    if (vt->size(0) != B || vt->size(2) != Hkv || vt->size(3) != D || v->size(1) + vt->size(1) != Sk || k_split % 64 != 0 ||
        k_split == 0 || vt->size(1) == 0 || v->stride(1) != vt->stride(1))
      return none();
  } else if (v->size(1) != Sk) {
    return none();
  }
  if (mask && (mask->dim() != 2 || mask->size(0) != B || mask->size(1) != Sk || !mask->is_contiguous() ||
               (mask->scalar_type() != at::kBool && mask->scalar_type() != at::kByte)))
    return none();
  if (split > Sq || B == 0 || Sq == 0 || Sk == 0) return none();
  Scratch ws;
  if (use_ws) {
    const size_t need = odit_attn_fwd_workspace_bytes(B, Sq, Sk, H, D);
    if (need > 0 && !attn_scratch(w, need, &ws)) return nullptr;
  }
  Tensor o = fresh({B, split < 0 ? Sq : split, H, D}, q->options()), ot, lse;
  if (split >= 0) ot = fresh({B, Sq - split, H, D}, q->options());
  if (want_lse) lse = fresh({B, H, Sq}, q->options().dtype(at::kFloat));
  void *head = o.data_ptr(), *tail = nullptr;
  int64_t n_head = split < 0 ? Sq : split;
  int cut = 0;
  if (split == 0) { head = ot.data_ptr(); n_head = Sq; }
  else if (split > 0 && split < Sq) { tail = ot.data_ptr(); cut = static_cast<int>(split); }
  const int64_t qs[3] = {q->stride(0), q->stride(1), q->stride(2)}, ks[3] = {k->stride(0), k->stride(1), k->stride(2)},
                vs[3] = {v->stride(0), v->stride(1), v->stride(2)}, os[3] = {n_head * H * D, H * D, D},
                ts[3] = {(Sq - cut) * H * D, H * D, D};
  int64_t vts[3] = {0, 0, 0};
  if (vt) { vts[0] = vt->stride(0); vts[1] = vt->stride(1); vts[2] = vt->stride(2); }
  if (unlocked([&] { return odit_attn_fwd_ex(ptr(q), ptr(k), ptr(v), ptr(vt), k_split, head, tail, cut, static_cast<const uint8_t*>(ptr(mask)),
                       want_lse ? lse.data_ptr<float>() : nullptr, B, Sq, Sk, H, Hkv, D, qs, ks, vs, vt ? vts : nullptr, os,
                       tail ? ts : nullptr, static_cast<float>(scale), dt, ws.p, ws.bytes, w.stream); }) != 0)
    return none();
  if (split < 0 && !want_lse) return wrap(std::move(o));
  if (split < 0) return wrap2(std::move(o), std::move(lse));
  if (!want_lse) return wrap2(std::move(o), std::move(ot));
  PyObject* r = PyTuple_New(3);
  PyTuple_SET_ITEM(r, 0, wrap(std::move(o)));
  PyTuple_SET_ITEM(r, 1, wrap(std::move(ot)));
  PyTuple_SET_ITEM(r, 2, wrap(std::move(lse)));
  return r;
  NATIVE_END
}

// ----------------------------------------------------------------------------------------------- linear
// rows of the last axis of t with one row stride (kernels._rows2d); false when they have none
bool rows_of(const Tensor& t, int64_t* rows, int64_t* ld) {
  const int64_t w = t.dim() > 0 ? t.size(-1) : 0;
  if (w == 0 || t.stride(-1) != 1) return false;
  *rows = t.numel() / w;
  if (t.is_contiguous()) { *ld = w; return true; }
  if (t.dim() != 2) return false;
  *ld = *rows > 1 ? t.stride(0) : w;
  return true;
}

// (t [n], dim, -log(max_period), scale, dtype code of the result, factor applied before in that type) -> [n, dim]
PyObject* py_time_sinusoid(PyObject*, PyObject* const* a, Py_ssize_t n) {
  NATIVE_BEGIN
  const Tensor* t;
  if (n != 6 || !(t = tensor_of(a[0]))) return none();
  const long dim = PyLong_AsLong(a[1]), code = PyLong_AsLong(a[4]);
  const double period = PyFloat_AsDouble(a[2]), scale = PyFloat_AsDouble(a[3]), pre = PyFloat_AsDouble(a[5]);
  if (PyErr_Occurred()) return nullptr;
  const Where w;
  const int dt = code_of(*t);
  if (dt < 0 || !w.holds(t) || t->dim() != 1 || !t->is_contiguous() || dim <= 0 || dim % 2 || code < 0 || code > 2) return none();
  Tensor out = fresh({t->size(0), dim}, t->options().dtype(code == ODIT_BF16 ? at::kBFloat16 : code == ODIT_F16 ? at::kHalf : at::kFloat));
  if (unlocked([&] { return odit_time_sinusoid(t->data_ptr(), out.data_ptr(), t->size(0), static_cast<int>(dim), static_cast<float>(period),
                         static_cast<float>(scale), static_cast<float>(pre), dt, static_cast<int>(code), w.stream); }) != 0)
    return none();
  return wrap(std::move(out));
  NATIVE_END
}

// Key masks and pairs of tensors stacked on the first axis, one launch. A list of (p, n): [B, S, ...] alike but for the second axis -> [2B, longer S,
// ...], rows past a shorter S zero; or (p, n, mask of p, mask of n): masks [B, S] or None (all true) -> [2B, longer S], false past the shorter. None
// where one is not taken.
PyObject* py_stack_pairs(PyObject*, PyObject* const* a, Py_ssize_t n) {
  NATIVE_BEGIN
  if (n != 1 || !PyList_Check(a[0]) || PyList_GET_SIZE(a[0]) < 1 || 2 * PyList_GET_SIZE(a[0]) > ODIT_PAD_PIECES) return none();
  const Where w;
  const Py_ssize_t count = PyList_GET_SIZE(a[0]);
  odit_pad_piece pieces[ODIT_PAD_PIECES];
  std::vector<Tensor> made;
  made.reserve(count);
  for (Py_ssize_t i = 0; i < count; ++i) {
    PyObject* item = PyList_GET_ITEM(a[0], i);
    if (!PyTuple_Check(item)) return none();
    const Py_ssize_t size = PyTuple_GET_SIZE(item);
    if (size != 2 && size != 4) return none();
    const Tensor* half[4] = {};
    for (Py_ssize_t j = 0; j < size; ++j) {
      PyObject* o = PyTuple_GET_ITEM(item, j);
      if (!optional_tensor(o, &half[j]) || (j < 2 && half[j] == nullptr)) return none();
      if (half[j] && (!THPVariable_CheckExact(o) || !w.holds(*half[j]) || !half[j]->is_contiguous() || half[j]->numel() == 0)) return none();
    }
    const Tensor &p = *half[0], &q = *half[1];
    if (code_of(p) < 0 || p.scalar_type() != q.scalar_type() || p.dim() != q.dim() || p.dim() < 1 || p.size(0) != q.size(0)) return none();
    const bool flat = p.dim() == 1;
    const int64_t B = flat ? 1 : p.size(0), S[2] = {flat ? p.size(0) : p.size(1), flat ? q.size(0) : q.size(1)}, longer = std::max(S[0], S[1]);
    int64_t inner = p.element_size();
    for (int64_t d = 2; d < p.dim(); ++d) {
      if (p.size(d) != q.size(d)) return none();
      inner *= p.size(d);
    }
    const Tensor* from[2] = {half[0], half[1]};
    if (size == 4) {
      if (flat) return none();
      inner = 1;
      for (int j = 0; j < 2; ++j) {
        from[j] = half[2 + j];
        if (from[j] && (from[j]->scalar_type() != at::kBool || from[j]->dim() != 2 || from[j]->size(0) != B || from[j]->size(1) != S[j])) return none();
      }
      made.push_back(fresh({2 * B, longer}, p.options().dtype(at::kBool)));
    } else {
      std::vector<int64_t> shape = p.sizes().vec();
      shape[0] *= 2;
      if (!flat) shape[1] = longer;
      made.push_back(fresh(shape, p.options()));
    }
    const int64_t pitch = longer * inner;
    for (int j = 0; j < 2; ++j)
      pieces[2 * i + j] = {ptr(from[j]), static_cast<char*>(made.back().data_ptr()) + j * B * pitch, B, S[j] * inner, S[j] * inner, pitch, 1, 0};
  }
  if (unlocked([&] { return odit_pad_rows(pieces, 2 * static_cast<int>(count), w.stream); }) != 0) return none();
  PyObject* r = PyTuple_New(count);
  if (r == nullptr) return nullptr;
  for (Py_ssize_t i = 0; i < count; ++i) PyTuple_SET_ITEM(r, i, wrap(std::move(made[i])));
  return r;
  NATIVE_END
}

// (x [1, S, C], shift and scale [n, C], index int32 [S], shift table, scale table float32 [C], eps): token s normed, with row index[s] of shift and scale
PyObject* py_adaln_rows(PyObject*, PyObject* const* a, Py_ssize_t n) {
  NATIVE_BEGIN
  const Tensor *x, *sh, *sc, *ix, *shb, *scb;
  if (n != 7 || !(x = tensor_of(a[0])) || !(sh = tensor_of(a[1])) || !(sc = tensor_of(a[2])) || !(ix = tensor_of(a[3])) || !(shb = tensor_of(a[4])) ||
      !(scb = tensor_of(a[5])))
    return none();
  const double eps = PyFloat_AsDouble(a[6]);
  if (PyErr_Occurred()) return nullptr;
  const Where w;
  const int dt = code_of(*x);
  for (const Tensor* t : {x, sh, sc, ix, shb, scb})
    if (!w.holds(t)) return none();
  if (dt < 0 || x->dim() != 3 || x->size(0) != 1 || !x->is_contiguous() || x->numel() == 0 || ix->scalar_type() != at::kInt || !ix->is_contiguous() ||
      ix->numel() != x->size(1) || x->size(1) >= (1ll << 31) || x->size(2) >= (1ll << 31))
    return none();
  const int64_t S = x->size(1), C = x->size(2);
  for (const Tensor* t : {sh, sc})
    if (t->scalar_type() != x->scalar_type() || t->dim() != 2 || t->size(1) != C || t->stride(1) != 1 || t->stride(0) != sh->stride(0) || t->stride(0) < C) return none();
  if (!f32_row(shb, C) || !f32_row(scb, C)) return none();
  Tensor out = fresh(x->sizes(), x->options());
  if (unlocked([&] { return odit_adaln_modulate_rows(x->data_ptr(), out.data_ptr(), sh->data_ptr(), sc->data_ptr(), ix->data_ptr<int32_t>(), shb->data_ptr<float>(),
                                                     scb->data_ptr<float>(), static_cast<int>(S), static_cast<int>(C), C, C, sh->stride(0), static_cast<float>(eps), dt,
                                                     dt, w.stream); }) != 0)
    return none();
  return wrap(std::move(out));
  NATIVE_END
}

// (bool mask [B, S], rows more) -> [B, S + more], true past S
PyObject* py_extend_mask(PyObject*, PyObject* const* a, Py_ssize_t n) {
  NATIVE_BEGIN
  const Tensor* m;
  if (n != 2 || !(m = tensor_of(a[0]))) return none();
  const int64_t more = PyLong_AsLong(a[1]);
  if (PyErr_Occurred()) return nullptr;
  const Where w;
  if (!w.holds(m) || m->scalar_type() != at::kBool || m->dim() != 2 || m->numel() == 0 || !m->is_contiguous() || more < 0) return none();
  const int64_t B = m->size(0), S = m->size(1);
  Tensor out = fresh({B, S + more}, m->options());
  const odit_pad_piece piece = {m->data_ptr(), out.data_ptr(), B, S, S, S + more, 1, 1};
  if (unlocked([&] { return odit_pad_rows(&piece, 1, w.stream); }) != 0) return none();
  return wrap(std::move(out));
  NATIVE_END
}

// (text ids [n, axes], image ids [m, axes], axis widths, theta) -> float32 (cos, sin), each [n + m, half]
PyObject* py_rope_tables(PyObject*, PyObject* const* a, Py_ssize_t n) {
  NATIVE_BEGIN
  const Tensor *t, *i;
  if (n != 4 || !(t = tensor_of(a[0])) || !(i = tensor_of(a[1])) || !PyTuple_Check(a[2])) return none();
  int axes[4], half = 0;
  const Py_ssize_t n_axes = PyTuple_GET_SIZE(a[2]);
  if (n_axes < 1 || n_axes > 4) return none();
  for (Py_ssize_t k = 0; k < n_axes; ++k) {
    axes[k] = static_cast<int>(PyLong_AsLong(PyTuple_GET_ITEM(a[2], k)));
    half += axes[k] / 2;
  }
  const double theta = PyFloat_AsDouble(a[3]);
  if (PyErr_Occurred()) return nullptr;
  const Where w;
  const int dt = code_of(*t);
  if (dt < 0 || !w.holds(t) || !w.holds(i) || t->scalar_type() != i->scalar_type() || t->dim() != 2 || i->dim() != 2 ||
      t->size(1) != n_axes || i->size(1) != n_axes || !t->is_contiguous() || !i->is_contiguous())
    return none();
  const int64_t rows = t->size(0) + i->size(0);
  Tensor c = fresh({rows, half}, t->options().dtype(at::kFloat)), s = fresh({rows, half}, t->options().dtype(at::kFloat));
  if (unlocked([&] { return odit_rope_tables(t->data_ptr(), t->size(0), i->data_ptr(), i->size(0), c.data_ptr<float>(), s.data_ptr<float>(), axes,
                       static_cast<int>(n_axes), theta, dt, w.stream); }) != 0)
    return none();
  return wrap2(std::move(c), std::move(s));
  NATIVE_END
}

// (positive, negative, scale, normalize)
PyObject* py_cfg_combine(PyObject*, PyObject* const* a, Py_ssize_t n) {
  NATIVE_BEGIN
  const Tensor *p, *q;
  if (n != 4 || !(p = tensor_of(a[0])) || !(q = tensor_of(a[1]))) return none();
  const double scale = PyFloat_AsDouble(a[2]);
  const int norm = PyObject_IsTrue(a[3]);
  if (PyErr_Occurred()) return nullptr;
  const Where w;
  const int dt = code_of(*p);
  if ((dt != ODIT_BF16 && dt != ODIT_F16) || !w.holds(p) || !w.holds(q) || p->dim() < 1 || p->numel() == 0 || p->sizes() != q->sizes() ||
      p->scalar_type() != q->scalar_type() || !p->is_contiguous() || !q->is_contiguous() || p->size(-1) >= (1ll << 31))
    return none();
  Tensor out = fresh(p->sizes(), p->options());
  if (unlocked([&] { return odit_cfg_combine(p->data_ptr(), q->data_ptr(), out.data_ptr(), p->numel() / p->size(-1), static_cast<int>(p->size(-1)),
                       static_cast<float>(scale), norm, dt, w.stream); }) != 0)
    return none();
  return wrap(std::move(out));
  NATIVE_END
}

// (x, v, dt)
PyObject* py_euler_step(PyObject*, PyObject* const* a, Py_ssize_t n) {
  NATIVE_BEGIN
  const Tensor *x, *v;
  if (n != 3 || !(x = tensor_of(a[0])) || !(v = tensor_of(a[1]))) return none();
  const double step = PyFloat_AsDouble(a[2]);
  if (PyErr_Occurred()) return nullptr;
  const Where w;
  const int dt = code_of(*x);
  if (dt < 0 || !w.holds(x) || !w.holds(v) || x->sizes() != v->sizes() || x->scalar_type() != v->scalar_type() ||
      !x->is_contiguous() || !v->is_contiguous())
    return none();
  Tensor out = fresh(x->sizes(), x->options());
  if (unlocked([&] { return odit_euler_step(x->data_ptr(), v->data_ptr(), out.data_ptr(), x->numel(), static_cast<float>(step), dt, w.stream); }) != 0) return none();
  return wrap(std::move(out));
  NATIVE_END
}

// (modulation parameters [B, ...] with 3 C per gated projection, list of the projections' biases [C]) -> float32 (gates, gates *
// biases), each [B, projections, C]
PyObject* py_gate_rows(PyObject*, PyObject* const* a, Py_ssize_t n) {
  NATIVE_BEGIN
  const Tensor *m, *first;
  if (n != 2 || !(m = tensor_of(a[0])) || !PyList_Check(a[1])) return none();
  const Py_ssize_t rows = PyList_GET_SIZE(a[1]);
  if (rows == 0 || rows > 65535 || !(first = tensor_of(PyList_GET_ITEM(a[1], 0)))) return none();
  const Where w;
  const int dt = code_of(*m);
  const int64_t C = first->numel(), B = m->dim() > 1 ? m->size(0) : 0;
  if ((dt != ODIT_BF16 && dt != ODIT_F16) || !w.holds(m) || B <= 0 || B >= 65536 || C <= 0 || C >= (1 << 30) || m->numel() != B * rows * 3 * C)
    return none();
  int64_t dense = 1;  // every batch row is dense
  for (int64_t d = m->dim() - 1; d > 0; --d) {
    if (m->size(d) != 1 && m->stride(d) != dense) return none();
    dense *= m->size(d);
  }
  std::vector<const void*> bias(static_cast<size_t>(rows));
  for (Py_ssize_t i = 0; i < rows; ++i) {
    const Tensor* t = tensor_of(PyList_GET_ITEM(a[1], i));
    if (!t || !w.holds(t) || t->dim() != 1 || t->size(0) != C || t->scalar_type() != m->scalar_type() || !t->is_contiguous()) return none();
    bias[static_cast<size_t>(i)] = t->data_ptr();
  }
  Tensor g = fresh({B, rows, C}, m->options().dtype(at::kFloat)), gb = fresh({B, rows, C}, m->options().dtype(at::kFloat));
  if (unlocked([&] { return odit_gate_rows(bias.data(), static_cast<int>(rows), m->data_ptr(), m->stride(0), static_cast<int>(B), static_cast<int>(C),
                       g.data_ptr<float>(), gb.data_ptr<float>(), dt, w.stream); }) != 0)
    return none();
  return wrap2(std::move(g), std::move(gb));
  NATIVE_END
}

// (rows, rows of the second problem, N, K): whether odit_linear_pair runs the kernel for small products
PyObject* py_pair_is_small(PyObject*, PyObject* const* a, Py_ssize_t n) {
  long v[4];
  if (n != 4) return none();
  for (int i = 0; i < 4; ++i) {
    v[i] = PyLong_AsLong(a[i]);
    if (PyErr_Occurred()) return nullptr;
    if (v[i] <= 0 || v[i] >= (1l << 31)) Py_RETURN_FALSE;
  }
  return PyBool_FromLong(odit_linear_pair_is_small(static_cast<int>(v[0]), static_cast<int>(v[1]), static_cast<int>(v[2]), static_cast<int>(v[3])));
}

// (x, weight, bias or None, silu of x first)
PyObject* py_linear_few(PyObject*, PyObject* const* a, Py_ssize_t n) {
  NATIVE_BEGIN
  const Tensor *x, *wt, *b;
  if (n != 4 || !(x = tensor_of(a[0])) || !(wt = tensor_of(a[1])) || !optional_tensor(a[2], &b)) return none();
  const Where w;
  if (!w.holds(x) || !w.holds(wt) || !w.holds(b)) return none();
  const int dt = code_of(*x);
  if (dt < 0 || x->dim() < 1 || wt->dim() != 2 || wt->stride(1) != 1 || wt->size(1) != x->size(-1) ||
      wt->scalar_type() != x->scalar_type())
    return none();
  const int64_t N = wt->size(0), K = wt->size(1);
  int64_t M, ldx;
  if (N == 0 || K == 0 || N >= (1ll << 31) || !rows_of(*x, &M, &ldx) || M == 0 || M > 16) return none();
  if (b && (b->numel() != N || !b->is_contiguous() || b->scalar_type() != x->scalar_type())) return none();
  std::vector<int64_t> shape(x->sizes().begin(), x->sizes().end());
  shape.back() = N;
  Tensor out = fresh(shape, x->options());
  if (unlocked([&] { return odit_linear_few(x->data_ptr(), wt->data_ptr(), ptr(b), out.data_ptr(), static_cast<int>(M), static_cast<int>(N),
                      static_cast<int>(K), ldx, N > 1 ? wt->stride(0) : K, N, dt, PyObject_IsTrue(a[3]), w.stream); }) != 0)
    return none();
  return wrap(std::move(out));
  NATIVE_END
}

// (x, weight, bias, gelu, residual, gate, gate_bias, prescaled, out, engine flags)
PyObject* py_linear(PyObject*, PyObject* const* a, Py_ssize_t n) {
  NATIVE_BEGIN
  const Tensor *x, *wt, *b, *r, *g, *gb, *o;
  if (n != 10 || !(x = tensor_of(a[0])) || !(wt = tensor_of(a[1])) || !optional_tensor(a[2], &b) || !optional_tensor(a[4], &r) ||
      !optional_tensor(a[5], &g) || !optional_tensor(a[6], &gb) || !optional_tensor(a[8], &o))
    return none();
  const int gelu = PyObject_IsTrue(a[3]), pre = PyObject_IsTrue(a[7]);
  const long flags = PyLong_AsLong(a[9]);
  if (PyErr_Occurred()) return nullptr;
  const Where w;
  for (const Tensor* t : {x, wt, b, r, g, gb, o})
    if (!w.holds(t)) return none();
  const int dt = code_of(*x);
  if (dt < 0 || x->dim() < 1 || wt->dim() != 2 || wt->stride(1) != 1 || wt->size(1) != x->size(-1) ||
      wt->scalar_type() != x->scalar_type())
    return none();
  const int64_t N = wt->size(0), K = wt->size(1);
  int64_t M, ldx, ldo, ldr = 0;
  if (N == 0 || K == 0 || !rows_of(*x, &M, &ldx) || M == 0 || M >= (1ll << 31)) return none();
  if (b && (b->numel() != N || !b->is_contiguous() || b->scalar_type() != x->scalar_type())) return none();
  auto same_rows = [&](const Tensor& t, int64_t* ld) {
    if (t.dim() != x->dim() || t.scalar_type() != x->scalar_type() || t.size(-1) != N) return false;
    for (int64_t d = 0; d + 1 < x->dim(); ++d)
      if (t.size(d) != x->size(d)) return false;
    int64_t rows;
    return rows_of(t, &rows, ld);
  };
  if ((o && !same_rows(*o, &ldo)) || (r && !same_rows(*r, &ldr))) return none();
  if (g && !r) return none();
  if (gelu && r) return none();
  int epi, gate_code = dt, rows_per_gate = 0;
  int64_t gstride = 0;
  const void* bias_ptr = ptr(b);
  if (!r) {
    epi = gelu ? (b ? ODIT_EPI_BIAS_GELU_TANH : ODIT_EPI_GELU_TANH) : (b ? ODIT_EPI_BIAS : ODIT_EPI_NONE);
  } else {
    epi = pre ? ODIT_EPI_GATED_RESIDUAL_PRE : ODIT_EPI_GATED_RESIDUAL;
    auto row_stride = [&](const Tensor& t, int64_t* st) {  // [N], or [B,N] / [B,1,N] with one row per batch row
      if (t.stride(-1) != 1 || t.size(-1) != N) return false;
      if (t.dim() == 1) { *st = -1; return true; }
      if (x->dim() < 2 || t.size(0) != x->size(0)) return false;
      if (t.dim() == 3 && t.size(1) != 1) return false;
      if (t.dim() > 3) return false;
      *st = t.size(0) > 1 ? t.stride(0) : -1;
      return true;
    };
    if (g) {
      if (!row_stride(*g, &gstride)) return none();
      if (g->scalar_type() != x->scalar_type() && g->scalar_type() != at::kFloat) return none();
      gate_code = code_of(*g);
      if (gstride >= 0) rows_per_gate = static_cast<int>(M / x->size(0)); else gstride = 0;
    }
    if (pre) {
      if (!g || gate_code != ODIT_F32) return none();
      bias_ptr = nullptr;
      if (gb) {
        int64_t bs;
        if (gb->dim() != g->dim() || gb->scalar_type() != at::kFloat || !row_stride(*gb, &bs)) return none();
        if (rows_per_gate > 0 && bs != gstride) return none();
        bias_ptr = gb->data_ptr();
      }
    } else if (gb) {
      return none();
    }
  }
  Scratch ws;
  if (!linear_scratch(w, &ws)) return nullptr;
  Tensor out;
  if (o) {
    out = *o;
  } else {
    auto sizes = x->sizes().vec();
    sizes.back() = N;
    out = fresh(sizes, x->options());
    ldo = N;
  }
  if (unlocked([&] { return odit_linear_rows(x->data_ptr(), wt->data_ptr(), bias_ptr, out.data_ptr(), ptr(r), ptr(g), M, N, K, ldx,
                       N > 1 ? wt->stride(0) : K, ldo, ldr, epi, gate_code, dt, rows_per_gate, gstride,
                       static_cast<unsigned>(flags), ws.p, ws.bytes, w.stream); }) != 0)
    return none();
  if (o) { Py_INCREF(a[8]); return a[8]; }
  return wrap(std::move(out));
  NATIVE_END
}

// ------------------------------------------------------------------------------------------------ blocks
// Reading a module tree. Everything below works on borrowed references.
struct Names {
  PyObject *modules, *parameters, *fwd_hooks, *pre_hooks, *forward, *weight, *bias, *eps, *elementwise_affine, *ref_rounding, *attention,
      *softmax_scale, *fused, *forward_hip, *kernel_takes_layer, *forward_method, *hidden_size, *variance_epsilon, *is_neox_style,
      *module, *bwd_hooks, *bwd_pre_hooks, *call, *call_impl, *wrapped_call_impl, *compiled_call_impl, *global_hooks[4];
};
Names g_name;
PyTypeObject *g_linear_type, *g_rmsnorm_type, *g_rownorm_type, *g_adaln_type, *g_attention_type, *g_attention_impl_type,
    *g_feed_forward_type, *g_gelu_type, *g_wan_ffn_type, *g_qwen_attention_type, *g_flux_attention_type, *g_flux_single_norm_type,
    *g_wan_self_type, *g_wan_cross_type, *g_time_embedding_type, *g_rotary_type, *g_text_projection_type;

PyObject* instance_dict(PyObject* m) {
  PyObject** d = m ? _PyObject_GetDictPtr(m) : nullptr;
  return d ? *d : nullptr;
}
PyObject* item(PyObject* dict, PyObject* name) { return dict && PyDict_Check(dict) ? PyDict_GetItem(dict, name) : nullptr; }

// the instance dict of a module without hooks or a replaced forward; `type`: its exact class (null: any)
PyObject* plain_module(PyObject* m, PyTypeObject* type) {
  if (m == nullptr || (type != nullptr && Py_TYPE(m) != type)) return nullptr;
  PyObject* d = instance_dict(m);
  if (d == nullptr) return nullptr;
  for (PyObject* h : {item(d, g_name.fwd_hooks), item(d, g_name.pre_hooks)})
    if (h == nullptr || !PyDict_Check(h) || PyDict_Size(h) != 0) return nullptr;
  if (item(d, g_name.forward) != nullptr) return nullptr;
  return d;
}
// child `name` of the module whose instance dict is `d`
PyObject* child(PyObject* d, const char* name) {
  PyObject* mods = item(d, g_name.modules);
  return mods && PyDict_Check(mods) ? PyDict_GetItemString(mods, name) : nullptr;
}
bool is_true(PyObject* d, PyObject* name) { return item(d, name) == Py_True; }
bool is_false(PyObject* d, PyObject* name) { return item(d, name) == Py_False; }
// the float attribute `name` of a module's instance dict
bool float_attr(PyObject* d, PyObject* name, double* v) {
  PyObject* o = item(d, name);
  if (!o || !PyFloat_Check(o)) return false;
  *v = PyFloat_AS_DOUBLE(o);
  return true;
}
const Tensor* parameter(PyObject* d, PyObject* name) {
  PyObject* p = item(item(d, g_name.parameters), name);
  return p && p != Py_None ? tensor_of(p) : nullptr;
}

// Whether a call of module `m` runs this package's code and torch's alone: no class of somebody else's in the tree, no hook, no forward and no layer's
// method put on a module.
bool own_tree(PyObject* m, const char* package, size_t length, int depth) {
  if (depth > 64) return false;  // (a module that holds itself)
  PyObject* d = plain_module(m, nullptr);
  PyObject* from = d ? item(Py_TYPE(m)->tp_dict, g_name.module) : nullptr;
  const char* name = from && PyUnicode_Check(from) ? PyUnicode_AsUTF8(from) : nullptr;
  if (name == nullptr) { PyErr_Clear(); return false; }
  if (strncmp(name, "torch.nn.modules.", 17) != 0 && (strncmp(name, package, length) != 0 || name[length] != '.')) return false;
  if (PyObject* f = item(d, g_name.forward_method))
    if (!PyMethod_Check(f) || PyMethod_GET_SELF(f) != m || PyMethod_GET_FUNCTION(f) != _PyType_Lookup(Py_TYPE(m), g_name.forward_hip)) return false;
  PyObject *children = item(d, g_name.modules), *child = nullptr;
  if (children == nullptr || !PyDict_Check(children)) return false;
  for (Py_ssize_t at = 0; PyDict_Next(children, &at, nullptr, &child);)
    if (child != Py_None && !own_tree(child, package, length, depth + 1)) return false;
  return true;
}
// (module, name of this package)
PyObject* py_own_tree(PyObject*, PyObject* const* a, Py_ssize_t n) {
  Py_ssize_t length = 0;
  const char* package = n == 2 && PyUnicode_Check(a[1]) ? PyUnicode_AsUTF8AndSize(a[1], &length) : nullptr;
  if (package == nullptr) { PyErr_Clear(); Py_RETURN_FALSE; }
  return PyBool_FromLong(own_tree(a[0], package, static_cast<size_t>(length), 0));
}

// ---- a layer's own call: what it holds is looked up here, where its class and the method that it was made with are this package's ----
PyObject *g_rmsnorm_hip, *g_adaln_hip, *g_rotary_hip;
// the instance dict of a layer of exactly `type` that calls `method`
PyObject* own_layer(PyObject* m, PyTypeObject* type, PyObject* method) {
  if (type == nullptr || Py_TYPE(m) != type) return nullptr;
  PyObject* d = instance_dict(m);
  PyObject* f = item(d, g_name.forward_method);
  return f && PyMethod_Check(f) && PyMethod_GET_FUNCTION(f) == method && PyMethod_GET_SELF(f) == m ? d : nullptr;
}
bool width_is(PyObject* d, int64_t n) {
  PyObject* o = item(d, g_name.hidden_size);
  return o && PyLong_CheckExact(o) && PyLong_AsLongLong(o) == n;
}
// (RMSNorm, x)
PyObject* py_rmsnorm_of(PyObject*, PyObject* const* a, Py_ssize_t n) {
  NATIVE_BEGIN
  const Tensor* x;
  PyObject* d = n == 2 ? own_layer(a[0], g_rmsnorm_type, g_rmsnorm_hip) : nullptr;
  const Tensor* w = d ? parameter(d, g_name.weight) : nullptr;
  double eps;
  if (!w || !(x = tensor_of(a[1])) || x->dim() < 1 || !width_is(d, x->size(-1)) || !float_attr(d, g_name.variance_epsilon, &eps)) return none();
  const Tensor held = *w;  // (another thread may replace the parameter meanwhile)
  return rmsnorm(x, &held, eps);
  NATIVE_END
}
// (AdaLayerNorm, x, modulation parameters)
PyObject* py_adaln_of(PyObject*, PyObject* const* a, Py_ssize_t n) {
  NATIVE_BEGIN
  const Tensor *x, *m;
  PyObject* d = n == 3 ? own_layer(a[0], g_adaln_type, g_adaln_hip) : nullptr;
  double eps;
  if (!d || !(x = tensor_of(a[1])) || !(m = tensor_of(a[2])) || x->dim() < 1 || !width_is(d, x->size(-1)) || !is_false(d, g_name.elementwise_affine) ||
      !float_attr(d, g_name.eps, &eps) || !(is_true(d, g_name.ref_rounding) || is_false(d, g_name.ref_rounding)))
    return none();
  return adaln_layer(x, m, eps, is_true(d, g_name.ref_rounding));
  NATIVE_END
}
// (RotaryEmbedding, x, cos, sin)
PyObject* py_rotary_of(PyObject*, PyObject* const* a, Py_ssize_t n) {
  NATIVE_BEGIN
  const Tensor *x, *cs, *sn;
  PyObject* d = n == 4 ? own_layer(a[0], g_rotary_type, g_rotary_hip) : nullptr;
  if (!d || !(x = tensor_of(a[1])) || !(cs = tensor_of(a[2])) || !(sn = tensor_of(a[3])) || cs->dim() == 3) return none();
  unsigned flags = 0;
  const std::pair<PyObject*, unsigned> of[2] = {{g_name.is_neox_style, ODIT_FLAG_NEOX}, {g_name.ref_rounding, ODIT_FLAG_REF_ROUNDING}};
  for (const auto& f : of) {
    if (is_true(d, f.first)) flags |= f.second;
    else if (!is_false(d, f.first)) return none();
  }
  return rotary(x, cs, sn, flags);
  NATIVE_END
}

// Whether a call of `m`, as torch makes it, would do nothing but call its class's own `forward`: no hook of any kind on it or on all modules, nothing compiled, no trace
// being taken, nobody following the thread's calls, and neither torch's way of calling modules (which torch.fx exchanges while it traces) nor the layer's forward replaced.
PyObject *g_module_type, *g_module_globals, *g_module_call[3], *g_rmsnorm_forward, *g_adaln_forward, *g_rotary_forward;
bool no_hooks(PyObject* dict, PyObject* name) {
  PyObject* h = item(dict, name);
  return h != nullptr && PyDict_Check(h) && PyDict_GET_SIZE(h) == 0;
}
bool calls_only(PyObject* m, PyObject* forward) {
  if (forward == nullptr || g_module_type == nullptr || g_module_globals == nullptr || item(Py_TYPE(m)->tp_dict, g_name.forward) != forward) return false;
  PyObject *d = instance_dict(m), *torch_way = reinterpret_cast<PyTypeObject*>(g_module_type)->tp_dict;
  for (PyObject* name : {g_name.fwd_hooks, g_name.pre_hooks, g_name.bwd_hooks, g_name.bwd_pre_hooks})
    if (!no_hooks(d, name)) return false;
  for (PyObject* name : g_name.global_hooks)
    if (!no_hooks(g_module_globals, name)) return false;
  // (torch finds these through the instance and all of its classes)
  if (item(torch_way, g_name.call) != g_module_call[0]) return false;
  PyObject* const ways[2] = {g_name.call_impl, g_name.wrapped_call_impl};
  for (int i = 0; i < 2; ++i)
    if (item(d, ways[i]) != nullptr || _PyType_Lookup(Py_TYPE(m), ways[i]) != g_module_call[i + 1]) return false;
  PyObject* compiled = item(d, g_name.compiled_call_impl);
  const PyThreadState* const thread = PyThreadState_Get();  // (a profiler or debugger that follows calls is shown torch's: torch.profiler's module events are those)
  return item(d, g_name.forward) == nullptr && (compiled == nullptr || compiled == Py_None) && _PyType_Lookup(Py_TYPE(m), g_name.compiled_call_impl) == Py_None &&
         thread->c_profilefunc == nullptr && thread->c_tracefunc == nullptr && !torch::jit::tracer::isTracing();
}
// (layer, its arguments): the whole call of an RMSNorm, an AdaLayerNorm or a RotaryEmbedding; None where torch has to make it
PyObject* py_layer_call(PyObject* self, PyObject* const* a, Py_ssize_t n) {
  if (n < 2) return none();
  PyTypeObject* const type = Py_TYPE(a[0]);
  if (type == g_rmsnorm_type) return calls_only(a[0], g_rmsnorm_forward) ? py_rmsnorm_of(self, a, n) : none();
  if (type == g_adaln_type) return calls_only(a[0], g_adaln_forward) ? py_adaln_of(self, a, n) : none();
  if (type == g_rotary_type) return calls_only(a[0], g_rotary_forward) ? py_rotary_of(self, a, n) : none();
  return none();
}

struct Lin {
  const void *w = nullptr, *b = nullptr;
  int64_t n = 0, k = 0, ldw = 0;
};

// The shared state of one block call: where it runs, its element type, and whether every operand so far was usable.
struct BlockCall {
  Where where;
  Scratch lin_ws;
  int dtype = -1;
  at::ScalarType st = at::kBFloat16;
  unsigned engine = 0;
  int rc = 0;  // first non-zero status of a C call
  mutable std::vector<Tensor> held;  // the parameters whose addresses were taken: another thread may replace them meanwhile

  BlockCall() { held.reserve(32); }

  bool operand(const Tensor& t) const { return where.holds(t) && t.scalar_type() == st; }

  bool linear(PyObject* m, Lin* out, bool need_bias = true) const {
    PyObject* d = plain_module(m, g_linear_type);
    const Tensor *w = d ? parameter(d, g_name.weight) : nullptr, *b = d ? parameter(d, g_name.bias) : nullptr;
    if (!w || !operand(*w) || w->dim() != 2 || w->stride(1) != 1 || (need_bias && !b)) return false;
    if (b && (!operand(*b) || !b->is_contiguous() || b->numel() != w->size(0))) return false;
    // (the library's kernels are chosen by sizes and strides and take the address for aligned; torch looks at it)
    if (!aligned16(w->data_ptr()) || (b && !aligned16(b->data_ptr()))) return false;
    held.push_back(*w);
    if (b) held.push_back(*b);
    *out = Lin{w->data_ptr(), ptr(b), w->size(0), w->size(1), w->size(0) > 1 ? w->stride(0) : w->size(1)};
    return true;
  }
  bool norm_weight(PyObject* m, PyTypeObject* type, int64_t n, const void** out, int* w_dtype) const {
    PyObject* d = plain_module(m, type);
    const Tensor* w = d ? parameter(d, g_name.weight) : nullptr;
    if (!w || !where.holds(*w) || !w->is_contiguous() || w->numel() != n) return false;
    const int c = code_of(*w);
    if (c != dtype && c != ODIT_F32) return false;
    if (*w_dtype >= 0 && *w_dtype != c) return false;
    *w_dtype = c;
    held.push_back(*w);
    *out = w->data_ptr();
    return true;
  }
  // projection with GELU(tanh) in its epilogue
  bool gelu_projection(PyObject* m, Lin* up) const {
    PyObject* d = plain_module(m, g_gelu_type);
    return d && is_true(d, g_name.fused) && linear(child(d, "proj"), up);
  }
  // gelu(tanh) projection and plain down-projection of a feed-forward
  bool feed_forward(PyObject* ff, Lin* up, Lin* down) const {
    PyObject* d = plain_module(ff, g_feed_forward_type);
    PyObject* net = d && is_true(d, g_name.fused) ? child(d, "net") : nullptr;
    PyObject* nd = net ? instance_dict(net) : nullptr;
    return nd && gelu_projection(child(nd, "0"), up) && linear(child(nd, "2"), down);
  }
  // an Attention layer whose backend object runs the kernel with its own scale
  bool attention(PyObject* m, double* scale) const {
    PyObject* d = plain_module(m, g_attention_type);
    PyObject* impl = d ? item(d, g_name.attention) : nullptr;
    if (!impl || Py_TYPE(impl) != g_attention_impl_type) return false;
    PyObject* id = instance_dict(impl);
    return id && item(id, g_name.forward) == nullptr && item(id, g_name.forward_hip) == nullptr && is_true(id, g_name.kernel_takes_layer) &&
           float_attr(id, g_name.softmax_scale, scale);
  }

  void check(int status) { if (rc == 0) rc = status; }

  // y[M,N] = x W^T + b with an optional GELU; rows dense
  void project(const void* x, const Lin& l, void* y, int64_t M, bool gelu) {
    if (rc != 0) return;
    const int epi = gelu ? (l.b ? ODIT_EPI_BIAS_GELU_TANH : ODIT_EPI_GELU_TANH) : (l.b ? ODIT_EPI_BIAS : ODIT_EPI_NONE);
    check(odit_linear_rows(x, l.w, l.b, y, nullptr, nullptr, M, l.n, l.k, l.k, l.ldw, l.n, 0, epi, dtype, dtype, 0, 0, engine,
                           lin_ws.p, lin_ws.bytes, where.stream));
  }
};

// (Linear module, x, silu of x first, engine flags): the module's projection of x with its own parameters as the module holds them now. None for a module that is not a plain torch Linear.
PyObject* py_project(PyObject*, PyObject* const* a, Py_ssize_t n) {
  NATIVE_BEGIN
  const Tensor* x;
  if (n != 4 || g_linear_type == nullptr || !(x = tensor_of(a[1]))) return none();
  const int silu = PyObject_IsTrue(a[2]);
  const long flags = PyLong_AsLong(a[3]);
  if (PyErr_Occurred()) return nullptr;
  BlockCall c;
  c.dtype = code_of(*x);
  c.st = x->scalar_type();
  Lin l;
  int64_t M, ldx;
  if ((c.dtype != ODIT_BF16 && c.dtype != ODIT_F16) || !c.operand(*x) || !aligned16(x->data_ptr()) || x->dim() < 1 || !c.linear(a[0], &l, false) ||
      x->size(-1) != l.k || l.n == 0 || l.k == 0 || l.n >= (1ll << 31) || !rows_of(*x, &M, &ldx) || M == 0 || M >= (1ll << 31))
    return none();
  auto sizes = x->sizes().vec();
  sizes.back() = l.n;
  Tensor out = fresh(sizes, x->options());
  const int few = unlocked([&] {
    return odit_linear_few(x->data_ptr(), l.w, l.b, out.data_ptr(), static_cast<int>(M), static_cast<int>(l.n), static_cast<int>(l.k), ldx,
                           l.ldw, l.n, c.dtype, silu, c.where.stream);
  });
  if (few == 0) return wrap(std::move(out));
  if (silu) return none();
  if (!linear_scratch(c.where, &c.lin_ws)) return nullptr;
  const int epi = l.b ? ODIT_EPI_BIAS : ODIT_EPI_NONE;
  const int rc = unlocked([&] {
    return odit_linear_rows(x->data_ptr(), l.w, l.b, out.data_ptr(), nullptr, nullptr, static_cast<int>(M), static_cast<int>(l.n),
                            static_cast<int>(l.k), ldx, l.ldw, l.n, 0, epi, c.dtype, c.dtype, 0, 0, static_cast<unsigned>(flags),
                            c.lin_ws.p, c.lin_ws.bytes, c.where.stream);
  });
  if (rc != 0) return none();
  return wrap(std::move(out));
  NATIVE_END
}

// (plain Linear, x [B, S, C], shift, scale [B, C] with rows equally far apart, eps, engine flags): the module's projection of the rows of x normed and
// modulated, in one launch; None where two are the way
PyObject* py_project_normed(PyObject*, PyObject* const* a, Py_ssize_t n) {
  NATIVE_BEGIN
  const Tensor *x, *sh, *sc;
  if (n != 6 || g_linear_type == nullptr || !(x = tensor_of(a[1])) || !(sh = tensor_of(a[2])) || !(sc = tensor_of(a[3]))) return none();
  const double eps = PyFloat_AsDouble(a[4]);
  const long flags = PyLong_AsLong(a[5]);
  if (PyErr_Occurred()) return nullptr;
  BlockCall c;
  c.dtype = code_of(*x);
  c.st = x->scalar_type();
  Lin l;
  if ((c.dtype != ODIT_BF16 && c.dtype != ODIT_F16) || !c.operand(*x) || x->dim() != 3 || !x->is_contiguous() || x->numel() == 0 || !aligned16(x->data_ptr()) ||
      !c.linear(a[0], &l, false) || x->size(2) != l.k || l.n == 0 || l.n >= (1ll << 31) || l.k >= (1ll << 31) || x->size(0) * x->size(1) >= (1ll << 31))
    return none();
  for (const Tensor* t : {sh, sc})
    if (!c.operand(*t) || t->dim() != 2 || t->size(0) != x->size(0) || t->size(1) != l.k || t->stride(1) != 1 || t->stride(0) != sh->stride(0)) return none();
  if (l.k > 256 && (l.n > 64 || l.k > 3072 || l.k % 1024 != 0)) return none();  // (widths that odit_linear_norm takes: nothing is allocated for others)
  Tensor out = fresh({x->size(0), x->size(1), l.n}, x->options());
  odit_linear_problem q = {x->data_ptr(), l.w, l.b, nullptr, nullptr, out.data_ptr(), static_cast<int>(x->size(0) * x->size(1)), 0, l.k, l.ldw, l.n, 0, 0};
  odit_row_norm r = {sh->data_ptr(), sc->data_ptr(), x->size(0) > 1 ? sh->stride(0) : 0, static_cast<int>(x->size(1)), static_cast<float>(eps)};
  if (unlocked([&] { return odit_linear_norm(&q, &r, static_cast<int>(l.n), static_cast<int>(l.k), l.b ? ODIT_EPI_BIAS : ODIT_EPI_NONE, c.dtype,
                                             static_cast<unsigned>(flags), c.where.stream); }) != 0)
    return none();
  return wrap(std::move(out));
  NATIVE_END
}

// (plain Linear, x, plain RMSNorm, its eps, plain Linear, y, engine flags): the first module's projection of x and the last one's of the normed y, in one
// launch; None where the kernel for small products is not the one
PyObject* py_project_stem(PyObject*, PyObject* const* a, Py_ssize_t n) {
  NATIVE_BEGIN
  const Tensor* x[2];
  if (n != 7 || g_linear_type == nullptr || g_rmsnorm_type == nullptr || !(x[0] = tensor_of(a[1])) || !(x[1] = tensor_of(a[5]))) return none();
  const double eps = PyFloat_AsDouble(a[3]);
  const long flags = PyLong_AsLong(a[6]);
  if (PyErr_Occurred()) return nullptr;
  BlockCall c;
  c.dtype = code_of(*x[0]);
  c.st = x[0]->scalar_type();
  Lin l[2];
  const void* weight = nullptr;
  int w_dtype = c.dtype;
  if ((c.dtype != ODIT_BF16 && c.dtype != ODIT_F16) || !c.linear(a[0], &l[0], false) || !c.linear(a[4], &l[1], false) || l[0].n != l[1].n || l[0].n == 0 ||
      l[0].n >= (1ll << 31) || !c.norm_weight(a[2], g_rmsnorm_type, l[1].k, &weight, &w_dtype))
    return none();
  odit_linear_problem q[2];
  Tensor out[2];
  for (int i = 0; i < 2; ++i) {
    if (!c.operand(*x[i]) || x[i]->dim() < 1 || !x[i]->is_contiguous() || x[i]->numel() == 0 || x[i]->size(-1) != l[i].k || l[i].k >= (1ll << 31) ||
        x[i]->numel() / l[i].k >= (1ll << 31) || !aligned16(x[i]->data_ptr()))
      return none();
    auto sizes = x[i]->sizes().vec();
    sizes.back() = l[i].n;
    out[i] = fresh(sizes, x[i]->options());
    q[i] = {x[i]->data_ptr(), l[i].w, l[i].b, nullptr, nullptr, out[i].data_ptr(), static_cast<int>(x[i]->numel() / l[i].k), 0, l[i].k, l[i].ldw, l[i].n, 0, 0};
  }
  const int K[2] = {static_cast<int>(l[0].k), static_cast<int>(l[1].k)};
  if (unlocked([&] { return odit_linear_stem(q, static_cast<int>(l[0].n), K, weight, static_cast<float>(eps), c.dtype, static_cast<unsigned>(flags),
                                             c.where.stream); }) != 0)
    return none();
  return wrap2(std::move(out[0]), std::move(out[1]));
  NATIVE_END
}

// (x, weight, bias or None, plain Linear): silu(x) W^T + bias of the weight and of the module's, each [rows of x, features], in one launch
PyObject* py_linear_few_pair(PyObject*, PyObject* const* a, Py_ssize_t n) {
  NATIVE_BEGIN
  const Tensor *x, *wt, *b;
  if (n != 4 || g_linear_type == nullptr || !(x = tensor_of(a[0])) || !(wt = tensor_of(a[1])) || !optional_tensor(a[2], &b)) return none();
  BlockCall c;
  c.dtype = code_of(*x);
  c.st = x->scalar_type();
  Lin l;
  int64_t M, ldx;
  if (c.dtype < 0 || !c.operand(*x) || !c.operand(*wt) || wt->dim() != 2 || wt->stride(1) != 1 || x->dim() != 2 || !c.linear(a[3], &l, false) ||
      x->size(1) != l.k || wt->size(1) != l.k || !rows_of(*x, &M, &ldx) || M < 1 || M > 16)
    return none();
  const int64_t N = wt->size(0), K = l.k;
  if (N < 1 || l.n < 1 || K < 1 || N >= (1ll << 30) || l.n >= (1ll << 30)) return none();
  if (b && (!c.operand(*b) || b->numel() != N || !b->is_contiguous())) return none();
  Tensor out = fresh({M, N}, x->options()), out2 = fresh({M, l.n}, x->options());
  const void *const w[2] = {wt->data_ptr(), l.w}, *const bias[2] = {ptr(b), l.b};
  void* const to[2] = {out.data_ptr(), out2.data_ptr()};
  const int features[2] = {static_cast<int>(N), static_cast<int>(l.n)};
  const int64_t ldw[2] = {N > 1 ? wt->stride(0) : K, l.ldw}, ldo[2] = {N, l.n};
  if (unlocked([&] { return odit_linear_few_pair(x->data_ptr(), w, bias, to, static_cast<int>(M), features, static_cast<int>(K), ldx, ldw, ldo, c.dtype, 1,
                                                 c.where.stream); }) != 0)
    return none();
  return Py_BuildValue("(NN)", wrap(std::move(out)), wrap(std::move(out2)));
  NATIVE_END
}

// (TimestepEmbedding, t [n], cosines and sines, - ln of the longest period, scale, type code of the rows, pre): linear_2(silu(linear_1(sinusoid of t))) in two launches
PyObject* py_time_embedding(PyObject*, PyObject* const* a, Py_ssize_t n) {
  NATIVE_BEGIN
  const Tensor* t;
  PyObject* const d = n == 7 && g_linear_type != nullptr && g_time_embedding_type != nullptr ? plain_module(a[0], g_time_embedding_type) : nullptr;
  if (d == nullptr || !(t = tensor_of(a[1]))) return none();
  const double period = PyFloat_AsDouble(a[3]), scale = PyFloat_AsDouble(a[4]), pre = PyFloat_AsDouble(a[6]);
  const long dim = PyLong_AsLong(a[2]), code = PyLong_AsLong(a[5]);
  if (PyErr_Occurred()) return nullptr;
  if (code != ODIT_BF16 && code != ODIT_F16) return none();
  BlockCall c;
  c.dtype = static_cast<int>(code);
  c.st = code == ODIT_BF16 ? at::kBFloat16 : at::kHalf;
  const int dt = code_of(*t);
  Lin l1, l2;
  if (dt < 0 || !c.where.holds(t) || t->dim() != 1 || !t->is_contiguous() || t->size(0) < 1 || t->size(0) > 16 ||
      !c.linear(child(d, "linear_1"), &l1, false) || !c.linear(child(d, "linear_2"), &l2, false) || l2.k != l1.n || l1.k != dim || dim < 2 || l1.n < 1 || l2.n < 1 ||
      l1.n >= (1ll << 30) || l2.n >= (1ll << 30))
    return none();
  const int M = static_cast<int>(t->size(0));
  const auto options = t->options().dtype(c.st);
  Tensor hidden = fresh({M, l1.n}, options), out = fresh({M, l2.n}, options);
  const int rc = unlocked([&] {
    const int first = odit_time_linear(t->data_ptr(), l1.w, l1.b, hidden.data_ptr(), M, static_cast<int>(l1.n), static_cast<int>(l1.k), l1.ldw, l1.n,
                                       static_cast<float>(period), static_cast<float>(scale), static_cast<float>(pre), dt, c.dtype, c.where.stream);
    return first != 0 ? first : odit_linear_few(hidden.data_ptr(), l2.w, l2.b, out.data_ptr(), M, static_cast<int>(l2.n), static_cast<int>(l2.k), l2.k, l2.ldw,
                                                l2.n, c.dtype, 1, c.where.stream);
  });
  if (rc != 0) return none();
  return wrap(std::move(out));
  NATIVE_END
}
// (timestep embedder, timesteps [M], guidance embedder or None, guidance [M] or None, text projection, pooled text [M, K], dim, neg_log_period, scale, pre): the
// sum of the embedders' results
PyObject* py_embed_sum(PyObject*, PyObject* const* a, Py_ssize_t n) {
  NATIVE_BEGIN
  const Tensor *t, *guidance, *pooled;
  if (n != 10 || g_linear_type == nullptr || g_time_embedding_type == nullptr || g_text_projection_type == nullptr || !(t = tensor_of(a[1])) ||
      !optional_tensor(a[3], &guidance) || (guidance == nullptr) != (a[2] == Py_None) || !(pooled = tensor_of(a[5])))
    return none();
  const long dim = PyLong_AsLong(a[6]);
  const double period = PyFloat_AsDouble(a[7]), scale = PyFloat_AsDouble(a[8]), pre = PyFloat_AsDouble(a[9]);
  if (PyErr_Occurred()) return nullptr;
  BlockCall c;
  c.dtype = code_of(*pooled);
  c.st = pooled->scalar_type();
  if ((c.dtype != ODIT_BF16 && c.dtype != ODIT_F16) || !c.where.holds(pooled) || pooled->dim() != 2 || pooled->stride(1) != 1 || pooled->size(0) < 1 ||
      pooled->size(0) > 4 || pooled->size(1) < 1 || pooled->size(1) >= (1 << 20))
    return none();
  const int M = static_cast<int>(pooled->size(0));
  const struct { PyObject* module; PyTypeObject* type; const Tensor* in; } of[3] = {
      {a[0], g_time_embedding_type, t}, {a[2], g_time_embedding_type, guidance}, {a[4], g_text_projection_type, pooled}};
  odit_embedder e[3];
  int count = 0;
  int64_t N = 0;
  for (const auto& m : of) {
    if (m.in == nullptr) continue;
    PyObject* const d = plain_module(m.module, m.type);
    const bool rows = m.in == pooled;
    Lin l1, l2;
    if (d == nullptr || !c.linear(child(d, "linear_1"), &l1, false) || !c.linear(child(d, "linear_2"), &l2, false) || l2.k != l1.n || l2.n != l1.n ||
        l1.k != (rows ? pooled->size(1) : dim) || l1.n < 1 || l1.n >= (1 << 20) || (count > 0 && l1.n != N))
      return none();
    if (!rows && (!c.where.holds(m.in) || code_of(*m.in) < 0 || m.in->dim() != 1 || m.in->size(0) != M || !m.in->is_contiguous())) return none();
    N = l1.n;
    e[count++] = odit_embedder{m.in->data_ptr(), rows ? (M > 1 ? pooled->stride(0) : l1.k) : 0, static_cast<int>(l1.k), rows ? -1 : code_of(*m.in),
                               static_cast<float>(period), static_cast<float>(scale), static_cast<float>(pre), l1.w, l1.b, l2.w, l2.b, l1.ldw, l2.ldw};
  }
  Tensor hidden = fresh({count, M, N}, pooled->options()), out = fresh({M, N}, pooled->options());
  if (unlocked([&] { return odit_embed_sum(e, count, M, static_cast<int>(N), hidden.data_ptr(), out.data_ptr(), c.dtype, c.where.stream); }) != 0) return none();
  return wrap(std::move(out));
  NATIVE_END
}

// (TimestepEmbedding, plain Linear time_proj, t [n], cosines and sines, - ln of the longest period, scale, type code of the rows) ->
// (linear_2(silu(linear_1(sinusoid of t))) [n, C], time_proj(silu of that) [n, P], the row int32 [n] of both that is a token's)
PyObject* py_time_tokens(PyObject*, PyObject* const* a, Py_ssize_t n) {
  NATIVE_BEGIN
  const Tensor* t;
  PyObject* const d = n == 7 && g_linear_type != nullptr && g_time_embedding_type != nullptr ? plain_module(a[0], g_time_embedding_type) : nullptr;
  if (d == nullptr || !(t = tensor_of(a[2]))) return none();
  const long dim = PyLong_AsLong(a[3]), code = PyLong_AsLong(a[6]);
  const double period = PyFloat_AsDouble(a[4]), scale = PyFloat_AsDouble(a[5]);
  if (PyErr_Occurred()) return nullptr;
  if (code != ODIT_BF16 && code != ODIT_F16) return none();
  BlockCall c;
  c.dtype = static_cast<int>(code);
  c.st = code == ODIT_BF16 ? at::kBFloat16 : at::kHalf;
  const int dt = code_of(*t);
  Lin l[3];
  if (dt < 0 || !c.where.holds(t) || t->dim() != 1 || !t->is_contiguous() || t->size(0) < 1 || t->size(0) >= (1 << 30) ||
      !c.linear(child(d, "linear_1"), &l[0], false) || !c.linear(child(d, "linear_2"), &l[1], false) || !c.linear(a[1], &l[2], false) || l[0].k != dim ||
      dim < 2 || l[1].k != l[0].n || l[1].n != l[0].n || l[2].k != l[1].n || l[0].n < 1 || l[2].n < 1 || l[0].n >= (1 << 30) || l[2].n >= (1 << 30))
    return none();
  if (!linear_scratch(c.where, &c.lin_ws)) return nullptr;
  const int N = static_cast<int>(t->size(0)), C = static_cast<int>(l[1].n), P = static_cast<int>(l[2].n);
  const auto options = t->options().dtype(c.st);
  const size_t bytes = odit_time_tokens_bytes(N, static_cast<int>(dim), C);
  Tensor temb = fresh({N, C}, options), proj = fresh({N, P}, options), index = fresh({N}, t->options().dtype(at::kInt)), scratch = fresh({static_cast<int64_t>(bytes)}, t->options().dtype(at::kByte));
  odit_time_tokens_args args = {};
  args.t = t->data_ptr();
  for (int i = 0; i < 3; ++i) { args.w[i] = l[i].w; args.bias[i] = l[i].b; args.ldw[i] = l[i].ldw; }
  args.temb = temb.data_ptr();
  args.proj = proj.data_ptr();
  args.index = index.data_ptr<int32_t>();
  args.n = N;
  args.K = static_cast<int>(dim);
  args.C = C;
  args.P = P;
  args.neg_log_period = static_cast<float>(period);
  args.scale = static_cast<float>(scale);
  if (unlocked([&] { return odit_time_tokens(&args, scratch.data_ptr(), bytes, dt, c.dtype, c.lin_ws.p, c.lin_ws.bytes, c.where.stream); }) != 0) return none();
  return Py_BuildValue("(NNN)", wrap(std::move(temb)), wrap(std::move(proj)), wrap(std::move(index)));
  NATIVE_END
}

// a gate row per batch entry (and, in the pre-scaled form, the gate times the projection's bias), or no gate at all
struct Gate {
  const void* gate = nullptr;   // element type `dtype`, or float32 when pre
  const void* gbias = nullptr;  // float32, pre only
  int64_t stride = 0;           // elements between batch entries
  bool pre = false;
  int code = 0;                 // element type of `gate` where not pre
};

// out = residual + gate * (x W^T + b), B batch entries of S rows. The hand-written GEMM takes one gate row per
// entry in one launch; for short entries the library's one launch per entry is slower than one launch over all rows
// followed by the gated-residual pass (`min_rows`), which needs the `tmp` rows. `clip` has the projection clip its rows of float16;
// true where it does.
bool project_gated(BlockCall& c, const void* x, const Lin& l, const void* residual, void* out, int64_t B, int64_t S, const Gate& g,
                   int64_t min_rows, void* tmp, const Gate& plain, bool clip = false) {
  if (c.rc != 0) return clip;
  const int M = static_cast<int>(B * S);
  const int epi = g.pre ? ODIT_EPI_GATED_RESIDUAL_PRE : ODIT_EPI_GATED_RESIDUAL;
  const int rows = g.gate && B > 1 ? static_cast<int>(S) : 0;
  const void* bias = g.pre ? g.gbias : l.b;
  const int gcode = g.pre ? ODIT_F32 : (g.gate ? g.code : c.dtype);
  if (rows > 0 && S < min_rows) {
    int own = 0, launches = 0;
    c.check(odit_linear_rows_plan(x, l.w, bias, out, residual, g.gate, M, l.n, l.k, l.k, l.ldw, l.n, l.n, epi, gcode, c.dtype, rows,
                                  g.stride, c.engine, c.lin_ws.p, c.lin_ws.bytes, &own, &launches));
    if (c.rc != 0) return clip;
    if (!own) {
      c.project(x, l, tmp, M, false);
      if (c.rc != 0) return clip;
      const int64_t st[2] = {S * l.n, l.n}, gs[2] = {plain.stride, 0};
      c.check(odit_gated_residual(residual, tmp, plain.gate, nullptr, out, B, S, l.n, st, st, st, gs, plain.code, c.dtype, 0u, c.where.stream));
      return false;
    }
  }
  c.check(odit_linear_rows(x, l.w, bias, out, residual, g.gate, M, l.n, l.k, l.k, l.ldw, l.n, l.n, epi, gcode, c.dtype, rows, g.stride,
                           c.engine | (clip ? ODIT_LINEAR_CLIP : 0u), c.lin_ws.p, c.lin_ws.bytes, c.where.stream));
  return clip;
}

// y[i] = x[i] W[i]^T + b[i] (GELU) for the two streams: one launch where that is the better way
void project_pair(BlockCall& c, const void* const x[2], const Lin l[2], void* const y[2], const int64_t M[2], bool gelu) {
  if (c.rc != 0) return;
  if (l[0].n == l[1].n && l[0].k == l[1].k && (l[0].b == nullptr) == (l[1].b == nullptr)) {
    odit_linear_problem q[2];
    for (int i = 0; i < 2; ++i)
      q[i] = {x[i], l[i].w, l[i].b, nullptr, nullptr, y[i], static_cast<int>(M[i]), 0, l[i].k, l[i].ldw, l[i].n, 0, 0};
    const int epi = gelu ? (l[0].b ? ODIT_EPI_BIAS_GELU_TANH : ODIT_EPI_GELU_TANH) : (l[0].b ? ODIT_EPI_BIAS : ODIT_EPI_NONE);
    const int rc = odit_linear_pair(q, l[0].n, l[0].k, epi, c.dtype, c.dtype, c.engine & ~static_cast<unsigned>(ODIT_LINEAR_HANDWRITTEN), c.lin_ws.p, c.lin_ws.bytes, c.where.stream);
    if (rc != ODIT_ENOTSUP) { c.check(rc); return; }
  }
  for (int i = 0; i < 2; ++i) c.project(x[i], l[i], y[i], M[i], gelu);
}

// out[i] = residual[i] + gate[i] * (x[i] W[i]^T + b[i]) for the two streams in one launch, clipped where `clip`; false when two calls are the better way
bool project_gated_pair(BlockCall& c, const void* const x[2], const Lin l[2], const void* const residual[2], void* const out[2], int64_t B,
                        const int64_t S[2], const Gate g[2], const bool clip[2]) {
  if (c.rc != 0) return true;
  if (l[0].n != l[1].n || l[0].k != l[1].k || g[0].pre != g[1].pre || g[0].code != g[1].code) return false;
  odit_linear_problem q[2];
  for (int i = 0; i < 2; ++i)
    q[i] = {x[i], l[i].w, g[i].pre ? g[i].gbias : l[i].b, residual[i], g[i].gate, out[i], static_cast<int>(B * S[i]), B > 1 ? static_cast<int>(S[i]) : 0,
            l[i].k, l[i].ldw, l[i].n, l[i].n, g[i].stride};
  const unsigned flags = (c.engine & ~static_cast<unsigned>(ODIT_LINEAR_HANDWRITTEN)) | (clip[0] ? ODIT_LINEAR_CLIP : 0u) | (clip[1] ? ODIT_LINEAR_CLIP2 : 0u);
  const int rc = odit_linear_pair(q, l[0].n, l[0].k, g[0].pre ? ODIT_EPI_GATED_RESIDUAL_PRE : ODIT_EPI_GATED_RESIDUAL, g[0].pre ? ODIT_F32 : g[0].code,
                                  c.dtype, flags, c.lin_ws.p, c.lin_ws.bytes, c.where.stream);
  if (rc == ODIT_ENOTSUP) return false;
  c.check(rc);
  return true;
}

// y[i] = x W[i]^T + b[i] for two projections of the same rows (GELU on the first where `gelu`): one launch where that is the better way
void project_fork(BlockCall& c, const void* x, const Lin l[2], void* const y[2], int64_t M, bool gelu) {
  if (c.rc != 0) return;
  if (l[0].k == l[1].k) {
    odit_linear_problem q[2];
    int n[2], epi[2];
    for (int i = 0; i < 2; ++i) {
      q[i] = {x, l[i].w, l[i].b, nullptr, nullptr, y[i], static_cast<int>(M), 0, l[i].k, l[i].ldw, l[i].n, 0, 0};
      n[i] = static_cast<int>(l[i].n);
      epi[i] = gelu && i == 0 ? (l[i].b ? ODIT_EPI_BIAS_GELU_TANH : ODIT_EPI_GELU_TANH) : (l[i].b ? ODIT_EPI_BIAS : ODIT_EPI_NONE);
    }
    const int rc = odit_linear_fork(q, n, static_cast<int>(l[0].k), epi, c.dtype, c.engine, c.lin_ws.p, c.lin_ws.bytes, c.where.stream);
    if (rc != ODIT_ENOTSUP) { c.check(rc); return; }
  }
  for (int i = 0; i < 2; ++i) c.project(x, l[i], y[i], M, gelu && i == 0);
}

// Three projections, of rows of their own, in one launch. launch false: whether that is expected to be the faster way (false: calls of
// their own are); true: what has been answered so, and is not asked again: the block's memory is laid out by the answer.
bool project_three(BlockCall& c, const void* const x[3], const Lin l[3], void* const y[3], const int64_t M[3], bool launch) {
  if (c.rc != 0) return true;
  if (l[0].k != l[1].k || l[0].k != l[2].k || (c.engine & ODIT_LINEAR_HANDWRITTEN)) return false;
  odit_linear_problem q[3];
  int n[3], epi[3];
  for (int i = 0; i < 3; ++i) {
    q[i] = {x[i], l[i].w, l[i].b, nullptr, nullptr, y[i], static_cast<int>(M[i]), 0, l[i].k, l[i].ldw, l[i].n, 0, 0};
    n[i] = static_cast<int>(l[i].n);
    epi[i] = l[i].b ? ODIT_EPI_BIAS : ODIT_EPI_NONE;
  }
  const int rc = odit_linear_three(q, n, static_cast<int>(l[0].k), epi, c.dtype, c.engine, launch ? ODIT_LAUNCH_ANSWERED : ODIT_LAUNCH_ASK, c.lin_ws.p, c.lin_ws.bytes, c.where.stream);
  if (rc == ODIT_ENOTSUP && !launch) return false;
  c.check(rc);
  return true;
}

// Two projections of which one or both go to query, key and value heads, in one launch: heads[i].q null is an ordinary output y[i]
// (GELU where `gelu`). launch as above; false: the projections and the pass behind them are the better way.
bool project_heads(BlockCall& c, const void* const x[2], const Lin l[2], void* const y[2], const int64_t M[2], const odit_head_output heads[2],
                   bool gelu, bool launch) {
  if (c.rc != 0) return true;
  if (l[0].k != l[1].k || (c.engine & ODIT_LINEAR_HANDWRITTEN)) return false;
  odit_linear_problem q[2];
  const odit_head_output* h[2];
  int n[2], epi[2];
  for (int i = 0; i < 2; ++i) {
    q[i] = {x[i], l[i].w, l[i].b, nullptr, nullptr, y[i], static_cast<int>(M[i]), 0, l[i].k, l[i].ldw, l[i].n, 0, 0};
    h[i] = heads[i].q ? &heads[i] : nullptr;
    n[i] = static_cast<int>(l[i].n);
    epi[i] = !h[i] && gelu ? (l[i].b ? ODIT_EPI_BIAS_GELU_TANH : ODIT_EPI_GELU_TANH) : (l[i].b ? ODIT_EPI_BIAS : ODIT_EPI_NONE);
  }
  const int rc = odit_linear_heads(q, n, static_cast<int>(l[0].k), epi, h, c.dtype, c.engine, launch ? ODIT_LAUNCH_ANSWERED : ODIT_LAUNCH_ASK, c.lin_ws.p, c.lin_ws.bytes, c.where.stream);
  if (rc == ODIT_ENOTSUP && !launch) return false;
  c.check(rc);
  return true;
}

// project_pair or, with heads, project_heads of two, of rows x[i] [B S[i], K] that are normed and modulated on the way: one launch in the place of
// two, or false. launch as above.
bool project_normed(BlockCall& c, const void* const x[2], const Lin l[2], void* const y[2], int64_t B, const int64_t S[2], const odit_row_norm norm[2],
                    const odit_head_output heads[2], bool gelu, bool launch) {
  if (c.rc != 0) return true;
  if (l[0].n != l[1].n || l[0].k != l[1].k || (l[0].b == nullptr) != (l[1].b == nullptr) || (c.engine & ODIT_LINEAR_HANDWRITTEN)) return false;
  odit_linear_problem q[2];
  const odit_head_output* h[2] = {heads, heads + 1};
  for (int i = 0; i < 2; ++i)
    q[i] = {x[i], l[i].w, l[i].b, nullptr, nullptr, y[i], static_cast<int>(B * S[i]), 0, l[i].k, l[i].ldw, l[i].n, 0, 0};
  const int epi = gelu ? (l[0].b ? ODIT_EPI_BIAS_GELU_TANH : ODIT_EPI_GELU_TANH) : (l[0].b ? ODIT_EPI_BIAS : ODIT_EPI_NONE);
  const int rc = odit_linear_pair_norm(q, norm, static_cast<int>(l[0].n), static_cast<int>(l[0].k), epi, heads ? h : nullptr, c.dtype, c.engine,
                                       launch ? ODIT_LAUNCH_ANSWERED : ODIT_LAUNCH_ASK, c.where.stream);
  if (rc == ODIT_ENOTSUP && !launch) return false;
  c.check(rc);
  return true;
}

// One allocation for a block's intermediate tensors. What is dead before another part begins shares its memory: after
// `mark`, every `rewind` starts laying out from there again, over what came since (all launches are on one stream). A Wan
// block of 2 x 32760 rows and width 5120 takes 4.7 GB this way; with every part apart it took 7.2.
struct Slab {
  Tensor t;
  size_t at = 0, marked = 0, size = 0;
  int esz;
  std::vector<std::pair<void**, size_t>> parts;
  explicit Slab(int esz_) : esz(esz_) {}
  void want(void** p, int64_t elements) {
    parts.emplace_back(p, at);
    at += (static_cast<size_t>(elements) * esz + 255) / 256 * 256;
    if (at > size) size = at;
  }
  void mark() { marked = at; }
  void rewind() { at = marked; }
  void allocate(const at::TensorOptions& opts) {
    t = at::empty({static_cast<int64_t>(size)}, opts.dtype(at::kByte));
    for (auto& p : parts) *p.first = static_cast<char*>(t.data_ptr()) + p.second;
  }
};

// ---- dual-stream block (Qwen-Image, Flux): stream 0 = image, 1 = text; joint rows are [text; image] -------------
struct DualBlock {
  Lin qkv[2], out[2], up[2], down[2];
  const void *nq[2], *nk[2];
  int w_dtype = -1;
  double scale = 0, eps_qk = 0, eps[2] = {0, 0};  // eps of the first and the second norm
  int64_t H = 0, D = 0;
};

struct ModRow {  // [B, 6C]: shift, scale, gate of the attention, then of the feed-forward
  const char* p;
  int64_t stride;
};

bool mod_row(const BlockCall& c, const Tensor* t, int64_t rows, int64_t C, ModRow* m) {
  if (!t || !c.operand(*t) || t->dim() != 2 || t->size(0) != rows || t->size(1) != 6 * C || t->stride(1) != 1) return false;
  m->p = static_cast<const char*>(t->data_ptr());
  m->stride = rows > 1 ? t->stride(0) : 0;
  return true;
}

bool f32_table(const BlockCall& c, const Tensor* t, int64_t rows, int64_t cols) {
  return t && c.where.holds(*t) && t->scalar_type() == at::kFloat && t->dim() == 2 && t->size(0) == rows && t->size(1) == cols && t->is_contiguous();
}

// gates / gate * bias rows: float32 [B, 2 (stream), 2 (attention, feed-forward), C]
bool gate_rows(const BlockCall& c, const Tensor* t, int64_t B, int64_t C) {
  return t && c.where.holds(*t) && t->scalar_type() == at::kFloat && t->dim() == 4 && t->size(0) == B && t->size(1) == 2 &&
         t->size(2) == 2 && t->size(3) == C && t->stride(3) == 1;
}

// x[2]: [B,S,C] dense; tables cos/sin per stream; key_mask [B, S_txt + S_img] or null; index: int32 [B, S_img] or null, the
// image stream's choice between modulation rows b and b + B. Returns false (nothing enqueued) when an operand is unusual;
// c.rc carries a C error.
bool run_dual(BlockCall& c, const DualBlock& k, const Tensor& img, const Tensor& txt, const ModRow mod[2], const Tensor* gates,
              const Tensor* gbias, const Tensor* const cos[2], const Tensor* const sin[2], const Tensor* mask, const Tensor* index,
              int64_t min_rows, bool clip[2], Tensor result[2]) {
  const Tensor* x[2] = {&img, &txt};
  const int64_t B = img.size(0), C = img.size(2), H = k.H, D = k.D, HD = H * D;
  const int64_t S[2] = {img.size(1), txt.size(1)}, Sj = S[0] + S[1];
  if (B * Sj >= (1ll << 31) || S[0] == 0 || S[1] == 0 || (D != 64 && D != 128)) return false;
  int64_t F[2];
  for (int i = 0; i < 2; ++i) {
    F[i] = k.up[i].n;
    if (k.qkv[i].k != C || k.qkv[i].n != 3 * HD || k.out[i].k != HD || k.out[i].n != C || k.up[i].k != C || k.down[i].k != F[i] ||
        k.down[i].n != C)
      return false;
    if (!f32_table(c, cos[i], S[i], cos[0]->size(1)) || !f32_table(c, sin[i], S[i], cos[0]->size(1))) return false;
  }
  if (mask && (!c.where.holds(*mask) || mask->dim() != 2 || mask->size(0) != B || mask->size(1) != Sj || !mask->is_contiguous() ||
               (mask->scalar_type() != at::kBool && mask->scalar_type() != at::kByte)))
    return false;
  if (index && (!c.where.holds(*index) || index->scalar_type() != at::kInt || index->dim() != 2 || index->size(0) != B || index->size(1) != S[0] ||
                !index->is_contiguous() || C % 8 != 0 || C > 8192))
    return false;
  const int32_t* idx = index ? index->data_ptr<int32_t>() : nullptr;
  const bool pre = gates != nullptr;
  if (pre && (!gate_rows(c, gates, B, C) || !gate_rows(c, gbias, B, C))) return false;
  for (int d = 0; pre && d < 3; ++d)
    if (gates->size(d) > 1 && gates->stride(d) != gbias->stride(d)) return false;
  const int esz = 2;
  const size_t attn_need = odit_attn_fwd_workspace_bytes(B, Sj, Sj, H, D);
  Scratch attn_ws;
  if (attn_need > 0 && !attn_scratch(c.where, attn_need, &attn_ws)) { c.rc = -100; return true; }
  const Unlocked others_run;  // to the end

  void *n[2], *qkv[2] = {nullptr, nullptr}, *jq, *jk, *jv = nullptr, *o[2], *u[2], *tmp;
  const int64_t M[2] = {B * S[0], B * S[1]};
  // the heads of both streams (image, text) as the projections may leave them: `at` is any aligned address while nothing is launched
  odit_head_output heads[2];
  auto heads_at = [&](void* q, void* kk, void* v) {
    for (int i = 0; i < 2; ++i)
      heads[i] = {q, kk, v, k.nq[i], k.nk[i], cos[i]->data_ptr<float>(), sin[i]->data_ptr<float>(), static_cast<int>(S[i]),
                  i == 0 ? static_cast<int>(S[1]) : 0, static_cast<int>(Sj), static_cast<int>(H), static_cast<int>(D), static_cast<float>(k.eps_qk)};
  };
  void* const at = img.data_ptr();
  heads_at(at, at, at);
  const void* const any[2] = {at, at};
  const bool fused = k.w_dtype == c.dtype && 2 * cos[0]->size(1) == D && project_heads(c, any, k.qkv, qkv, M, heads, false, false);
  if (c.rc != 0) return true;
  // the norms in the projections' launches (those of a small model)
  auto mod_at = [&](int stream, int col) { return mod[stream].p + col * C * esz; };
  auto row_norms = [&](int which, odit_row_norm r[2]) {
    for (int i = 0; i < 2; ++i)
      r[i] = {mod_at(i, 3 * which), mod_at(i, 3 * which + 1), mod[i].stride, static_cast<int>(S[i]), static_cast<float>(k.eps[which])};
  };
  odit_row_norm rn[2];
  void* const anywhere[2] = {at, at};
  row_norms(0, rn);
  const bool normed_qkv = !idx && project_normed(c, any, k.qkv, anywhere, B, S, rn, fused ? heads : nullptr, false, false);
  row_norms(1, rn);
  const bool normed_up = !idx && project_normed(c, any, k.up, anywhere, B, S, rn, nullptr, true, false);
  if (c.rc != 0) return true;
  // values are read where the projections left them when the text rows are whole key tiles and 32-bit offsets reach them
  const bool v_in_place = !fused && S[1] % 64 == 0 && (Sj + 64) * 3 * HD * esz < (1ll << 31);
  Slab slab(esz);
  for (int i = 0; i < 2; ++i) {
    slab.want(&n[i], B * S[i] * C);
    slab.want(&o[i], B * S[i] * HD);
  }
  slab.mark();  // up to the attention
  for (int i = 0; i < 2 && !fused; ++i) slab.want(&qkv[i], B * S[i] * 3 * HD);
  slab.want(&jq, B * Sj * HD);
  slab.want(&jk, B * Sj * HD);
  if (!v_in_place) slab.want(&jv, B * Sj * HD);
  slab.rewind();  // behind it
  for (int i = 0; i < 2; ++i) slab.want(&u[i], B * S[i] * F[i]);
  slab.want(&tmp, B * (S[0] > S[1] ? S[0] : S[1]) * C);
  slab.allocate(img.options());
  for (int i = 0; i < 2; ++i) result[i] = at::empty({B, S[i], C}, img.options());

  const int64_t rows[2][2] = {{S[0] * C, C}, {S[1] * C, C}};
  auto norm = [&](int stream, const void* src, int which) {
    if (c.rc != 0) return;
    c.check(odit_adaln_modulate(src, n[stream], mod_at(stream, 3 * which), mod_at(stream, 3 * which + 1), stream == 0 ? idx : nullptr, nullptr, nullptr,
                                nullptr, nullptr, B, S[stream], C, rows[stream], rows[stream], mod[stream].stride, 0,
                                static_cast<float>(k.eps[which]), c.dtype, c.dtype, 0u, c.where.stream));
  };
  auto norms = [&](const void* const src[2], int which) {
    const void *sh[2] = {mod_at(0, 3 * which), mod_at(1, 3 * which)}, *sc[2] = {mod_at(0, 3 * which + 1), mod_at(1, 3 * which + 1)};
    const int Si[2] = {static_cast<int>(S[0]), static_cast<int>(S[1])};
    const int64_t st[4] = {S[0] * C, C, S[1] * C, C}, ms[2] = {mod[0].stride, mod[1].stride};
    void* dst[2] = {n[0], n[1]};
    c.check(odit_adaln_modulate_pair(src, dst, sh, sc, B, Si, C, st, st, ms, static_cast<float>(k.eps[which]), c.dtype, c.dtype, 0u, c.where.stream));
  };
  // image rows with a gate per token: the projection, then residual + gate (and the second norm behind the first of them)
  auto indexed = [&](const void* a, const Lin& l, const void* residual, void* out, int which) {
    c.project(a, l, tmp, B * S[0], false);
    if (c.rc != 0) return;
    const int64_t st[2] = {mod[0].stride, 0};
    c.check(odit_gated_residual_adaln(residual, tmp, mod_at(0, 3 * which + 2), nullptr, out, which == 0 ? mod_at(0, 3) : nullptr,
                                      which == 0 ? mod_at(0, 4) : nullptr, nullptr, nullptr, nullptr, nullptr, which == 0 ? n[0] : nullptr, idx, B,
                                      S[0], C, st, st, static_cast<float>(k.eps[1]), c.dtype, c.dtype, c.where.stream));
  };
  auto gate_of = [&](int stream, int which, Gate* plain) {
    Gate g;
    g.gate = mod[stream].p + (which * 3 + 2) * C * esz;
    g.stride = mod[stream].stride;
    g.code = c.dtype;
    *plain = g;
    if (pre) {
      const int64_t off = stream * gates->stride(1) + which * gates->stride(2);
      g.gate = gates->data_ptr<float>() + off;
      g.gbias = gbias->data_ptr<float>() + off;
      g.stride = B > 1 ? gates->stride(0) : 0;
      g.pre = true;
    }
    return g;
  };

  const void* src[2] = {x[0]->data_ptr(), x[1]->data_ptr()};
  if (idx) {
    norm(0, src[0], 0);
    norm(1, src[1], 0);
  } else if (!normed_qkv) {
    norms(src, 0);
  }
  heads_at(jq, jk, jv);
  row_norms(0, rn);
  if (normed_qkv) {
    project_normed(c, src, k.qkv, qkv, B, S, rn, fused ? heads : nullptr, false, true);
  } else if (fused) {
    project_heads(c, n, k.qkv, qkv, M, heads, false, true);
  } else {
    project_pair(c, n, k.qkv, qkv, M, false);
  }
  if (c.rc == 0 && !fused) {  // problem 0 = text rows [0, S_txt), problem 1 = image rows
    auto part = [&](int stream, int which) { return static_cast<char*>(qkv[stream]) + which * HD * esz; };
    const void *qi[2] = {part(1, 0), part(0, 0)}, *ki[2] = {part(1, 1), part(0, 1)},
               *vi[2] = {v_in_place ? nullptr : part(1, 2), v_in_place ? nullptr : part(0, 2)}, *wq[2] = {k.nq[1], k.nq[0]},
               *wk[2] = {k.nk[1], k.nk[0]};
    const float *cs[2] = {cos[1]->data_ptr<float>(), cos[0]->data_ptr<float>()}, *sn[2] = {sin[1]->data_ptr<float>(), sin[0]->data_ptr<float>()};
    const int Si[2] = {static_cast<int>(S[1]), static_cast<int>(S[0])}, off[2] = {0, static_cast<int>(S[1])};
    const int64_t st[4] = {S[1] * 3 * HD, 3 * HD, S[0] * 3 * HD, 3 * HD};
    c.check(odit_qknorm_rope_pair(qi, ki, vi, jq, jk, v_in_place ? nullptr : jv, wq, wk, cs, sn, B, Si, H, D,
                                  static_cast<int>(2 * cos[0]->size(1)), st, off, Sj, static_cast<float>(k.eps_qk), ODIT_NORM_HEAD, k.w_dtype,
                                  c.dtype, 0u, c.where.stream));
  }
  if (c.rc == 0) {
    const int64_t js[3] = {Sj * HD, HD, D}, vt[3] = {S[1] * 3 * HD, 3 * HD, D}, vi[3] = {S[0] * 3 * HD, 3 * HD, D},
                  ot[3] = {S[1] * HD, HD, D}, oi[3] = {S[0] * HD, HD, D};
    const void* v0 = v_in_place ? static_cast<char*>(qkv[1]) + 2 * HD * esz : jv;
    const void* v1 = v_in_place ? static_cast<char*>(qkv[0]) + 2 * HD * esz : nullptr;
    c.check(odit_attn_fwd_ex(jq, jk, v0, v1, v_in_place ? static_cast<int>(S[1]) : 0, o[1], o[0], static_cast<int>(S[1]),
                             static_cast<const uint8_t*>(ptr(mask)), nullptr, B, Sj, Sj, H, H, D, js, js, v_in_place ? vt : js,
                             v_in_place ? vi : nullptr, ot, oi, static_cast<float>(k.scale), c.dtype, attn_ws.p, attn_ws.bytes,
                             c.where.stream));
  }
  void* res[2] = {result[0].data_ptr(), result[1].data_ptr()};
  Gate plain;
  // (`to`: the streams to clip in float16; false behind it for one that is left to the caller)
  auto gated = [&](const void* const a[2], const Lin l[2], const void* const residual[2], int which, bool to[2]) {
    const Gate g[2] = {gate_of(0, which, &plain), gate_of(1, which, &plain)};
    if (!idx && project_gated_pair(c, a, l, residual, res, B, S, g, to)) return;
    for (int i = 0; i < 2; ++i) {
      if (i == 0 && idx) { indexed(a[0], l[0], residual[0], res[0], which); to[0] = false; continue; }
      gate_of(i, which, &plain);
      to[i] = project_gated(c, a[i], l[i], residual[i], res[i], B, S[i], g[i], min_rows, tmp, plain, to[i]);
    }
  };
  bool unclipped[2] = {false, false};
  gated(o, k.out, src, 0, unclipped);
  const void* mid[2] = {res[0], res[1]};
  if (idx) norm(1, mid[1], 1);
  else if (c.rc == 0 && !normed_up) norms(mid, 1);
  row_norms(1, rn);
  if (normed_up) project_normed(c, mid, k.up, u, B, S, rn, nullptr, true, true);
  else project_pair(c, n, k.up, u, M, true);
  gated(u, k.down, mid, 1, clip);
  return true;
}

// an AdaLayerNorm without affine and reference rounding
bool plain_adaln(PyObject* m, double* eps) {
  PyObject* d = plain_module(m, g_adaln_type);
  return d && is_false(d, g_name.elementwise_affine) && is_false(d, g_name.ref_rounding) && float_attr(d, g_name.eps, eps);
}

// to_qkv, add_kv_proj, the four head norms, the attention layer
bool dual_attention(const BlockCall& c, PyObject* attn, PyTypeObject* type, DualBlock* k) {
  PyObject* d = plain_module(attn, type);
  if (!d || !is_false(d, g_name.ref_rounding) || (type == g_qwen_attention_type && !is_true(d, g_name.fused)) || !c.linear(child(d, "to_qkv"), &k->qkv[0]) || !c.linear(child(d, "add_kv_proj"), &k->qkv[1]) ||
      !c.linear(child(d, "to_add_out"), &k->out[1]) || !c.attention(child(d, "attn"), &k->scale) || !float_attr(d, g_name.eps, &k->eps_qk))
    return false;
  const char* names[4] = {"norm_q", "norm_added_q", "norm_k", "norm_added_k"};
  for (int i = 0; i < 4; ++i) {
    const void** out = i < 2 ? &k->nq[i] : &k->nk[i - 2];
    if (!c.norm_weight(child(d, names[i]), g_rmsnorm_type, k->D, out, &k->w_dtype)) return false;
  }
  return true;
}

bool block_input(BlockCall& c, const Tensor* x) {
  if (!x || x->dim() != 3 || !x->is_contiguous() || !c.where.holds(*x) || !aligned16(x->data_ptr())) return false;
  const int dt = code_of(*x);
  if (dt != ODIT_BF16 && dt != ODIT_F16) return false;
  c.dtype = dt;
  c.st = x->scalar_type();
  return linear_scratch(c.where, &c.lin_ws);
}

// The answer of a block function after a C call that did not succeed. A refusal (an operand, a workspace or a problem that a
// kernel does not take) leaves the block to Python, which has other ways for some of them and raises for the rest: what has
// been launched wrote this call's own tensors only. Anything else, and a refusal behind a write to the caller's tensor, raises.
PyObject* block_failed(int rc, bool caller_written = false) {
  if (PyErr_Occurred()) return nullptr;
  if (!caller_written && (rc == ODIT_EINVAL || rc == ODIT_ENOTSUP || rc == ODIT_EWORKSPACE)) return none();
  return PyErr_Format(PyExc_RuntimeError, "native block: a kernel call failed with status %d: %s", rc, odit_last_error());
}

// Arguments of the two dual-stream blocks: (block, heads, head_dim, hidden_states, encoder_hidden_states, img mods [B,6C], txt mods [B,6C],
// gates, gate * bias (float32 [B,2,2,C] or None), img cos, img sin, txt cos, txt sin, key mask or None, min rows, engine flags,
// modulation index int32 [B,S_img] or None (then the img mods are [2B,6C] and there are no gates)).
// -> (encoder_hidden_states, hidden_states) or None
PyObject* dual_block(PyObject* const* a, Py_ssize_t n, bool flux) {
  NATIVE_BEGIN
  if (n != 17) return none();
  BlockCall c;
  DualBlock k;
  const Tensor *img = tensor_of(a[3]), *txt = tensor_of(a[4]), *m0 = tensor_of(a[5]), *m1 = tensor_of(a[6]), *gates, *gbias, *mask, *index;
  k.H = PyLong_AsLong(a[1]);
  k.D = PyLong_AsLong(a[2]);
  const int64_t min_rows = PyLong_AsLong(a[14]);
  c.engine = static_cast<unsigned>(PyLong_AsLong(a[15]));
  if (PyErr_Occurred()) return nullptr;
  if (!optional_tensor(a[7], &gates) || !optional_tensor(a[8], &gbias) || !optional_tensor(a[13], &mask) || !optional_tensor(a[16], &index) ||
      (index && gates))
    return none();
  const Tensor *cos[2] = {tensor_of(a[9]), tensor_of(a[11])}, *sin[2] = {tensor_of(a[10]), tensor_of(a[12])};
  if (!cos[0] || !cos[1] || !sin[0] || !sin[1] || cos[0]->dim() != 2) return none();
  if (!block_input(c, img)) return PyErr_Occurred() ? nullptr : none();
  if (!txt || txt->dim() != 3 || !txt->is_contiguous() || !c.operand(*txt) || txt->size(0) != img->size(0) || txt->size(2) != img->size(2)) return none();
  const int64_t B = img->size(0), C = img->size(2);
  ModRow mod[2];
  if (!mod_row(c, m0, index ? 2 * B : B, C, &mod[0]) || !mod_row(c, m1, B, C, &mod[1])) return none();
  PyObject* d = instance_dict(a[0]);
  PyObject* attn = d ? child(d, "attn") : nullptr;
  if (!attn || !dual_attention(c, attn, flux ? g_flux_attention_type : g_qwen_attention_type, &k)) return none();
  PyObject* attn_d = instance_dict(attn);
  if (!flux) {
    double e[4];
    if (!plain_adaln(child(d, "img_norm1"), &e[0]) || !plain_adaln(child(d, "txt_norm1"), &e[1]) ||
        !plain_adaln(child(d, "img_norm2"), &e[2]) || !plain_adaln(child(d, "txt_norm2"), &e[3]) || e[0] != e[1] || e[2] != e[3])
      return none();
    k.eps[0] = e[0];
    k.eps[1] = e[2];
    if (!c.linear(child(attn_d, "to_out"), &k.out[0]) || !c.feed_forward(child(d, "img_mlp"), &k.up[0], &k.down[0]) ||
        !c.feed_forward(child(d, "txt_mlp"), &k.up[1], &k.down[1]))
      return none();
  } else {
    PyObject *n1 = instance_dict(child(d, "norm1")), *n2 = instance_dict(child(d, "norm2")), *outs = instance_dict(child(attn_d, "to_out"));
    if (!n1 || !n2 || !outs || !float_attr(n1, g_name.eps, &k.eps[0]) || !float_attr(n2, g_name.eps, &k.eps[1])) return none();
    if (!c.linear(child(outs, "0"), &k.out[0]) || !c.feed_forward(child(d, "ff"), &k.up[0], &k.down[0]) ||
        !c.feed_forward(child(d, "ff_context"), &k.up[1], &k.down[1]))
      return none();
  }
  Tensor out[2];
  // the reference clips both streams after every Qwen block, the text's after every Flux block; the last projections do it on the way
  const bool wanted[2] = {c.dtype == ODIT_F16 && !flux, c.dtype == ODIT_F16};
  bool clipped[2] = {wanted[0], wanted[1]};
  if (!run_dual(c, k, *img, *txt, mod, gates, gbias, cos, sin, mask, index, min_rows, clipped, out)) return none();
  if (c.rc != 0) return block_failed(c.rc);
  for (int i = 0; i < 2; ++i) {
    if (!wanted[i] || clipped[i]) continue;
    const Unlocked others_run;
    out[i].clamp_(-65504, 65504);
  }
  return wrap2(std::move(out[1]), std::move(out[0]));
  NATIVE_END
}
PyObject* py_qwen_block(PyObject*, PyObject* const* a, Py_ssize_t n) { return dual_block(a, n, false); }
PyObject* py_flux_block(PyObject*, PyObject* const* a, Py_ssize_t n) { return dual_block(a, n, true); }

// ---- Flux single-stream block on a joint sequence ------------------------------------------------------------
// (block, heads, head_dim, x [B,S,C], mods [B,3C], gate, gate * bias (float32 [B,C]), cos, sin, in_place, engine flags) -> x or None
PyObject* py_flux_single_block(PyObject*, PyObject* const* a, Py_ssize_t n) {
  NATIVE_BEGIN
  if (n != 11) return none();
  BlockCall c;
  const Tensor *x = tensor_of(a[3]), *mod = tensor_of(a[4]), *gate = tensor_of(a[5]), *gbias = tensor_of(a[6]), *cos = tensor_of(a[7]), *sin = tensor_of(a[8]);
  const int64_t H = PyLong_AsLong(a[1]), D = PyLong_AsLong(a[2]);
  const int in_place = PyObject_IsTrue(a[9]);
  c.engine = static_cast<unsigned>(PyLong_AsLong(a[10]));
  if (PyErr_Occurred()) return nullptr;
  if (!x || !mod || !gate || !gbias || !cos || !sin || cos->dim() != 2) return none();
  if (!block_input(c, x)) return PyErr_Occurred() ? nullptr : none();
  const int64_t B = x->size(0), S = x->size(1), C = x->size(2), HD = H * D;
  if (B * S >= (1ll << 31) || S == 0 || (D != 64 && D != 128) || !c.operand(*mod) || mod->dim() != 2 || mod->size(0) != B || mod->size(1) != 3 * C || mod->stride(1) != 1) return none();
  for (const Tensor* t : {gate, gbias})
    if (!c.where.holds(*t) || t->scalar_type() != at::kFloat || t->dim() != 2 || t->size(0) != B || t->size(1) != C || t->stride(1) != 1) return none();
  if (B > 1 && gate->stride(0) != gbias->stride(0)) return none();
  if (!f32_table(c, cos, S, cos->size(1)) || !f32_table(c, sin, S, cos->size(1))) return none();
  PyObject* d = instance_dict(a[0]);
  PyObject *norm = d ? plain_module(child(d, "norm"), g_flux_single_norm_type) : nullptr, *attn = d ? plain_module(child(d, "attn"), g_flux_attention_type) : nullptr;
  Lin qkv, up, down;
  double eps, eps_qk, scale;
  const void *wq, *wk;
  int w_dtype = -1;
  if (!norm || !is_false(norm, g_name.ref_rounding) || !attn || !is_false(attn, g_name.ref_rounding) || !float_attr(norm, g_name.eps, &eps) || !float_attr(attn, g_name.eps, &eps_qk) || !c.linear(child(attn, "to_qkv"), &qkv) ||
      !c.attention(child(attn, "attn"), &scale) || !c.norm_weight(child(attn, "norm_q"), g_rmsnorm_type, D, &wq, &w_dtype) ||
      !c.norm_weight(child(attn, "norm_k"), g_rmsnorm_type, D, &wk, &w_dtype) || !c.linear(child(d, "proj_mlp"), &up) ||
      !c.linear(child(d, "proj_out"), &down))
    return none();
  const int64_t F = up.n;
  if (HD != C || qkv.k != C || qkv.n != 3 * HD || up.k != C || down.k != C + F || down.n != C) return none();
  const size_t attn_need = odit_attn_fwd_workspace_bytes(B, S, S, H, D);
  Scratch attn_ws;
  if (attn_need > 0 && !attn_scratch(c.where, attn_need, &attn_ws)) return nullptr;
  std::optional<Unlocked> others_run(std::in_place);
  const int esz = 2;
  void *nx, *q3 = nullptr, *q, *k, *v = nullptr, *o, *u;
  Slab slab(esz);
  const Lin both[2] = {up, qkv};
  const int64_t M[2] = {B * S, B * S};
  odit_head_output heads[2] = {};
  auto heads_at = [&](void* q_, void* k_, void* v_) {
    heads[1] = {q_, k_, v_, wq, wk, cos->data_ptr<float>(), sin->data_ptr<float>(), static_cast<int>(S), 0, static_cast<int>(S), static_cast<int>(H),
                static_cast<int>(D), static_cast<float>(eps_qk)};
  };
  void* const at = x->data_ptr();
  heads_at(at, at, at);
  const void* const any[2] = {at, at};
  void* const any_out[2] = {at, at};
  const bool fused = w_dtype == c.dtype && 2 * cos->size(1) == D && project_heads(c, any, both, any_out, M, heads, true, false);
  slab.want(&nx, B * S * C);
  if (fused) slab.want(&v, B * S * HD);
  else slab.want(&q3, B * S * 3 * HD);
  slab.want(&q, B * S * HD);
  slab.want(&k, B * S * HD);
  slab.want(&o, B * S * HD);
  slab.want(&u, B * S * F);
  slab.allocate(x->options());
  Tensor out = in_place ? *x : at::empty({B, S, C}, x->options());
  const int64_t ms = B > 1 ? mod->stride(0) : 0, rs[2] = {S * C, C};
  const char* mp = static_cast<const char*>(mod->data_ptr());
  c.check(odit_adaln_modulate(x->data_ptr(), nx, mp, mp + C * esz, nullptr, nullptr, nullptr, nullptr, nullptr, B, S, C, rs, rs, ms, 0,
                              static_cast<float>(eps), c.dtype, c.dtype, 0u, c.where.stream));
  void* const into[2] = {u, q3};
  if (fused) {
    heads_at(q, k, v);
    const void* const rows[2] = {nx, nx};
    project_heads(c, rows, both, into, M, heads, true, true);
  } else {
    project_fork(c, nx, both, into, B * S, true);
  }
  const int64_t st[2] = {S * 3 * HD, 3 * HD};
  char* qp = static_cast<char*>(q3);
  if (c.rc == 0 && !fused)
    c.check(odit_qknorm_rope(qp, qp + HD * esz, nullptr, q, k, nullptr, wq, wk, cos->data_ptr<float>(), sin->data_ptr<float>(), B, S, H, D,
                             static_cast<int>(2 * cos->size(1)), st, 0, S, static_cast<float>(eps_qk), ODIT_NORM_HEAD, w_dtype, c.dtype, 0u,
                             c.where.stream));
  if (c.rc == 0) {
    const int64_t ds[3] = {S * HD, HD, D}, vs[3] = {S * 3 * HD, 3 * HD, D};
    c.check(odit_attn_fwd_ex(q, k, fused ? v : qp + 2 * HD * esz, nullptr, 0, o, nullptr, 0, nullptr, nullptr, B, S, S, H, H, D, ds, ds, fused ? ds : vs,
                             nullptr, ds, nullptr, static_cast<float>(scale), c.dtype, attn_ws.p, attn_ws.bytes, c.where.stream));
  }
  // gate * proj_out(cat([attention, mlp])) + x: one reduction over both, or two accumulating products over the two column
  // ranges of the weight
  Gate g;
  g.gate = gate->data_ptr();
  g.gbias = gbias->data_ptr();
  g.stride = B > 1 ? gate->stride(0) : 0;
  g.pre = true;
  Lin wm = down, wa = down;
  wm.w = static_cast<const char*>(down.w) + C * esz;
  wm.k = F;
  wa.k = C;
  bool written = false;
  const int joined = c.rc != 0 ? c.rc : odit_linear_join(o, u, down.w, g.gbias, out.data_ptr(), x->data_ptr(), g.gate, static_cast<int>(B * S),
                                                         static_cast<int>(C), static_cast<int>(C), static_cast<int>(F), C, F, down.ldw, C, C,
                                                         ODIT_EPI_GATED_RESIDUAL_PRE, ODIT_F32, c.dtype, B > 1 ? static_cast<int>(S) : 0, g.stride,
                                                         c.engine | ODIT_LINEAR_CLIP, c.lin_ws.p, c.lin_ws.bytes, c.where.stream);
  if (joined != ODIT_ENOTSUP) {
    c.check(joined);
  } else {
    project_gated(c, u, wm, x->data_ptr(), out.data_ptr(), B, S, g, 0, nullptr, Gate());
    written = in_place && c.rc == 0;
    g.gbias = nullptr;
    project_gated(c, o, wa, out.data_ptr(), out.data_ptr(), B, S, g, 0, nullptr, Gate(), true);  // (no gated-residual pass at min_rows 0)
  }
  others_run.reset();
  if (c.rc != 0) return block_failed(c.rc, written);
  if (in_place) { Py_INCREF(a[3]); return a[3]; }
  return wrap(std::move(out));
  NATIVE_END
}

// ---- Wan block: self-attention, cross-attention to the text, feed-forward ------------------------------------------
// (block, heads, head_dim, x [B,S,C], context [B,T,C], mod float32 [B,6,C] or None, gate * bias float32 [B,2,C] or None, temb [B,S,6,C] or None,
//  table float32 [6,C] or None, norm2 weight, norm2 bias (float32 [C] or None), cos, sin, min rows, engine flags, index int32 [S] or None: with one
//  video, token s has row index[s] of temb [1,rows,6,C]) -> x or None
// (gate * bias rows lie as far apart from batch entry to batch entry as the mod rows)
PyObject* py_wan_block(PyObject*, PyObject* const* a, Py_ssize_t n) {
  NATIVE_BEGIN
  if (n != 16) return none();
  BlockCall c;
  const Tensor* index;
  if (!optional_tensor(a[15], &index)) return none();
  const Tensor *x = tensor_of(a[3]), *ctx = tensor_of(a[4]), *mod, *gb, *temb, *table, *lw, *lb, *cos = tensor_of(a[11]), *sin = tensor_of(a[12]);
  const int64_t H = PyLong_AsLong(a[1]), D = PyLong_AsLong(a[2]);
  const int64_t min_rows = PyLong_AsLong(a[13]);
  c.engine = static_cast<unsigned>(PyLong_AsLong(a[14]));
  if (PyErr_Occurred()) return nullptr;
  if (!optional_tensor(a[5], &mod) || !optional_tensor(a[6], &gb) || !optional_tensor(a[7], &temb) || !optional_tensor(a[8], &table) ||
      !optional_tensor(a[9], &lw) || !optional_tensor(a[10], &lb) || !ctx || !cos || !sin || cos->dim() != 2)
    return none();
  if (!block_input(c, x)) return PyErr_Occurred() ? nullptr : none();
  const int64_t B = x->size(0), S = x->size(1), C = x->size(2), HD = H * D, T = ctx->dim() == 3 ? ctx->size(1) : 0;
  // A batch (in the video pipelines a CFG pair) keeps the library's own kernels, what stands in for the one of them that is never run, or those a tuning call chose. Another order of
  // summation is neither better nor worse: against a float32 model the guided noise of 16 batches is 2.03e-2 to 2.8e-2 off (bf16;
  // fp16 2.6e-3 to 3.5e-3) whichever kernels ran. But guidance (scale 5) multiplies the difference of the two rows, so two orders
  // are as far from each other, and results of earlier versions are reproduced. It costs 12 % at B=2 S=3536 and 0 to 7 %
  // elsewhere; at S=3220 it gains 7 %. One video takes whatever is expected to be the fastest: its text's keys and values, in one
  // launch with the queries' projection or in one of their own (project_three, by the number of rows of both), are summed as whole tiles or in up
  // to four parts, so that their last bit can depend on the video's size. Whole tiles give the library's bits; against float64, 512 rows, both
  // are 1.6537107e-3 off (bf16), 2.070324e-4 and 2.070321e-4 (fp16): the one rounding of the result.
  if (B > 1) c.engine |= ODIT_LINEAR_FIRST;
  if (B * S >= (1ll << 31) || S == 0 || T == 0 || (D != 64 && D != 128) || !c.operand(*ctx) || !ctx->is_contiguous() || ctx->size(0) != B || ctx->size(2) != C || HD != C) return none();
  const bool per_token = temb != nullptr;
  if (per_token) {
    if (!table || !c.operand(*temb) || temb->dim() != 4 || temb->size(0) != B || (!index && temb->size(1) != S) || temb->size(2) != 6 || temb->size(3) != C ||
        temb->stride(3) != 1 || !c.where.holds(*table) || table->scalar_type() != at::kFloat || !table->is_contiguous() || table->numel() != 6 * C)
      return none();
  } else {
    if (index || !mod || !gb || !c.where.holds(*mod) || !c.where.holds(*gb) || mod->scalar_type() != at::kFloat || gb->scalar_type() != at::kFloat ||
        mod->dim() != 3 || mod->size(0) != B || mod->size(1) != 6 || mod->size(2) != C || mod->stride(2) != 1 || gb->dim() != 3 || gb->size(0) != B ||
        gb->size(1) != 2 || gb->size(2) != C || gb->stride(2) != 1 || (B > 1 && gb->stride(0) != mod->stride(0)))
      return none();
  }
  if (index && (B != 1 || !c.where.holds(*index) || index->scalar_type() != at::kInt || index->dim() != 1 || index->size(0) != S || !index->is_contiguous() ||
                temb->stride(1) < C || C % 8 != 0 || C > 8192 || temb->stride(1) % 8 != 0 || temb->stride(2) % 8 != 0 || !aligned16(temb->data_ptr()) ||
                !aligned16(table->data_ptr())))
    return none();
  if ((lw == nullptr) != (lb == nullptr) || !f32_row(lw, C) || !f32_row(lb, C) || !c.where.holds(lw) || !c.where.holds(lb)) return none();
  if (!f32_table(c, cos, S, cos->size(1)) || !f32_table(c, sin, S, cos->size(1))) return none();
  PyObject* d = instance_dict(a[0]);
  PyObject *a1 = d ? plain_module(child(d, "attn1"), g_wan_self_type) : nullptr, *a2 = d ? plain_module(child(d, "attn2"), g_wan_cross_type) : nullptr,
           *ffn = d ? plain_module(child(d, "ffn"), g_wan_ffn_type) : nullptr;
  if (!a1 || !a2 || !ffn) return none();
  Lin qkv, out1, q2, k2, v2, out2, up, down;
  double eps, scale1, scale2, eps_n[4];
  const void* nw[4];
  int w_dtype = -1;
  if (!float_attr(d, g_name.eps, &eps) || !c.linear(child(a1, "to_qkv"), &qkv) || !c.linear(child(a1, "to_out"), &out1) ||
      !c.linear(child(a2, "to_q"), &q2) || !c.linear(child(a2, "to_k"), &k2) || !c.linear(child(a2, "to_v"), &v2) ||
      !c.linear(child(a2, "to_out"), &out2) || !c.gelu_projection(child(ffn, "net_0"), &up) || !c.linear(child(ffn, "net_2"), &down) ||
      !c.attention(child(a1, "attn"), &scale1) || !c.attention(child(a2, "attn"), &scale2))
    return none();
  if (PyObject* mods2 = item(a2, g_name.modules); mods2 && PyDict_GetItemString(mods2, "add_k_proj") != nullptr &&
      PyDict_GetItemString(mods2, "add_k_proj") != Py_None)
    return none();  // image-conditioned cross-attention
  PyObject* norms[4] = {child(a1, "norm_q"), child(a1, "norm_k"), child(a2, "norm_q"), child(a2, "norm_k")};
  for (int i = 0; i < 4; ++i) {
    if (!c.norm_weight(norms[i], g_rownorm_type, HD, &nw[i], &w_dtype) || !float_attr(instance_dict(norms[i]), g_name.eps, &eps_n[i])) return none();
  }
  if (eps_n[0] != eps_n[1]) return none();
  const int64_t F = up.n;
  if (qkv.k != C || qkv.n != 3 * HD || out1.k != HD || out1.n != C || q2.k != C || q2.n != HD || k2.k != C || k2.n != HD || v2.k != C ||
      v2.n != HD || out2.k != HD || out2.n != C || up.k != C || down.k != F || down.n != C)
    return none();
  const size_t need1 = odit_attn_fwd_workspace_bytes(B, S, S, H, D), need2 = odit_attn_fwd_workspace_bytes(B, S, T, H, D);
  Scratch ws;
  const size_t need = need1 > need2 ? need1 : need2;
  if (need > 0 && !attn_scratch(c.where, need, &ws)) return nullptr;
  std::optional<Unlocked> others_run(std::in_place);
  const int esz = 2;
  void *nx, *q3, *q, *k, *o, *u, *kc, *kn, *vc, *y;
  // the text's keys and values with the self-attention's projection where that is expected to be faster (asked with addresses that stand
  // in for the ones to come)
  const Lin three[3] = {qkv, k2, v2};
  const int64_t three_rows[3] = {B * S, B * T, B * T};
  const void* const any[3] = {ctx->data_ptr(), ctx->data_ptr(), ctx->data_ptr()};
  void* const any_out[3] = {ctx->data_ptr(), ctx->data_ptr(), ctx->data_ptr()};
  const bool early = project_three(c, any, three, any_out, three_rows, false);
  if (c.rc != 0) {
    others_run.reset();
    return block_failed(c.rc);
  }
  Slab slab(esz);
  slab.want(&nx, B * S * C);
  slab.want(&q, B * S * HD);
  slab.want(&k, B * S * HD);
  slab.want(&o, B * S * HD);
  if (early) {
    slab.want(&kc, B * T * HD);
    slab.want(&vc, B * T * HD);
  }
  slab.mark();
  slab.want(&q3, B * S * 3 * HD);  // self-attention
  slab.rewind();
  slab.want(&kn, B * T * HD);  // cross-attention
  if (!early) {
    slab.want(&kc, B * T * HD);
    slab.want(&vc, B * T * HD);
  }
  slab.rewind();
  slab.want(&u, B * S * F);  // feed-forward
  slab.allocate(x->options());
  y = q;  // a projection's rows on their way to a residual: q is dead behind either attention (HD = C)
  Tensor out = at::empty({B, S, C}, x->options());
  const int64_t rs[2] = {S * C, C};
  const char* tp = per_token ? static_cast<const char*>(temb->data_ptr()) : nullptr;
  auto modulate = [&](const void* src, int row) {  // rows `row` (shift) and row + 1 (scale)
    if (index) {
      const float* tab = table->data_ptr<float>();
      c.check(odit_adaln_modulate_rows(src, nx, tp + row * temb->stride(2) * esz, tp + (row + 1) * temb->stride(2) * esz, index->data_ptr<int32_t>(), tab + row * C,
                                       tab + (row + 1) * C, static_cast<int>(S), static_cast<int>(C), C, C, temb->stride(1), static_cast<float>(eps), c.dtype,
                                       c.dtype, c.where.stream));
    } else if (per_token) {
      const float* tab = table->data_ptr<float>();
      c.check(odit_adaln_modulate(src, nx, tp + row * temb->stride(2) * esz, tp + (row + 1) * temb->stride(2) * esz, nullptr, nullptr, nullptr,
                                  tab + row * C, tab + (row + 1) * C, B, S, C, rs, rs, B > 1 ? temb->stride(0) : 0, S > 1 ? temb->stride(1) : C,
                                  static_cast<float>(eps), c.dtype, c.dtype, 0u, c.where.stream));
    } else {
      const float* m = mod->data_ptr<float>();
      c.check(odit_adaln_modulate(src, nx, m + row * mod->stride(1), m + (row + 1) * mod->stride(1), nullptr, nullptr, nullptr, nullptr, nullptr, B, S, C,
                                  rs, rs, B > 1 ? mod->stride(0) : 0, 0, static_cast<float>(eps), ODIT_F32, c.dtype, 0u, c.where.stream));
    }
  };
  // out = residual + gate row * (src W^T + b)
  const bool norm2_fused = per_token && lw && C % 8 == 0 && C <= 8192;  // with the residual in front of it
  auto gated = [&](const void* src, const Lin& l, const void* residual, int row, int which) {
    if (c.rc != 0) return;
    if (per_token) {
      c.project(src, l, y, B * S, false);
      const int64_t gs[2] = {B > 1 ? temb->stride(0) : 0, S > 1 ? temb->stride(1) : 0}, none[2] = {0, 0};
      if (c.rc == 0 && index) {
        const bool norm = which == 0 && norm2_fused;
        c.check(odit_gated_residual_adaln_rows(residual, y, tp + row * temb->stride(2) * esz, table->data_ptr<float>() + row * C, out.data_ptr(),
                                               norm ? lw->data_ptr<float>() : nullptr, norm ? lb->data_ptr<float>() : nullptr, norm ? nx : nullptr,
                                               index->data_ptr<int32_t>(), static_cast<int>(S), static_cast<int>(C), temb->stride(1), static_cast<float>(eps), c.dtype,
                                               c.where.stream));
        return;
      }
      if (c.rc == 0 && which == 0 && norm2_fused)
        c.check(odit_gated_residual_adaln(residual, y, tp + row * temb->stride(2) * esz, table->data_ptr<float>() + row * C, out.data_ptr(), nullptr,
                                          nullptr, nullptr, nullptr, lw->data_ptr<float>(), lb->data_ptr<float>(), nx, nullptr, B, S, C, gs, none,
                                          static_cast<float>(eps), c.dtype, c.dtype, c.where.stream));
      else if (c.rc == 0)
        c.check(odit_gated_residual(residual, y, tp + row * temb->stride(2) * esz, table->data_ptr<float>() + row * C, out.data_ptr(), B, S, C, rs, rs, rs,
                                    gs, c.dtype, c.dtype, 0u, c.where.stream));
      return;
    }
    Gate g, plain;
    plain.gate = g.gate = mod->data_ptr<float>() + row * mod->stride(1);
    plain.stride = g.stride = B > 1 ? mod->stride(0) : 0;
    plain.code = ODIT_F32;
    g.gbias = gb->data_ptr<float>() + which * gb->stride(1);
    g.pre = true;
    project_gated(c, src, l, residual, out.data_ptr(), B, S, g, min_rows, y, plain);
  };
  modulate(x->data_ptr(), 0);
  if (early) {
    const void* const rows[3] = {nx, ctx->data_ptr(), ctx->data_ptr()};
    void* const into[3] = {q3, kc, vc};
    project_three(c, rows, three, into, three_rows, true);
  } else {
    c.project(nx, qkv, q3, B * S, false);
  }
  char* qp = static_cast<char*>(q3);
  const int64_t st3[2] = {S * 3 * HD, 3 * HD}, st1[2] = {S * HD, HD}, stc[2] = {T * HD, HD};
  if (c.rc == 0)
    c.check(odit_qknorm_rope(qp, qp + HD * esz, nullptr, q, k, nullptr, nw[0], nw[1], cos->data_ptr<float>(), sin->data_ptr<float>(), B, S, H, D,
                             static_cast<int>(2 * cos->size(1)), st3, 0, S, static_cast<float>(eps_n[0]), ODIT_NORM_ROW, w_dtype, c.dtype, 0u,
                             c.where.stream));
  const int64_t ds[3] = {S * HD, HD, D}, vs[3] = {S * 3 * HD, 3 * HD, D}, cs3[3] = {T * HD, HD, D};
  if (c.rc == 0)
    c.check(odit_attn_fwd_ex(q, k, qp + 2 * HD * esz, nullptr, 0, o, nullptr, 0, nullptr, nullptr, B, S, S, H, H, D, ds, ds, vs, nullptr, ds, nullptr,
                             static_cast<float>(scale1), c.dtype, need1 > 0 ? ws.p : nullptr, need1 > 0 ? ws.bytes : 0, c.where.stream));
  gated(o, out1, x->data_ptr(), 2, 0);
  const void* n2 = out.data_ptr();
  if (norm2_fused) {
    n2 = nx;
  } else if (c.rc == 0 && lw) {
    c.check(odit_adaln_modulate(out.data_ptr(), nx, nullptr, nullptr, nullptr, lw->data_ptr<float>(), lb->data_ptr<float>(), nullptr, nullptr, B, S, C, rs,
                                rs, 0, 0, static_cast<float>(eps), c.dtype, c.dtype, 0u, c.where.stream));
    n2 = nx;
  }
  c.project(n2, q2, k, B * S, false);
  if (!early) {
    const Lin kv[2] = {k2, v2};
    void* const kv_out[2] = {kc, vc};
    project_fork(c, ctx->data_ptr(), kv, kv_out, B * T, false);
  }
  if (c.rc == 0)
    c.check(odit_qknorm_rope(k, nullptr, nullptr, q, nullptr, nullptr, nw[2], nullptr, nullptr, nullptr, B, S, H, D, 0, st1, 0, S,
                             static_cast<float>(eps_n[2]), ODIT_NORM_ROW, w_dtype, c.dtype, 0u, c.where.stream));
  if (c.rc == 0)
    c.check(odit_qknorm_rope(kc, nullptr, nullptr, kn, nullptr, nullptr, nw[3], nullptr, nullptr, nullptr, B, T, H, D, 0, stc, 0, T,
                             static_cast<float>(eps_n[3]), ODIT_NORM_ROW, w_dtype, c.dtype, 0u, c.where.stream));
  if (c.rc == 0)
    c.check(odit_attn_fwd_ex(q, kn, vc, nullptr, 0, o, nullptr, 0, nullptr, nullptr, B, S, T, H, H, D, ds, cs3, cs3, nullptr, ds, nullptr,
                             static_cast<float>(scale2), c.dtype, need2 > 0 ? ws.p : nullptr, need2 > 0 ? ws.bytes : 0, c.where.stream));
  project_gated(c, o, out2, out.data_ptr(), out.data_ptr(), B, S, Gate(), 0, nullptr, Gate());  // no gate on this residual
  if (c.rc == 0) modulate(out.data_ptr(), 3);
  c.project(nx, up, u, B * S, true);
  gated(u, down, out.data_ptr(), 5, 1);
  others_run.reset();
  if (c.rc != 0) return block_failed(c.rc);
  return wrap(std::move(out));
  NATIVE_END
}

// -------------------------------------------------------------------------------------------- module
// (linear scratch, attention scratch)
PyObject* py_configure(PyObject*, PyObject* const* a, Py_ssize_t n) {
  if (n != 2) { PyErr_SetString(PyExc_TypeError, "configure takes two callables"); return nullptr; }
  Py_INCREF(a[0]); Py_INCREF(a[1]);
  Py_XSETREF(g_linear_scratch_fn, a[0]);
  Py_XSETREF(g_attn_scratch_fn, a[1]);
  Py_RETURN_NONE;
}

// the classes whose instances the block functions recognise, by name
PyObject* py_classes(PyObject*, PyObject* const* a, Py_ssize_t n) {
  if (n != 1 || !PyDict_Check(a[0])) { PyErr_SetString(PyExc_TypeError, "classes takes a dict"); return nullptr; }
  const struct { const char* name; PyTypeObject** slot; } want[] = {
      {"Linear", &g_linear_type}, {"RMSNorm", &g_rmsnorm_type}, {"DistributedRMSNorm", &g_rownorm_type}, {"AdaLayerNorm", &g_adaln_type},
      {"Attention", &g_attention_type}, {"AttentionImpl", &g_attention_impl_type}, {"FeedForward", &g_feed_forward_type},
      {"ApproxGELU", &g_gelu_type}, {"WanFeedForward", &g_wan_ffn_type}, {"QwenImageCrossAttention", &g_qwen_attention_type},
      {"FluxAttention", &g_flux_attention_type},
      {"AdaLayerNormZeroSingle", &g_flux_single_norm_type}, {"WanSelfAttention", &g_wan_self_type}, {"WanCrossAttention", &g_wan_cross_type},
      {"TimestepEmbedding", &g_time_embedding_type}, {"RotaryEmbedding", &g_rotary_type},
      {"PixArtAlphaTextProjection", &g_text_projection_type}};
  for (const auto& w : want) {
    PyObject* t = PyDict_GetItemString(a[0], w.name);
    if (t == nullptr) continue;
    if (!PyType_Check(t)) { PyErr_SetString(PyExc_TypeError, w.name); return nullptr; }
    Py_INCREF(t);
    Py_XSETREF(*w.slot, reinterpret_cast<PyTypeObject*>(t));
  }
  const struct { const char* name; PyObject** slot; } methods[] = {
      {"RMSNorm.forward_hip", &g_rmsnorm_hip}, {"AdaLayerNorm.forward_hip", &g_adaln_hip}, {"RotaryEmbedding.forward_hip", &g_rotary_hip},
      {"RMSNorm.forward", &g_rmsnorm_forward}, {"AdaLayerNorm.forward", &g_adaln_forward}, {"RotaryEmbedding.forward", &g_rotary_forward},
      {"Module", &g_module_type}, {"Module.globals", &g_module_globals}, {"Module.__call__", &g_module_call[0]},
      {"Module._call_impl", &g_module_call[1]}, {"Module._wrapped_call_impl", &g_module_call[2]}};
  for (const auto& w : methods) {
    PyObject* f = PyDict_GetItemString(a[0], w.name);
    if (f == nullptr) continue;
    Py_INCREF(f);
    Py_XSETREF(*w.slot, f);
  }
  Py_RETURN_NONE;
}

bool intern_names() {
  const struct { const char* s; PyObject** slot; } want[] = {
      {"_modules", &g_name.modules}, {"_parameters", &g_name.parameters}, {"_forward_hooks", &g_name.fwd_hooks},
      {"_forward_pre_hooks", &g_name.pre_hooks}, {"forward", &g_name.forward}, {"weight", &g_name.weight}, {"bias", &g_name.bias},
      {"eps", &g_name.eps}, {"elementwise_affine", &g_name.elementwise_affine}, {"ref_rounding", &g_name.ref_rounding},
      {"attention", &g_name.attention}, {"softmax_scale", &g_name.softmax_scale}, {"fused", &g_name.fused},
      {"forward_hip", &g_name.forward_hip}, {"kernel_takes_layer", &g_name.kernel_takes_layer}, {"_forward_method", &g_name.forward_method},
      {"hidden_size", &g_name.hidden_size}, {"variance_epsilon", &g_name.variance_epsilon}, {"is_neox_style", &g_name.is_neox_style},
      {"__module__", &g_name.module}, {"_backward_hooks", &g_name.bwd_hooks}, {"_backward_pre_hooks", &g_name.bwd_pre_hooks}, {"__call__", &g_name.call},
      {"_call_impl", &g_name.call_impl}, {"_wrapped_call_impl", &g_name.wrapped_call_impl}, {"_compiled_call_impl", &g_name.compiled_call_impl},
      {"_global_forward_hooks", &g_name.global_hooks[0]}, {"_global_forward_pre_hooks", &g_name.global_hooks[1]},
      {"_global_backward_hooks", &g_name.global_hooks[2]}, {"_global_backward_pre_hooks", &g_name.global_hooks[3]}};
  for (const auto& w : want)
    if ((*w.slot = PyUnicode_InternFromString(w.s)) == nullptr) return false;
  return true;
}

#define NATIVE_FN(name, fn) {name, reinterpret_cast<PyCFunction>(reinterpret_cast<void*>(fn)), METH_FASTCALL, nullptr}
PyMethodDef kMethods[] = {
    NATIVE_FN("configure", &py_configure),
    NATIVE_FN("silu", &py_unary<odit_silu>),
    NATIVE_FN("gelu_tanh", &py_unary<odit_gelu_tanh>),
    NATIVE_FN("adaln", &py_adaln),
    NATIVE_FN("adaln_layer", &py_adaln_layer),
    NATIVE_FN("adaln_pair", &py_adaln_pair),
    NATIVE_FN("qknorm_rope", &py_qknorm_rope),
    NATIVE_FN("qknorm_rope_pair", &py_qknorm_rope_pair),
    NATIVE_FN("rmsnorm", &py_rmsnorm),
    NATIVE_FN("rmsnorm_of", &py_rmsnorm_of),
    NATIVE_FN("adaln_of", &py_adaln_of),
    NATIVE_FN("rotary_of", &py_rotary_of),
    NATIVE_FN("layer_call", &py_layer_call),
    NATIVE_FN("own_tree", &py_own_tree),
    NATIVE_FN("rotary", &py_rotary),
    NATIVE_FN("attn", &py_attn),
    NATIVE_FN("linear", &py_linear),
    NATIVE_FN("pair_is_small", &py_pair_is_small),
    NATIVE_FN("linear_few", &py_linear_few),
    NATIVE_FN("linear_few_pair", &py_linear_few_pair),
    NATIVE_FN("time_embedding", &py_time_embedding),
    NATIVE_FN("embed_sum", &py_embed_sum),
    NATIVE_FN("time_tokens", &py_time_tokens),
    NATIVE_FN("project_normed", &py_project_normed),
    NATIVE_FN("project_stem", &py_project_stem),
    NATIVE_FN("project", &py_project),
    NATIVE_FN("time_sinusoid", &py_time_sinusoid),
    NATIVE_FN("rope_tables", &py_rope_tables),
    NATIVE_FN("stack_pairs", &py_stack_pairs),
    NATIVE_FN("extend_mask", &py_extend_mask),
    NATIVE_FN("adaln_rows", &py_adaln_rows),
    NATIVE_FN("cfg_combine", &py_cfg_combine),
    NATIVE_FN("euler_step", &py_euler_step),
    NATIVE_FN("gate_rows", &py_gate_rows),
    NATIVE_FN("classes", &py_classes),
    NATIVE_FN("qwen_block", &py_qwen_block),
    NATIVE_FN("flux_block", &py_flux_block),
    NATIVE_FN("flux_single_block", &py_flux_single_block),
    NATIVE_FN("wan_block", &py_wan_block),
    {nullptr, nullptr, 0, nullptr}};

PyModuleDef kModule = {PyModuleDef_HEAD_INIT, "_native", "native host path of the kernel wrappers", -1, kMethods,
                       nullptr, nullptr, nullptr, nullptr};

}  // namespace

PyMODINIT_FUNC PyInit__native(void) { return intern_names() ? PyModule_Create(&kModule) : nullptr; }
