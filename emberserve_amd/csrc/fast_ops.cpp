// The per-call host path of the row ops and of decode attention as a CPython extension: what
// the Python wrappers do before a launch (operand checks, output allocation, raw pointers
// and strides, the ctypes call) in one native call.
//
// Every function answers an ordinary call and returns None for anything else, with nothing
// launched: the Python wrapper then takes its own path, which converts, raises or runs the
// eager form. Ordinary means: plain CUDA tensors of one device, which is the current one
// (no subclass, no functorch or dispatch-mode wrapper, no tracing), the dtypes and strides
// the kernels read as they are, EMBERSERVE_FUSED_OPS not "0", EMBERSERVE_CHECK_INDICES not
// "1", and an entry point that accepted the call. A launch that fails is raised. No state is
// kept but the entry points' addresses (set once per loaded library).
//
// What bounded the small calls was this host work: about 16 us a launch in Python and ctypes,
// 5 here, 3-4 of them the launch itself. Measured (wall per pass, launches back to back): the
// four row ops of a Qwen2.5-0.5B layer at one token 67.7 -> 25.8 us, of a Qwen2.5-7B layer at
// 339 tokens 68.3 -> 26.7, an MLA layer's three at 5003 tokens 49.3 -> 25.9, paged decode of 32
// sequences (14q/2kv x 64, up to 2048 keys) 15.0 -> 8.6.
#include <Python.h>

#include <ATen/PythonTorchFunctionTLS.h>
#include <ATen/core/Tensor.h>
#include <ATen/ops/empty.h>
#include <c10/core/impl/LocalDispatchKeySet.h>
#include <c10/core/impl/TorchDispatchModeTLS.h>
#include <c10/hip/HIPFunctions.h>
#include <c10/hip/HIPStream.h>
#include <torch/csrc/Exceptions.h>
#include <torch/csrc/autograd/python_variable.h>
#include <torch/csrc/jit/frontend/tracer.h>

#include <cstdlib>
#include <cstring>
#include <initializer_list>
#include <stdexcept>
#include <string>

#include "../../include/ember_ops.h"

namespace {

// The library's entry points, from the loaded libember_ops.so (`bind`).
struct Entry {
  const char* name;
  void* fn;
};
enum {
  kRmsnorm, kAddRmsnorm, kRope, kSilu, kEmbedding, kQkNormRope, kMlaLatentRope, kRopeKvCache, kMlaLatentRopeCache,
  kPagedDecode, kMlaDecode, kStatusString, kEntries
};
Entry g_entry[kEntries] = {
    {"ember_rmsnorm", nullptr}, {"ember_fused_add_rmsnorm", nullptr}, {"ember_rope", nullptr},
    {"ember_silu_and_mul", nullptr}, {"ember_embedding", nullptr}, {"ember_qk_norm_rope", nullptr},
    {"ember_mla_latent_rope", nullptr}, {"ember_rope_kv_cache", nullptr}, {"ember_mla_latent_rope_cache", nullptr},
    {"ember_paged_decode_shared", nullptr}, {"ember_mla_decode", nullptr}, {"ember_status_string", nullptr}};
bool g_bound = false;

#define ENTRY(i, f) reinterpret_cast<decltype(&f)>(g_entry[i].fn)

const c10::DispatchKeySet kWrapped({c10::DispatchKey::Python, c10::DispatchKey::FuncTorchBatched,
                                    c10::DispatchKey::FuncTorchGradWrapper, c10::DispatchKey::Functionalize,
                                    c10::DispatchKey::Conjugate, c10::DispatchKey::Negative,
                                    c10::DispatchKey::ZeroTensor});

bool env_is(const char* name, const char* value) {
  const char* v = std::getenv(name);
  return v != nullptr && std::strcmp(v, value) == 0;
}

// One call's view of its operands: `ok` stays true while the call is an ordinary one.
struct Call {
  bool ok;
  c10::DeviceIndex dev = -1;

  Call() {
    ok = g_bound && !at::impl::torch_function_mode_enabled() && !c10::impl::TorchDispatchModeTLS::any_modes_set() &&
         !c10::impl::tls_is_dispatch_key_included(c10::DispatchKey::FuncTorchDynamicLayerFrontMode) &&
         !torch::jit::tracer::isTracing() && !env_is("EMBERSERVE_FUSED_OPS", "0") &&
         !env_is("EMBERSERVE_CHECK_INDICES", "1");
  }

  // The operand behind `o` when it is a plain strided CUDA tensor on the current device.
  const at::Tensor* tensor(PyObject* o) {
    if (!ok || !THPVariable_CheckExact(o)) return fail();
    const at::Tensor& t = THPVariable_Unpack(o);
    if (!t.defined() || !t.is_cuda() || t.layout() != c10::kStrided || t.key_set().has_any(kWrapped)) return fail();
    if (dev < 0) {
      dev = t.device().index();
      if (dev != c10::hip::current_device()) return fail();
    } else if (t.device().index() != dev) {
      return fail();
    }
    return &t;
  }
  const at::Tensor* fail() {
    ok = false;
    return nullptr;
  }
  void need(bool c) { ok = ok && c; }

  void* stream() const { return c10::hip::getCurrentHIPStream(dev).stream(); }
};

int dtype_tag(const at::Tensor& t) {
  switch (t.scalar_type()) {
    case at::kFloat: return EMBER_F32;
    case at::kHalf: return EMBER_F16;
    case at::kBFloat16: return EMBER_BF16;
    default: return -1;
  }
}

// A tensor as rows of its last dim: unit inner stride, one row stride.
struct Rows {
  int64_t rows = 0, width = 0, stride = 0;
  bool ok = false;
  explicit Rows(const at::Tensor& t) {
    const int64_t dim = t.dim();
    if (dim < 1 || t.numel() == 0) return;
    width = t.size(-1);
    rows = t.numel() / width;
    if (dim == 2 && t.stride(1) == 1) {
      stride = t.stride(0);
      ok = true;
    } else if (t.is_contiguous()) {
      stride = width;
      ok = true;
    }
  }
};

bool weight_ok(const at::Tensor& w, const at::Tensor& x, int64_t n) {
  return (w.scalar_type() == x.scalar_type() || w.scalar_type() == at::kFloat) && w.is_contiguous() && w.numel() == n;
}

bool tables_ok(const at::Tensor& cos, const at::Tensor& sin, const at::Tensor& pos, int64_t n, int64_t d) {
  return cos.scalar_type() == at::kFloat && sin.scalar_type() == at::kFloat && cos.dim() == 2 && sin.dim() == 2 &&
         cos.stride(1) == 1 && sin.stride(1) == 1 && cos.sizes() == sin.sizes() && cos.size(1) >= d / 2 &&
         cos.stride(0) == sin.stride(0) && pos.scalar_type() == at::kLong && pos.is_contiguous() && pos.numel() == n;
}

bool slots_ok(const at::Tensor& slots, int64_t n) {
  return slots.scalar_type() == at::kLong && slots.is_contiguous() && slots.numel() == n;
}

// A paged cache [blocks, block, ...] as flat slots: (slots, slot stride).
bool flat_slots(const at::Tensor& c, int64_t tail, int64_t& n, int64_t& stride) {
  if (c.dim() != tail + 2 || c.size(1) < 2 || c.stride(0) != c.size(1) * c.stride(1)) return false;
  n = c.size(0) * c.size(1);
  stride = c.stride(1);
  return true;
}

bool as_float(PyObject* o, double& v) {
  v = PyFloat_AsDouble(o);
  if (v == -1.0 && PyErr_Occurred()) {
    PyErr_Clear();
    return false;
  }
  return true;
}

// Runs the entry point without the GIL, as ctypes does.
template <typename F>
int launch(F&& f) {
  int st;
  Py_BEGIN_ALLOW_THREADS
  st = f();
  Py_END_ALLOW_THREADS
  return st;
}

// Whether entry point `e` answered the call: false for a refusal, which comes before any launch.
// A failed launch is raised, as the wrappers raise it: the kernel may have been enqueued (the
// status is the thread's last HIP error, which can be an earlier call's), and a second run
// would rotate in-place operands twice.
bool answered(int st, int e) {
  if (st == EMBER_OK) return true;
  if (st == EMBER_EINVAL || st == EMBER_EALIGN || st == EMBER_ENODEV || st == EMBER_ETOOBIG) return false;
  throw std::runtime_error(std::string("emberserve_amd: ") + g_entry[e].name + " failed: " +
                           ENTRY(kStatusString, ember_status_string)(st) + " (status " + std::to_string(st) + ")");
}

PyObject* pair(PyObject* a, PyObject* b) {  // steals both
  PyObject* t = a != nullptr && b != nullptr ? PyTuple_New(2) : nullptr;
  if (t == nullptr) {
    Py_XDECREF(a);
    Py_XDECREF(b);
    return nullptr;
  }
  PyTuple_SET_ITEM(t, 0, a);
  PyTuple_SET_ITEM(t, 1, b);
  return t;
}

PyObject* bind(PyObject*, PyObject* arg) {  // {name: address}
  g_bound = false;
  for (Entry& e : g_entry) {
    PyObject* v = PyDict_GetItemString(arg, e.name);
    void* p = v != nullptr ? PyLong_AsVoidPtr(v) : nullptr;
    if (p == nullptr) {
      if (!PyErr_Occurred()) PyErr_Format(PyExc_KeyError, "no address of %s", e.name);
      return nullptr;
    }
    e.fn = p;
  }
  g_bound = true;
  Py_RETURN_NONE;
}

// (x, weight, eps) -> out
PyObject* rmsnorm(PyObject*, PyObject* const* a, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  if (n != 3) Py_RETURN_NONE;
  Call c;
  const at::Tensor* x = c.tensor(a[0]);
  const at::Tensor* w = c.tensor(a[1]);
  double eps;
  if (!c.ok || !as_float(a[2], eps)) Py_RETURN_NONE;
  const Rows r(*x);
  const int tag = dtype_tag(*x);
  if (!r.ok || tag < 0 || !weight_ok(*w, *x, r.width)) Py_RETURN_NONE;
  at::Tensor out = at::empty(x->sizes(), x->options());
  void* s = c.stream();
  const int st = launch([&] {
    return ENTRY(kRmsnorm, ember_rmsnorm)(x->data_ptr(), r.stride, w->data_ptr(), dtype_tag(*w), out.data_ptr(),
                                          r.width, r.rows, r.width, static_cast<float>(eps), tag, s);
  });
  if (!answered(st, kRmsnorm)) Py_RETURN_NONE;
  return THPVariable_Wrap(std::move(out));
  END_HANDLE_TH_ERRORS
}

// (x, residual, weight, eps) -> (normed, new residual)
PyObject* add_rmsnorm(PyObject*, PyObject* const* a, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  if (n != 4) Py_RETURN_NONE;
  Call c;
  const at::Tensor* x = c.tensor(a[0]);
  const at::Tensor* res = c.tensor(a[1]);
  const at::Tensor* w = c.tensor(a[2]);
  double eps;
  if (!c.ok || !as_float(a[3], eps)) Py_RETURN_NONE;
  const Rows r(*x), q(*res);
  const int tag = dtype_tag(*x);
  if (!r.ok || !q.ok || tag < 0 || res->scalar_type() != x->scalar_type() || res->sizes() != x->sizes() ||
      !weight_ok(*w, *x, r.width))
    Py_RETURN_NONE;
  at::Tensor out = at::empty(x->sizes(), x->options());
  at::Tensor sum = at::empty(x->sizes(), x->options());
  void* s = c.stream();
  const int st = launch([&] {
    return ENTRY(kAddRmsnorm, ember_fused_add_rmsnorm)(x->data_ptr(), r.stride, res->data_ptr(), q.stride,
                                                       w->data_ptr(), dtype_tag(*w), out.data_ptr(), r.width,
                                                       sum.data_ptr(), r.width, r.rows, r.width,
                                                       static_cast<float>(eps), tag, s);
  });
  if (!answered(st, kAddRmsnorm)) Py_RETURN_NONE;
  return pair(THPVariable_Wrap(std::move(out)), THPVariable_Wrap(std::move(sum)));
  END_HANDLE_TH_ERRORS
}

// (x) -> out
PyObject* silu_and_mul(PyObject*, PyObject* arg) {
  HANDLE_TH_ERRORS
  Call c;
  const at::Tensor* x = c.tensor(arg);
  if (!c.ok) Py_RETURN_NONE;
  const Rows r(*x);
  const int tag = dtype_tag(*x);
  if (!r.ok || tag < 0 || r.width % 2 != 0) Py_RETURN_NONE;
  const int64_t inter = r.width / 2;
  c10::SmallVector<int64_t, 5> sizes(x->sizes().begin(), x->sizes().end());
  sizes.back() = inter;
  at::Tensor out = at::empty(sizes, x->options());
  void* s = c.stream();
  const int st = launch([&] {
    return ENTRY(kSilu, ember_silu_and_mul)(x->data_ptr(), r.stride, out.data_ptr(), inter, r.rows, inter, tag, s);
  });
  if (!answered(st, kSilu)) Py_RETURN_NONE;
  return THPVariable_Wrap(std::move(out));
  END_HANDLE_TH_ERRORS
}

// (ids, weight) -> rows
PyObject* embedding(PyObject*, PyObject* const* a, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  if (n != 2) Py_RETURN_NONE;
  Call c;
  const at::Tensor* ids = c.tensor(a[0]);
  const at::Tensor* w = c.tensor(a[1]);
  if (!c.ok) Py_RETURN_NONE;
  if (ids->scalar_type() != at::kLong || !ids->is_contiguous() || ids->numel() == 0 || w->dim() != 2 ||
      w->numel() == 0 || w->stride(1) != 1)
    Py_RETURN_NONE;
  c10::SmallVector<int64_t, 5> sizes(ids->sizes().begin(), ids->sizes().end());
  sizes.push_back(w->size(1));
  at::Tensor out = at::empty(sizes, w->options());
  void* s = c.stream();
  const int st = launch([&] {
    return ENTRY(kEmbedding, ember_embedding)(static_cast<const int64_t*>(ids->data_ptr()), ids->numel(),
                                              w->data_ptr(), w->size(0), w->size(1), w->stride(0), out.data_ptr(),
                                              w->size(1), static_cast<int64_t>(w->element_size()), s);
  });
  if (!answered(st, kEmbedding)) Py_RETURN_NONE;
  return THPVariable_Wrap(std::move(out));
  END_HANDLE_TH_ERRORS
}

// q [N, H, D] and k [N, Hkv, D]: unit stride in an even D, one dtype, N > 0.
bool heads_ok(const at::Tensor& q, const at::Tensor& k) {
  return q.dim() == 3 && k.dim() == 3 && q.numel() > 0 && k.numel() > 0 && q.stride(2) == 1 && k.stride(2) == 1 &&
         q.size(2) % 2 == 0 && k.size(0) == q.size(0) && k.size(2) == q.size(2) && k.scalar_type() == q.scalar_type();
}

// (q, k, cos, sin, positions) -> (q, k)
PyObject* rope(PyObject*, PyObject* const* a, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  if (n != 5) Py_RETURN_NONE;
  Call c;
  const at::Tensor *q = c.tensor(a[0]), *k = c.tensor(a[1]), *cos = c.tensor(a[2]), *sin = c.tensor(a[3]),
                   *pos = c.tensor(a[4]);
  if (!c.ok || !heads_ok(*q, *k) || !tables_ok(*cos, *sin, *pos, q->size(0), q->size(2))) Py_RETURN_NONE;
  const int tag = dtype_tag(*q);
  if (tag < 0) Py_RETURN_NONE;
  void* s = c.stream();
  const int st = launch([&] {
    return ENTRY(kRope, ember_rope)(q->data_ptr(), q->stride(0), q->stride(1), q->size(1), k->data_ptr(),
                                    k->stride(0), k->stride(1), k->size(1), q->size(2),
                                    static_cast<const float*>(cos->data_ptr()),
                                    static_cast<const float*>(sin->data_ptr()), cos->size(0), cos->stride(0),
                                    static_cast<const int64_t*>(pos->data_ptr()), q->size(0), tag, s);
  });
  if (!answered(st, kRope)) Py_RETURN_NONE;
  return pair(Py_NewRef(a[0]), Py_NewRef(a[1]));
  END_HANDLE_TH_ERRORS
}

// (q, k, q_weight, k_weight, eps, cos, sin, positions) -> (q, k)
PyObject* qk_norm_rope(PyObject*, PyObject* const* a, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  if (n != 8) Py_RETURN_NONE;
  Call c;
  const at::Tensor *q = c.tensor(a[0]), *k = c.tensor(a[1]), *qw = c.tensor(a[2]), *kw = c.tensor(a[3]),
                   *cos = c.tensor(a[5]), *sin = c.tensor(a[6]), *pos = c.tensor(a[7]);
  double eps;
  if (!c.ok || !as_float(a[4], eps) || !heads_ok(*q, *k)) Py_RETURN_NONE;
  const int64_t d = q->size(2);
  const int tag = dtype_tag(*q);
  if (tag < 0 || !tables_ok(*cos, *sin, *pos, q->size(0), d) || !weight_ok(*qw, *q, d) || !weight_ok(*kw, *q, d) ||
      qw->scalar_type() != kw->scalar_type())
    Py_RETURN_NONE;
  void* s = c.stream();
  const int st = launch([&] {
    return ENTRY(kQkNormRope, ember_qk_norm_rope)(
        q->data_ptr(), q->stride(0), q->stride(1), q->size(1), k->data_ptr(), k->stride(0), k->stride(1), k->size(1),
        d, qw->data_ptr(), kw->data_ptr(), dtype_tag(*qw), static_cast<float>(eps),
        static_cast<const float*>(cos->data_ptr()), static_cast<const float*>(sin->data_ptr()), cos->size(0),
        cos->stride(0), static_cast<const int64_t*>(pos->data_ptr()), q->size(0), tag, s);
  });
  if (!answered(st, kQkNormRope)) Py_RETURN_NONE;
  return pair(Py_NewRef(a[0]), Py_NewRef(a[1]));
  END_HANDLE_TH_ERRORS
}

// (q, k, v, cos, sin, positions, slots, k_cache, v_cache, q_weight, k_weight, eps) -> (q, k)
PyObject* rope_kv_cache(PyObject*, PyObject* const* a, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  if (n != 12) Py_RETURN_NONE;
  Call c;
  const at::Tensor *q = c.tensor(a[0]), *k = c.tensor(a[1]), *v = c.tensor(a[2]), *cos = c.tensor(a[3]),
                   *sin = c.tensor(a[4]), *pos = c.tensor(a[5]), *slots = c.tensor(a[6]), *kc = c.tensor(a[7]),
                   *vc = c.tensor(a[8]);
  const bool norm = a[9] != Py_None;
  const at::Tensor *qw = nullptr, *kw = nullptr;
  if (norm) {
    qw = c.tensor(a[9]);
    kw = c.tensor(a[10]);
  }
  double eps;
  if (!c.ok || !as_float(a[11], eps) || !heads_ok(*q, *k)) Py_RETURN_NONE;
  const int64_t t = q->size(0), d = q->size(2), hk = k->size(1);
  const int tag = dtype_tag(*q);
  int64_t nslots = 0, slot_stride = 0;
  if (tag < 0 || v->sizes() != k->sizes() || v->stride(2) != 1 || v->scalar_type() != q->scalar_type() ||
      !tables_ok(*cos, *sin, *pos, t, d) || !slots_ok(*slots, t) || kc->scalar_type() != q->scalar_type() ||
      vc->scalar_type() != q->scalar_type() || kc->sizes() != vc->sizes() || kc->strides() != vc->strides() ||
      !flat_slots(*kc, 2, nslots, slot_stride) || kc->size(2) != hk || kc->size(3) != d)
    Py_RETURN_NONE;
  if (norm && (!weight_ok(*qw, *q, d) || !weight_ok(*kw, *q, d) || qw->scalar_type() != kw->scalar_type()))
    Py_RETURN_NONE;
  void* s = c.stream();
  const int st = launch([&] {
    return ENTRY(kRopeKvCache, ember_rope_kv_cache)(
        q->data_ptr(), q->stride(0), q->stride(1), q->size(1), k->data_ptr(), k->stride(0), k->stride(1), hk,
        v->data_ptr(), v->stride(0), v->stride(1), d, norm ? qw->data_ptr() : nullptr, norm ? kw->data_ptr() : nullptr,
        norm ? dtype_tag(*qw) : 0, static_cast<float>(eps), static_cast<const float*>(cos->data_ptr()),
        static_cast<const float*>(sin->data_ptr()), cos->size(0), cos->stride(0),
        static_cast<const int64_t*>(pos->data_ptr()), static_cast<const int64_t*>(slots->data_ptr()), t,
        kc->data_ptr(), vc->data_ptr(), nslots, slot_stride, kc->stride(2), tag, s);
  });
  if (!answered(st, kRopeKvCache)) Py_RETURN_NONE;
  return pair(Py_NewRef(a[0]), Py_NewRef(a[1]));
  END_HANDLE_TH_ERRORS
}

// The MLA operands c [N, R], k_pe [N, Dr], q_pe [N, H, Dr], weight [R].
bool mla_ok(const at::Tensor& c, const at::Tensor& kp, const at::Tensor& qp, const at::Tensor& w) {
  return c.dim() == 2 && kp.dim() == 2 && qp.dim() == 3 && c.numel() > 0 && qp.numel() > 0 && kp.size(0) == c.size(0) &&
         qp.size(0) == c.size(0) && kp.size(1) == qp.size(2) && qp.size(2) % 2 == 0 && c.stride(1) == 1 &&
         kp.stride(1) == 1 && qp.stride(2) == 1 && kp.scalar_type() == c.scalar_type() &&
         qp.scalar_type() == c.scalar_type() && weight_ok(w, c, c.size(1));
}

// (c, k_pe, q_pe, weight, eps, cos, sin, positions) -> (q_pe, latent)
PyObject* mla_latent_rope(PyObject*, PyObject* const* a, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  if (n != 8) Py_RETURN_NONE;
  Call call;
  const at::Tensor *c = call.tensor(a[0]), *kp = call.tensor(a[1]), *qp = call.tensor(a[2]), *w = call.tensor(a[3]),
                   *cos = call.tensor(a[5]), *sin = call.tensor(a[6]), *pos = call.tensor(a[7]);
  double eps;
  if (!call.ok || !as_float(a[4], eps) || !mla_ok(*c, *kp, *qp, *w)) Py_RETURN_NONE;
  const int64_t t = c->size(0), r = c->size(1), dr = qp->size(2);
  const int tag = dtype_tag(*c);
  if (tag < 0 || !tables_ok(*cos, *sin, *pos, t, dr)) Py_RETURN_NONE;
  at::Tensor latent = at::empty({t, r + dr}, c->options());
  void* s = call.stream();
  const int st = launch([&] {
    return ENTRY(kMlaLatentRope, ember_mla_latent_rope)(
        c->data_ptr(), c->stride(0), r, kp->data_ptr(), kp->stride(0), qp->data_ptr(), qp->stride(0), qp->stride(1),
        qp->size(1), dr, w->data_ptr(), dtype_tag(*w), static_cast<float>(eps),
        static_cast<const float*>(cos->data_ptr()), static_cast<const float*>(sin->data_ptr()), cos->size(0),
        cos->stride(0), static_cast<const int64_t*>(pos->data_ptr()), t, latent.data_ptr(), r + dr, tag, s);
  });
  if (!answered(st, kMlaLatentRope)) Py_RETURN_NONE;
  return pair(Py_NewRef(a[2]), THPVariable_Wrap(std::move(latent)));
  END_HANDLE_TH_ERRORS
}

// (c, k_pe, q_pe, weight, eps, cos, sin, positions, slots, cache, return_latent) -> (q_pe, latent or None)
PyObject* mla_latent_rope_cache(PyObject*, PyObject* const* a, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  if (n != 11) Py_RETURN_NONE;
  Call call;
  const at::Tensor *c = call.tensor(a[0]), *kp = call.tensor(a[1]), *qp = call.tensor(a[2]), *w = call.tensor(a[3]),
                   *cos = call.tensor(a[5]), *sin = call.tensor(a[6]), *pos = call.tensor(a[7]),
                   *slots = call.tensor(a[8]), *cache = call.tensor(a[9]);
  double eps;
  if (!call.ok || !as_float(a[4], eps) || !mla_ok(*c, *kp, *qp, *w)) Py_RETURN_NONE;
  const int keep = PyObject_IsTrue(a[10]);
  if (keep < 0) return nullptr;
  const int64_t t = c->size(0), r = c->size(1), dr = qp->size(2);
  const int tag = dtype_tag(*c);
  int64_t nslots = 0, slot_stride = 0;
  if (tag < 0 || !tables_ok(*cos, *sin, *pos, t, dr) || !slots_ok(*slots, t) ||
      cache->scalar_type() != c->scalar_type() || !flat_slots(*cache, 1, nslots, slot_stride) ||
      cache->size(2) != r + dr || cache->stride(2) != 1)
    Py_RETURN_NONE;
  at::Tensor latent;
  if (keep) latent = at::empty({t, r + dr}, c->options());
  void* s = call.stream();
  const int st = launch([&] {
    return ENTRY(kMlaLatentRopeCache, ember_mla_latent_rope_cache)(
        c->data_ptr(), c->stride(0), r, kp->data_ptr(), kp->stride(0), qp->data_ptr(), qp->stride(0), qp->stride(1),
        qp->size(1), dr, w->data_ptr(), dtype_tag(*w), static_cast<float>(eps),
        static_cast<const float*>(cos->data_ptr()), static_cast<const float*>(sin->data_ptr()), cos->size(0),
        cos->stride(0), static_cast<const int64_t*>(pos->data_ptr()), t, keep ? latent.data_ptr() : nullptr,
        keep ? r + dr : 0, static_cast<const int64_t*>(slots->data_ptr()), cache->data_ptr(), nslots, slot_stride, tag,
        s);
  });
  if (!answered(st, kMlaLatentRopeCache)) Py_RETURN_NONE;
  return pair(Py_NewRef(a[2]), keep ? THPVariable_Wrap(std::move(latent)) : Py_NewRef(Py_None));
  END_HANDLE_TH_ERRORS
}

// The split count and workspace of a decode call, from the Python module's own rule and
// scratch cache: `plan(*shape)` -> (num_splits, workspace or None). False on a Python error.
struct Plan {
  int64_t splits = 1;
  void* ws = nullptr;
  int64_t ws_bytes = 0;
  PyObject* held = nullptr;
  ~Plan() { Py_XDECREF(held); }
  bool resolve(PyObject* plan, std::initializer_list<int64_t> shape, PyObject* q) {
    PyObject* args = PyTuple_New(static_cast<Py_ssize_t>(shape.size()) + 1);
    if (args == nullptr) return false;
    Py_ssize_t i = 0;
    for (int64_t v : shape) PyTuple_SET_ITEM(args, i++, PyLong_FromLongLong(v));
    PyTuple_SET_ITEM(args, i, Py_NewRef(q));
    held = PyObject_CallObject(plan, args);
    Py_DECREF(args);
    if (held == nullptr) return false;
    splits = PyLong_AsLongLong(PyTuple_GetItem(held, 0));
    if (PyErr_Occurred()) return false;
    PyObject* w = PyTuple_GetItem(held, 1);
    if (w == nullptr) return false;
    if (w != Py_None) {
      const at::Tensor& t = THPVariable_Unpack(w);
      ws = t.data_ptr();
      ws_bytes = static_cast<int64_t>(t.nbytes());
    }
    return true;
  }
};

bool block_tables_ok(const at::Tensor& bt, const at::Tensor& ctx, int64_t b) {
  return bt.dim() == 2 && bt.size(0) == b && bt.numel() > 0 && bt.scalar_type() == at::kInt && bt.stride(1) == 1 &&
         ctx.dim() == 1 && ctx.size(0) == b && ctx.scalar_type() == at::kInt && ctx.stride(0) == 1;
}

// (q, k_cache, v_cache, block_tables, context_lens, scale, plan) -> out
PyObject* paged_decode(PyObject*, PyObject* const* a, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  if (n != 7) Py_RETURN_NONE;
  Call c;
  const at::Tensor *q = c.tensor(a[0]), *kc = c.tensor(a[1]), *vc = c.tensor(a[2]), *bt = c.tensor(a[3]),
                   *ctx = c.tensor(a[4]);
  double scale;
  if (!c.ok || std::getenv("EMBERSERVE_TRITON_VARIANT") != nullptr || !as_float(a[5], scale)) Py_RETURN_NONE;
  if (q->dim() != 3 || q->numel() == 0 || !q->is_contiguous() || kc->dim() != 4 || kc->numel() == 0 ||
      vc->sizes() != kc->sizes() || !block_tables_ok(*bt, *ctx, q->size(0)))
    Py_RETURN_NONE;
  const int64_t b = q->size(0), h = q->size(1), d = q->size(2), hk = kc->size(2), bs = kc->size(1);
  const int tag = dtype_tag(*q), ctag = dtype_tag(*kc);
  if ((d != 64 && d != 128) || kc->size(3) != d || kc->stride(3) != 1 || vc->stride(3) != 1 || bs % 16 != 0 ||
      h % hk != 0 || tag < 0 || ctag < 0 || vc->scalar_type() != kc->scalar_type())
    Py_RETURN_NONE;
  Plan p;
  if (!p.resolve(a[6], {b, h, d, hk, bt->size(1) * bs}, a[0])) return nullptr;
  at::Tensor out = at::empty(q->sizes(), q->options());
  void* s = c.stream();
  const int st = launch([&] {
    return ENTRY(kPagedDecode, ember_paged_decode_shared)(
        q->data_ptr(), q->stride(0), q->stride(1), tag, kc->data_ptr(), vc->data_ptr(), kc->size(0), bs, hk, d,
        kc->stride(0), kc->stride(1), kc->stride(2), vc->stride(0), vc->stride(1), vc->stride(2), ctag,
        static_cast<const int32_t*>(bt->data_ptr()), bt->stride(0), bt->size(1),
        static_cast<const int32_t*>(ctx->data_ptr()), b, h, static_cast<float>(scale), p.splits, 0, p.ws, p.ws_bytes,
        out.data_ptr(), out.stride(0), out.stride(1), s);
  });
  if (!answered(st, kPagedDecode)) Py_RETURN_NONE;
  return THPVariable_Wrap(std::move(out));
  END_HANDLE_TH_ERRORS
}

// (q_c, q_pe, cache, block_tables, context_lens, scale, plan) -> out_c
PyObject* mla_decode(PyObject*, PyObject* const* a, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  if (n != 7) Py_RETURN_NONE;
  Call c;
  const at::Tensor *qc = c.tensor(a[0]), *qp = c.tensor(a[1]), *lat = c.tensor(a[2]), *bt = c.tensor(a[3]),
                   *ctx = c.tensor(a[4]);
  double scale;
  if (!c.ok || !as_float(a[5], scale)) Py_RETURN_NONE;
  if (qc->dim() != 3 || qp->dim() != 3 || qc->numel() == 0 || qp->size(0) != qc->size(0) ||
      qp->size(1) != qc->size(1) || lat->dim() != 3 || lat->numel() == 0 || !block_tables_ok(*bt, *ctx, qc->size(0)))
    Py_RETURN_NONE;
  const int64_t b = qc->size(0), h = qc->size(1), dl = qc->size(2), dr = qp->size(2), bs = lat->size(1);
  const int tag = dtype_tag(*qc);
  if (dl != 512 || dr != 64 || lat->size(2) != dl + dr || tag < 0 || qp->scalar_type() != qc->scalar_type() ||
      lat->scalar_type() != qc->scalar_type() || qc->stride(2) != 1 || qp->stride(2) != 1 || lat->stride(2) != 1 ||
      bs % 16 != 0)
    Py_RETURN_NONE;
  Plan p;
  if (!p.resolve(a[6], {b, h, dl, bt->size(1) * bs}, a[0])) return nullptr;
  at::Tensor out = at::empty({b, h, dl}, qc->options());
  void* s = c.stream();
  const int st = launch([&] {
    return ENTRY(kMlaDecode, ember_mla_decode)(
        qc->data_ptr(), qc->stride(0), qc->stride(1), qp->data_ptr(), qp->stride(0), qp->stride(1), tag,
        lat->data_ptr(), lat->size(0), bs, dl, dr, lat->stride(0), lat->stride(1), tag,
        static_cast<const int32_t*>(bt->data_ptr()), bt->stride(0), bt->size(1),
        static_cast<const int32_t*>(ctx->data_ptr()), b, h, static_cast<float>(scale), p.splits, p.ws, p.ws_bytes,
        out.data_ptr(), out.stride(0), out.stride(1), s);
  });
  if (!answered(st, kMlaDecode)) Py_RETURN_NONE;
  return THPVariable_Wrap(std::move(out));
  END_HANDLE_TH_ERRORS
}

#define FAST(f) {#f, reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)()>(f)), METH_FASTCALL, nullptr}
PyMethodDef kMethods[] = {
    {"bind", bind, METH_O, nullptr}, {"silu_and_mul", silu_and_mul, METH_O, nullptr},
    FAST(rmsnorm), FAST(add_rmsnorm), FAST(embedding), FAST(rope), FAST(qk_norm_rope), FAST(rope_kv_cache),
    FAST(mla_latent_rope), FAST(mla_latent_rope_cache), FAST(paged_decode), FAST(mla_decode),
    {nullptr, nullptr, 0, nullptr}};
PyModuleDef kModule = {PyModuleDef_HEAD_INIT, "_fast", nullptr, -1, kMethods, nullptr, nullptr, nullptr, nullptr};

}  // namespace

PyMODINIT_FUNC PyInit__fast(void) {
  PyObject* m = PyModule_Create(&kModule);
  // the ABI version (ember_abi_version) of the header this was compiled against
  if (m != nullptr && PyModule_AddIntConstant(m, "ABI_VERSION", 20) != 0) {
    Py_DECREF(m);
    return nullptr;
  }
  return m;
}
