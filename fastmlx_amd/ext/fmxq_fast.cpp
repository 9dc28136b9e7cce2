// fmxq_fast.cpp -- the call path of the torch wrappers (fastmlx_amd/ops.py) in C++.
//
// A decode-sized call is bound by the host: ops.quantized_matmul of a 2048 x 2048
// product took 10.2 us a call through Python checks, torch.empty and ctypes for 2.6 us
// of kernel.  Each function here takes the same tensors, checks them as ops.py does,
// allocates the result and calls the C ABI: that call 10.5 -> 4.9 us, a small
// dequantize and quantize pair 22.5 -> 11.0 us, most of it the two HIP launches.
//
// A function returns None, with nothing enqueued, for anything but the plain case: an
// argument that ops.py would refuse, a tensor subclass, a functorch wrapper, an active
// dispatch or function mode, or sizes of zero.  ops.py then runs its own path, which
// raises the error or handles the call.  A nonzero status of the library is raised from
// here, as ops.py raises it: a second attempt would enqueue again what the first had
// launched, and an error of the device, reported once, would be lost.
#define PY_SSIZE_T_CLEAN
#include <Python.h>

#include <ATen/ATen.h>
#include <ATen/PythonTorchFunctionTLS.h>
#include <c10/core/impl/TorchDispatchModeTLS.h>
#include <c10/hip/HIPStream.h>
#include <torch/csrc/autograd/python_variable.h>

#include "../../include/fmxq.h"

namespace {

constexpr int kBf16Like = 1, kU32Like = 2, kBf16 = 4, kF32 = 8;

bool type_ok(at::ScalarType t, int kinds) {
  switch (t) {
    case at::kBFloat16: return (kinds & (kBf16Like | kBf16)) != 0;
    case at::kShort:
    case at::kUInt16: return (kinds & kBf16Like) != 0;
    case at::kInt:
    case at::kUInt32: return (kinds & kU32Like) != 0;
    case at::kFloat: return (kinds & kF32) != 0;
    default: return false;
  }
}

// No mode that watches tensor creation or calls is active.
bool plain_mode() {
  return !c10::impl::TorchDispatchModeTLS::any_modes_set() &&
         !at::impl::torch_function_mode_enabled();
}

// One call's arguments: after the first that is out of the ordinary, `ok` is false and
// every later request returns nothing.
struct Call {
  bool ok = plain_mode();

  // A plain, contiguous, non-empty device tensor of one of the kinds.
  const at::Tensor* tensor(PyObject* o, int kinds) {
    if (!ok || !THPVariable_CheckExact(o)) return fail();
    const at::Tensor& t = THPVariable_Unpack(o);
    constexpr c10::DispatchKeySet odd({c10::DispatchKey::Python, c10::DispatchKey::FuncTorchBatched,
                                       c10::DispatchKey::FuncTorchGradWrapper,
                                       c10::DispatchKey::Functionalize, c10::DispatchKey::Conjugate,
                                       c10::DispatchKey::Negative, c10::DispatchKey::ZeroTensor});
    if (!t.defined() || !t.is_cuda() || t.layout() != at::kStrided || t.key_set().has_any(odd) ||
        !type_ok(t.scalar_type(), kinds) || t.numel() == 0 || !t.is_contiguous())
      return fail();
    return &t;
  }
  template <class T = uint16_t>
  T* ptr(PyObject* o, int kinds) {
    const at::Tensor* t = tensor(o, kinds);
    return t ? static_cast<T*>(t->data_ptr()) : nullptr;
  }
  uint16_t* opt(PyObject* o, int kinds) { return o == Py_None ? nullptr : ptr(o, kinds); }
  // A (w, scales, biases) triple.
  struct Triple {
    const at::Tensor* w = nullptr;
    uint32_t* wp = nullptr;
    uint16_t *s = nullptr, *b = nullptr;
  };
  Triple triple(PyObject* o) {
    Triple r;
    if (!ok || !(PyTuple_CheckExact(o) || PyList_CheckExact(o)) || PySequence_Fast_GET_SIZE(o) != 3) {
      fail();
      return r;
    }
    r.w = tensor(PySequence_Fast_GET_ITEM(o, 0), kU32Like);
    r.s = ptr(PySequence_Fast_GET_ITEM(o, 1), kBf16Like);
    r.b = ptr(PySequence_Fast_GET_ITEM(o, 2), kBf16Like);
    if (r.w) r.wp = static_cast<uint32_t*>(r.w->data_ptr());
    return r;
  }
  bool integer(PyObject* o, int64_t* v) {
    if (!ok || !PyLong_CheckExact(o)) return fail() != nullptr;
    *v = PyLong_AsLongLong(o);
    if (*v == -1 && PyErr_Occurred()) {
      PyErr_Clear();
      return fail() != nullptr;
    }
    return true;
  }
  bool format(PyObject* group, PyObject* bits, int64_t* g, int64_t* b) {
    if (!integer(group, g) || !integer(bits, b)) return false;
    if ((*b != 4 && *b != 8) || (*g != 32 && *g != 64 && *g != 128)) return fail() != nullptr;
    return true;
  }
  const at::Tensor* fail() {
    ok = false;
    return nullptr;
  }
};

at::Tensor make(const at::Tensor& like, at::IntArrayRef sizes, at::ScalarType t) {
  return at::empty(sizes, like.options().dtype(t).requires_grad(false));
}

void* stream_of(const at::Tensor& t) {
  return c10::hip::getCurrentHIPStream(t.device().index()).stream();
}

// Run f() without the GIL; its status 0 means enqueued, another sets the Python error
// that fastmlx_amd._lib.check raises for it.
template <class F>
bool enqueue(F&& f) {
  int rc;
  Py_BEGIN_ALLOW_THREADS;
  rc = f();
  Py_END_ALLOW_THREADS;
  if (rc == FMXQ_OK) return true;
  if (PyObject* lib = PyImport_ImportModule("fastmlx_amd._lib")) {
    Py_XDECREF(PyObject_CallMethod(lib, "check", "i", rc));
    Py_DECREF(lib);
  }
  return false;
}

// C++ exceptions (out of memory in an allocation) leave through Python's path, which
// meets the same condition and raises it.
template <class F>
PyObject* guarded(F&& f) {
  try {
    PyObject* r = f();
    if (r || PyErr_Occurred()) return r;
  } catch (...) {
    PyErr_Clear();
  }
  Py_RETURN_NONE;
}

// (x, w, scales, biases, bias | None, out | None, group_size, bits)
PyObject* quantized_matmul(PyObject*, PyObject* const* a, Py_ssize_t n) {
  return guarded([&]() -> PyObject* {
    if (n != 8) return nullptr;
    Call c;
    int64_t group, bits;
    const at::Tensor* x = c.tensor(a[0], kBf16Like);
    const at::Tensor* w = c.tensor(a[1], kU32Like);
    const uint16_t *s = c.ptr(a[2], kBf16Like), *b = c.ptr(a[3], kBf16Like);
    const uint16_t* bias = c.opt(a[4], kBf16Like);
    uint16_t* y = c.opt(a[5], kBf16Like);
    if (!c.format(a[6], a[7], &group, &bits) || x->dim() < 1 || w->dim() != 2) return nullptr;
    const int64_t K = x->size(-1), N = w->size(0), M = x->numel() / K;
    if (w->size(1) * 32 / bits != K) return nullptr;
    at::Tensor out;
    if (!y) {
      at::DimVector sizes(x->sizes());
      sizes.back() = N;
      out = make(*x, sizes, at::kBFloat16);
      y = static_cast<uint16_t*>(out.data_ptr());
    }
    const uint16_t* xp = static_cast<uint16_t*>(x->data_ptr());
    const uint32_t* wp = static_cast<uint32_t*>(w->data_ptr());
    void* st = stream_of(*x);
    if (!enqueue([&] {
          return bias ? fmxq_quantized_matmul_bias(xp, wp, s, b, bias, y, M, N, K, true, (int)group,
                                                   (int)bits, st)
                      : fmxq_quantized_matmul(xp, wp, s, b, y, M, N, K, true, (int)group, (int)bits, st);
        }))
      return nullptr;
    return out.defined() ? THPVariable_Wrap(std::move(out)) : Py_NewRef(a[5]);
  });
}

// (w, scales, biases, out | None, group_size, bits)
PyObject* dequantize(PyObject*, PyObject* const* a, Py_ssize_t n) {
  return guarded([&]() -> PyObject* {
    if (n != 6) return nullptr;
    Call c;
    int64_t group, bits;
    const at::Tensor* w = c.tensor(a[0], kU32Like);
    const uint16_t *s = c.ptr(a[1], kBf16Like), *b = c.ptr(a[2], kBf16Like);
    uint16_t* y = c.opt(a[3], kBf16Like);
    if (!c.format(a[4], a[5], &group, &bits) || w->dim() < 1) return nullptr;
    const int64_t K = w->size(-1) * 32 / bits, rows = w->numel() / w->size(-1);
    at::Tensor out;
    if (!y) {
      at::DimVector sizes(w->sizes());
      sizes.back() = K;
      out = make(*w, sizes, at::kBFloat16);
      y = static_cast<uint16_t*>(out.data_ptr());
    }
    const uint32_t* wp = static_cast<uint32_t*>(w->data_ptr());
    void* st = stream_of(*w);
    if (!enqueue([&] { return fmxq_dequantize(wp, s, b, y, rows, K, (int)group, (int)bits, st); }))
      return nullptr;
    return out.defined() ? THPVariable_Wrap(std::move(out)) : Py_NewRef(a[3]);
  });
}

// (w, group_size, bits) -> (wq, scales, biases)
PyObject* quantize(PyObject*, PyObject* const* a, Py_ssize_t n) {
  return guarded([&]() -> PyObject* {
    if (n != 3) return nullptr;
    Call c;
    int64_t group, bits;
    const at::Tensor* w = c.tensor(a[0], kBf16Like);
    if (!c.format(a[1], a[2], &group, &bits) || w->dim() < 1) return nullptr;
    const int64_t K = w->size(-1), rows = w->numel() / K;
    if (K % group) return nullptr;
    at::DimVector sizes(w->sizes());
    sizes.back() = K * bits / 32;
    at::Tensor wq = make(*w, sizes, at::kInt);
    sizes.back() = K / group;
    at::Tensor s = make(*w, sizes, at::kBFloat16), b = make(*w, sizes, at::kBFloat16);
    const uint16_t* wp = static_cast<uint16_t*>(w->data_ptr());
    void* st = stream_of(*w);
    if (!enqueue([&] {
          return fmxq_quantize(wp, static_cast<uint32_t*>(wq.data_ptr()),
                               static_cast<uint16_t*>(s.data_ptr()),
                               static_cast<uint16_t*>(b.data_ptr()), rows, K, (int)group, (int)bits, st);
        }))
      return nullptr;
    return Py_BuildValue("(NNN)", THPVariable_Wrap(std::move(wq)), THPVariable_Wrap(std::move(s)),
                         THPVariable_Wrap(std::move(b)));
  });
}

// (x, inds, gate, up, down, weights, shared expert triples | None, shared | None,
// shared_gate | None, out | None, group_size, bits): moe_layer with the triples,
// switch_glu_combine without.
PyObject* moe_layer(PyObject*, PyObject* const* a, Py_ssize_t n) {
  return guarded([&]() -> PyObject* {
    if (n != 12) return nullptr;
    Call c;
    int64_t group, bits;
    const at::Tensor *x = c.tensor(a[0], kBf16Like), *inds = c.tensor(a[1], kU32Like);
    const auto g = c.triple(a[2]), u = c.triple(a[3]), d = c.triple(a[4]);
    const uint16_t* wts = c.ptr(a[5], kBf16Like);
    Call::Triple sh[3];
    const bool own = a[6] != Py_None;
    if (own) {
      if (!(PyTuple_CheckExact(a[6]) || PyList_CheckExact(a[6])) || PySequence_Fast_GET_SIZE(a[6]) != 3)
        return nullptr;
      for (int i = 0; i < 3; ++i) sh[i] = c.triple(PySequence_Fast_GET_ITEM(a[6], i));
    }
    const uint16_t *shared = c.opt(a[7], kBf16Like), *sgate = c.opt(a[8], kBf16Like);
    uint16_t* y = c.opt(a[9], kBf16Like);
    if (!c.format(a[10], a[11], &group, &bits) || x->dim() != 2 || inds->dim() < 1 || g.w->dim() < 2)
      return nullptr;
    const int64_t T = x->size(0), D = x->size(1), k = inds->size(-1), E = g.w->size(0), I = g.w->size(1);
    at::Tensor out;
    if (!y) {
      out = make(*x, {T, D}, at::kBFloat16);
      y = static_cast<uint16_t*>(out.data_ptr());
    }
    const uint16_t* xp = static_cast<uint16_t*>(x->data_ptr());
    const uint32_t* ip = static_cast<uint32_t*>(inds->data_ptr());
    void* st = stream_of(*x);
    if (!enqueue([&] {
          return own ? fmxq_moe_layer(xp, ip, g.wp, g.s, g.b, u.wp, u.s, u.b, d.wp, d.s, d.b, wts,
                                      sh[0].wp, sh[0].s, sh[0].b, sh[1].wp, sh[1].s, sh[1].b, sh[2].wp,
                                      sh[2].s, sh[2].b, sgate, y, T, k, E, D, I, (int)group, (int)bits, st)
                     : fmxq_switch_glu_combine(xp, ip, g.wp, g.s, g.b, u.wp, u.s, u.b, d.wp, d.s, d.b,
                                               wts, shared, sgate, y, T, k, E, D, I, (int)group,
                                               (int)bits, st);
        }))
      return nullptr;
    return out.defined() ? THPVariable_Wrap(std::move(out)) : Py_NewRef(a[9]);
  });
}

// (logits, top_k, norm_topk_prob, weights in bf16) -> (inds, weights)
PyObject* route_softmax_topk(PyObject*, PyObject* const* a, Py_ssize_t n) {
  return guarded([&]() -> PyObject* {
    if (n != 4 || !PyBool_Check(a[2]) || !PyBool_Check(a[3])) return nullptr;
    Call c;
    int64_t k;
    const at::Tensor* x = c.tensor(a[0], kBf16 | kF32);
    if (!c.integer(a[1], &k) || x->dim() != 2 || k < 1 || k > 64) return nullptr;
    const int64_t T = x->size(0), E = x->size(1);
    const bool wb = a[3] == Py_True, norm = a[2] == Py_True;
    at::Tensor inds = make(*x, {T, k}, at::kInt);
    at::Tensor w = make(*x, {T, k}, wb ? at::kBFloat16 : at::kFloat);
    void* st = stream_of(*x);
    if (!enqueue([&] {
          return fmxq_route_softmax_topk(x->data_ptr(), x->scalar_type() == at::kBFloat16, T, E, (int)k,
                                         norm, static_cast<uint32_t*>(inds.data_ptr()), w.data_ptr(),
                                         wb, st);
        }))
      return nullptr;
    return Py_BuildValue("(NN)", THPVariable_Wrap(std::move(inds)), THPVariable_Wrap(std::move(w)));
  });
}

// (gates, bias | None, top_k, n_group, topk_group, scale, norm, weights in bf16)
PyObject* route_group_topk(PyObject*, PyObject* const* a, Py_ssize_t n) {
  return guarded([&]() -> PyObject* {
    if (n != 8 || !PyFloat_CheckExact(a[5]) || !PyBool_Check(a[6]) || !PyBool_Check(a[7])) return nullptr;
    Call c;
    int64_t k, ng, tg;
    const at::Tensor* x = c.tensor(a[0], kBf16 | kF32);
    const float* bias = a[1] == Py_None ? nullptr : c.ptr<float>(a[1], kF32);
    if (!c.integer(a[2], &k) || !c.integer(a[3], &ng) || !c.integer(a[4], &tg) || x->dim() != 2 ||
        k < 1 || k > 64 || ng < 1 || ng > 64 || tg < 1 || tg > 64)
      return nullptr;
    const int64_t T = x->size(0), E = x->size(1);
    const float scale = (float)PyFloat_AS_DOUBLE(a[5]);
    const bool norm = a[6] == Py_True, wb = a[7] == Py_True;
    at::Tensor inds = make(*x, {T, k}, at::kInt);
    at::Tensor w = make(*x, {T, k}, wb ? at::kBFloat16 : at::kFloat);
    void* st = stream_of(*x);
    if (!enqueue([&] {
          return fmxq_route_group_topk(x->data_ptr(), x->scalar_type() == at::kBFloat16, bias, T, E,
                                       (int)k, (int)ng, (int)tg, scale, norm,
                                       static_cast<uint32_t*>(inds.data_ptr()), w.data_ptr(), wb, st);
        }))
      return nullptr;
    return Py_BuildValue("(NN)", THPVariable_Wrap(std::move(inds)), THPVariable_Wrap(std::move(w)));
  });
}

#define FMXQ_FAST(f) {#f, reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)(void)>(f)), METH_FASTCALL, nullptr}
PyMethodDef methods[] = {FMXQ_FAST(quantized_matmul), FMXQ_FAST(dequantize),       FMXQ_FAST(quantize),
                         FMXQ_FAST(moe_layer),        FMXQ_FAST(route_softmax_topk), FMXQ_FAST(route_group_topk),
                         {nullptr, nullptr, 0, nullptr}};
PyModuleDef module = {PyModuleDef_HEAD_INIT, "_fast", nullptr, -1, methods, nullptr, nullptr, nullptr, nullptr};

}  // namespace

PyMODINIT_FUNC PyInit__fast(void) { return PyModule_Create(&module); }
