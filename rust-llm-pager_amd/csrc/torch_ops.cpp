// Call path of the operator API for plain tensors: the Python functions of
// pager_hf/streaming_attention.py hand their arguments to these before anything else.
//
// Each function checks that its arguments are what the kernels take as they are (exact
// torch.Tensor objects without functorch, functionalization or lazy-bit keys, one GPU, one
// dtype, contiguous, matching shapes), allocates the workspace or outputs from torch's current
// allocator, and calls the C entry point of libpgr.so. It returns the entry point's status, or
// None where any check fails: the caller then runs its general Python path, which converts,
// copies or refuses as it always has. So this file decides nothing but speed: checks in Python,
// one attribute object at a time, and a ctypes call of 19 arguments held the GPU up. A call of one
// query (init, fold, finalize; 28/4 heads, D 128, fp16, 64 tokens) 30.6 -> 16.8 us, 4133 tokens
// the same; the two-pass run of 12 calls (32/4, D 64, batch 4, 8209 tokens) 151 -> 84.6 us.
//
// libpgr.so's entry points come as addresses (bind), so that the library the Python package has
// loaded is the one called.
#include <Python.h>

#include <ATen/ATen.h>
#include <ATen/detail/CUDAHooksInterface.h>
#include <c10/core/Allocator.h>
#include <c10/core/DeviceGuard.h>
#include <c10/core/impl/TorchDispatchModeTLS.h>
#include <ATen/PythonTorchFunctionTLS.h>
#include <torch/csrc/Device.h>
#include <torch/csrc/Dtype.h>
#include <torch/csrc/autograd/python_variable.h>

#include <cmath>
#include <cstdint>
#include <exception>

namespace {

using Tensor = at::Tensor;

size_t (*g_workspace_bytes)(int64_t, int64_t, int64_t, int64_t, int64_t, int, int64_t);
int (*g_step)(const void*, const void*, const void*, const int32_t*, const int32_t*, float*, float*, float*, int64_t,
              int64_t, int64_t, int64_t, int64_t, int, float, float, void*, size_t, void*);
int (*g_stats)(const void*, const void*, const int32_t*, const int32_t*, float*, float*, int64_t, int64_t, int64_t,
               int64_t, int64_t, int, float, float, void*, size_t, void*);
int (*g_accumulate)(const void*, const void*, const void*, const int32_t*, const int32_t*, const float*, const float*,
                    float*, float*, int64_t, int64_t, int64_t, int64_t, int64_t, int64_t, int64_t, int64_t, int, float,
                    float, void*, size_t, void*);
int (*g_fold_fixed)(const void*, const void*, const void*, const int32_t*, const float*, const float*, float*, int64_t,
                    int64_t, int64_t, int64_t, int64_t, int, float, float, void*, size_t, void*);
int (*g_state_init)(float*, float*, float*, int64_t, int64_t, void*);
int (*g_finalize)(const float*, const float*, void*, int64_t, int64_t, int, void*);
PyObject* g_raw_stream;     // torch._C._cuda_getCurrentRawStream
PyObject* g_out_of_memory;  // torch.OutOfMemoryError

enum Mode : int { kFold = 0, kStats = 1, kAccumulate = 2, kFoldFixed = 3 };  // PGR_MODE_* (pgr.h)

// The dispatch keys of an ordinary GPU tensor. A tensor with any other key (functorch wrappers,
// functionalization, Python subclasses, the negative bit) takes the general path.
bool plain_keys(const Tensor& t) {
  static const c10::DispatchKeySet allowed =
      c10::DispatchKeySet({c10::DispatchKey::CUDA, c10::DispatchKey::ADInplaceOrView}) |
      c10::getAutogradRelatedKeySetFromBackend(c10::BackendComponent::CUDABit) |
      c10::getAutocastRelatedKeySetFromBackend(c10::BackendComponent::CUDABit);
  return (t.key_set().raw_repr() & ~allowed.raw_repr()) == 0;  // (operator- would keep backend bits)
}

const Tensor* plain(PyObject* o) {
  if (!THPVariable_CheckExact(o)) return nullptr;
  const Tensor& t = THPVariable_Unpack(o);
  return t.defined() && t.is_cuda() && plain_keys(t) && t.has_storage() && t.is_contiguous() ? &t : nullptr;
}

bool is_f32(const Tensor* t, const c10::Device& dev, at::IntArrayRef shape) {
  return t && t->scalar_type() == at::kFloat && t->device() == dev && t->sizes() == shape;
}

// An optional 0/1 mask: *out is its data or null. False: not in the form the kernels read.
bool mask(PyObject* o, const c10::Device& dev, at::IntArrayRef shape, const int32_t** out) {
  *out = nullptr;
  if (o == Py_None) return true;
  const Tensor* t = plain(o);
  if (!t || t->scalar_type() != at::kInt || t->device() != dev || t->sizes() != shape) return false;
  *out = t->const_data_ptr<int32_t>();
  return true;
}

// None or an exact Python float.
bool number(PyObject* o, double none_value, double* out) {
  if (o == Py_None) {
    *out = none_value;
    return true;
  }
  if (PyFloat_CheckExact(o)) {
    *out = PyFloat_AS_DOUBLE(o);
    return true;
  }
  return false;
}

bool integer(PyObject* o, int64_t* out) {
  if (!PyLong_CheckExact(o)) return false;
  int overflow = 0;
  *out = PyLong_AsLongLongAndOverflow(o, &overflow);
  return overflow == 0;
}

bool current_stream(const c10::Device& dev, void** out) {
  PyObject* idx = PyLong_FromLong(dev.index());
  if (!idx) return false;
  PyObject* s = PyObject_CallFunctionObjArgs(g_raw_stream, idx, nullptr);
  Py_DECREF(idx);
  if (!s) return false;
  *out = PyLong_AsVoidPtr(s);
  Py_DECREF(s);
  return !PyErr_Occurred();
}

// Everything a launch needs, resolved while the GIL is held.
struct Call {
  const void *q, *k, *v = nullptr;
  float *m, *l, *acc = nullptr;
  const int32_t *valid = nullptr, *active = nullptr;
  int64_t b, hq, hkv, tc, d;
  int code;
  float scale, softcap;
  void* stream;
  c10::Device dev{c10::DeviceType::CUDA};
};

int dtype_code(at::ScalarType t) {
  return t == at::kHalf ? 0 : t == at::kBFloat16 ? 1 : t == at::kFloat ? 2 : -1;  // PGR_DTYPE_*
}

float* f32(const Tensor* t) { return static_cast<float*>(t->mutable_data_ptr()); }

// The operands that every mode takes; v and acc are null for the statistics pass.
bool prepare(Call& c, PyObject* q_, PyObject* k_, PyObject* v_, PyObject* m_, PyObject* l_, PyObject* acc_,
             PyObject* valid_, PyObject* active_, PyObject* scale_, PyObject* softcap_) {
  const Tensor *q = plain(q_), *k = plain(k_);
  if (!q || !k || q->dim() != 3 || k->dim() != 4) return false;
  c.dev = q->device();
  c.b = q->size(0);
  c.hq = q->size(1);
  c.d = q->size(2);
  c.hkv = k->size(1);
  c.tc = k->size(2);
  c.code = dtype_code(q->scalar_type());
  if (c.code < 0 || k->scalar_type() != q->scalar_type() || k->device() != c.dev) return false;
  if (c.b <= 0 || c.tc <= 0 || c.hkv <= 0 || c.hq <= 0 || c.hq % c.hkv != 0 || c.hq / c.hkv > 16 ||
      k->size(0) != c.b || k->size(3) != c.d)
    return false;
  if (v_) {
    const Tensor* v = plain(v_);
    if (!v || v->scalar_type() != q->scalar_type() || v->device() != c.dev || v->sizes() != k->sizes()) return false;
    c.v = v->const_data_ptr();
  }
  const Tensor *m = plain(m_), *l = plain(l_), *acc = acc_ ? plain(acc_) : nullptr;
  if (!is_f32(m, c.dev, {c.b, c.hq}) || !is_f32(l, c.dev, {c.b, c.hq})) return false;
  if (acc_ && !is_f32(acc, c.dev, {c.b, c.hq, c.d})) return false;
  if (!mask(valid_, c.dev, {c.b, c.tc}, &c.valid)) return false;
  if (active_ && !mask(active_, c.dev, {c.b}, &c.active)) return false;
  double scale = 0.0, softcap = 0.0;
  if (!number(scale_, 1.0 / std::pow((double)c.d, 0.5), &scale) || !number(softcap_, 0.0, &softcap)) return false;
  c.scale = (float)scale;
  c.softcap = (float)softcap;
  c.q = q->const_data_ptr();
  c.k = k->const_data_ptr();
  c.m = f32(m);
  c.l = f32(l);
  if (acc_) c.acc = f32(acc);
  return true;
}

// Runs `launch(workspace, bytes)` with the workspace of the call's mode. New reference or null.
template <class F>
PyObject* run(Call& c, int mode, int64_t tpb, F launch) {
  if (!current_stream(c.dev, &c.stream)) return nullptr;
  int rc = 0;
  {
    const c10::DeviceGuard guard(c.dev);
    const size_t bytes = g_workspace_bytes(c.b, c.hq, c.hkv, c.tc, c.d, mode, tpb);
    // Freed on return, behind this stream's work, as a tensor of this size would be, and from the
    // allocator that torch.empty uses (c10::GetAllocator is the native one also where
    // torch.cuda.memory.change_current_allocator has put another in its place).
    const c10::DataPtr ws =
        at::detail::getCUDAHooks().getCUDADeviceAllocator()->allocate(bytes ? bytes : 1);
    Py_BEGIN_ALLOW_THREADS;
    rc = launch(ws.get(), bytes);
    Py_END_ALLOW_THREADS;
  }
  return PyLong_FromLong(rc);
}

// C++ exceptions (an allocation that fails, a torch check) end as Python exceptions.
template <class F>
PyObject* guarded(F body) {
  try {
    return body();
  } catch (const c10::OutOfMemoryError& e) {
    PyErr_SetString(g_out_of_memory, e.what_without_backtrace());
  } catch (const std::exception& e) {
    PyErr_SetString(PyExc_RuntimeError, e.what());
  } catch (...) {
    PyErr_SetString(PyExc_RuntimeError, "unknown C++ exception");
  }
  return nullptr;
}

bool ready(Py_ssize_t n, Py_ssize_t want) {
  if (n == want && g_raw_stream) return true;
  PyErr_SetString(PyExc_TypeError, g_raw_stream ? "wrong number of arguments" : "bind was not called");
  return false;
}

// A torch dispatch or function mode sees what the general path calls.
bool modes_active() {
  return c10::impl::TorchDispatchModeTLS::any_modes_set() || at::impl::torch_function_mode_enabled();
}

// step(q, k, v, m, l, acc, valid, active, scale, softcap)
PyObject* py_step(PyObject*, PyObject* const* a, Py_ssize_t n) {
  if (!ready(n, 10)) return nullptr;
  return guarded([&]() -> PyObject* {
    Call c;
    if (modes_active() || !prepare(c, a[0], a[1], a[2], a[3], a[4], a[5], a[6], a[7], a[8], a[9])) Py_RETURN_NONE;
    return run(c, kFold, 16, [&](void* ws, size_t bytes) {
      return g_step(c.q, c.k, c.v, c.valid, c.active, c.m,
                    c.l, c.acc, c.b, c.hq, c.hkv, c.tc, c.d, c.code, c.scale, c.softcap, ws,
                    bytes, c.stream);
    });
  });
}

// stats_step(q, k, m, l, valid, active, scale, softcap)
PyObject* py_stats(PyObject*, PyObject* const* a, Py_ssize_t n) {
  if (!ready(n, 8)) return nullptr;
  return guarded([&]() -> PyObject* {
    Call c;
    if (modes_active() || !prepare(c, a[0], a[1], nullptr, a[2], a[3], nullptr, a[4], a[5], a[6], a[7]))
      Py_RETURN_NONE;
    return run(c, kStats, 16, [&](void* ws, size_t bytes) {
      return g_stats(c.q, c.k, c.valid, c.active, c.m, c.l, c.b, c.hq,
                     c.hkv, c.tc, c.d, c.code, c.scale, c.softcap, ws, bytes, c.stream);
    });
  });
}

// accumulate_step(q, k, v, m, l, acc, block_mass, block_id_offset, tokens_per_block, valid,
// active, scale, softcap)
PyObject* py_accumulate(PyObject*, PyObject* const* a, Py_ssize_t n) {
  if (!ready(n, 13)) return nullptr;
  return guarded([&]() -> PyObject* {
    Call c;
    int64_t offset = 0, tpb = 0;
    if (modes_active() || !prepare(c, a[0], a[1], a[2], a[3], a[4], a[5], a[9], a[10], a[11], a[12]) ||
        !integer(a[7], &offset) || !integer(a[8], &tpb) || tpb <= 0)
      Py_RETURN_NONE;
    const Tensor* mass = plain(a[6]);
    if (!mass || mass->scalar_type() != at::kFloat || mass->device() != c.dev || mass->dim() != 3 ||
        mass->size(0) != c.b || mass->size(1) != c.hq)
      Py_RETURN_NONE;
    const int64_t max_blocks = mass->size(2);
    float* const mass_data = f32(mass);
    return run(c, kAccumulate, tpb, [&](void* ws, size_t bytes) {
      return g_accumulate(c.q, c.k, c.v, c.valid, c.active,
                          c.m, c.l, c.acc, mass_data, max_blocks, offset, tpb, c.b, c.hq, c.hkv, c.tc,
                          c.d, c.code, c.scale, c.softcap, ws, bytes, c.stream);
    });
  });
}

// fold_fixed_step(q, k, v, m, l, acc, valid, scale, softcap)
PyObject* py_fold_fixed(PyObject*, PyObject* const* a, Py_ssize_t n) {
  if (!ready(n, 9)) return nullptr;
  return guarded([&]() -> PyObject* {
    Call c;
    if (modes_active() || !prepare(c, a[0], a[1], a[2], a[3], a[4], a[5], a[6], nullptr, a[7], a[8])) Py_RETURN_NONE;
    return run(c, kFoldFixed, 16, [&](void* ws, size_t bytes) {
      return g_fold_fixed(c.q, c.k, c.v, c.valid, c.m,
                          c.l, c.acc, c.b, c.hq, c.hkv, c.tc, c.d, c.code, c.scale, c.softcap,
                          ws, bytes, c.stream);
    });
  });
}

// state_init(batch, query_heads, head_dim, device) -> (status, m, l, acc) or None. The device has
// an index and torch's GPU state exists: the caller sees to both.
PyObject* py_state_init(PyObject*, PyObject* const* a, Py_ssize_t n) {
  if (!ready(n, 4)) return nullptr;
  return guarded([&]() -> PyObject* {
    int64_t b = 0, hq = 0, d = 0;
    if (modes_active() || !THPDevice_Check(a[3])) Py_RETURN_NONE;
    const c10::Device dev = reinterpret_cast<THPDevice*>(a[3])->device;
    if (!dev.is_cuda() || !dev.has_index() || !integer(a[0], &b) || !integer(a[1], &hq) || !integer(a[2], &d) ||
        b <= 0 || hq <= 0 || d <= 0)
      Py_RETURN_NONE;
    void* stream = nullptr;
    if (!current_stream(dev, &stream)) return nullptr;
    const c10::DeviceGuard guard(dev);
    const auto opt = at::TensorOptions().dtype(at::kFloat).device(dev);
    Tensor m = at::empty({b, hq}, opt), l = at::empty({b, hq}, opt), acc = at::empty({b, hq, d}, opt);
    if (!plain_keys(m)) Py_RETURN_NONE;  // a mode or transform is active: the general path
    float *pm = f32(&m), *pl = f32(&l), *pacc = f32(&acc);
    int rc = 0;
    Py_BEGIN_ALLOW_THREADS;
    rc = g_state_init(pm, pl, pacc, b * hq, d, stream);
    Py_END_ALLOW_THREADS;
    return Py_BuildValue("(iNNN)", rc, THPVariable_Wrap(m), THPVariable_Wrap(l), THPVariable_Wrap(acc));
  });
}

// finalize(acc, l, dtype) -> (status, out) or None
PyObject* py_finalize(PyObject*, PyObject* const* a, Py_ssize_t n) {
  if (!ready(n, 3)) return nullptr;
  return guarded([&]() -> PyObject* {
    const Tensor *acc = plain(a[0]), *l = plain(a[1]);
    if (modes_active() || !acc || !l || !THPDtype_Check(a[2]) || acc->dim() < 1) Py_RETURN_NONE;
    const at::ScalarType type = reinterpret_cast<THPDtype*>(a[2])->scalar_type;
    const int code = dtype_code(type);
    if (code < 0 || acc->numel() == 0 || !is_f32(acc, acc->device(), acc->sizes()) ||
        !is_f32(l, acc->device(), acc->sizes().slice(0, acc->dim() - 1)))
      Py_RETURN_NONE;
    void* stream = nullptr;
    if (!current_stream(acc->device(), &stream)) return nullptr;
    const c10::DeviceGuard guard(acc->device());
    Tensor out = at::empty(acc->sizes(), at::TensorOptions().dtype(type).device(acc->device()));
    if (!plain_keys(out)) Py_RETURN_NONE;
    const float *pacc = f32(acc), *pl = f32(l);
    void* pout = out.mutable_data_ptr();
    const int64_t rows = l->numel(), d = acc->size(-1);
    int rc = 0;
    Py_BEGIN_ALLOW_THREADS;
    rc = g_finalize(pacc, pl, pout, rows, d, code, stream);
    Py_END_ALLOW_THREADS;
    return Py_BuildValue("(iN)", rc, THPVariable_Wrap(out));
  });
}

// bind(workspace_bytes, step, stats, accumulate, fold_fixed, state_init, finalize: addresses;
// raw_stream: callable(device index) -> hipStream_t; out_of_memory: exception class)
PyObject* py_bind(PyObject*, PyObject* args) {
  unsigned long long p[7];
  PyObject *raw = nullptr, *oom = nullptr;
  if (!PyArg_ParseTuple(args, "KKKKKKKOO", &p[0], &p[1], &p[2], &p[3], &p[4], &p[5], &p[6], &raw, &oom))
    return nullptr;
  auto set = [](auto& fn, unsigned long long addr) { fn = reinterpret_cast<std::decay_t<decltype(fn)>>(addr); };
  set(g_workspace_bytes, p[0]);
  set(g_step, p[1]);
  set(g_stats, p[2]);
  set(g_accumulate, p[3]);
  set(g_fold_fixed, p[4]);
  set(g_state_init, p[5]);
  set(g_finalize, p[6]);
  Py_INCREF(raw);
  Py_XSETREF(g_raw_stream, raw);
  Py_INCREF(oom);
  Py_XSETREF(g_out_of_memory, oom);
  Py_RETURN_NONE;
}

PyMethodDef methods[] = {
    {"bind", py_bind, METH_VARARGS, nullptr},
    {"step", (PyCFunction)(void (*)(void))py_step, METH_FASTCALL, nullptr},
    {"stats_step", (PyCFunction)(void (*)(void))py_stats, METH_FASTCALL, nullptr},
    {"accumulate_step", (PyCFunction)(void (*)(void))py_accumulate, METH_FASTCALL, nullptr},
    {"fold_fixed_step", (PyCFunction)(void (*)(void))py_fold_fixed, METH_FASTCALL, nullptr},
    {"state_init", (PyCFunction)(void (*)(void))py_state_init, METH_FASTCALL, nullptr},
    {"finalize", (PyCFunction)(void (*)(void))py_finalize, METH_FASTCALL, nullptr},
    {nullptr, nullptr, 0, nullptr},
};

PyModuleDef module = {PyModuleDef_HEAD_INIT, "_pgr_ops", nullptr, -1, methods, nullptr, nullptr, nullptr, nullptr};

}  // namespace

PyMODINIT_FUNC PyInit__pgr_ops() { return PyModule_Create(&module); }
