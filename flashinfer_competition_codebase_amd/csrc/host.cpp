// host.cpp - the Python entry points' call path in native code (CPython
// extension module _gdn_host).
//
// A small call's time is its host path: a 6-token prefill's kernel takes 4.4
// us, and the Python checks of its twelve tensors, the workspace, the stream
// and the 22-argument ctypes call made it 20.3 us a call; a value-returning
// decode step of a few heads took 16.1.  These functions make the same checks,
// allocations and call: 5.5-6.4 and 6.2 us.  They are a fast path only: arguments
// outside what they accept (anything the Python path would refuse, convert or
// treat specially) return None, nothing done, and the Python path takes the
// call from the start, so its errors and conversions stay as they are.
// Nothing is kept between calls.

#define PY_SSIZE_T_CLEAN
#include <Python.h>

#include <ATen/core/Tensor.h>
#include <ATen/ops/empty.h>
#include <ATen/ops/zeros.h>
#include <c10/core/impl/VirtualGuardImpl.h>
#include <c10/hip/HIPStream.h>
#include <torch/csrc/Exceptions.h>
#include <torch/csrc/autograd/python_variable.h>

#include <cmath>
#include <cstdint>

#include "gdn_decode.h"
#include "gdn_prefill.h"

namespace {

constexpr int64_t kDim = 128;

// The library functions, bound by bind_prefill and bind_decode.
decltype(&gdn_prefill) g_prefill;
decltype(&gdn_prefill_workspace_bytes) g_workspace;
decltype(&gdn_decode_steps) g_decode;

// A plain strided tensor in device memory: no subclass, and none of the
// wrappers of tracing, vmap or functionalisation (their data is elsewhere).
const at::Tensor* plain(PyObject* obj) {
  if (!THPVariable_CheckExact(obj)) return nullptr;
  const at::Tensor& t = THPVariable_Unpack(obj);
  if (!t.defined() || t.layout() != c10::kStrided || !t.is_cuda() || !t.has_storage())
    return nullptr;
  const c10::DispatchKeySet ks = t.key_set();
  for (const c10::DispatchKey key :
       {c10::DispatchKey::Python, c10::DispatchKey::FuncTorchBatched,
        c10::DispatchKey::FuncTorchGradWrapper, c10::DispatchKey::Functionalize,
        c10::DispatchKey::Negative, c10::DispatchKey::Conjugate})
    if (ks.has(key)) return nullptr;
  return &t;
}

bool is(const at::Tensor* t, c10::ScalarType type, c10::IntArrayRef shape) {
  return t != nullptr && t->scalar_type() == type && t->sizes() == shape && t->is_contiguous();
}

// The scale argument: None and 0 mean 1 / sqrt(128); only Python numbers here.
bool scale_of(PyObject* obj, float* out) {
  double x;
  if (obj == Py_None) {
    x = 0.0;
  } else if (PyFloat_CheckExact(obj)) {
    x = PyFloat_AS_DOUBLE(obj);
  } else {
    return false;
  }
  *out = static_cast<float>(x == 0.0 ? 1.0 / std::sqrt(static_cast<double>(kDim)) : x);
  return true;
}

bool one_device(const at::Tensor* first, std::initializer_list<const at::Tensor*> others) {
  for (const at::Tensor* t : others)
    if (t != nullptr && t->device() != first->device()) return false;
  return true;
}

// The current stream of the tensors' device, if that device is current (else
// the Python path, which switches to it).
bool stream_of(const at::Tensor* t, c10::Stream* stream) {
  const c10::impl::VirtualGuardImpl impl(c10::DeviceType::CUDA);
  if (impl.getDevice() != t->device()) return false;
  *stream = impl.getStream(t->device());
  return true;
}

bool ranges_overlap(const at::Tensor* x, const at::Tensor* y) {
  const auto x0 = reinterpret_cast<uintptr_t>(x->const_data_ptr());
  const auto y0 = reinterpret_cast<uintptr_t>(y->const_data_ptr());
  return x0 < y0 + y->nbytes() && y0 < x0 + x->nbytes();
}

// A tensor the call reads.
template <typename T>
const T* ptr(const at::Tensor* t) {
  return t == nullptr ? nullptr : static_cast<const T*>(t->const_data_ptr());
}

// A tensor the call writes: one that shares its memory until it is written (a
// lazy clone) gets its own first, on the current stream.
template <typename T>
T* out_ptr(const at::Tensor* t) {
  return static_cast<T*>(t->mutable_data_ptr());
}

PyObject* code_of(int code) {
  return PyLong_FromLong(code);
}

// prefill(q, k, v, state, A_log, a, dt_bias, b, cu_seqlens, scale, output,
// new_state, use_qk_l2norm): the library's return code, or with output and
// new_state None (both allocated here, output zeroed) (code, output,
// new_state); None for the Python path.
PyObject* prefill(PyObject*, PyObject* const* args, Py_ssize_t nargs) {
  HANDLE_TH_ERRORS
  if (nargs != 13) {
    PyErr_SetString(PyExc_TypeError, "prefill takes 13 arguments");
    return nullptr;
  }
  const at::Tensor *q = plain(args[0]), *k = plain(args[1]), *v = plain(args[2]);
  if (g_prefill == nullptr || q == nullptr || v == nullptr || q->dim() != 3 || v->dim() != 3)
    Py_RETURN_NONE;
  const at::Tensor* state = nullptr;
  if (args[3] != Py_None && (state = plain(args[3])) == nullptr) Py_RETURN_NONE;
  const at::Tensor *A_log = plain(args[4]), *a = plain(args[5]), *dt_bias = plain(args[6]),
                   *b = plain(args[7]), *cu = plain(args[8]);
  const int64_t L = q->size(0), H = q->size(1), HV = v->size(1);
  if (cu == nullptr || cu->dim() != 1 || cu->numel() < 2 || !is(cu, at::kInt, cu->sizes()))
    Py_RETURN_NONE;
  const int64_t N = cu->numel() - 1;
  constexpr int64_t kMax = 0x7fffffff;
  if (H <= 0 || HV <= 0 || HV % H != 0 || L > kMax || N > kMax || HV > 65535) Py_RETURN_NONE;
  float scale;
  if (!is(q, at::kBFloat16, {L, H, kDim}) || !is(k, at::kBFloat16, {L, H, kDim}) ||
      !is(v, at::kBFloat16, {L, HV, kDim}) ||
      (state != nullptr && !is(state, at::kFloat, {N, HV, kDim, kDim})) ||
      !is(A_log, at::kFloat, {HV}) || !is(dt_bias, at::kFloat, {HV}) ||
      !is(a, at::kBFloat16, {L, HV}) || !is(b, at::kBFloat16, {L, HV}) ||
      !scale_of(args[9], &scale))
    Py_RETURN_NONE;
  if (!PyBool_Check(args[12])) Py_RETURN_NONE;
  const bool allocate = args[10] == Py_None && args[11] == Py_None;
  const at::Tensor* output = allocate ? nullptr : plain(args[10]);
  const at::Tensor* new_state = allocate ? nullptr : plain(args[11]);
  if (!allocate && (!is(output, at::kBFloat16, {L, HV, kDim}) ||
                    !is(new_state, at::kFloat, {N, HV, kDim, kDim})))
    Py_RETURN_NONE;
  if (!one_device(q, {k, v, state, A_log, a, dt_bias, b, cu, output, new_state})) Py_RETURN_NONE;
  c10::Stream stream(c10::Stream::DEFAULT, q->device());
  if (!stream_of(q, &stream)) Py_RETURN_NONE;
  if (!allocate) {
    out_ptr<void>(output);                         // before any pointer is compared
    const void* const d = out_ptr<void>(new_state);
    if (state != nullptr && d != state->const_data_ptr() && ranges_overlap(new_state, state))
      Py_RETURN_NONE;
  }
  const int n = static_cast<int>(N), l = static_cast<int>(L), h = static_cast<int>(H),
            hv = static_cast<int>(HV);
  const size_t need = g_workspace(l, n, h, hv);
  if (need == 0) Py_RETURN_NONE;
  at::Tensor out_t, state_t, workspace;
  if (allocate) {
    out_t = at::zeros({L, HV, kDim}, q->options().requires_grad(false));
    state_t = at::empty({N, HV, kDim, kDim}, A_log->options().requires_grad(false));
    output = &out_t;
    new_state = &state_t;
  }
  // The workspace is the current stream's, as the launch is: freed here, its
  // memory is reused in that stream's order.
  workspace = at::empty({static_cast<int64_t>(need + 256)},
                        q->options().dtype(at::kByte).requires_grad(false));
  void* const ws = reinterpret_cast<void*>(
      (reinterpret_cast<uintptr_t>(workspace.data_ptr()) + 255) & ~static_cast<uintptr_t>(255));
  void* const hip_stream = c10::hip::getCurrentHIPStream(q->device().index()).stream();
  const int l2 = args[12] == Py_True;
  // the pointers before the interpreter lock is released: an accessor may throw
  const void *qp = ptr<void>(q), *kp = ptr<void>(k), *vp = ptr<void>(v), *ap = ptr<void>(a),
             *bp = ptr<void>(b);
  const float *sp = ptr<float>(state), *lp = ptr<float>(A_log), *dp = ptr<float>(dt_bias);
  const int32_t* const cp = ptr<int32_t>(cu);
  void* const op = out_ptr<void>(output);
  float* const np = out_ptr<float>(new_state);
  int code;
  Py_BEGIN_ALLOW_THREADS;
  code = g_prefill(qp, kp, vp, sp, lp, ap, dp, bp, cp, scale, op, np, l, n, h, hv, kDim, kDim, l2,
                   ws, need, hip_stream);
  Py_END_ALLOW_THREADS;
  // as the Python path: cu_seqlens may be another stream's tensor
  cu->record_stream(stream);
  if (!allocate) return code_of(code);
  PyObject* const r = PyTuple_New(3);
  if (r == nullptr) return nullptr;
  PyTuple_SET_ITEM(r, 0, code_of(code));
  PyTuple_SET_ITEM(r, 1, THPVariable_Wrap(out_t));
  PyTuple_SET_ITEM(r, 2, THPVariable_Wrap(state_t));
  return r;
  END_HANDLE_TH_ERRORS
}

// decode_run(q, k, v, state, A_log, a, dt_bias, b, scale, use_qk_l2norm):
// (code, output, new_state), both allocated here, or None for the Python path.
PyObject* decode_run(PyObject*, PyObject* const* args, Py_ssize_t nargs) {
  HANDLE_TH_ERRORS
  if (nargs != 10) {
    PyErr_SetString(PyExc_TypeError, "decode_run takes 10 arguments");
    return nullptr;
  }
  const at::Tensor *q = plain(args[0]), *k = plain(args[1]), *v = plain(args[2]);
  if (g_decode == nullptr || q == nullptr || v == nullptr || q->dim() != 4 || v->dim() != 4)
    Py_RETURN_NONE;
  const at::Tensor* state = nullptr;
  if (args[3] != Py_None && (state = plain(args[3])) == nullptr) Py_RETURN_NONE;
  const at::Tensor *A_log = plain(args[4]), *a = plain(args[5]), *dt_bias = plain(args[6]),
                   *b = plain(args[7]);
  const int64_t B = q->size(0), T = q->size(1), H = q->size(2), HV = v->size(2);
  constexpr int64_t kMax = 0x7fffffff;
  if (B < 1 || T < 1 || H <= 0 || HV <= 0 || HV % H != 0 || B > kMax || T > kMax || HV > kMax)
    Py_RETURN_NONE;
  const bool bf16 = state != nullptr && state->scalar_type() == at::kBFloat16;
  auto gate = [&](const at::Tensor* t) {
    return is(t, at::kBFloat16, {B, T, HV}) || (T == 1 && is(t, at::kBFloat16, {B, HV}));
  };
  float scale;
  if (!is(q, at::kBFloat16, {B, T, H, kDim}) || !is(k, at::kBFloat16, {B, T, H, kDim}) ||
      !is(v, at::kBFloat16, {B, T, HV, kDim}) ||
      (state != nullptr &&
       !is(state, bf16 ? at::kBFloat16 : at::kFloat, {B, HV, kDim, kDim})) ||
      !is(A_log, at::kFloat, {HV}) || !is(dt_bias, at::kFloat, {HV}) || !gate(a) || !gate(b) ||
      !scale_of(args[8], &scale) || !PyBool_Check(args[9]) ||
      !one_device(q, {k, v, state, A_log, a, dt_bias, b}))
    Py_RETURN_NONE;
  c10::Stream stream(c10::Stream::DEFAULT, q->device());
  if (!stream_of(q, &stream)) Py_RETURN_NONE;
  const at::Tensor output = at::empty({B, T, HV, kDim}, q->options().requires_grad(false));
  const at::Tensor new_state =
      at::empty({B, HV, kDim, kDim}, (bf16 ? q : A_log)->options().requires_grad(false));
  void* const hip_stream = c10::hip::getCurrentHIPStream(q->device().index()).stream();
  const int l2 = args[9] == Py_True;
  const void *qp = ptr<void>(q), *kp = ptr<void>(k), *vp = ptr<void>(v), *sp = ptr<void>(state),
             *ap = ptr<void>(a), *bp = ptr<void>(b);
  const float *lp = ptr<float>(A_log), *dp = ptr<float>(dt_bias);
  void *const op = out_ptr<void>(&output), *const np = out_ptr<void>(&new_state);
  int code;
  Py_BEGIN_ALLOW_THREADS;
  code = g_decode(qp, kp, vp, sp, lp, ap, dp, bp, scale, op, np, static_cast<int>(B),
                  static_cast<int>(T), static_cast<int>(H), static_cast<int>(HV), kDim, kDim, bf16,
                  l2, hip_stream);
  Py_END_ALLOW_THREADS;
  PyObject* const r = PyTuple_New(3);
  if (r == nullptr) return nullptr;
  PyTuple_SET_ITEM(r, 0, code_of(code));
  PyTuple_SET_ITEM(r, 1, THPVariable_Wrap(output));
  PyTuple_SET_ITEM(r, 2, THPVariable_Wrap(new_state));
  return r;
  END_HANDLE_TH_ERRORS
}

// bind_prefill(gdn_prefill, gdn_prefill_workspace_bytes) and
// bind_decode(gdn_decode_steps): addresses.
PyObject* bind_prefill(PyObject*, PyObject* args) {
  unsigned long long p, w;
  if (!PyArg_ParseTuple(args, "KK", &p, &w)) return nullptr;
  g_prefill = reinterpret_cast<decltype(g_prefill)>(static_cast<uintptr_t>(p));
  g_workspace = reinterpret_cast<decltype(g_workspace)>(static_cast<uintptr_t>(w));
  Py_RETURN_NONE;
}

PyObject* bind_decode(PyObject*, PyObject* args) {
  unsigned long long p;
  if (!PyArg_ParseTuple(args, "K", &p)) return nullptr;
  g_decode = reinterpret_cast<decltype(g_decode)>(static_cast<uintptr_t>(p));
  Py_RETURN_NONE;
}

PyMethodDef kMethods[] = {
    {"prefill", reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)()>(prefill)),
     METH_FASTCALL, nullptr},
    {"decode_run", reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)()>(decode_run)),
     METH_FASTCALL, nullptr},
    {"bind_prefill", bind_prefill, METH_VARARGS, nullptr},
    {"bind_decode", bind_decode, METH_VARARGS, nullptr},
    {nullptr, nullptr, 0, nullptr}};

PyModuleDef kModule = {PyModuleDef_HEAD_INIT, "_gdn_host", nullptr, -1, kMethods};

}  // namespace

// torch_version: the torch that the module was compiled against (its inline
// accessors know that one's object layouts), for the importer to compare.
PyMODINIT_FUNC PyInit__gdn_host(void) {
  PyObject* const m = PyModule_Create(&kModule);
  if (m != nullptr && PyModule_AddStringConstant(m, "torch_version", GDN_TORCH_VERSION) != 0) {
    Py_DECREF(m);
    return nullptr;
  }
  return m;
}
