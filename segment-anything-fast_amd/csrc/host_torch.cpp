// The per-call host work of the hot entry points as native code: reading shapes, strides and
// pointers out of torch tensors, allocating outputs and workspaces and calling the C ABI.  Done in
// Python (ops.py) this costs 20-30 us per call, several times what a small call runs on the GPU
// (a Linear over 7 tokens: 7 us of kernels); here it is 2-3 us plus the launches.
//
// Every function returns None for a call it does not cover - a CPU tensor, another type, a strided
// view, a shape the C ABI refuses, a call that somebody watches (plain_call) - and the caller then takes
// the Python route, whose checks and error texts stay the one definition of what is accepted.
//
// The C ABI is reached through pointers that bind() receives from the ctypes handle, so that one
// copy of libsamfast.so serves both (also when SAMFAST_LIB names another file).
#define PY_SSIZE_T_CLEAN
#include <Python.h>

#include <ATen/ATen.h>
#include <ATen/hip/EmptyTensor.h>
#include <ATen/PythonTorchFunctionTLS.h>
#include <c10/core/GradMode.h>
#include <c10/core/impl/LocalDispatchKeySet.h>
#include <c10/hip/HIPFunctions.h>
#include <c10/hip/HIPStream.h>
#include <torch/csrc/PyInterpreter.h>
#include <torch/csrc/autograd/python_variable.h>

#include "samfast.h"

namespace {

decltype(&samfast_linear_i8) p_linear_i8;
decltype(&samfast_linear_i8_workspace) p_linear_i8_workspace;
decltype(&samfast_linear_i8_one_launch) p_linear_i8_one_launch;
decltype(&samfast_linear_i8_sparse24) p_linear_i8_sparse24;
decltype(&samfast_attn_relpos_bias_fwd) p_attn_bias;

struct Bound { const char* name; void** slot; };
const Bound kBound[] = {
    {"samfast_linear_i8", reinterpret_cast<void**>(&p_linear_i8)},
    {"samfast_linear_i8_workspace", reinterpret_cast<void**>(&p_linear_i8_workspace)},
    {"samfast_linear_i8_one_launch", reinterpret_cast<void**>(&p_linear_i8_one_launch)},
    {"samfast_linear_i8_sparse24", reinterpret_cast<void**>(&p_linear_i8_sparse24)},
    {"samfast_attn_relpos_bias_fwd", reinterpret_cast<void**>(&p_attn_bias)},
};

PyObject* device_context = nullptr;  // the mode of `with torch.device(..)` and torch.set_default_device, set by bind()

// Function modes see calls in Python; the one that only gives factory functions their device need not see these.
bool function_mode_watches() {
  using at::impl::PythonTorchFunctionTLS;
  if (!at::impl::torch_function_mode_enabled()) return false;
  for (int64_t i = 0; i < PythonTorchFunctionTLS::stack_len(); ++i) {
    PyObject* mode = PythonTorchFunctionTLS::get_stack_at(i)->ptr(getPyInterpreter());
    if (reinterpret_cast<PyObject*>(Py_TYPE(mode)) != device_context) return true;
  }
  return false;
}

// Whether nobody but the kernels has to see this thread's calls: a launch on raw pointers passes by tracers,
// functional transforms (vmap, grad, functionalization) and dispatch and function modes.  All but the last stand as
// dispatch keys that the thread has included beyond the default ones.
bool plain_call() {
  return (c10::impl::tls_local_dispatch_key_set().included_ | c10::default_included_set) == c10::default_included_set &&
         !function_mode_watches();
}

// A tensor that is its memory and nothing more: no wrapper of a transform, subclass, conjugate or negative view, sparse or
// nested layout, no forward-mode tangent.
bool plain_tensor(const at::Tensor& t) {
  constexpr c10::DispatchKeySet expected = c10::DispatchKeySet(
      {c10::DispatchKey::Dense, c10::DispatchKey::ADInplaceOrView, c10::DispatchKey::AutogradFunctionality,
       c10::DispatchKey::AutocastCUDA, c10::DispatchKey::AutocastCPU});
  const c10::DispatchKeySet keys(c10::DispatchKeySet::RAW, t.key_set().raw_repr() & ~static_cast<uint64_t>(c10::full_backend_mask));
  return (keys | expected) == expected && !t._fw_grad(/*level=*/0).defined();
}

// a plain strided GPU tensor on the current device (the launches go to its current stream)
bool on_current_gpu(const at::Tensor& t, c10::DeviceIndex dev) {
  return t.defined() && t.is_cuda() && t.layout() == at::kStrided && t.device().index() == dev && plain_tensor(t);
}

// (exactly a Tensor or Parameter: a subclass may override what happens to it)
const at::Tensor* tensor_arg(PyObject* o) { return THPVariable_CheckExact(o) ? &THPVariable_Unpack(o) : nullptr; }

void* stream_of(c10::DeviceIndex dev) { return c10::hip::getCurrentHIPStream(dev).stream(); }

const void* ptr(const at::Tensor& t) { return t.const_data_ptr(); }

// at::empty without its way through the dispatcher (0.72 -> 0.49 us): whoever has to see the allocation there is one of those whose
// calls are declined above, and what is allocated here is written in full.
at::Tensor new_tensor(at::IntArrayRef sizes, at::ScalarType type, c10::DeviceIndex dev) {
  return at::detail::empty_cuda(sizes, type, c10::Device(c10::kCUDA, dev), std::nullopt);
}

// What the dense and the sparse Linear share: x is (..., K) contiguous bf16, sw_bits / bias_bits are
// the fp32 scales and bias as the modules hold them (int32 bit patterns).  Fills y and the workspace.
struct LinearCall {
  const at::Tensor *x, *sw, *bias;
  int64_t M, N, K;
  at::Tensor y, work;
  const float* sw_ptr() const { return static_cast<const float*>(ptr(*sw)); }
  const float* bias_ptr() const { return bias ? static_cast<const float*>(ptr(*bias)) : nullptr; }
  void* work_ptr() const { return work.defined() ? work.data_ptr() : nullptr; }

  bool accept(c10::DeviceIndex dev) const {
    return on_current_gpu(*x, dev) && on_current_gpu(*sw, dev) && (!bias || on_current_gpu(*bias, dev)) &&
           x->scalar_type() == at::kBFloat16 && x->dim() >= 1 && x->is_contiguous() && x->numel() > 0 &&
           K > 0 && x->size(-1) == K && N <= INT32_MAX && K <= INT32_MAX &&
           sw->scalar_type() == at::kInt && sw->is_contiguous() && sw->numel() == N &&
           (!bias || (bias->scalar_type() == at::kInt && bias->is_contiguous() && bias->numel() == N));
  }
  void allocate(int64_t need, c10::DeviceIndex dev) {
    c10::SmallVector<int64_t, 5> shape(x->sizes().begin(), x->sizes().end());
    shape.back() = N;
    y = new_tensor(shape, at::kBFloat16, dev);
    if (need > 0) work = new_tensor({need}, at::kByte, dev);
  }
};

// bytes of workspace of a call whose output is its own
int64_t workspace(const LinearCall& c, int layout) {
  const int N = static_cast<int>(c.N), K = static_cast<int>(c.K);
  return p_linear_i8_one_launch(c.M, N, K, layout) == 1 ? 0 : p_linear_i8_workspace(c.M, N, K, layout);
}

// The entry of a module's buffers by that name, borrowed; None where there is none
PyObject* buffer(PyObject* buffers, PyObject* name) {
  PyObject* v = PyDict_GetItemWithError(buffers, name);
  if (!v && PyErr_Occurred()) throw python_error();
  return v ? v : Py_None;
}
PyObject* name_of(const char* s) { return PyUnicode_InternFromString(s); }

// linear(x, wq, layout, sw_bits, bias_bits or None): the whole int8 Linear on bf16 rows.
// wq is (N, K), or (K/64, N, 64) for layout 1.
PyObject* host_linear(PyObject*, PyObject* const* args, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  if (n != 5 || !plain_call()) Py_RETURN_NONE;
  const at::Tensor* wq = tensor_arg(args[1]);
  const int layout = static_cast<int>(PyLong_AsLong(args[2]));
  const bool kb = layout == SAMFAST_LAYOUT_KB64;
  LinearCall c = {tensor_arg(args[0]), tensor_arg(args[3]), tensor_arg(args[4])};
  if (!c.x || !c.x->is_cuda() || !wq || !c.sw || (args[4] != Py_None && !c.bias)) Py_RETURN_NONE;
  const c10::DeviceIndex dev = c10::hip::current_device();
  if (!on_current_gpu(*wq, dev) || wq->scalar_type() != at::kChar || wq->dim() != (kb ? 3 : 2) || !wq->is_contiguous()) Py_RETURN_NONE;
  c.N = wq->size(kb ? 1 : 0);
  c.K = kb ? wq->size(0) * 64 : wq->size(1);
  if (!c.accept(dev)) Py_RETURN_NONE;
  c.M = c.x->numel() / c.K;
  const int64_t need = workspace(c, layout);
  if (need < 0) Py_RETURN_NONE;
  c.allocate(need, dev);
  const int rc = p_linear_i8(ptr(*c.x), c.K, static_cast<const int8_t*>(ptr(*wq)), c.sw_ptr(), c.bias_ptr(), c.y.data_ptr(), c.N,
                             c.work_ptr(), c.M, static_cast<int>(c.N), static_cast<int>(c.K), SAMFAST_BF16, layout, stream_of(dev));
  if (rc != SAMFAST_OK) Py_RETURN_NONE;
  return THPVariable_Wrap(std::move(c.y));
  END_HANDLE_TH_ERRORS
}

// sparse_linear(x, wc, widx, sw_bits, bias_bits or None): the same with the packed 2:4 weight
PyObject* host_sparse_linear(PyObject*, PyObject* const* args, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  if (n != 5 || !plain_call()) Py_RETURN_NONE;
  const at::Tensor *wc = tensor_arg(args[1]), *widx = tensor_arg(args[2]);
  LinearCall c = {tensor_arg(args[0]), tensor_arg(args[3]), tensor_arg(args[4])};
  if (!c.x || !c.x->is_cuda() || !wc || !widx || !c.sw || (args[4] != Py_None && !c.bias)) Py_RETURN_NONE;
  const c10::DeviceIndex dev = c10::hip::current_device();
  if (!on_current_gpu(*wc, dev) || !on_current_gpu(*widx, dev) || wc->scalar_type() != at::kChar || widx->scalar_type() != at::kInt ||
      wc->dim() != 3 || widx->dim() != 3 || !wc->is_contiguous() || !widx->is_contiguous() || wc->size(2) != 32 ||
      widx->size(0) != wc->size(0) || widx->size(1) != wc->size(1) || widx->size(2) != 2)
    Py_RETURN_NONE;
  c.N = wc->size(1);
  c.K = wc->size(0) * 64;
  if (!c.accept(dev)) Py_RETURN_NONE;
  c.M = c.x->numel() / c.K;
  const int64_t need = workspace(c, SAMFAST_LAYOUT_SPARSE24);
  if (need < 0) Py_RETURN_NONE;
  c.allocate(need, dev);
  const int rc = p_linear_i8_sparse24(ptr(*c.x), c.K, static_cast<const int8_t*>(ptr(*wc)), static_cast<const int32_t*>(ptr(*widx)),
                                      c.sw_ptr(), c.bias_ptr(), c.y.data_ptr(), c.N, c.work_ptr(), c.M, static_cast<int>(c.N),
                                      static_cast<int>(c.K), SAMFAST_BF16, stream_of(dev));
  if (rc != SAMFAST_OK) Py_RETURN_NONE;
  return THPVariable_Wrap(std::move(c.y));
  END_HANDLE_TH_ERRORS
}

// module_linear(x, buffers), module_sparse_linear(x, buffers): the same with the buffers of the module as they stand
PyObject* host_module_linear(PyObject* self, PyObject* const* args, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  static PyObject *const wq = name_of("wq"), *const sw = name_of("sw_bits"), *const bias = name_of("bias_bits"), *const layout = PyLong_FromLong(SAMFAST_LAYOUT_ROWMAJOR);
  if (n != 2 || !PyDict_Check(args[1])) Py_RETURN_NONE;
  PyObject* const call[5] = {args[0], buffer(args[1], wq), layout, buffer(args[1], sw), buffer(args[1], bias)};
  return host_linear(self, call, 5);
  END_HANDLE_TH_ERRORS
}
PyObject* host_module_sparse_linear(PyObject* self, PyObject* const* args, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  static PyObject *const wc = name_of("wc"), *const widx = name_of("widx"), *const sw = name_of("sw_bits"), *const bias = name_of("bias_bits");
  if (n != 2 || !PyDict_Check(args[1])) Py_RETURN_NONE;
  PyObject* const call[5] = {args[0], buffer(args[1], wc), buffer(args[1], widx), buffer(args[1], sw), buffer(args[1], bias)};
  return host_sparse_linear(self, call, 5);
  END_HANDLE_TH_ERRORS
}

// attention(q, k, v, rel_h (B, nH, N, gh, 1), rel_w (B, nH, N, 1, gw), scale): attention with the
// caller's bias factors, read through their strides; returns a contiguous (B, nH, N, hd) tensor
PyObject* host_attention(PyObject*, PyObject* const* args, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  if (n != 6 || !plain_call()) Py_RETURN_NONE;
  const at::Tensor* t[5];
  const c10::DeviceIndex dev = c10::hip::current_device();
  for (int i = 0; i < 5; ++i) {
    t[i] = tensor_arg(args[i]);
    if (!t[i] || !on_current_gpu(*t[i], dev) || t[i]->dim() != (i < 3 ? 4 : 5) || t[i]->scalar_type() != t[0]->scalar_type()) Py_RETURN_NONE;
    if (t[i]->requires_grad() && c10::GradMode::is_enabled()) Py_RETURN_NONE;
  }
  const at::Tensor &q = *t[0], &k = *t[1], &v = *t[2], &rh = *t[3], &rw = *t[4];
  const int64_t B = q.size(0), nH = q.size(1), N = q.size(2), hd = q.size(3), gh = rh.size(3), gw = rw.size(4);
  const bool half = q.scalar_type() == at::kBFloat16 || q.scalar_type() == at::kHalf;
  if (!half || k.sizes() != q.sizes() || v.sizes() != q.sizes() || B == 0 || B > INT32_MAX || nH > INT32_MAX || hd > 128 || gh > 64 || gw > 64 || gh * gw != N)
    Py_RETURN_NONE;
  for (const at::Tensor* b : {&rh, &rw})
    if (b->size(0) != B || b->size(1) != nH || b->size(2) != N) Py_RETURN_NONE;
  if (rh.size(4) != 1 || rw.size(3) != 1 || q.stride(3) != 1 || k.stride(3) != 1 || v.stride(3) != 1 || rh.stride(3) != 1 || rw.stride(4) != 1)
    Py_RETURN_NONE;
  const double scale = PyFloat_AsDouble(args[5]);
  at::Tensor out = new_tensor({B, nH, N, hd}, q.scalar_type(), dev);
  const int rc = p_attn_bias(ptr(q), ptr(k), ptr(v), ptr(rh), ptr(rw), out.data_ptr(), static_cast<int>(B), static_cast<int>(nH),
                             static_cast<int>(gh), static_cast<int>(gw), static_cast<int>(hd), q.stride(0), q.stride(1), q.stride(2),
                             k.stride(0), k.stride(1), k.stride(2), v.stride(0), v.stride(1), v.stride(2), nH * N * hd, N * hd, hd,
                             rh.stride(0), rh.stride(1), rh.stride(2), rw.stride(0), rw.stride(1), rw.stride(2),
                             q.scalar_type() == at::kHalf ? SAMFAST_F16 : SAMFAST_BF16, static_cast<float>(scale), stream_of(dev));
  if (rc != SAMFAST_OK) Py_RETURN_NONE;
  return THPVariable_Wrap(std::move(out));
  END_HANDLE_TH_ERRORS
}

// plain(tensor): whether a launch that only the kernels see may stand for operations on this tensor
PyObject* host_plain(PyObject*, PyObject* arg) {
  const at::Tensor* t = tensor_arg(arg);
  return PyBool_FromLong(t && plain_call() && plain_tensor(*t));
}

// bind({name: address}): the C ABI functions used above
PyObject* host_bind(PyObject*, PyObject* table) {
  for (const Bound& b : kBound) {
    PyObject* v = PyDict_GetItemString(table, b.name);  // borrowed
    if (!v) return PyErr_Format(PyExc_KeyError, "samfast: %s is not in the table", b.name);
    void* p = PyLong_AsVoidPtr(v);
    if (!p) return PyErr_Occurred() ? nullptr : PyErr_Format(PyExc_ValueError, "samfast: %s has no address", b.name);
    *b.slot = p;
  }
  if (!device_context) {
    PyObject* module = PyImport_ImportModule("torch.utils._device");
    if (!module) return nullptr;
    device_context = PyObject_GetAttrString(module, "DeviceContext");  // kept
    Py_DECREF(module);
    if (!device_context) return nullptr;
  }
  Py_RETURN_NONE;
}

PyObject* host_bound_names(PyObject*, PyObject*) {
  PyObject* out = PyList_New(0);
  for (const Bound& b : kBound) {
    PyObject* s = PyUnicode_FromString(b.name);
    PyList_Append(out, s);
    Py_DECREF(s);
  }
  return out;
}

PyCFunction fastcall(PyObject* (*f)(PyObject*, PyObject* const*, Py_ssize_t)) {
  return reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)()>(f));
}
PyMethodDef kMethods[] = {
    {"bind", host_bind, METH_O, nullptr},
    {"bound_names", host_bound_names, METH_NOARGS, nullptr},
    {"plain", host_plain, METH_O, nullptr},
    {"linear", fastcall(host_linear), METH_FASTCALL, nullptr},
    {"sparse_linear", fastcall(host_sparse_linear), METH_FASTCALL, nullptr},
    {"module_linear", fastcall(host_module_linear), METH_FASTCALL, nullptr},
    {"module_sparse_linear", fastcall(host_module_sparse_linear), METH_FASTCALL, nullptr},
    {"attention", fastcall(host_attention), METH_FASTCALL, nullptr},
    {nullptr, nullptr, 0, nullptr},
};
PyModuleDef kModule = {PyModuleDef_HEAD_INIT, "_samfast_host", nullptr, -1, kMethods, nullptr, nullptr, nullptr, nullptr};

}  // namespace

PyMODINIT_FUNC PyInit__samfast_host() { return PyModule_Create(&kModule); }
