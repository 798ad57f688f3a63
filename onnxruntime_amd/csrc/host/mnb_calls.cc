// The operators' calls from Python in native code: the module onnxruntime_amd._calls.
//
// One function for each operator: it looks a call over, makes the result, asks for the scratch and enters the C ABI of
// libmnb_mi355x.so, whose entry points it is given as addresses.  A call that is not the plain one (a subclass of Tensor, a wrapper of
// functorch, rows that have to be copied, an input of another type or shape, a torch function mode) returns None before anything is
// launched, and the caller goes through the Python path, which does the same with every check and message.  Errors of the library
// are raised.  Nothing is kept between calls.
//
// Why: products of a few rows are over in 4 to 8 us, and the Python path needs 8.3 to 9.0 us a call, of which 2.0 are torch.empty,
// 0.8 the conversion of sixteen arguments by ctypes, 0.5 the question for the scratch's size and 1.2 checks and attributes; the launch
// itself takes 3.  Now 4.1 to 4.6 us a call: a router of one token 9.0 -> 4.7 to 5.9 us by the host, one row of 4096 x 4096 in fp32 8.4 ->
// 6.7, the projections of a decoder layer 41 to 44 -> 33 (20.7 of the host's).  A call that is declined pays 0.25 us for the attempt (three
// dimensions, 9.5 -> 9.8).
#define PY_SSIZE_T_CLEAN
#include <Python.h>

#include <ATen/PythonTorchFunctionTLS.h>
#include <ATen/ops/empty.h>
#include <c10/hip/HIPStream.h>
#include <torch/csrc/Exceptions.h>
#include <torch/csrc/autograd/python_variable.h>
#include <torch/version.h>

#include <array>
#include <cstring>

#include "mnb_mi355x.h"

namespace {

struct Ref {  // an owned reference
  PyObject* p = nullptr;
  ~Ref() { Py_XDECREF(p); }
};

PyObject* g_workspace = nullptr;  // "_get_workspace"
PyObject* g_device = nullptr;     // "device"

// The arguments of a call by position.  A number that does not convert leaves a Python error behind.
struct Args {
  PyObject* const* v;
  template <class F>
  F fn(int i) const { return reinterpret_cast<F>(PyLong_AsVoidPtr(v[i])); }
  int64_t integer(int i) const { return PyLong_AsLongLong(v[i]); }
};

// The plan of a variant, copied from the object that holds it: it may be replaced, and freed, by another thread during the call.
bool plan_of(PyObject* o, MnbVariantPlan* plan) {
  Py_buffer view;
  if (PyObject_GetBuffer(o, &view, PyBUF_SIMPLE) != 0) return false;
  const bool fits = view.len == (Py_ssize_t)sizeof(*plan);
  if (fits) memcpy(plan, view.buf, sizeof(*plan));
  else PyErr_Format(PyExc_TypeError, "a plan of %zu bytes expected, %zd given", sizeof(*plan), view.len);
  PyBuffer_Release(&view);
  return fits;
}

// A plain strided tensor of the GPU with memory of its own; nullptr: one for the Python path.
const at::Tensor* plain(PyObject* o) {
  if (!THPVariable_CheckExact(o)) return nullptr;
  const at::Tensor& t = THPVariable_Unpack(o);
  if (!t.defined() || !t.is_cuda() || t.layout() != at::kStrided || !t.has_storage() || t.is_conj() || t.is_neg() ||
      t._is_zerotensor() || t.key_set().has_any(c10::python_ks | c10::DispatchKeySet(c10::DispatchKey::Functionalize)))
    return nullptr;
  return &t;
}

bool type_of(int64_t dtype, at::ScalarType* type) {
  switch (dtype) {
    case 1: *type = at::kFloat; return true;
    case 10: *type = at::kHalf; return true;
    case 16: *type = at::kBFloat16; return true;
    default: return false;
  }
}

// Activations: rows of K adjacent elements, at least one.
const at::Tensor* rows(PyObject* o, int64_t K, int64_t dtype) {
  const at::Tensor* a = plain(o);
  at::ScalarType type;
  if (a == nullptr || !type_of(dtype, &type) || a->scalar_type() != type || a->dim() != 2 || a->size(1) != K ||
      a->stride(1) != 1 || a->size(0) <= 0)
    return nullptr;
  return a;
}

void* stream_of(const at::Tensor& a) { return c10::hip::getCurrentHIPStream(a.device().index()).stream(); }

// The operator's own scratch on the stream: op._get_workspace(device, bytes, stream).  False with a Python error set.
bool scratch(PyObject* op, PyObject* a, size_t bytes, void* stream, Ref& held, void** ptr) {
  *ptr = nullptr;
  if (bytes == 0) return true;
  Ref device, size, handle;
  device.p = PyObject_GetAttr(a, g_device);
  size.p = PyLong_FromSize_t(bytes);
  handle.p = PyLong_FromVoidPtr(stream);
  if (!device.p || !size.p || !handle.p) return false;
  PyObject* const args[] = {op, device.p, size.p, handle.p};
  held.p = PyObject_VectorcallMethod(g_workspace, args, 4 | PY_VECTORCALL_ARGUMENTS_OFFSET, nullptr);
  if (!held.p) return false;
  if (held.p != Py_None) *ptr = THPVariable_Unpack(held.p).data_ptr();
  return true;
}

// What the entry point has reported, raised as the Python path raises it.  (None would have the call made again: its first launches may
// be under way or recorded in a graph by then, and an error that hipGetLastError has handed out once is not there a second time.)
PyObject* failed(int rc) {
  Ref lib;
  lib.p = PyImport_ImportModule("onnxruntime_amd._lib");
  return lib.p ? PyObject_CallMethod(lib.p, "check", "i", rc) : nullptr;
}

bool expect(Py_ssize_t n, Py_ssize_t want) {
  if (n == want) return true;
  PyErr_Format(PyExc_TypeError, "%zd arguments expected, %zd given", want, n);
  return false;
}

// A bias of N values, or none.
bool bias_of(PyObject* o, int64_t N, void** ptr) {
  *ptr = nullptr;
  if (o == Py_None) return true;
  const at::Tensor* t = plain(o);
  if (t == nullptr || t->dim() != 1 || t->size(0) != N) return false;
  *ptr = t->data_ptr();
  return true;
}

// (gemm, workspace_size, N, K, bits, block_size, has_zero_points, dtype, a, packed, bias, op) -> Y or None
PyObject* linear(PyObject*, PyObject* const* v, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  if (!expect(n, 12)) return nullptr;
  const Args args{v};
  const auto gemm = args.fn<decltype(&MnbGemm)>(0);
  const auto need = args.fn<decltype(&MnbGemmWorkspaceSize)>(1);
  const int64_t N = args.integer(2), K = args.integer(3);
  const int bits = (int)args.integer(4), block = (int)args.integer(5), zp = PyObject_IsTrue(v[6]), dtype = (int)args.integer(7);
  if (PyErr_Occurred()) return nullptr;
  const at::Tensor *a = rows(v[8], K, dtype), *packed = plain(v[9]);
  void* bias;
  if (!gemm || !need || N <= 0 || a == nullptr || packed == nullptr || !bias_of(v[10], N, &bias) || at::impl::torch_function_mode_enabled())
    Py_RETURN_NONE;
  const int64_t M = a->size(0);
  at::Tensor y = at::empty({M, N}, a->options());
  void* const s = stream_of(*a);
  const size_t bytes = need((size_t)M, (size_t)N, (size_t)K, bits, block, zp, dtype);
  Ref held;
  void* ws;
  if (!scratch(v[11], v[8], bytes, s, held, &ws)) return nullptr;
  const void *pa = a->data_ptr(), *pw = packed->data_ptr();
  const size_t lda = M > 1 ? (size_t)a->stride(0) : (size_t)K;
  void* const py = y.data_ptr();
  int rc;
  Py_BEGIN_ALLOW_THREADS
  rc = gemm((size_t)M, (size_t)N, (size_t)K, bits, block, zp, dtype, pa, lda, pw, bias, py, (size_t)N, ws, bytes, s);
  Py_END_ALLOW_THREADS
  if (rc != MNB_OK) return failed(rc);
  return THPVariable_Wrap(std::move(y));
  END_HANDLE_TH_ERRORS
}

// (gemm, workspace_size, plan, N, K, dtype, a, packed, bias, op) -> Y or None
PyObject* variant(PyObject*, PyObject* const* v, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  if (!expect(n, 10)) return nullptr;
  const Args args{v};
  const auto gemm = args.fn<decltype(&MnbVariantGemm)>(0);
  const auto need = args.fn<decltype(&MnbVariantGemmWorkspaceSize)>(1);
  const int64_t N = args.integer(3), K = args.integer(4), dtype = args.integer(5);
  MnbVariantPlan plan;
  if (PyErr_Occurred() || !plan_of(v[2], &plan)) return nullptr;
  const at::Tensor *a = rows(v[6], K, dtype), *packed = plain(v[7]);
  void* bias;
  if (!gemm || !need || N <= 0 || a == nullptr || packed == nullptr || !bias_of(v[8], N, &bias) ||
      at::impl::torch_function_mode_enabled())
    Py_RETURN_NONE;
  const int64_t M = a->size(0);
  at::Tensor y = at::empty({M, N}, a->options());
  void* const s = stream_of(*a);
  const size_t bytes = need(&plan, (size_t)M);
  Ref held;
  void* ws;
  if (!scratch(v[9], v[6], bytes, s, held, &ws)) return nullptr;
  const void *pa = a->data_ptr(), *pw = packed->data_ptr();
  const size_t lda = M > 1 ? (size_t)a->stride(0) : (size_t)K;
  void* const py = y.data_ptr();
  int rc;
  Py_BEGIN_ALLOW_THREADS
  rc = gemm(&plan, (size_t)M, pa, lda, pw, bias, py, (size_t)N, ws, bytes, s);
  Py_END_ALLOW_THREADS
  if (rc != MNB_OK) return failed(rc);
  return THPVariable_Wrap(std::move(y));
  END_HANDLE_TH_ERRORS
}

// The normalisation in front of a fused operator.
struct Prologue {
  MnbNormPrologue norm{};
  bool has = false;
  at::Tensor sum;  // input_skip_bias_sum, where it is wanted
};

// False: a call for the Python path.
bool prologue(const at::Tensor& a, int64_t K, PyObject* skip_o, PyObject* norm_o, bool want_sum, double epsilon, Prologue* out) {
  if (norm_o == Py_None) return skip_o == Py_None && !want_sum;
  const at::Tensor* norm = plain(norm_o);
  if (norm == nullptr || norm->dim() != 1 || norm->size(0) != K || !norm->is_contiguous()) return false;
  out->has = true;
  out->norm.norm_scale_dev = norm->data_ptr();
  out->norm.epsilon = (float)epsilon;
  if (skip_o == Py_None) return !want_sum;
  const at::Tensor* skip = plain(skip_o);
  if (skip == nullptr || skip->dim() != 2 || skip->size(1) != K || skip->size(0) <= 0 || !skip->is_contiguous() ||
      a.size(0) % skip->size(0) != 0)
    return false;
  out->norm.skip_dev = skip->data_ptr();
  out->norm.ld_skip = (size_t)K;
  out->norm.skip_rows = (size_t)skip->size(0);
  if (want_sum) {
    out->sum = at::empty({a.size(0), K}, a.options());
    out->norm.skip_sum_dev = out->sum.data_ptr();
    out->norm.ld_skip_sum = (size_t)K;
  }
  return true;
}

// (gemm, workspace_size, N, K, bits, block_size, dtype, epsilon, a, packed, skip, norm_scale, want_skip_sum, op) -> Y, (Y, sum) or None
PyObject* mlp(PyObject*, PyObject* const* v, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  if (!expect(n, 14)) return nullptr;
  const Args args{v};
  const auto gemm = args.fn<decltype(&MnbMlpGemm)>(0);
  const auto need = args.fn<decltype(&MnbMlpWorkspaceSize)>(1);
  const int64_t N = args.integer(2), K = args.integer(3);
  const int bits = (int)args.integer(4), block = (int)args.integer(5), dtype = (int)args.integer(6);
  const double epsilon = PyFloat_AsDouble(v[7]);
  const int want = PyObject_IsTrue(v[12]);
  if (PyErr_Occurred()) return nullptr;
  const at::Tensor *a = rows(v[8], K, dtype), *packed = plain(v[9]);
  Prologue pro;
  if (!gemm || !need || N <= 0 || a == nullptr || packed == nullptr || at::impl::torch_function_mode_enabled() ||
      !prologue(*a, K, v[10], v[11], want != 0, epsilon, &pro))
    Py_RETURN_NONE;
  const int64_t M = a->size(0);
  at::Tensor y = at::empty({M, N}, a->options());
  void* const s = stream_of(*a);
  const size_t bytes = need((size_t)M, (size_t)N, (size_t)K, bits, block, dtype, pro.has);
  Ref held;
  void* ws;
  if (!scratch(v[13], v[8], bytes, s, held, &ws)) return nullptr;
  const void *pa = a->data_ptr(), *pw = packed->data_ptr();
  const size_t lda = M > 1 ? (size_t)a->stride(0) : (size_t)K;
  void* const py = y.data_ptr();
  int rc;
  Py_BEGIN_ALLOW_THREADS
  rc = gemm((size_t)M, (size_t)N, (size_t)K, bits, block, dtype, pa, lda, pro.has ? &pro.norm : nullptr, pw, 0, py, (size_t)N, ws,
            bytes, s);
  Py_END_ALLOW_THREADS
  if (rc != MNB_OK) return failed(rc);
  Ref first;
  first.p = THPVariable_Wrap(std::move(y));
  if (!first.p) return nullptr;
  if (!want) return std::exchange(first.p, nullptr);
  Ref second;
  second.p = THPVariable_Wrap(std::move(pro.sum));
  return second.p ? PyTuple_Pack(2, first.p, second.p) : nullptr;
  END_HANDLE_TH_ERRORS
}

// (gemm, workspace_size, Nq, Nkv, K, bits, block_size, dtype, epsilon, a, packed, skip, norm_scale, want_skip_sum, op)
// -> (Q, K, V), (Q, K, V, sum) or None
PyObject* qkv(PyObject*, PyObject* const* v, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  if (!expect(n, 15)) return nullptr;
  const Args args{v};
  const auto gemm = args.fn<decltype(&MnbQkvGemm)>(0);
  const auto need = args.fn<decltype(&MnbQkvWorkspaceSize)>(1);
  const int64_t Nq = args.integer(2), Nkv = args.integer(3), K = args.integer(4);
  const int bits = (int)args.integer(5), block = (int)args.integer(6), dtype = (int)args.integer(7);
  const double epsilon = PyFloat_AsDouble(v[8]);
  const int want = PyObject_IsTrue(v[13]);
  if (PyErr_Occurred()) return nullptr;
  const at::Tensor *a = rows(v[9], K, dtype), *packed = plain(v[10]);
  Prologue pro;
  if (!gemm || !need || Nq <= 0 || Nkv <= 0 || a == nullptr || packed == nullptr || at::impl::torch_function_mode_enabled() ||
      !prologue(*a, K, v[11], v[12], want != 0, epsilon, &pro))
    Py_RETURN_NONE;
  const int64_t M = a->size(0);
  std::array<at::Tensor, 3> out;
  for (int i = 0; i < 3; ++i) out[i] = at::empty({M, i == 0 ? Nq : Nkv}, a->options());
  void* const s = stream_of(*a);
  const size_t bytes = need((size_t)M, (size_t)Nq, (size_t)Nkv, (size_t)K, bits, block, dtype, pro.has);
  Ref held;
  void* ws;
  if (!scratch(v[14], v[9], bytes, s, held, &ws)) return nullptr;
  const void *pa = a->data_ptr(), *pw = packed->data_ptr();
  const size_t lda = M > 1 ? (size_t)a->stride(0) : (size_t)K;
  void *const o0 = out[0].data_ptr(), *const o1 = out[1].data_ptr(), *const o2 = out[2].data_ptr();
  int rc;
  Py_BEGIN_ALLOW_THREADS
  rc = gemm((size_t)M, (size_t)Nq, (size_t)Nkv, (size_t)K, bits, block, dtype, pa, lda, pro.has ? &pro.norm : nullptr, pw, o0,
            (size_t)Nq, o1, (size_t)Nkv, o2, (size_t)Nkv, ws, bytes, s);
  Py_END_ALLOW_THREADS
  if (rc != MNB_OK) return failed(rc);
  Ref result;
  result.p = PyTuple_New(want ? 4 : 3);
  if (!result.p) return nullptr;
  for (int i = 0; i < (want ? 4 : 3); ++i) {
    PyObject* const t = THPVariable_Wrap(i < 3 ? std::move(out[i]) : std::move(pro.sum));
    if (!t) return nullptr;
    PyTuple_SET_ITEM(result.p, i, t);
  }
  return std::exchange(result.p, nullptr);
  END_HANDLE_TH_ERRORS
}

// (quantize, dtype, bits, block_size, symmetric, w) -> (B, scales, zero points or None) or None
PyObject* quantize(PyObject*, PyObject* const* v, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  if (!expect(n, 6)) return nullptr;
  const Args args{v};
  const auto run = args.fn<decltype(&MnbQuantizeBlockwise)>(0);
  const int64_t dtype = args.integer(1), bits = args.integer(2), block = args.integer(3);
  const int symmetric = PyObject_IsTrue(v[4]);
  if (PyErr_Occurred()) return nullptr;
  at::ScalarType type;
  const at::Tensor* w = plain(v[5]);
  if (!run || !type_of(dtype, &type) || w == nullptr || w->scalar_type() != type || w->dim() != 2 || w->size(0) <= 0 || w->size(1) <= 0 ||
      w->stride(1) != 1 || (bits != 2 && bits != 4 && bits != 8) || block <= 0 || block > 256 || at::impl::torch_function_mode_enabled())
    Py_RETURN_NONE;
  const int64_t K = w->size(0), N = w->size(1), blocks = (K + block - 1) / block;
  const at::TensorOptions bytes = w->options().dtype(at::kByte);
  at::Tensor b = at::empty({N, blocks, block * bits / 8}, bytes), scales = at::empty({N, blocks}, w->options()), zp;
  if (!symmetric) zp = at::empty({N, (blocks * bits + 7) / 8}, bytes);
  void *const pb = b.data_ptr(), *const ps = scales.data_ptr(), *const pz = symmetric ? nullptr : zp.data_ptr();
  const void* const pw = w->data_ptr();
  const size_t ld = K > 1 ? (size_t)w->stride(0) : (size_t)N;
  void* const s = stream_of(*w);
  int rc;
  Py_BEGIN_ALLOW_THREADS
  rc = run(pb, ps, pz, pw, (int)block, (int)bits, (size_t)K, (size_t)N, ld, (int)dtype, s);
  Py_END_ALLOW_THREADS
  if (rc != MNB_OK) return failed(rc);
  Ref first, second, third;
  first.p = THPVariable_Wrap(std::move(b));
  second.p = THPVariable_Wrap(std::move(scales));
  if (symmetric) Py_INCREF(third.p = Py_None);
  else third.p = THPVariable_Wrap(std::move(zp));
  return first.p && second.p && third.p ? PyTuple_Pack(3, first.p, second.p, third.p) : nullptr;
  END_HANDLE_TH_ERRORS
}

#define MNB_METHOD(f) {#f, reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)()>(f)), METH_FASTCALL, nullptr}
PyMethodDef g_methods[] = {MNB_METHOD(linear), MNB_METHOD(variant), MNB_METHOD(mlp), MNB_METHOD(qkv), MNB_METHOD(quantize),
                            {nullptr, nullptr, 0, nullptr}};
PyModuleDef g_module = {PyModuleDef_HEAD_INIT, "_calls", nullptr, -1, g_methods, nullptr, nullptr, nullptr, nullptr};

}  // namespace

PyMODINIT_FUNC PyInit__calls() {
  g_workspace = PyUnicode_InternFromString("_get_workspace");
  g_device = PyUnicode_InternFromString("device");
  PyObject* const module = g_workspace && g_device ? PyModule_Create(&g_module) : nullptr;
  if (module && PyModule_AddStringConstant(module, "TORCH_VERSION", TORCH_VERSION) != 0) {
    Py_DECREF(module);
    return nullptr;
  }
  return module;
}
