// The host side of a small call in one native function each: what bounds a projection of one or a few rows, and the
// torch op, is not the GPU but the way to its launches.  us on the host a call of 4096x4096, one row: 20.7 through
// ctypes, of which checks of eight tensors 3.5, two allocations 3.4 and the marshalling of twenty arguments 2; 14.7 here.  (The
// op 11.9 and 7.5.)
//
// A function takes a call whose operands are ordinary tensors that fit, and returns None for any other: the Python
// wrapper then looks at its operands one by one and raises, copies or goes another way.  Nothing is kept
// between calls but the addresses of the library's entry points (bind).
#define PY_SSIZE_T_CLEAN
#include <Python.h>

#include <ATen/core/Tensor.h>
#include <ATen/ops/empty.h>
#include <c10/core/impl/TorchDispatchModeTLS.h>
#include <c10/core/impl/VirtualGuardImpl.h>
#include <torch/csrc/autograd/python_variable.h>

#include "../../include/qtip_hip.h"

namespace {

decltype(&qtip_linear) run_linear = nullptr, run_linear_long = nullptr;
decltype(&qtip_linear_workspace_bytes) linear_bytes = nullptr, linear_long_bytes = nullptr;
decltype(&qtip_decompress_matvec) run_matvec = nullptr;
decltype(&qtip_linear_rows) run_rows = nullptr;

// a tensor that a launch can be given: strided, contiguous GPU memory behind no wrapper (batches, fake or traced tensors)
const at::Tensor* plain(PyObject* o, at::ScalarType type, int64_t numel) {
  if (!THPVariable_Check(o)) return nullptr;
  const at::Tensor& t = THPVariable_Unpack(o);
  constexpr c10::DispatchKeySet wrappers({c10::DispatchKey::Python, c10::DispatchKey::FuncTorchBatched,
                                          c10::DispatchKey::FuncTorchGradWrapper, c10::DispatchKey::Functionalize});
  if (!t.defined() || !t.is_cuda() || t.layout() != at::kStrided || t.key_set().has_any(wrappers) || t.scalar_type() != type ||
      !t.has_storage() || !t.is_contiguous() || t.numel() != numel)
    return nullptr;
  return &t;
}

// packed words in one of the types that they come in
const at::Tensor* packed_words(PyObject* o, int64_t bytes) {
  if (!THPVariable_Check(o)) return nullptr;
  const at::ScalarType type = THPVariable_Unpack(o).scalar_type();
  const bool ok = type == at::kShort || type == at::kUInt16 || type == at::kInt || type == at::kByte;
  const int64_t size = ok ? (int64_t)c10::elementSize(type) : 0;
  return ok && bytes % size == 0 ? plain(o, type, bytes / size) : nullptr;
}

// sign bits of a table order: true where they are there as needed, null for order 1
bool sign_bits(PyObject* o, long order, long n, c10::Device dev, const uint32_t*& bits) {
  bits = nullptr;
  if (order < 1 || n % order || ((n / order) & (n / order - 1))) return false;
  if (order == 1) return true;
  if (!THPVariable_Check(o)) return false;
  const at::Tensor* t = plain(o, at::kInt, THPVariable_Unpack(o).numel());
  if (!t || t->device() != dev || t->numel() * 32 < order * order) return false;
  bits = (const uint32_t*)t->data_ptr();
  return true;
}

bool here(c10::Device dev) {
  return !c10::impl::dispatch_mode_enabled() && c10::impl::VirtualGuardImpl(dev.type()).getDevice().index() == dev.index();
}

bool shape_ok(long m, long k, long bits) { return m > 0 && k > 0 && !((m | k) & 31) && bits >= 2 && bits <= 4; }

PyObject* failed(int rc) { return PyLong_FromLong(rc); }  // (the wrapper raises)

// linear(x, packed, tlut, su, sv, had_in, order_in, had_out, order_out, m, k, bits, scale_in, scale_out, long_sums,
// copy_rows, stream[, pre_mode, norm_weight, eps, residual]) -> tensor, an error code, or None.  From copy_rows rows on
// operands must start on 16 bytes.  With the last four: fp16 rows through qtip_linear_rows.
PyObject* linear(PyObject*, PyObject* const* a, Py_ssize_t nargs) {
  const bool fused = nargs == 21;
  if ((nargs != 17 && !fused) || !run_linear) {
    PyErr_SetString(PyExc_TypeError, "linear: 17 or 21 arguments, behind bind()");
    return nullptr;
  }
  const long pre_mode = fused ? PyLong_AsLong(a[17]) : 0;
  const double eps = fused ? PyFloat_AsDouble(a[19]) : 0.;
  const long order_in = PyLong_AsLong(a[6]), order_out = PyLong_AsLong(a[8]), m = PyLong_AsLong(a[9]), k = PyLong_AsLong(a[10]),
             bits = PyLong_AsLong(a[11]), copy_rows = PyLong_AsLong(a[15]);
  const double scale_in = PyFloat_AsDouble(a[12]), scale_out = PyFloat_AsDouble(a[13]);
  const int long_sums = PyObject_IsTrue(a[14]);
  void* stream = PyLong_AsVoidPtr(a[16]);
  if (PyErr_Occurred()) return nullptr;
  try {
    if (!shape_ok(m, k, bits) || !THPVariable_Check(a[0])) Py_RETURN_NONE;
    const at::Tensor& xt = THPVariable_Unpack(a[0]);
    if (xt.dim() != 2) Py_RETURN_NONE;
    const int64_t rows = xt.sym_sizes()[0].is_symbolic() ? 0 : xt.size(0);
    const at::ScalarType type = xt.scalar_type();
    const int64_t width = pre_mode == 2 ? 2 * k : k;  // [gate | up]
    if (rows < (fused ? 2 : 1) || rows > 65535 || xt.size(1) != width || (type != at::kHalf && (type != at::kFloat || fused)))
      Py_RETURN_NONE;
    const at::Tensor *x = plain(a[0], type, rows * width), *packed = packed_words(a[1], m * k / 8 * bits),
                     *tlut = plain(a[2], at::kHalf, 1024), *su = plain(a[3], at::kHalf, k), *sv = plain(a[4], at::kFloat, m);
    if (!x || !packed || !tlut || !su || !sv) Py_RETURN_NONE;
    const c10::Device dev = packed->device();
    const uint32_t *had_in, *had_out;
    if (x->device() != dev || tlut->device() != dev || su->device() != dev || sv->device() != dev ||
        !sign_bits(a[5], order_in, k, dev, had_in) || !sign_bits(a[7], order_out, m, dev, had_out) || !here(dev))
      Py_RETURN_NONE;
    const void *xp = x->data_ptr(), *pp = packed->data_ptr(), *tp = tlut->data_ptr(), *up = su->data_ptr();
    const float* vp = (const float*)sv->data_ptr();
    const void *np = nullptr, *rp = nullptr;
    if (fused) {
      const at::Tensor *norm = a[18] == Py_None ? nullptr : plain(a[18], at::kHalf, k),
                       *res = a[20] == Py_None ? nullptr : plain(a[20], at::kHalf, rows * m);
      if ((a[18] != Py_None && (!norm || norm->device() != dev)) || (a[20] != Py_None && (!res || res->device() != dev)))
        Py_RETURN_NONE;
      if (norm) np = norm->data_ptr();
      if (res) rp = res->data_ptr();
      if (((uintptr_t)np | (uintptr_t)rp) & 15) Py_RETURN_NONE;
    }
    if (rows >= copy_rows && (((uintptr_t)xp | (uintptr_t)up | (uintptr_t)vp) & 15)) Py_RETURN_NONE;
    const int dtype = type == at::kHalf ? QTIP_F16 : QTIP_F32;
    const size_t need = (long_sums ? linear_long_bytes : linear_bytes)((int)m, (int)k, (int)bits, (int)rows, (int)order_in, dtype);
    const at::Tensor out = at::empty({rows, m}, x->options().requires_grad(false));
    const at::Tensor ws = at::empty({(int64_t)need}, x->options().dtype(at::kByte).requires_grad(false));
    void *op = out.data_ptr(), *wp = ws.data_ptr();
    int rc;
    Py_BEGIN_ALLOW_THREADS;
    if (fused)
      rc = run_rows(op, xp, pp, tp, up, vp, had_in, (int)order_in, had_out, (int)order_out, (int)m, (int)k, (int)bits, (int)rows,
                    (float)scale_in, (float)scale_out, (int)pre_mode, np, (float)eps, rp, long_sums, wp, need, stream);
    else
      rc = (long_sums ? run_linear_long : run_linear)(op, xp, dtype, pp, tp, up, vp, had_in, (int)order_in, had_out,
                                                      (int)order_out, (int)m, (int)k, (int)bits, (int)rows, (float)scale_in,
                                                      (float)scale_out, wp, need, stream);
    Py_END_ALLOW_THREADS;
    return rc ? failed(rc) : THPVariable_Wrap(out);
  } catch (const std::exception&) {  // (out of memory among them: the wrapper's way meets it again, and raises)
    Py_RETURN_NONE;
  }
}

// matvec(packed, x, tlut, m, k, bits, workspace, its bytes, stream) -> (1, m) fp32 tensor, an error code, or None
PyObject* matvec(PyObject*, PyObject* const* a, Py_ssize_t nargs) {
  if (nargs != 9 || !run_matvec) {
    PyErr_SetString(PyExc_TypeError, "matvec: 9 arguments, behind bind()");
    return nullptr;
  }
  const long m = PyLong_AsLong(a[3]), k = PyLong_AsLong(a[4]), bits = PyLong_AsLong(a[5]);
  void *ws = PyLong_AsVoidPtr(a[6]), *stream = PyLong_AsVoidPtr(a[8]);
  const size_t ws_bytes = PyLong_AsSize_t(a[7]);
  if (PyErr_Occurred()) return nullptr;
  try {
    if (!shape_ok(m, k, bits)) Py_RETURN_NONE;
    const at::Tensor *packed = packed_words(a[0], m * k / 8 * bits), *x = plain(a[1], at::kHalf, k),
                     *tlut = plain(a[2], at::kHalf, 1024);
    if (!packed || !x || !tlut) Py_RETURN_NONE;
    const c10::Device dev = packed->device();
    if (x->device() != dev || tlut->device() != dev || !here(dev)) Py_RETURN_NONE;
    const void *xp = x->data_ptr(), *pp = packed->data_ptr(), *tp = tlut->data_ptr();
    const at::Tensor out = at::empty({1, m}, x->options().dtype(at::kFloat).requires_grad(false));
    float* op = (float*)out.data_ptr();
    int rc;
    Py_BEGIN_ALLOW_THREADS;
    rc = run_matvec(op, pp, xp, tp, (int)m, (int)k, (int)bits, ws, ws_bytes, stream);
    Py_END_ALLOW_THREADS;
    return rc ? failed(rc) : THPVariable_Wrap(out);
  } catch (const std::exception&) {
    Py_RETURN_NONE;
  }
}

// bind(addresses of qtip_linear, qtip_linear_long, their workspace sizes, qtip_decompress_matvec, qtip_linear_rows)
PyObject* bind(PyObject*, PyObject* const* a, Py_ssize_t nargs) {
  if (nargs != 6) {
    PyErr_SetString(PyExc_TypeError, "bind: 6 addresses");
    return nullptr;
  }
  void* p[6];
  for (int i = 0; i < 6; ++i) p[i] = PyLong_AsVoidPtr(a[i]);
  if (PyErr_Occurred()) return nullptr;
  run_linear = (decltype(run_linear))p[0];
  run_linear_long = (decltype(run_linear_long))p[1];
  linear_bytes = (decltype(linear_bytes))p[2];
  linear_long_bytes = (decltype(linear_long_bytes))p[3];
  run_matvec = (decltype(run_matvec))p[4];
  run_rows = (decltype(run_rows))p[5];
  Py_RETURN_NONE;
}

PyMethodDef methods[] = {{"linear", (PyCFunction)(void*)linear, METH_FASTCALL, nullptr},
                         {"matvec", (PyCFunction)(void*)matvec, METH_FASTCALL, nullptr},
                         {"bind", (PyCFunction)(void*)bind, METH_FASTCALL, nullptr},
                         {nullptr, nullptr, 0, nullptr}};
PyModuleDef module = {PyModuleDef_HEAD_INIT, "_qtip_host", nullptr, -1, methods, nullptr, nullptr, nullptr, nullptr};

}  // namespace

// (abi_version, torch_version: of the header and of the torch that this was compiled against, for the loader to compare)
PyMODINIT_FUNC PyInit__qtip_host() {
  PyObject* m = PyModule_Create(&module);
  if (m && (PyModule_AddIntConstant(m, "abi_version", QTIP_ABI_VERSION) ||
            PyModule_AddStringConstant(m, "torch_version", QTIP_TORCH_VERSION))) {
    Py_DECREF(m);
    return nullptr;
  }
  return m;
}
