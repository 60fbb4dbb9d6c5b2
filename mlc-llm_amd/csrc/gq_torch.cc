// The dense operators' way from a Python call to a kernel launch, in native code: argument checks, the output and scratch
// allocation, the current stream and the C ABI call of linear / linear_silu_mul / embedding_take, one Python call each.
//
// What it replaces took 13 us of interpreter time per projection (a torch.cuda.Stream object, three Python checks per tensor, two
// ctypes calls), which is more than a decode projection takes on the GPU: a one-row 4096 x 4096 linear took 14.0 us per call for
// a 4.3 us kernel (7.3 us this way), and every decode step of one to a few rows was bound by it (34 linears of an 8-layer step with
// one row: 455 -> 332 us, with 3-bit weights 449 -> 277).
//
// A function returns the output tensor, or the C ABI's (negative) code as an int, or None where the arguments are not what it
// expects: plain strided tensors on the GPU of the types and shapes that the operator takes, no torch function mode.  The caller
// then runs the Python route, which accepts or refuses them in its own words; nothing is accepted here that is refused there.
#include <Python.h>

#include <ATen/Functions.h>
#include <ATen/PythonTorchFunctionTLS.h>
#include <c10/hip/HIPStream.h>
#include <torch/csrc/Dtype.h>
#include <torch/csrc/Exceptions.h>
#include <torch/csrc/autograd/python_variable.h>

#include <optional>

#include "../../include/mi355gq.h"

namespace {

using at::ScalarType;
using at::Tensor;

// A plain tensor in GPU memory; a subclass may mean anything by its methods and goes to the Python route.
const Tensor* plain(PyObject* o) {
  if (!THPVariable_CheckExact(o)) return nullptr;
  const Tensor& t = THPVariable_Unpack(o);
  return t.defined() && t.layout() == at::kStrided && t.is_cuda() && t.is_contiguous() ? &t : nullptr;
}

// the model dtypes -> the C ABI's codes, -1 for anything else
int model_code(ScalarType t) {
  switch (t) {
    case ScalarType::Half: return MI355GQ_F16;
    case ScalarType::Float: return MI355GQ_F32;
    case ScalarType::BFloat16: return MI355GQ_BF16;
    default: return -1;
  }
}

bool small_int(PyObject* o, int* out) {
  if (!PyLong_CheckExact(o)) return false;
  int overflow = 0;
  const long v = PyLong_AsLongAndOverflow(o, &overflow);
  if (overflow || v < 1 || v > 1 << 20) return false;
  *out = static_cast<int>(v);
  return true;
}

struct Packed {
  const Tensor *words, *scales;
  int bits, group;
};

// q_weight [N, words(K)] and q_scale [N, groups(K)] of `dtype`
bool packed_fits(const Packed& p, int64_t n, int64_t k, ScalarType dtype) {
  if (p.bits > 32 || p.words->dim() != 2 || p.scales->dim() != 2 || p.scales->scalar_type() != dtype) return false;
  const ScalarType w = p.words->scalar_type();
  if (w != ScalarType::Int && w != ScalarType::UInt32) return false;
  const int64_t groups = (k + p.group - 1) / p.group, words = (p.group / (32 / p.bits)) * groups;
  return p.words->size(0) == n && p.words->size(1) == words && p.scales->size(0) == n && p.scales->size(1) == groups;
}

bool packed_args(PyObject* const* a, Packed* p) {
  p->words = plain(a[0]);
  p->scales = plain(a[1]);
  return p->words && p->scales && small_int(a[2], &p->bits) && small_int(a[3], &p->group);
}

void* current_stream() { return c10::hip::getCurrentHIPStream().stream(); }

// leading sizes of x, then `last`
c10::SmallVector<int64_t, 6> with_last(const Tensor& x, int64_t last) {
  c10::SmallVector<int64_t, 6> s(x.sizes().begin(), x.sizes().end());
  s.back() = last;
  return s;
}

int64_t leading_rows(const Tensor& x) {
  int64_t m = 1;
  for (int64_t d = 0; d + 1 < x.dim(); ++d) m *= x.size(d);
  return m;
}

// scratch for one call, given back to the allocator when it goes (the kernels that use it are on the same stream)
struct Scratch {
  Tensor t;
  void* ptr = nullptr;
  Scratch(const Tensor& like, int64_t bytes) {
    if (bytes == 0) return;
    t = at::empty({bytes}, like.options().dtype(at::kByte));
    ptr = t.mutable_data_ptr();
  }
};

PyObject* result(int rc, const Tensor& out) { return rc == MI355GQ_OK ? THPVariable_Wrap(out) : PyLong_FromLong(rc); }

// linear(x, q_weight, q_scale, bits, group_size, bias | None, out_dtype, out | None, residual | None)
PyObject* linear(PyObject*, PyObject* const* a, Py_ssize_t nargs) {
  HANDLE_TH_ERRORS
  Packed p;
  if (nargs != 9 || at::impl::torch_function_mode_enabled()) Py_RETURN_NONE;
  const Tensor* x = plain(a[0]);
  if (!x || x->dim() < 1 || !packed_args(a + 1, &p) || !THPDtype_Check(a[6])) Py_RETURN_NONE;
  const ScalarType dtype = x->scalar_type();
  const int code = model_code(dtype);
  const int64_t k = x->size(-1), n = p.words->dim() ? p.words->size(0) : -1, m = leading_rows(*x);
  if (code < 0 || !packed_fits(p, n, k, dtype)) Py_RETURN_NONE;
  ScalarType out_dtype = reinterpret_cast<THPDtype*>(a[6])->scalar_type;
  if (out_dtype == ScalarType::Half) out_dtype = dtype;  // the signature's default: a model's own dtype
  if (out_dtype != dtype && out_dtype != ScalarType::Float) Py_RETURN_NONE;
  const Tensor *bias = nullptr, *given = nullptr, *residual = nullptr;
  if (a[5] != Py_None) {
    bias = plain(a[5]);
    if (!bias || bias->scalar_type() != dtype || bias->dim() != 1 || bias->size(0) != n) Py_RETURN_NONE;
  }
  const auto shape = with_last(*x, n);
  if (a[7] != Py_None) {
    given = plain(a[7]);
    if (!given || given->scalar_type() != out_dtype || given->sizes() != at::IntArrayRef(shape)) Py_RETURN_NONE;
  }
  if (a[8] != Py_None) {
    residual = plain(a[8]);
    if (!residual || residual->scalar_type() != dtype || residual->sizes() != at::IntArrayRef(shape)) Py_RETURN_NONE;
  }
  Tensor out;
  int rc;
  {
    pybind11::gil_scoped_release release;
    out = given ? *given : at::empty(shape, x->options().dtype(out_dtype));
    const int64_t bytes = mi355gq_linear_dt_workspace_bytes(m, n, k, p.bits, p.group, code);
    Scratch ws(*x, bytes);
    const void *xp = x->const_data_ptr(), *wp = p.words->const_data_ptr(), *sp = p.scales->const_data_ptr(),
               *bp = bias ? bias->const_data_ptr() : nullptr;
    void* yp = out.mutable_data_ptr();
    const int oc = model_code(out_dtype);
    if (residual)
      rc = mi355gq_linear_residual_dt(xp, wp, sp, bp, residual->const_data_ptr(), m, n, k, p.bits, p.group, code, oc, yp, ws.ptr,
                                      bytes, current_stream());
    else
      rc = mi355gq_linear_dt(xp, wp, sp, bp, m, n, k, p.bits, p.group, code, oc, yp, ws.ptr, bytes, current_stream());
  }
  return result(rc, out);
  END_HANDLE_TH_ERRORS
}

// linear_silu_mul(x, q_weight, q_scale, bits, group_size)
PyObject* linear_silu_mul(PyObject*, PyObject* const* a, Py_ssize_t nargs) {
  HANDLE_TH_ERRORS
  Packed p;
  if (nargs != 5 || at::impl::torch_function_mode_enabled()) Py_RETURN_NONE;
  const Tensor* x = plain(a[0]);
  if (!x || x->dim() < 1 || !packed_args(a + 1, &p)) Py_RETURN_NONE;
  const ScalarType dtype = x->scalar_type();
  const int code = model_code(dtype);
  const int64_t k = x->size(-1), n = p.words->dim() ? p.words->size(0) : -1, m = leading_rows(*x);
  if (code < 0 || !packed_fits(p, n, k, dtype) || n % 2) Py_RETURN_NONE;
  Tensor out;
  int rc;
  {
    pybind11::gil_scoped_release release;
    out = at::empty(with_last(*x, n / 2), x->options());
    const int64_t bytes = mi355gq_linear_silu_mul_dt_workspace_bytes(m, n, k, p.bits, p.group, code);
    Scratch ws(*x, bytes);
    rc = mi355gq_linear_silu_mul_dt(x->const_data_ptr(), p.words->const_data_ptr(), p.scales->const_data_ptr(), m, n, k, p.bits,
                                    p.group, code, out.mutable_data_ptr(), ws.ptr, bytes, current_stream());
  }
  return result(rc, out);
  END_HANDLE_TH_ERRORS
}

// embedding_take(ids, q_weight, q_scale, k, bits, group_size)
PyObject* embedding_take(PyObject*, PyObject* const* a, Py_ssize_t nargs) {
  HANDLE_TH_ERRORS
  Packed p;
  PyObject* packed[4];
  int k = 0;
  if (nargs != 6 || at::impl::torch_function_mode_enabled()) Py_RETURN_NONE;
  packed[0] = a[1], packed[1] = a[2], packed[2] = a[4], packed[3] = a[5];
  const Tensor* ids = plain(a[0]);
  if (!ids || ids->scalar_type() != ScalarType::Int || !packed_args(packed, &p) || !small_int(a[3], &k)) Py_RETURN_NONE;
  const ScalarType dtype = p.scales->scalar_type();
  const int code = model_code(dtype);
  const int64_t rows = p.words->dim() ? p.words->size(0) : -1;
  if (code < 0 || !packed_fits(p, rows, k, dtype)) Py_RETURN_NONE;
  Tensor out;
  int rc;
  {
    pybind11::gil_scoped_release release;
    c10::SmallVector<int64_t, 6> shape(ids->sizes().begin(), ids->sizes().end());
    shape.push_back(k);
    out = at::empty(shape, p.scales->options());
    rc = mi355gq_embedding_take_dt(ids->const_data_ptr(), ids->numel(), p.words->const_data_ptr(), p.scales->const_data_ptr(), rows,
                                   k, p.bits, p.group, code, out.mutable_data_ptr(), current_stream());
  }
  return result(rc, out);
  END_HANDLE_TH_ERRORS
}

// the current HIP stream of the current device, as a number
PyObject* stream(PyObject*, PyObject*) {
  HANDLE_TH_ERRORS
  return PyLong_FromVoidPtr(current_stream());
  END_HANDLE_TH_ERRORS
}

#define GQ_FAST(fn) reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)()>(fn)), METH_FASTCALL
PyMethodDef kMethods[] = {
    {"linear", GQ_FAST(linear), nullptr},
    {"linear_silu_mul", GQ_FAST(linear_silu_mul), nullptr},
    {"embedding_take", GQ_FAST(embedding_take), nullptr},
    {"stream", stream, METH_NOARGS, nullptr},
    {nullptr, nullptr, 0, nullptr},
};
PyModuleDef kModule = {PyModuleDef_HEAD_INIT, "_mi355gq_torch", nullptr, -1, kMethods, nullptr, nullptr, nullptr, nullptr};

}  // namespace

PyMODINIT_FUNC PyInit__mi355gq_torch() { return PyModule_Create(&kModule); }
