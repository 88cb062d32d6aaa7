// fagq_py.cpp - CPython binding of the operators' per-call paths.
//
// Small calls are bound by the host: in Python the checks (some 30 tensor
// attribute reads), the outputs' allocation and a 16-argument ctypes call cost
// 5 to 11 us against kernels of 3 to 8.  This module does the same checks on the
// tensors' C++ metadata, allocates through ATen and calls the library through
// function pointers handed over from the ctypes binding at import, so both
// bindings reach the one library.  us per call, Python path -> this one:
// functional quantizer 4 x 8192 8.1 -> 6.6, GEMM 32 x 4096 x 7168 11.6 -> 8.2, DSA 1 x 8 x 129 x
// 1021 11.2 -> 5.5.
//
//   launch(x, residual, gamma, residual_out, norm_out, x_q, x_scale, eps,
//          group_size, rounding, stream) -> int
//     The drop-in for src/task01_fused_add_rmsnorm_group_quant.py:1731-1741.
//     rounding: -1 = the format's default (fp8 RNE, int8 truncation),
//               0 = RNE, 1 = truncation, anything else = invalid.
//     Returns fagq_launch's status, or kArgError when a tensor argument is
//     rejected here (the Python layer then raises its detailed error).
//   quant(...) (with a list of tensors the multi-input form), gemm(...), dsa(...),
//     mla(...): the other operators, allocation included.  They return the outputs
//     (dsa and mla: 0), the library's status as an int where it is an error, or
//     kArgError for any argument that the Python layer should look at: it then takes
//     the call from the start, with the same results and its own wording of the errors.
//     Nothing is allocated or launched before all arguments are accepted.  The
//     allocations (which may reach hipMalloc, or wait for the device to free cached
//     blocks) and the launch run without the GIL, as torch's and ctypes' own calls do.
//
// In all of them the caller passes the current stream of the tensors' device
// and has made that device current.
#include <Python.h>

#include <ATen/ATen.h>
#include <torch/csrc/Exceptions.h>
#include <torch/csrc/autograd/python_variable.h>

#include <algorithm>
#include <cstdint>
#include <vector>

#include "fagq.h"
#include "fagq_dsa.h"
#include "fagq_gemm.h"
#include "fagq_mla.h"

namespace {

constexpr int kArgError = 1000;

using LaunchFn = int (*)(const void*, const void*, const void*, void*, void*, void*, void*, int64_t,
                         int64_t, int64_t, float, int, int, int, int, void*);
using TypedLaunchFn = int (*)(const void*, const void*, const void*, void*, void*, void*, void*,
                              int64_t, int64_t, int64_t, float, int, int, int, int, int, int,
                              void*);
LaunchFn g_launch = nullptr;
TypedLaunchFn g_launch_typed = nullptr;
decltype(&fagq_launch_parts) g_parts = nullptr;
decltype(&fagq_gemm_launch) g_gemm = nullptr;
decltype(&fagq_dsa_topk_launch) g_dsa = nullptr;
decltype(&fagq_mla_bwd_workspace_bytes) g_mla_bytes = nullptr;
decltype(&fagq_mla_bwd_launch) g_mla = nullptr;

bool is_tensor(PyObject* o) { return THPVariable_Check(o); }

// A contiguous tensor of element type `st` and `shape` on CUDA device `dev`.
bool rows_ok(const at::Tensor& t, at::IntArrayRef shape, c10::DeviceIndex dev,
             at::ScalarType st) {
  return t.scalar_type() == st && t.sizes() == shape && t.is_cuda() && t.get_device() == dev &&
         t.is_contiguous();
}

// fagq_dtype code of an element type, -1 for others.
int dtype_code(at::ScalarType st) {
  switch (st) {
    case at::kBFloat16: return FAGQ_DT_BF16;
    case at::kHalf: return FAGQ_DT_F16;
    case at::kFloat: return FAGQ_DT_F32;
    default: return -1;
  }
}

PyObject* launch(PyObject*, PyObject* const* args, Py_ssize_t nargs) {
  if (nargs != 11) {
    PyErr_SetString(PyExc_TypeError, "launch() takes 11 arguments");
    return nullptr;
  }
  if (!g_launch) {
    PyErr_SetString(PyExc_RuntimeError, "launch(): bind() has not been called");
    return nullptr;
  }
  for (int i : {0, 1, 2, 3, 5, 6})
    if (!is_tensor(args[i])) return PyLong_FromLong(kArgError);
  const bool has_norm = args[4] != Py_None;
  if (has_norm && !is_tensor(args[4])) return PyLong_FromLong(kArgError);
  // Numbers of other types (a float group size, say) go to the Python checks.
  if (!PyFloat_Check(args[7]) || !PyLong_Check(args[8]) || !PyLong_Check(args[9]) ||
      !PyLong_Check(args[10]))
    return PyLong_FromLong(kArgError);
  const double eps = PyFloat_AS_DOUBLE(args[7]);
  const long long G = PyLong_AsLongLong(args[8]);
  const long rounding = PyLong_AsLong(args[9]);
  void* stream = PyLong_AsVoidPtr(args[10]);
  if (PyErr_Occurred()) {
    PyErr_Clear();
    return PyLong_FromLong(kArgError);
  }

  const at::Tensor& x = THPVariable_Unpack(args[0]);
  const at::Tensor& residual = THPVariable_Unpack(args[1]);
  const at::Tensor& gamma = THPVariable_Unpack(args[2]);
  const at::Tensor& residual_out = THPVariable_Unpack(args[3]);
  const at::Tensor& x_q = THPVariable_Unpack(args[5]);
  const at::Tensor& x_scale = THPVariable_Unpack(args[6]);
  if (x.dim() != 2 || !x.is_cuda()) return PyLong_FromLong(kArgError);
  const c10::DeviceIndex dev = x.get_device();
  const auto shape = x.sizes();
  const int64_t M = shape[0], D = shape[1];
  const int64_t dshape[1] = {D};
  // x, gamma and norm_out share the activation type, residual and
  // residual_out the residual stream's; the library checks the pair.
  const at::ScalarType at_ = x.scalar_type(), rt = residual.scalar_type();
  const int act = dtype_code(at_), res = dtype_code(rt);
  if (act < 0 || res < 0) return PyLong_FromLong(kArgError);
  if (!rows_ok(x, shape, dev, at_) || !rows_ok(residual, shape, dev, rt) ||
      !rows_ok(residual_out, shape, dev, rt) ||
      !rows_ok(gamma, at::IntArrayRef(dshape, 1), dev, at_))
    return PyLong_FromLong(kArgError);
  if (has_norm && !rows_ok(THPVariable_Unpack(args[4]), shape, dev, at_))
    return PyLong_FromLong(kArgError);
  if (G <= 0 || D % G != 0) return PyLong_FromLong(kArgError);

  int qf;
  if (x_q.scalar_type() == at::kFloat8_e4m3fn)
    qf = FAGQ_Q_FP8_E4M3FN;
  else if (x_q.scalar_type() == at::kChar)
    qf = FAGQ_Q_INT8;
  else
    return PyLong_FromLong(kArgError);
  if (x_q.sizes() != shape || !x_q.is_cuda() || x_q.get_device() != dev || !x_q.is_contiguous())
    return PyLong_FromLong(kArgError);

  int sf;
  if (x_scale.scalar_type() == at::kFloat)
    sf = FAGQ_SCALE_F32;
  else if (x_scale.scalar_type() == at::kByte)
    sf = FAGQ_SCALE_UE8M0;
  else
    return PyLong_FromLong(kArgError);
  const int64_t groups = D / G;
  if (x_scale.dim() != 2 || x_scale.size(0) != M || x_scale.size(1) != groups ||
      !x_scale.is_cuda() || x_scale.get_device() != dev)
    return PyLong_FromLong(kArgError);
  int layout;
  if (x_scale.is_contiguous())
    layout = FAGQ_LAYOUT_ROW_MAJOR;
  else if (x_scale.stride(0) == 1 && x_scale.stride(1) == M)
    layout = FAGQ_LAYOUT_COL_MAJOR;
  else
    return PyLong_FromLong(kArgError);

  int rnd;
  if (rounding == -1)
    rnd = qf == FAGQ_Q_FP8_E4M3FN ? FAGQ_ROUND_RNE : FAGQ_ROUND_TRUNC;
  else if (rounding == 0)
    rnd = FAGQ_ROUND_RNE;
  else if (rounding == 1 && qf == FAGQ_Q_INT8)
    rnd = FAGQ_ROUND_TRUNC;
  else
    return PyLong_FromLong(kArgError);
  if (M == 0) return PyLong_FromLong(FAGQ_OK);

  void* norm = has_norm ? THPVariable_Unpack(args[4]).data_ptr() : nullptr;
  if (act == FAGQ_DT_BF16 && res == FAGQ_DT_BF16)
    return PyLong_FromLong(g_launch(x.data_ptr(), residual.data_ptr(), gamma.data_ptr(),
                                    residual_out.data_ptr(), norm, x_q.data_ptr(),
                                    x_scale.data_ptr(), M, D, G, (float)eps, qf, sf, layout, rnd,
                                    stream));
  if (!g_launch_typed) return PyLong_FromLong(kArgError);
  const int st = g_launch_typed(x.data_ptr(), residual.data_ptr(), gamma.data_ptr(),
                                residual_out.data_ptr(), norm, x_q.data_ptr(), x_scale.data_ptr(),
                                M, D, G, (float)eps, qf, sf, layout, rnd, act, res, stream);
  // An unsupported type pair goes to the Python checks, which word the error.
  return PyLong_FromLong(st == FAGQ_E_FORMAT ? kArgError : st);
}

// ------------------------------------------------------------------ with allocation

PyObject* arg_error() { return PyLong_FromLong(kArgError); }

// Releases the GIL for its scope, also when an exception leaves it.  The argument
// objects outlive the call (the caller's frame holds them); their data pointers
// are read before.
struct NoGil {
  PyThreadState* const state = PyEval_SaveThread();
  NoGil() = default;
  NoGil(const NoGil&) = delete;
  NoGil& operator=(const NoGil&) = delete;
  ~NoGil() { PyEval_RestoreThread(state); }
};

// Plain tensors only: a subclass may override what the Python layer calls.
bool is_plain(PyObject* o) { return THPVariable_CheckExact(o); }

// An int argument in [lo, hi].
bool int_arg(PyObject* o, long long lo, long long hi, long long* out) {
  if (!PyLong_CheckExact(o)) return false;
  *out = PyLong_AsLongLong(o);
  if (*out == -1 && PyErr_Occurred()) {
    PyErr_Clear();
    return false;
  }
  return *out >= lo && *out <= hi;
}

// A float argument: a Python float (NaN and infinities too) or int.
bool float_arg(PyObject* o, double* out) {
  if (!PyFloat_CheckExact(o) && !PyLong_CheckExact(o)) return false;
  *out = PyFloat_AsDouble(o);
  if (*out == -1.0 && PyErr_Occurred()) {
    PyErr_Clear();
    return false;
  }
  return true;
}

bool stream_arg(PyObject* o, void** out) {
  if (!PyLong_CheckExact(o)) return false;
  *out = PyLong_AsVoidPtr(o);
  if (PyErr_Occurred()) {
    PyErr_Clear();
    return false;
  }
  return true;
}

// Code and scale tensors of the functional forms.
at::Tensor empty_codes(c10::Device device, int64_t M, int64_t D, bool fp8) {
  return at::empty({M, D}, at::TensorOptions(device).dtype(fp8 ? at::kFloat8_e4m3fn : at::kChar));
}
at::Tensor empty_scale(c10::Device device, int64_t M, int64_t groups, bool ue8m0, bool col_major) {
  const auto o = at::TensorOptions(device).dtype(ue8m0 ? at::kByte : at::kFloat);
  // The strides of empty({groups, M}).t(), which are at least 1 where M is 0.
  return col_major ? at::empty_strided({M, groups}, {1, std::max<int64_t>(M, 1)}, o)
                   : at::empty({M, groups}, o);
}

PyObject* three(const at::Tensor& a, const at::Tensor& b, const at::Tensor& c) {
  PyObject* t = PyTuple_New(3);
  if (!t) return nullptr;
  const at::Tensor* v[3] = {&a, &b, &c};
  for (int i = 0; i < 3; ++i) {
    PyObject* o = THPVariable_Wrap(*v[i]);
    if (!o) {
      Py_DECREF(t);
      return nullptr;
    }
    PyTuple_SET_ITEM(t, i, o);
  }
  return t;
}

// quant(x or [x, ...], residual, weight, eps, group_size, fp8, col_major, ue8m0,
//       rounding, inplace, stream) -> (residual_out, q, scale): the functional
// form, or with a list the multi-input form.
PyObject* quant(PyObject*, PyObject* const* args, Py_ssize_t nargs) {
  HANDLE_TH_ERRORS
  if (nargs != 11) {
    PyErr_SetString(PyExc_TypeError, "quant() takes 11 arguments");
    return nullptr;
  }
  const bool multi = PyList_CheckExact(args[0]);
  if (!g_launch || !g_launch_typed || !g_parts) return arg_error();
  const Py_ssize_t n = multi ? PyList_GET_SIZE(args[0]) : 1;
  if (n < 1 || n > FAGQ_MAX_PARTS) return arg_error();
  PyObject* xs[FAGQ_MAX_PARTS];
  for (Py_ssize_t i = 0; i < n; ++i) {
    xs[i] = multi ? PyList_GET_ITEM(args[0], i) : args[0];
    if (!is_plain(xs[i])) return arg_error();
  }
  long long G, fp8, col, ue, rounding, inplace;
  void* stream;
  if (!is_plain(args[1]) || !is_plain(args[2]) || !PyFloat_CheckExact(args[3]) ||
      !int_arg(args[4], 1, INT32_MAX, &G) || !int_arg(args[5], 0, 1, &fp8) ||
      !int_arg(args[6], 0, 1, &col) || !int_arg(args[7], 0, 1, &ue) ||
      !int_arg(args[8], -1, 1, &rounding) || !int_arg(args[9], 0, 1, &inplace) ||
      !stream_arg(args[10], &stream))
    return arg_error();
  const at::Tensor& x = THPVariable_Unpack(xs[0]);
  const at::Tensor& residual = THPVariable_Unpack(args[1]);
  const at::Tensor& weight = THPVariable_Unpack(args[2]);
  if (x.dim() != 2 || !x.is_cuda()) return arg_error();
  const c10::DeviceIndex dev = x.get_device();
  const auto shape = x.sizes();
  const int64_t M = shape[0], D = shape[1], dshape[1] = {D};
  const at::ScalarType at_ = x.scalar_type(), rt = residual.scalar_type();
  const int act = dtype_code(at_), res = dtype_code(rt);
  if (act < 0 || res < 0 || D % G != 0) return arg_error();
  if (multi && (act != FAGQ_DT_BF16 || res != FAGQ_DT_BF16)) return arg_error();
  for (Py_ssize_t i = 0; i < n; ++i)
    if (!rows_ok(THPVariable_Unpack(xs[i]), shape, dev, at_)) return arg_error();
  if (!rows_ok(residual, shape, dev, rt) ||
      !rows_ok(weight, at::IntArrayRef(dshape, 1), dev, at_))
    return arg_error();
  if (fp8 && rounding == 1) return arg_error();
  const int qf = fp8 ? FAGQ_Q_FP8_E4M3FN : FAGQ_Q_INT8;
  const int rnd = fp8 || rounding == 0 ? FAGQ_ROUND_RNE : FAGQ_ROUND_TRUNC;
  const int sf = ue ? FAGQ_SCALE_UE8M0 : FAGQ_SCALE_F32;
  const int64_t groups = D / G;

  // The list is the caller's to change once the GIL is released: its tensors are held.
  std::vector<at::Tensor> held;
  if (multi) held.reserve(n);
  const void* ptrs[FAGQ_MAX_PARTS];
  for (Py_ssize_t i = 0; i < n; ++i) {
    const at::Tensor& t = THPVariable_Unpack(xs[i]);
    if (multi) held.push_back(t);
    ptrs[i] = t.data_ptr();
  }
  const void* const rp = residual.data_ptr();
  const void* const wp = weight.data_ptr();
  const float eps = (float)PyFloat_AS_DOUBLE(args[3]);
  const c10::Device device = x.device();
  at::Tensor residual_out, q, scale;
  int st = FAGQ_OK;
  {
    NoGil no_gil;
    residual_out = inplace ? residual : at::empty_like(residual);
    q = empty_codes(device, M, D, fp8);
    scale = empty_scale(device, M, groups, ue, col);
    if (M != 0) {
      // A [M, groups] tensor with one row or column is both: row-major, as in Python.
      const int layout = scale.is_contiguous() ? FAGQ_LAYOUT_ROW_MAJOR : FAGQ_LAYOUT_COL_MAJOR;
      if (multi)
        st = g_parts(ptrs, (int)n, rp, wp, residual_out.data_ptr(), q.data_ptr(), scale.data_ptr(),
                     M, D, G, eps, qf, sf, layout, rnd, stream);
      else if (act == FAGQ_DT_BF16 && res == FAGQ_DT_BF16)
        st = g_launch(ptrs[0], rp, wp, residual_out.data_ptr(), nullptr, q.data_ptr(),
                      scale.data_ptr(), M, D, G, eps, qf, sf, layout, rnd, stream);
      else
        st = g_launch_typed(ptrs[0], rp, wp, residual_out.data_ptr(), nullptr, q.data_ptr(),
                            scale.data_ptr(), M, D, G, eps, qf, sf, layout, rnd, act, res, stream);
    }
  }
  // A type pair the library refuses goes to the Python checks.
  if (st == FAGQ_E_FORMAT && !(act == FAGQ_DT_BF16 && res == FAGQ_DT_BF16)) return arg_error();
  if (st != FAGQ_OK) return PyLong_FromLong(st);
  return three(residual_out, q, scale);   // inplace: the caller's own tensor object
  END_HANDLE_TH_ERRORS
}

// gemm(a_q, a_scale, b_q, b_scale, out or None, stream) -> out
PyObject* gemm(PyObject*, PyObject* const* args, Py_ssize_t nargs) {
  HANDLE_TH_ERRORS
  if (nargs != 6) {
    PyErr_SetString(PyExc_TypeError, "gemm() takes 6 arguments");
    return nullptr;
  }
  if (!g_gemm) return arg_error();
  for (int i = 0; i < 4; ++i)
    if (!is_plain(args[i])) return arg_error();
  const bool has_out = args[4] != Py_None;
  void* stream;
  if ((has_out && !is_plain(args[4])) || !stream_arg(args[5], &stream)) return arg_error();
  const at::Tensor& a = THPVariable_Unpack(args[0]);
  const at::Tensor& as = THPVariable_Unpack(args[1]);
  const at::Tensor& b = THPVariable_Unpack(args[2]);
  const at::Tensor& bs = THPVariable_Unpack(args[3]);
  if (a.dim() != 2 || b.dim() != 2 || !a.is_cuda()) return arg_error();
  const c10::DeviceIndex dev = a.get_device();
  const int64_t M = a.size(0), K = a.size(1), N = b.size(0), kb = K / 128, nb = (N + 127) / 128;
  if (b.size(1) != K || K % 128 != 0 || N % 16 != 0) return arg_error();
  const int64_t ashape[2] = {M, K}, bshape[2] = {N, K}, sshape[2] = {nb, kb}, cshape[2] = {M, N};
  auto scale_format = [](const at::Tensor& t) {
    return t.scalar_type() == at::kFloat  ? FAGQ_SCALE_F32
           : t.scalar_type() == at::kByte ? FAGQ_SCALE_UE8M0
                                          : -1;
  };
  const int asf = scale_format(as), bsf = scale_format(bs);
  if (asf < 0 || bsf < 0 || !rows_ok(a, ashape, dev, at::kFloat8_e4m3fn) ||
      !rows_ok(b, bshape, dev, at::kFloat8_e4m3fn) || !rows_ok(bs, sshape, dev, bs.scalar_type()) ||
      as.dim() != 2 || as.size(0) != M || as.size(1) != kb || !as.is_cuda() ||
      as.get_device() != dev)
    return arg_error();
  int layout;
  if (as.is_contiguous()) layout = FAGQ_LAYOUT_ROW_MAJOR;
  else if (as.stride(0) == 1 && as.stride(1) == M) layout = FAGQ_LAYOUT_COL_MAJOR;
  else return arg_error();
  if (has_out && !rows_ok(THPVariable_Unpack(args[4]), cshape, dev, at::kBFloat16)) return arg_error();
  const void* const p[4] = {a.data_ptr(), as.data_ptr(), b.data_ptr(), bs.data_ptr()};
  const c10::Device device = a.device();
  at::Tensor out;
  if (has_out) out = THPVariable_Unpack(args[4]);
  int st;
  {
    NoGil no_gil;
    if (!has_out) out = at::empty({M, N}, at::TensorOptions(device).dtype(at::kBFloat16));
    st = g_gemm(p[0], p[1], p[2], p[3], out.data_ptr(), M, N, K, asf, layout, bsf, stream);
  }
  if (st != FAGQ_OK) return PyLong_FromLong(st);
  return THPVariable_Wrap(out);
  END_HANDLE_TH_ERRORS
}

// dsa(scores, page_table, q_pos, kv_lens, out_blocks, out_pages, block_size,
//     top_k, stream) -> status
PyObject* dsa(PyObject*, PyObject* const* args, Py_ssize_t nargs) {
  HANDLE_TH_ERRORS
  if (nargs != 9) {
    PyErr_SetString(PyExc_TypeError, "dsa() takes 9 arguments");
    return nullptr;
  }
  if (!g_dsa) return arg_error();
  for (int i = 0; i < 6; ++i)
    if (!is_plain(args[i])) return arg_error();
  long long bs, k;
  void* stream;
  if (!int_arg(args[6], INT64_MIN, INT64_MAX, &bs) || !int_arg(args[7], INT64_MIN, INT64_MAX, &k) ||
      !stream_arg(args[8], &stream))
    return arg_error();
  const at::Tensor& s = THPVariable_Unpack(args[0]);
  if (s.dim() != 4 || !s.is_cuda() || !s.is_contiguous()) return arg_error();
  const c10::DeviceIndex dev = s.get_device();
  const int64_t B = s.size(0), H = s.size(1), Q = s.size(2), NB = s.size(3);
  const int sdt = s.scalar_type() == at::kFloat      ? FAGQ_DSA_F32
                  : s.scalar_type() == at::kBFloat16 ? FAGQ_DSA_BF16
                                                     : -1;
  const at::Tensor* t[5];
  for (int i = 0; i < 5; ++i) t[i] = &THPVariable_Unpack(args[1 + i]);
  const at::ScalarType it = t[1]->scalar_type();
  if (sdt < 0 || (it != at::kInt && it != at::kLong)) return arg_error();
  const int64_t pt[2] = {B, NB}, qp[2] = {B, Q}, kv[1] = {B}, ob[4] = {B, H, Q, k};
  if (!rows_ok(*t[0], pt, dev, at::kInt) || !rows_ok(*t[1], qp, dev, it) ||
      !rows_ok(*t[2], at::IntArrayRef(kv, 1), dev, it) || !rows_ok(*t[3], ob, dev, at::kInt) ||
      !rows_ok(*t[4], ob, dev, at::kInt))
    return arg_error();
  void* p[6] = {s.data_ptr()};
  for (int i = 0; i < 5; ++i) p[1 + i] = t[i]->data_ptr();
  int st;
  {
    NoGil no_gil;
    st = g_dsa(p[0], sdt, p[1], p[2], p[3], it == at::kLong ? FAGQ_DSA_I64 : FAGQ_DSA_I32, p[4],
               p[5], B, H, Q, NB, bs, k, stream);
  }
  return PyLong_FromLong(st);
  END_HANDLE_TH_ERRORS
}

// mla(q, c_kv, out, do, lse, dq, dc_kv, sm_scale, stream) -> status; the
// workspace is allocated here (a caller's own goes through Python).
PyObject* mla(PyObject*, PyObject* const* args, Py_ssize_t nargs) {
  HANDLE_TH_ERRORS
  if (nargs != 9) {
    PyErr_SetString(PyExc_TypeError, "mla() takes 9 arguments");
    return nullptr;
  }
  if (!g_mla || !g_mla_bytes) return arg_error();
  for (int i = 0; i < 7; ++i)
    if (!is_plain(args[i])) return arg_error();
  double sm_scale;
  void* stream;
  if (!float_arg(args[7], &sm_scale) || !stream_arg(args[8], &stream)) return arg_error();
  const at::Tensor* t[7];
  for (int i = 0; i < 7; ++i) t[i] = &THPVariable_Unpack(args[i]);
  if (t[0]->dim() != 4 || !t[0]->is_cuda()) return arg_error();
  const c10::DeviceIndex dev = t[0]->get_device();
  const auto qs = t[0]->sizes();
  const int64_t B = qs[0], H = qs[1], S = qs[2], D = qs[3];
  const int64_t cs[3] = {B, S, D}, ls[3] = {B, H, S};
  auto grad_code = [](const at::Tensor& g) {
    return g.scalar_type() == at::kFloat      ? FAGQ_MLA_F32
           : g.scalar_type() == at::kBFloat16 ? FAGQ_MLA_BF16
                                              : -1;
  };
  const int dq = grad_code(*t[5]), dc = grad_code(*t[6]);
  if (dq < 0 || dc < 0 || !rows_ok(*t[0], qs, dev, at::kBFloat16) ||
      !rows_ok(*t[1], cs, dev, at::kBFloat16) || !rows_ok(*t[2], qs, dev, at::kBFloat16) ||
      !rows_ok(*t[3], qs, dev, at::kBFloat16) || !rows_ok(*t[4], ls, dev, at::kFloat) ||
      !rows_ok(*t[5], qs, dev, t[5]->scalar_type()) || !rows_ok(*t[6], cs, dev, t[6]->scalar_type()))
    return arg_error();
  const int64_t need = g_mla_bytes(B, S, D);
  if (need < 0) return arg_error();
  void* p[7];
  for (int i = 0; i < 7; ++i) p[i] = t[i]->data_ptr();
  const c10::Device device = t[0]->device();
  int st;
  {
    NoGil no_gil;
    const at::Tensor ws = at::empty({std::max<int64_t>(need, 16)},
                                    at::TensorOptions(device).dtype(at::kByte));
    st = g_mla(p[0], p[1], p[2], p[3], static_cast<const float*>(p[4]), p[5], p[6], ws.data_ptr(),
               ws.numel(), B, H, S, D, (float)sm_scale, dq, dc, stream);
  }
  return PyLong_FromLong(st);
  END_HANDLE_TH_ERRORS
}

// bind_all(addresses of fagq_launch_parts, fagq_gemm_launch,
// fagq_dsa_topk_launch, fagq_mla_bwd_workspace_bytes, fagq_mla_bwd_launch).
PyObject* bind_all(PyObject*, PyObject* const* args, Py_ssize_t nargs) {
  if (nargs != 5) {
    PyErr_SetString(PyExc_TypeError, "bind_all() takes 5 arguments");
    return nullptr;
  }
  void* p[5];
  for (int i = 0; i < 5; ++i) {
    p[i] = PyLong_AsVoidPtr(args[i]);
    if (PyErr_Occurred()) return nullptr;
    if (!p[i]) {
      PyErr_SetString(PyExc_ValueError, "bind_all(): null function address");
      return nullptr;
    }
  }
  g_parts = reinterpret_cast<decltype(g_parts)>(p[0]);
  g_gemm = reinterpret_cast<decltype(g_gemm)>(p[1]);
  g_dsa = reinterpret_cast<decltype(g_dsa)>(p[2]);
  g_mla_bytes = reinterpret_cast<decltype(g_mla_bytes)>(p[3]);
  g_mla = reinterpret_cast<decltype(g_mla)>(p[4]);
  Py_RETURN_NONE;
}

// bind(address of fagq_launch, address of fagq_launch_typed) in the loaded
// libfagq.so.
PyObject* bind(PyObject*, PyObject* const* args, Py_ssize_t nargs) {
  if (nargs != 2) {
    PyErr_SetString(PyExc_TypeError, "bind() takes 2 arguments");
    return nullptr;
  }
  void* p = PyLong_AsVoidPtr(args[0]);
  void* pt = PyLong_AsVoidPtr(args[1]);
  if (PyErr_Occurred()) return nullptr;
  if (!p || !pt) {
    PyErr_SetString(PyExc_ValueError, "bind(): null function address");
    return nullptr;
  }
  g_launch = reinterpret_cast<LaunchFn>(p);
  g_launch_typed = reinterpret_cast<TypedLaunchFn>(pt);
  Py_RETURN_NONE;
}

PyMethodDef kMethods[] = {
    {"launch", reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)(void)>(&launch)),
     METH_FASTCALL, "Checks the operator's tensors and calls fagq_launch; returns its status."},
    {"bind", reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)(void)>(&bind)),
     METH_FASTCALL, "Sets the addresses of fagq_launch and fagq_launch_typed."},
    {"quant", reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)(void)>(&quant)),
     METH_FASTCALL, "The functional and multi-input quantizer: allocates and launches."},
    {"gemm", reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)(void)>(&gemm)),
     METH_FASTCALL, "The fp8 block-scaled GEMM: allocates (without an out) and launches."},
    {"dsa", reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)(void)>(&dsa)),
     METH_FASTCALL, "The DSA top-k page-table transform; returns its status."},
    {"mla", reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)(void)>(&mla)),
     METH_FASTCALL, "The MLA backward with a workspace of its own; returns its status."},
    {"bind_all", reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)(void)>(&bind_all)),
     METH_FASTCALL, "Sets the addresses of the other entry points."},
    {nullptr, nullptr, 0, nullptr}};

PyModuleDef kModule = {PyModuleDef_HEAD_INIT, "_fagq_py", "Per-call binding of the operators.", -1,
                       kMethods, nullptr, nullptr, nullptr, nullptr};

}  // namespace

PyMODINIT_FUNC PyInit__fagq_py(void) {
  PyObject* m = PyModule_Create(&kModule);
  if (m && PyModule_AddIntConstant(m, "ARG_ERROR", kArgError) != 0) {
    Py_DECREF(m);
    return nullptr;
  }
  return m;
}
