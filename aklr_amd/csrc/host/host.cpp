// aklr_amd._host: the ops' per-call host work in native code, for the calls a serving loop makes.
//
// Each function takes a call's positional and keyword arguments as the op received them and returns its
// outputs, or None where the general Python path has to decide: a call outside the contract, a disabled or
// traced op, out=, trans_b=False, a tensor subclass, an active torch mode, a missing or unknown argument.
// It serves exactly what that path would serve, in the same way: the checks of aklr_amd/gemm.py and
// aklr_amd/quant.py, then torch's allocator for outputs and scratch and the C ABI on the current stream.
// Nothing is kept between calls, and the GIL is released around allocation and launch.
//
// Why: a decode GEMM takes 3 to 20 us on the GPU, and its call took 12 to 17 us on the host (argument
// binding, about forty tensor attribute reads, two environment lookups, a ctypes call of 21 arguments), so
// a loop of layers was bound by Python. One quantizer call of 8 x 7168 12.4 -> 4.6 us, one GEMM call of
// 333 x 3072 x 1536 17.5 -> 7.6 (the GPU's time now), quantizer and MXFP4 GEMM of 8 x 10240 x 8192 31.0 -> 14.1.
#include <ATen/Context.h>
#include <ATen/PythonTorchFunctionTLS.h>
#include <ATen/core/Tensor.h>
#include <ATen/ops/empty.h>
#include <c10/core/impl/TorchDispatchModeTLS.h>
#include <c10/hip/HIPStream.h>
#include <torch/csrc/Dtype.h>
#include <torch/csrc/Exceptions.h>
#include <torch/csrc/autograd/python_variable.h>

#include <cstdlib>
#include <cstring>
#include <optional>

#include "../../../include/aklr_amd.h"

namespace {

constexpr int64_t kMaxM = 1 << 20, kMaxN = 262144, kMaxK = 65536;              // aklr_amd/gemm.py
constexpr int64_t kMaxTokens = 131072, kMaxHidden = 21504, kMaxHidden4 = 65536;  // aklr_amd/quant.py

// The arguments of one call by parameter position, nullptr where not given. False: the general path binds
// them (and raises what it raises).
bool bind(PyObject* const* argv, Py_ssize_t argc, const char* const* names, int count, int positional, int required,
          PyObject** out) {
  if (argc != 2 || !PyTuple_CheckExact(argv[0]) || !PyDict_CheckExact(argv[1])) return false;
  for (int i = 0; i < count; ++i) out[i] = nullptr;
  const Py_ssize_t n = PyTuple_GET_SIZE(argv[0]);
  if (n > positional) return false;
  for (Py_ssize_t i = 0; i < n; ++i) out[i] = PyTuple_GET_ITEM(argv[0], i);
  PyObject *key, *value;
  Py_ssize_t pos = 0;
  while (PyDict_Next(argv[1], &pos, &key, &value)) {
    int at = -1;
    for (int i = 0; i < count && at < 0; ++i)
      if (PyUnicode_CompareWithASCIIString(key, names[i]) == 0) at = i;
    if (at < 0 || out[at]) return false;
    out[at] = value;
  }
  for (int i = 0; i < required; ++i)
    if (!out[i]) return false;
  return true;
}

bool set_and_not_zero(const char* name) {
  const char* v = std::getenv(name);
  return v && *v && std::strcmp(v, "0") != 0;
}

// Whether anything may look at, or change, what a call does: the general path's business.
bool watched() {
  return set_and_not_zero("AKLR_DISABLE") || set_and_not_zero("AKLR_TRACE") || at::impl::torch_function_mode_enabled() ||
         c10::impl::TorchDispatchModeTLS::any_modes_set() || at::globalContext().deterministicAlgorithms();
}

// A plain dense GPU tensor (no subclass, no functional wrapper), 16-byte aligned.
const at::Tensor* plain(PyObject* o) {
  if (!THPVariable_CheckExact(o)) return nullptr;
  const at::Tensor& t = THPVariable_Unpack(o);
  if (!t.defined() || t.layout() != at::kStrided || !t.device().is_cuda() || !t.has_storage()) return nullptr;
  if (t.unsafeGetTensorImpl()->is_python_dispatch()) return nullptr;
  if (reinterpret_cast<uintptr_t>(t.const_data_ptr()) % 16 != 0) return nullptr;
  return &t;
}

bool is_true_attr(PyObject* o, PyObject* name, bool* out) {
  PyObject* v = nullptr;
#if PY_VERSION_HEX >= 0x030D0000
  if (PyObject_GetOptionalAttr(o, name, &v) < 0) return false;
#else
  if (_PyObject_LookupAttr(o, name, &v) < 0) return false;  // the same function before it was public
#endif
  *out = v == Py_True;
  Py_XDECREF(v);
  return true;
}

PyObject *s_is_shuffled, *s_is_row_major;

bool str_is(PyObject* o, const char* s) { return PyUnicode_CheckExact(o) && PyUnicode_CompareWithASCIIString(o, s) == 0; }

bool is_none(PyObject* o) { return o == nullptr || o == Py_None; }

// block_size: the default, or a tuple of two ints equal to it
bool block_ok(PyObject* o) {
  if (!o) return true;
  if (!PyTuple_CheckExact(o) || PyTuple_GET_SIZE(o) != 2) return false;
  for (int i = 0; i < 2; ++i) {
    PyObject* v = PyTuple_GET_ITEM(o, i);
    if (!PyLong_CheckExact(v) || PyLong_AsLong(v) != 128) return PyErr_Clear(), false;
  }
  return true;
}

bool out_type(PyObject* o, at::ScalarType* t) {
  if (is_none(o)) return *t = at::kBFloat16, true;
  if (!THPDtype_Check(o)) return false;
  *t = reinterpret_cast<THPDtype*>(o)->scalar_type;
  return *t == at::kBFloat16 || *t == at::kHalf;
}

int out_code(at::ScalarType t) { return t == at::kBFloat16 ? AKLR_OUT_BF16 : AKLR_OUT_F16; }

hipStream_t stream_of(const at::Tensor& t) { return c10::hip::getCurrentHIPStream(t.device().index()).stream(); }

at::Tensor make(at::IntArrayRef size, at::ScalarType type, const at::Tensor& like) {
  return at::empty(size, at::TensorOptions().dtype(type).device(like.device()));
}

// The outputs of a launch, or the exception aklr_amd._lib.check raises for its status.
PyObject* status_error(int status, const char* what) {
  PyObject* m = PyImport_ImportModule("aklr_amd._lib");
  if (!m) return nullptr;
  PyObject* r = PyObject_CallMethod(m, "check", "is", status, what);
  Py_DECREF(m);
  if (r) {
    Py_DECREF(r);
    PyErr_Format(PyExc_RuntimeError, "%s: status %d", what, status);
  }
  return nullptr;
}

PyObject* pair(const at::Tensor& a, const at::Tensor& b) {
  PyObject* x = THPVariable_Wrap(a);
  PyObject* y = THPVariable_Wrap(b);
  PyObject* r = x && y ? PyTuple_Pack(2, x, y) : nullptr;
  Py_XDECREF(x);
  Py_XDECREF(y);
  return r;
}

// ---------------------------------------------------------------------------------------------
// quantizers
const at::Tensor* activations(PyObject* o, int64_t multiple, int64_t max_hidden) {
  const at::Tensor* x = plain(o);
  if (!x || x->dim() != 2 || x->scalar_type() != at::kBFloat16 || !x->is_contiguous()) return nullptr;
  const int64_t t = x->size(0), h = x->size(1);
  return t >= 1 && t <= kMaxTokens && h >= multiple && h <= max_hidden && h % multiple == 0 ? x : nullptr;
}

PyObject* quant_fp8(PyObject*, PyObject* const* argv, Py_ssize_t argc) {
  HANDLE_TH_ERRORS
  static const char* const names[] = {"x"};
  PyObject* a[1];
  if (!bind(argv, argc, names, 1, 1, 1, a) || watched()) Py_RETURN_NONE;
  const at::Tensor* x = activations(a[0], 128, kMaxHidden);
  if (!x) Py_RETURN_NONE;
  const int64_t t = x->size(0), h = x->size(1);
  at::Tensor q, s;
  int st;
  {
    pybind11::gil_scoped_release no_gil;
    q = make({t, h}, at::kFloat8_e4m3fn, *x);
    s = make({h / 128, t}, at::kFloat, *x);
    st = aklr_per_group_quant_fp8(x->const_data_ptr(), h, q.mutable_data_ptr(), static_cast<float*>(s.mutable_data_ptr()),
                                  t, h, stream_of(*x));
  }
  return st == AKLR_OK ? pair(q, s) : status_error(st, "per_group_quant_fp8");
  END_HANDLE_TH_ERRORS
}

PyObject* quant_mxfp8(PyObject*, PyObject* const* argv, Py_ssize_t argc) {
  HANDLE_TH_ERRORS
  static const char* const names[] = {"x"};
  PyObject* a[1];
  if (!bind(argv, argc, names, 1, 1, 1, a) || watched()) Py_RETURN_NONE;
  const at::Tensor* x = activations(a[0], 32, kMaxHidden);
  if (!x) Py_RETURN_NONE;
  const int64_t t = x->size(0), h = x->size(1);
  at::Tensor q, s;
  int st;
  {
    pybind11::gil_scoped_release no_gil;
    q = make({t, h}, at::kFloat8_e4m3fn, *x);
    s = make({t, h / 32}, at::kByte, *x);
    st = aklr_per_group_quant_mxfp8(x->const_data_ptr(), h, q.mutable_data_ptr(),
                                    static_cast<uint8_t*>(s.mutable_data_ptr()), t, h, stream_of(*x));
  }
  return st == AKLR_OK ? pair(q, s) : status_error(st, "per_group_quant_mxfp8");
  END_HANDLE_TH_ERRORS
}

PyObject* quant_mxfp4(PyObject*, PyObject* const* argv, Py_ssize_t argc) {
  HANDLE_TH_ERRORS
  static const char* const names[] = {"x", "shuffle"};
  PyObject* a[2];
  if (!bind(argv, argc, names, 2, 2, 1, a) || watched()) Py_RETURN_NONE;
  if (a[1] && a[1] != Py_True && a[1] != Py_False) Py_RETURN_NONE;
  const bool shuffle = a[1] == Py_True;
  const at::Tensor* x = activations(a[0], 32, kMaxHidden4);
  if (!x) Py_RETURN_NONE;
  const int64_t t = x->size(0), h = x->size(1), g = h / 32;
  at::Tensor q, s;
  int st;
  {
    pybind11::gil_scoped_release no_gil;
    q = make({t, h / 2}, at::kFloat4_e2m1fn_x2, *x);
    s = make({shuffle ? (t + 255) / 256 * 256 : t, shuffle ? (g + 7) / 8 * 8 : g}, at::kFloat8_e8m0fnu, *x);
    st = aklr_dynamic_mxfp4_quant(x->const_data_ptr(), h, static_cast<uint8_t*>(q.mutable_data_ptr()),
                                  static_cast<uint8_t*>(s.mutable_data_ptr()), t, h,
                                  shuffle ? AKLR_SCALES_SHUFFLED : AKLR_SCALES_ROW_MAJOR, stream_of(*x));
  }
  return st == AKLR_OK ? pair(q, s) : status_error(st, "dynamic_mxfp4_quant");
  END_HANDLE_TH_ERRORS
}

// ---------------------------------------------------------------------------------------------
// GEMMs
bool gemm_dims(int64_t m, int64_t n, int64_t k, int64_t k_multiple) {
  return m >= 1 && m <= kMaxM && n >= 16 && n <= kMaxN && n % 16 == 0 && k >= k_multiple && k <= kMaxK && k % k_multiple == 0;
}

// bias: none, or fp32 [n] on the operands' device
bool bias_ok(PyObject* o, int64_t n, const at::Tensor& like, const float** data) {
  *data = nullptr;
  if (is_none(o)) return true;
  const at::Tensor* b = plain(o);
  if (!b || b->scalar_type() != at::kFloat || b->dim() != 1 || b->size(0) != n || !b->is_contiguous() ||
      b->device() != like.device())
    return false;
  *data = static_cast<const float*>(b->const_data_ptr());
  return true;
}

bool shape_is(const at::Tensor& t, int64_t r, int64_t c) { return t.dim() == 2 && t.size(0) == r && t.size(1) == c; }

PyObject* gemm_fp8(PyObject*, PyObject* const* argv, Py_ssize_t argc) {
  HANDLE_TH_ERRORS
  static const char* const names[] = {"a", "b", "a_scale", "b_scale", "block_size", "scale_major_mode", "trans_b",
                                      "bias", "out_dtype", "out", "operand_format"};
  PyObject* p[11];
  if (!bind(argv, argc, names, 11, 10, 4, p) || watched()) Py_RETURN_NONE;
  if (!block_ok(p[4]) || (p[6] && p[6] != Py_True) || !is_none(p[9])) Py_RETURN_NONE;
  const bool mn = p[5] && str_is(p[5], "MN");
  if (p[5] && !mn && !str_is(p[5], "K")) Py_RETURN_NONE;
  const bool pre = p[10] && str_is(p[10], "none:preshuffled");
  if (p[10] && !pre && !str_is(p[10], "none:none")) Py_RETURN_NONE;
  at::ScalarType ot;
  const at::Tensor *a = plain(p[0]), *b = plain(p[1]), *sa = plain(p[2]), *sb = plain(p[3]);
  if (!a || !b || !sa || !sb || !out_type(p[8], &ot)) Py_RETURN_NONE;
  bool shuffled = false, row_major_scale = false;
  if (!is_true_attr(p[1], s_is_shuffled, &shuffled) || !is_true_attr(p[2], s_is_row_major, &row_major_scale)) return nullptr;
  if (!pre && shuffled) Py_RETURN_NONE;
  const auto type = a->scalar_type();
  if ((type != at::kFloat8_e4m3fn && type != at::kFloat8_e5m2) || b->scalar_type() != type) Py_RETURN_NONE;
  if (pre && (mn || !is_none(p[7]) || type != at::kFloat8_e4m3fn)) Py_RETURN_NONE;
  if (sa->scalar_type() != at::kFloat || sb->scalar_type() != at::kFloat || a->dim() != 2 || b->dim() != 2) Py_RETURN_NONE;
  const int64_t m = a->size(0), k = a->size(1), n = b->size(0), kb = k / 128;
  if (b->size(1) != k || !gemm_dims(m, n, k, 128) || !a->is_contiguous() || !b->is_contiguous()) Py_RETURN_NONE;
  // preshuffled weights with a_scale not marked row-major: the column-major bytes in the logical shape
  const bool column_major = pre && !row_major_scale;
  if (!shape_is(*sa, mn ? kb : m, mn ? m : kb) || !sa->is_contiguous()) Py_RETURN_NONE;
  if (!shape_is(*sb, (n + 127) / 128, kb) || !sb->is_contiguous()) Py_RETURN_NONE;
  if (b->device() != a->device() || sa->device() != a->device() || sb->device() != a->device()) Py_RETURN_NONE;
  const float* bias;
  if (!bias_ok(p[7], n, *a, &bias)) Py_RETURN_NONE;
  at::Tensor out, ws;
  int st;
  {
    pybind11::gil_scoped_release no_gil;
    out = make({m, n}, ot, *a);
    const size_t bytes = aklr_gemm_a8w8_blockscale_workspace_bytes(m, n, k);
    if (bytes) ws = make({static_cast<int64_t>(bytes)}, at::kByte, *a);
    st = aklr_gemm_a8w8_blockscale(
        a->const_data_ptr(), a->stride(0), b->const_data_ptr(), pre ? k : b->stride(0),
        static_cast<const float*>(sa->const_data_ptr()),
        mn || column_major ? 1 : kb, mn || column_major ? m : 1, static_cast<const float*>(sb->const_data_ptr()),
        sb->stride(0), bias, out.mutable_data_ptr(), n, m, n, k,
        type == at::kFloat8_e4m3fn ? AKLR_FP8_E4M3FN : AKLR_FP8_E5M2, pre ? AKLR_B_PRESHUFFLE_16x16 : AKLR_B_ROW_MAJOR,
        out_code(ot), bytes ? ws.mutable_data_ptr() : nullptr, bytes, stream_of(*a));
  }
  return st == AKLR_OK ? THPVariable_Wrap(out) : status_error(st, "gemm_a8w8_blockwise_scaled");
  END_HANDLE_TH_ERRORS
}

PyObject* quant_gemm_fp8(PyObject*, PyObject* const* argv, Py_ssize_t argc) {
  HANDLE_TH_ERRORS
  static const char* const names[] = {"x", "b", "b_scale", "bias", "out_dtype", "out", "operand_format"};
  PyObject* p[7];
  if (!bind(argv, argc, names, 7, 6, 3, p) || watched()) Py_RETURN_NONE;
  if (!is_none(p[5])) Py_RETURN_NONE;
  const bool pre = p[6] && str_is(p[6], "none:preshuffled");
  if (p[6] && !pre && !str_is(p[6], "none:none")) Py_RETURN_NONE;
  at::ScalarType ot;
  const at::Tensor *x = plain(p[0]), *b = plain(p[1]), *sb = plain(p[2]);
  if (!x || !b || !sb || !out_type(p[4], &ot)) Py_RETURN_NONE;
  bool shuffled = false;
  if (!is_true_attr(p[1], s_is_shuffled, &shuffled)) return nullptr;
  if (!pre && shuffled) Py_RETURN_NONE;
  if (x->scalar_type() != at::kBFloat16 || b->scalar_type() != at::kFloat8_e4m3fn || sb->scalar_type() != at::kFloat ||
      x->dim() != 2 || b->dim() != 2)
    Py_RETURN_NONE;
  const int64_t m = x->size(0), k = x->size(1), n = b->size(0);
  if (b->size(1) != k || !gemm_dims(m, n, k, 128)) Py_RETURN_NONE;
  if (!shape_is(*sb, (n + 127) / 128, k / 128) || !sb->is_contiguous() || !b->is_contiguous()) Py_RETURN_NONE;
  if (x->stride(1) != 1 || x->stride(0) < k || x->stride(0) % 8 != 0) Py_RETURN_NONE;
  if (b->device() != x->device() || sb->device() != x->device()) Py_RETURN_NONE;
  const float* bias;
  if (!bias_ok(p[3], n, *x, &bias)) Py_RETURN_NONE;
  at::Tensor out, ws;
  int st;
  {
    pybind11::gil_scoped_release no_gil;
    out = make({m, n}, ot, *x);
    const size_t bytes = aklr_quant_gemm_a8w8_blockscale_workspace_bytes(m, n, k);
    if (bytes) ws = make({static_cast<int64_t>(bytes)}, at::kByte, *x);
    st = aklr_quant_gemm_a8w8_blockscale(x->const_data_ptr(), x->stride(0), b->const_data_ptr(),
                                         pre ? k : b->stride(0), static_cast<const float*>(sb->const_data_ptr()), sb->stride(0), bias,
                                         out.mutable_data_ptr(), n, m, n, k,
                                         pre ? AKLR_B_PRESHUFFLE_16x16 : AKLR_B_ROW_MAJOR, out_code(ot),
                                         bytes ? ws.mutable_data_ptr() : nullptr, bytes, stream_of(*x));
  }
  return st == AKLR_OK ? THPVariable_Wrap(out) : status_error(st, "quant_gemm_a8w8_blockwise_scaled");
  END_HANDLE_TH_ERRORS
}

bool float_is(PyObject* o, double v) { return !o || (PyFloat_CheckExact(o) && PyFloat_AS_DOUBLE(o) == v); }

PyObject* gemm_mxfp4(PyObject*, PyObject* const* argv, Py_ssize_t argc) {
  HANDLE_TH_ERRORS
  static const char* const names[] = {"a", "b", "a_scale", "b_scale", "alpha", "beta", "trans_b", "bias", "out_dtype",
                                      "out", "operand_format"};
  PyObject* p[11];
  if (!bind(argv, argc, names, 11, 10, 4, p) || watched()) Py_RETURN_NONE;
  if (!float_is(p[4], 1.0) || !float_is(p[5], 0.0) || (p[6] && p[6] != Py_True) || !is_none(p[9])) Py_RETURN_NONE;
  const bool pre = !p[10] || str_is(p[10], "none:preshuffled");
  if (!pre && !str_is(p[10], "none:none")) Py_RETURN_NONE;
  at::ScalarType ot;
  const at::Tensor *a = plain(p[0]), *b = plain(p[1]), *sa = plain(p[2]), *sb = plain(p[3]);
  if (!a || !b || !sa || !sb || !out_type(p[8], &ot)) Py_RETURN_NONE;
  const auto code = [](const at::Tensor& t) { return t.scalar_type() == at::kFloat4_e2m1fn_x2 || t.scalar_type() == at::kByte; };
  const auto scale = [](const at::Tensor& t) { return t.scalar_type() == at::kFloat8_e8m0fnu || t.scalar_type() == at::kByte; };
  if (!code(*a) || !code(*b) || !scale(*sa) || !scale(*sb) || a->dim() != 2 || b->dim() != 2) Py_RETURN_NONE;
  const int64_t m = a->size(0), kh = a->size(1), n = b->size(0), k = 2 * kh, g = k / 32;
  if (b->size(1) != kh || !gemm_dims(m, n, k, 64)) Py_RETURN_NONE;
  const int64_t cols = pre ? (g + 7) / 8 * 8 : g;
  if (!shape_is(*sa, pre ? (m + 255) / 256 * 256 : m, cols) || !shape_is(*sb, pre ? (n + 255) / 256 * 256 : n, cols)) Py_RETURN_NONE;
  for (const at::Tensor* t : {a, b, sa, sb})
    if (!t->is_contiguous() || t->device() != a->device()) Py_RETURN_NONE;
  const float* bias;
  if (!bias_ok(p[7], n, *a, &bias)) Py_RETURN_NONE;
  at::Tensor out, ws;
  int st;
  {
    pybind11::gil_scoped_release no_gil;
    out = make({m, n}, ot, *a);
    const size_t bytes = aklr_gemm_a4w4_mxfp4_workspace_bytes(m, n, k);
    if (bytes) ws = make({static_cast<int64_t>(bytes)}, at::kByte, *a);
    const auto u8 = [](const at::Tensor& t) { return static_cast<const uint8_t*>(t.const_data_ptr()); };
    st = aklr_gemm_a4w4_mxfp4(u8(*a), a->stride(0), u8(*b), b->stride(0), u8(*sa), sa->stride(0), u8(*sb), sb->stride(0),
                              bias, out.mutable_data_ptr(), n, m, n, k,
                              pre ? AKLR_B_PRESHUFFLE_16x16 : AKLR_B_ROW_MAJOR,
                              pre ? AKLR_SCALES_SHUFFLED : AKLR_SCALES_ROW_MAJOR, out_code(ot),
                              bytes ? ws.mutable_data_ptr() : nullptr, bytes, stream_of(*a));
  }
  return st == AKLR_OK ? THPVariable_Wrap(out) : status_error(st, "gemm_a4w4_mxfp4");
  END_HANDLE_TH_ERRORS
}

#define AKLR_HOST_FN(name) \
  {#name, reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)()>(name)), METH_FASTCALL, nullptr}
PyMethodDef kMethods[] = {AKLR_HOST_FN(quant_fp8), AKLR_HOST_FN(quant_mxfp8), AKLR_HOST_FN(quant_mxfp4),
                          AKLR_HOST_FN(gemm_fp8), AKLR_HOST_FN(quant_gemm_fp8), AKLR_HOST_FN(gemm_mxfp4),
                          {nullptr, nullptr, 0, nullptr}};
PyModuleDef kModule = {PyModuleDef_HEAD_INIT, "_host", "the ops' per-call host work", -1, kMethods,
                       nullptr, nullptr, nullptr, nullptr};

}  // namespace

// The checks above read torch's own objects, whose layout belongs to one version.
static bool same_torch() {
  PyObject* torch = PyImport_ImportModule("torch");
  PyObject* version = torch ? PyObject_GetAttrString(torch, "__version__") : nullptr;
  Py_XDECREF(torch);
  if (!version) return false;
  const bool same = PyUnicode_Check(version) && PyUnicode_CompareWithASCIIString(version, AKLR_TORCH_VERSION) == 0;
  if (!same) PyErr_Format(PyExc_ImportError, "built with torch %s, not %S", AKLR_TORCH_VERSION, version);
  Py_DECREF(version);
  return same;
}

PyMODINIT_FUNC PyInit__host() {
  if (!same_torch()) return nullptr;
  if (aklr_abi_version() != 1) {
    PyErr_SetString(PyExc_ImportError, "libaklr_amd.so ABI version does not match aklr_amd._host");
    return nullptr;
  }
  s_is_shuffled = PyUnicode_InternFromString("is_shuffled");
  s_is_row_major = PyUnicode_InternFromString("is_row_major");
  if (!s_is_shuffled || !s_is_row_major) return nullptr;
  return PyModule_Create(&kModule);
}
