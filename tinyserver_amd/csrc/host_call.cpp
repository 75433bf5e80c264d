// The Python side of libtsa.so's calls: _tsa_host.call(entry, *args) turns
// tensors into tsa_view structs, calls the C entry point and returns its
// status. Packing a view in Python and passing it through ctypes costs about
// 1 us a tensor, which bounds the eager calls of small batches: the fused
// decode step (12 tensors) took 17.3 us a call with 9.0 us of GPU work.
//
// Arguments are told apart by type, in the C entry point's order: a tensor or
// None is a view (None: NULL), a float a double, an int an integer or a
// pointer. Only exact torch.Tensor and Parameter objects are taken here: with
// any other tensor type the result is None and the caller takes the general
// (ctypes) route.
#include <Python.h>
#include <torch/csrc/Exceptions.h>
#include <torch/csrc/autograd/python_variable.h>

#include "tsa_api.h"

namespace {

enum Entry { kDecode, kDecodeStep, kNormRope, kNormRopeStore, kPrefill, kMixed, kSample, kSampleWs };
struct Shape { const char* name; int views, doubles, ints; };
constexpr Shape kShapes[] = {
    {"tsa_paged_decode", 6, 1, 4},      {"tsa_paged_decode_step", 12, 2, 4}, {"tsa_qk_norm_rope", 8, 1, 1},
    {"tsa_qk_norm_rope_store", 14, 1, 1}, {"tsa_varlen_prefill", 6, 1, 4},   {"tsa_mixed_attention", 11, 2, 6},
    {"tsa_sample_tokens", 6, 0, 1},     {"tsa_sample_tokens_ws", 6, 0, 3},
};
constexpr int kEntries = sizeof(kShapes) / sizeof(kShapes[0]);
constexpr int kMaxViews = 16, kMaxDoubles = 4, kMaxInts = 8;

// A tensor's view, as _lib.view describes it. False with a Python error set
// for a rank or dtype that has none.
bool make_view(const at::Tensor& t, tsa_view& v) {
  const int64_t nd = t.dim();
  if (nd > 4) {
    PyErr_Format(PyExc_ValueError, "tensors of rank > 4 are not supported (got %lld)", static_cast<long long>(nd));
    return false;
  }
  switch (t.scalar_type()) {
    case at::kBFloat16: v.dtype = TSA_BF16; break;
    case at::kHalf: v.dtype = TSA_F16; break;
    case at::kFloat: v.dtype = TSA_F32; break;
    case at::kInt: v.dtype = TSA_I32; break;
    case at::kLong: v.dtype = TSA_I64; break;
    default:
      PyErr_Format(PyExc_ValueError, "unsupported dtype %s", c10::toString(t.scalar_type()));
      return false;
  }
  v.data = t.numel() ? t.data_ptr() : nullptr;
  v.ndim = static_cast<int32_t>(nd);
  const auto sizes = t.sizes(), strides = t.strides();
  for (int64_t d = 0; d < 4; ++d) {
    v.size[d] = d < nd ? sizes[d] : 0;
    v.stride[d] = d < nd ? strides[d] : 0;
  }
  return true;
}

int run(int e, const tsa_view* const* v, const double* d, const int64_t* i) {
  auto p = [&](int k) { return reinterpret_cast<void*>(i[k]); };
  auto i32 = [&](int k) { return static_cast<int32_t>(i[k]); };
  switch (e) {
    case kDecode:
      return tsa_paged_decode(v[0], v[1], v[2], v[3], v[4], v[5], d[0], p(0), static_cast<size_t>(i[1]), i32(2), p(3));
    case kDecodeStep:
      return tsa_paged_decode_step(v[0], v[1], v[2], v[3], v[4], v[5], v[6], v[7], d[0], v[8], v[9], v[10], v[11], d[1],
                                   p(0), static_cast<size_t>(i[1]), i32(2), p(3));
    case kNormRope:
      return tsa_qk_norm_rope(v[0], v[1], v[2], v[3], v[4], v[5], v[6], v[7], d[0], p(0));
    case kNormRopeStore:
      return tsa_qk_norm_rope_store(v[0], v[1], v[2], v[3], v[4], v[5], v[6], v[7], v[8], d[0], v[9], v[10], v[11],
                                    v[12], v[13], p(0));
    case kPrefill:
      return tsa_varlen_prefill(v[0], v[1], v[2], v[3], v[4], v[5], i[0], i[1], i32(2), d[0], p(3));
    case kMixed:
      return tsa_mixed_attention(v[0], v[1], v[2], v[3], v[4], i[0], d[0], v[5], v[6], v[7], v[8], v[9], v[10], d[1],
                                 p(1), static_cast<size_t>(i[2]), i32(3), i32(4), p(5));
    case kSample:
      return tsa_sample_tokens(v[0], v[1], v[2], v[3], v[4], v[5], p(0));
    default:
      return tsa_sample_tokens_ws(v[0], v[1], v[2], v[3], v[4], v[5], p(0), static_cast<size_t>(i[1]), p(2));
  }
}

PyObject* call(PyObject*, PyObject* const* args, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  const long e = n > 0 ? PyLong_AsLong(args[0]) : -1;
  if (e == -1 && PyErr_Occurred()) return nullptr;
  if (e < 0 || e >= kEntries) {
    PyErr_SetString(PyExc_ValueError, "no such entry point");
    return nullptr;
  }
  tsa_view views[kMaxViews];
  const tsa_view* pv[kMaxViews];
  double d[kMaxDoubles];
  int64_t ints[kMaxInts];
  int nv = 0, nd = 0, ni = 0;
  for (Py_ssize_t k = 1; k < n; ++k) {
    PyObject* const a = args[k];
    if (nv == kMaxViews || nd == kMaxDoubles || ni == kMaxInts) break;  // (the count below then differs)
    if (a == Py_None) {
      pv[nv++] = nullptr;
    } else if (PyFloat_Check(a)) {
      d[nd++] = PyFloat_AS_DOUBLE(a);
    } else if (PyLong_Check(a)) {
      int over = 0;
      int64_t x = PyLong_AsLongLongAndOverflow(a, &over);
      if (over > 0) x = static_cast<int64_t>(PyLong_AsUnsignedLongLong(a));  // (a handle past 2^63)
      if (PyErr_Occurred()) return nullptr;
      ints[ni++] = x;
    } else if (THPVariable_CheckExact(a)) {
      if (!make_view(THPVariable_Unpack(a), views[nv])) return nullptr;
      pv[nv] = &views[nv];
      ++nv;
    } else {
      Py_RETURN_NONE;
    }
  }
  const Shape& s = kShapes[e];
  if (nv != s.views || nd != s.doubles || ni != s.ints) {
    PyErr_Format(PyExc_TypeError, "%s takes %d tensors, %d floats and %d ints", s.name, s.views, s.doubles, s.ints);
    return nullptr;
  }
  int rc;
  Py_BEGIN_ALLOW_THREADS
  rc = run(static_cast<int>(e), pv, d, ints);
  Py_END_ALLOW_THREADS
  return PyLong_FromLong(rc);
  END_HANDLE_TH_ERRORS
}

// The index of the one GPU every given tensor (None aside) lives on, or -1
// where that does not hold or cannot be said here (the caller finds out
// which and raises).
PyObject* device_index(PyObject*, PyObject* const* args, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  long idx = -1;
  for (Py_ssize_t k = 0; k < n; ++k) {
    if (args[k] == Py_None) continue;
    if (!THPVariable_CheckExact(args[k])) return PyLong_FromLong(-1);
    const at::Device dev = THPVariable_Unpack(args[k]).device();
    if (!dev.is_cuda() || !dev.has_index() || (idx >= 0 && dev.index() != idx)) return PyLong_FromLong(-1);
    idx = dev.index();
  }
  return PyLong_FromLong(idx);
  END_HANDLE_TH_ERRORS
}

// The entry points call() knows, in order.
PyObject* entries(PyObject*, PyObject*) {
  PyObject* t = PyTuple_New(kEntries);
  for (int e = 0; t && e < kEntries; ++e) PyTuple_SET_ITEM(t, e, PyUnicode_FromString(kShapes[e].name));
  return t;
}

PyMethodDef kMethods[] = {
    {"call", reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)()>(call)), METH_FASTCALL, nullptr},
    {"device_index", reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)()>(device_index)), METH_FASTCALL, nullptr},
    {"entries", entries, METH_NOARGS, nullptr},
    {nullptr, nullptr, 0, nullptr},
};
PyModuleDef kModule = {PyModuleDef_HEAD_INIT, "_tsa_host", nullptr, -1, kMethods, nullptr, nullptr, nullptr, nullptr};

}  // namespace

PyMODINIT_FUNC PyInit__tsa_host() { return PyModule_Create(&kModule); }
