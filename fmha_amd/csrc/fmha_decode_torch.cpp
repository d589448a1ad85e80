// fmha_decode_torch.cpp -- the accepted calls of the tensor interface
// (fmha_amd/decode.py) in native code: argument checks, output and workspace,
// the call of the C ABI on torch's current stream.
//
// Each function here takes its Python namesake's arguments by position and
// returns the output tensor, or an int, the error code of a call that the
// library rejected, or None where anything is not plainly acceptable: an
// argument of another type, a shape, stride, device or dtype that a check
// refuses, a tensor subclass, a functorch wrapper, an active torch function
// or dispatch mode.  The caller then runs the Python form, which has the
// error messages and stays the reference for what is accepted.
//
// Why: a call of the Python form spends about 8 us in attribute lookups and
// ctypes before its launch, more than a small call's kernel (µs among other
// calls, B=10 16/16 D=128 lengths up to 16: 10.5 in Python, 5.3
// here).
#define PY_SSIZE_T_CLEAN
#include <Python.h>

#include <ATen/PythonTorchFunctionTLS.h>
#include <ATen/core/Tensor.h>
#include <ATen/hip/impl/HIPStreamMasqueradingAsCUDA.h>
#include <ATen/ops/empty.h>
#include <c10/core/impl/TorchDispatchModeTLS.h>
#include <torch/csrc/autograd/python_variable.h>

#include <cmath>
#include <cstdint>
#include <exception>
#include <optional>

#include "fmha_decode.h"

namespace {

constexpr int64_t kShortRows = FMHA_DECODE_MAX_SEQLEN_KV;

// Entry points of the library the Python side has loaded (bind).
struct Library {
  decltype(&fmha_decode_fwd) fwd = nullptr;
  decltype(&fmha_decode_fwd_fast) fwd_fast = nullptr;
  decltype(&fmha_decode_fwd_fp32_weights) fwd_fp32_weights = nullptr;
  decltype(&fmha_decode_fwd_exact) fwd_exact = nullptr;
  decltype(&fmha_decode_fwd_uniform) fwd_uniform = nullptr;
  decltype(&fmha_decode_fwd_uniform_fast) fwd_uniform_fast = nullptr;
  decltype(&fmha_decode_fwd_strided) fwd_strided = nullptr;
  decltype(&fmha_decode_fwd_paged) fwd_paged = nullptr;
  decltype(&fmha_decode_splitkv_workspace_size) workspace_size = nullptr;
  decltype(&fmha_decode_fwd_splitkv) splitkv = nullptr;
  decltype(&fmha_decode_fwd_splitkv_strided) splitkv_strided = nullptr;
  decltype(&fmha_decode_fwd_splitkv_paged) splitkv_paged = nullptr;
} g_lib;

// Thrown where the Python form has to look at the call.
struct NotPlain {};
inline void need(bool ok) {
  if (!ok) throw NotPlain{};
}

// A strided GPU tensor of exactly torch.Tensor (or Parameter), with no wrapper
// whose data pointer is not the data.
const at::Tensor& plain(PyObject* o) {
  need(THPVariable_CheckExact(o));
  const at::Tensor& t = THPVariable_Unpack(o);
  need(t.defined() && t.is_cuda() && t.layout() == at::kStrided);
  static const c10::DispatchKeySet wrapped({c10::DispatchKey::Python, c10::DispatchKey::PythonTLSSnapshot,
                                            c10::DispatchKey::FuncTorchBatched, c10::DispatchKey::FuncTorchGradWrapper,
                                            c10::DispatchKey::Functionalize, c10::DispatchKey::Batched,
                                            c10::DispatchKey::Conjugate, c10::DispatchKey::Negative,
                                            c10::DispatchKey::ZeroTensor});
  need(!t.key_set().has_any(wrapped));
  return t;
}

int32_t small(int64_t x) {
  need(x >= INT32_MIN && x <= INT32_MAX);
  return (int32_t)x;
}

bool flag(PyObject* o) {
  need(o == Py_True || o == Py_False);
  return o == Py_True;
}

int32_t integer(PyObject* o) {
  need(PyLong_CheckExact(o));
  int overflow = 0;
  const long long x = PyLong_AsLongLongAndOverflow(o, &overflow);
  need(overflow == 0 && !(x == -1 && PyErr_Occurred()));
  return small(x);
}

// The call's query, its output and what they say of the shape.
struct Call {
  const at::Tensor& q;
  int32_t B, Hq, D;
  at::Tensor out;
  PyObject* given_out;  // the caller's, or null
  float scale;
  void* stream;

  Call(PyObject* q_, PyObject* scale_, PyObject* out_) : q(plain(q_)) {
    need(!c10::impl::TorchDispatchModeTLS::any_modes_set() && !at::impl::torch_function_mode_enabled());
    const int64_t dims = q.dim();
    need((dims == 3 || (dims == 4 && q.size(2) == 1)) && q.scalar_type() == at::kBFloat16 && q.is_contiguous());
    B = small(q.size(0));
    Hq = small(q.size(1));
    D = small(q.size(dims - 1));
    need(D > 0);
    if (scale_ == Py_None) {
      scale = (float)(1.0 / std::sqrt((double)D));
    } else {
      need(PyFloat_CheckExact(scale_));
      scale = (float)PyFloat_AS_DOUBLE(scale_);
    }
    if (out_ == Py_None) {
      given_out = nullptr;
    } else {
      out = plain(out_);
      need(out.scalar_type() == at::kHalf && out.sizes() == q.sizes() && out.is_contiguous() && here(out));
      given_out = out_;
    }
    stream = c10::hip::getCurrentHIPStreamMasqueradingAsCUDA(q.device().index()).stream();
  }
  bool here(const at::Tensor& t) const { return t.device() == q.device(); }
  // After every check: the output, allocated where none was given.
  void* output() {
    if (!given_out) out = at::empty(q.sizes(), q.options().dtype(at::kHalf).requires_grad(false));
    return out.data_ptr();
  }
  const int32_t* lengths(PyObject* o, int64_t n) const {
    const at::Tensor& t = plain(o);
    need(t.scalar_type() == at::kInt && t.numel() == n && here(t) && t.is_contiguous());
    return static_cast<const int32_t*>(t.data_ptr());
  }
  at::Tensor workspace(PyObject* o, int32_t hkv, int32_t rows) const {
    if (o != Py_None) {
      const at::Tensor& t = plain(o);
      need(t.scalar_type() == at::kByte && here(t) && t.is_contiguous());
      return t;
    }
    const size_t n = g_lib.workspace_size(B, Hq, hkv, rows, D);
    return at::empty({(int64_t)(n > 1 ? n : 1)}, q.options().dtype(at::kByte).requires_grad(false));
  }
  // K or V of this dtype and device.
  const at::Tensor& cache(PyObject* o) const {
    const at::Tensor& t = plain(o);
    need(t.scalar_type() == at::kBFloat16 && here(t));
    return t;
  }
  PyObject* result(int rc) {
    if (rc != 0) return PyLong_FromLong(rc);
    if (!given_out) return THPVariable_Wrap(out);
    Py_INCREF(given_out);
    return given_out;
  }
};

// Runs the library call without the interpreter lock, as ctypes does.
template <class F>
int unlocked(F f) {
  PyThreadState* s = PyEval_SaveThread();
  const int rc = f();
  PyEval_RestoreThread(s);
  return rc;
}

PyObject* decode(PyObject* const* a) {
  Call c(a[0], a[5], a[6]);
  const at::Tensor &k = c.cache(a[1]), &v = c.cache(a[2]);
  const bool fp32 = flag(a[7]), exact = flag(a[8]), fast = flag(a[9]);
  need((int)fp32 + (int)exact + (int)fast <= 1);
  need((k.dim() == 3 || k.dim() == 4) && k.is_contiguous() && v.is_contiguous() && k.sizes() == v.sizes() &&
       k.size(-1) == c.D);
  const int32_t hkv = small(k.size(-2));
  need(hkv > 0);
  if (a[3] != Py_None) {
    need(k.dim() == 3);
    const int32_t* cu = c.lengths(a[3], (int64_t)c.B + 1);
    void* o = c.output();
    const auto f = fp32 ? g_lib.fwd_fp32_weights : exact ? g_lib.fwd_exact : fast ? g_lib.fwd_fast : g_lib.fwd;
    return c.result(unlocked([&] {
      return f(c.stream, c.q.data_ptr(), k.data_ptr(), v.data_ptr(), o, cu, c.B, c.Hq, hkv, 1, c.D, c.D, c.scale);
    }));
  }
  need(!fp32 && !(exact && c.Hq / hkv > 2));
  int32_t rows;
  if (a[4] == Py_None) {
    need(k.dim() == 4 && k.size(0) == c.B);
    rows = small(k.size(1));
  } else {
    rows = integer(a[4]);
    need(rows >= 0);
  }
  need(k.numel() == (int64_t)c.B * rows * hkv * c.D);
  void* o = c.output();
  const auto f = fast ? g_lib.fwd_uniform_fast : g_lib.fwd_uniform;
  return c.result(unlocked([&] {
    return f(c.stream, c.q.data_ptr(), k.data_ptr(), v.data_ptr(), o, rows, c.B, c.Hq, hkv, 1, c.D, c.D, c.scale);
  }));
}

PyObject* splitkv(PyObject* const* a) {
  Call c(a[0], a[5], a[6]);
  const at::Tensor &k = c.cache(a[1]), &v = c.cache(a[2]);
  need(k.dim() == 3 && k.is_contiguous() && v.is_contiguous() && k.sizes() == v.sizes() && k.size(2) == c.D);
  const int32_t* cu = c.lengths(a[3], (int64_t)c.B + 1);
  const int32_t hkv = small(k.size(1)), rows = integer(a[4]);
  const at::Tensor ws = c.workspace(a[7], hkv, rows);
  void* o = c.output();
  return c.result(unlocked([&] {
    return g_lib.splitkv(c.stream, c.q.data_ptr(), k.data_ptr(), v.data_ptr(), o, cu, rows, c.B, c.Hq, hkv, 1, c.D, c.D,
                         c.scale, ws.data_ptr(), (size_t)ws.numel());
  }));
}

PyObject* strided(PyObject* const* a) {
  Call c(a[0], a[4], a[5]);
  const at::Tensor &k = c.cache(a[1]), &v = c.cache(a[2]);
  need(k.dim() == 4 && k.size(0) == c.B && k.size(3) == c.D && k.stride(3) == 1 && k.sizes() == v.sizes() &&
       k.strides() == v.strides());
  const int32_t rows = small(k.size(1)), hkv = small(k.size(2));
  const int32_t* lens = a[3] == Py_None ? nullptr : c.lengths(a[3], c.B);
  if (rows > kShortRows) {
    const at::Tensor ws = c.workspace(a[6], hkv, rows);
    void* o = c.output();
    return c.result(unlocked([&] {
      return g_lib.splitkv_strided(c.stream, c.q.data_ptr(), k.data_ptr(), v.data_ptr(), o, lens, rows, k.stride(0),
                                   k.stride(1), k.stride(2), c.B, c.Hq, hkv, 1, c.D, c.D, c.scale, ws.data_ptr(),
                                   (size_t)ws.numel());
    }));
  }
  void* o = c.output();
  return c.result(unlocked([&] {
    return g_lib.fwd_strided(c.stream, c.q.data_ptr(), k.data_ptr(), v.data_ptr(), o, lens, rows, k.stride(0),
                             k.stride(1), k.stride(2), c.B, c.Hq, hkv, 1, c.D, c.D, c.scale);
  }));
}

PyObject* paged(PyObject* const* a) {
  Call c(a[0], a[5], a[6]);
  const at::Tensor &k = c.cache(a[1]), &v = c.cache(a[2]);
  need(k.dim() == 4 && k.is_contiguous() && v.is_contiguous() && k.sizes() == v.sizes() && k.size(3) == c.D);
  const at::Tensor& table = plain(a[3]);
  need(table.scalar_type() == at::kInt && table.dim() == 2 && table.size(0) == c.B && table.stride(1) == 1 &&
       c.here(table));
  const int32_t* bt = static_cast<const int32_t*>(table.data_ptr());
  const int32_t bt_stride = small(table.stride(0)), page = small(k.size(1)), hkv = small(k.size(2));
  const int32_t* lens = c.lengths(a[4], c.B);
  need(lens != nullptr);
  if (a[7] != Py_None) {
    const int32_t rows = integer(a[7]);
    const at::Tensor ws = c.workspace(a[8], hkv, rows);
    void* o = c.output();
    return c.result(unlocked([&] {
      return g_lib.splitkv_paged(c.stream, c.q.data_ptr(), k.data_ptr(), v.data_ptr(), o, bt, bt_stride, lens, page,
                                 rows, c.B, c.Hq, hkv, 1, c.D, c.D, c.scale, ws.data_ptr(), (size_t)ws.numel());
    }));
  }
  void* o = c.output();
  return c.result(unlocked([&] {
    return g_lib.fwd_paged(c.stream, c.q.data_ptr(), k.data_ptr(), v.data_ptr(), o, bt, bt_stride, lens, page, c.B,
                           c.Hq, hkv, 1, c.D, c.D, c.scale);
  }));
}

// n positional arguments; no C++ exception leaves.
template <PyObject* (*F)(PyObject* const*), Py_ssize_t N>
PyObject* entry(PyObject*, PyObject* const* args, Py_ssize_t n) {
  if (n != N || !g_lib.fwd) {
    PyErr_Format(PyExc_TypeError, "%zd arguments expected after bind(), got %zd", N, n);
    return nullptr;
  }
  try {
    return F(args);
  } catch (const NotPlain&) {
    PyErr_Clear();
  } catch (const c10::OutOfMemoryError&) {
    // The Python form raises it as torch does.
  } catch (const std::exception&) {
  }
  Py_RETURN_NONE;
}

// bind(addresses): those of Library's members, in order.
PyObject* bind(PyObject*, PyObject* const* args, Py_ssize_t n) {
  constexpr Py_ssize_t kCount = sizeof(Library) / sizeof(void*);
  if (n != kCount) {
    PyErr_Format(PyExc_TypeError, "bind takes %zd addresses, got %zd", kCount, n);
    return nullptr;
  }
  void* p[kCount];
  for (Py_ssize_t i = 0; i < n; ++i) {
    p[i] = PyLong_AsVoidPtr(args[i]);
    if (!p[i]) {
      if (!PyErr_Occurred()) PyErr_SetString(PyExc_ValueError, "null address");
      return nullptr;
    }
  }
  static_assert(sizeof(Library) == sizeof(p), "Library holds function pointers only");
  __builtin_memcpy(static_cast<void*>(&g_lib), p, sizeof(p));
  Py_RETURN_NONE;
}

#define FMHA_DECODE_METHOD(name, fn) {name, reinterpret_cast<PyCFunction>(fn), METH_FASTCALL, nullptr}
PyMethodDef methods[] = {
    FMHA_DECODE_METHOD("bind", static_cast<PyObject* (*)(PyObject*, PyObject* const*, Py_ssize_t)>(bind)),
    FMHA_DECODE_METHOD("decode", (entry<decode, 10>)),
    FMHA_DECODE_METHOD("splitkv", (entry<splitkv, 8>)),
    FMHA_DECODE_METHOD("strided", (entry<strided, 7>)),
    FMHA_DECODE_METHOD("paged", (entry<paged, 9>)),
    {nullptr, nullptr, 0, nullptr},
};
PyModuleDef module = {PyModuleDef_HEAD_INIT, "_host", nullptr, -1, methods, nullptr, nullptr, nullptr, nullptr};

}  // namespace

PyMODINIT_FUNC PyInit__host(void) { return PyModule_Create(&module); }
