// The operators of beam/_C.py for the ordinary call: plain torch tensors, no tile named, nothing to report.
//
// A call of a small product is bound by the host: through ctypes, 5.1 us for gemmrc at 64^3, of which the launch takes 3.3 and
// the rest is attribute look-ups on three tensors and the conversion of ten arguments.  Here the tensors' fields are read
// where they lie.  Same machine, us for a call returning, through ctypes -> here: gemmrc and matmul 5.1 -> 3.1, split-K 6.0 ->
// 3.6, GEMM+LayerNorm 7.1 -> 3.8 (checked, with the wait for the result, 19.3 -> 15.4), GEMM and SiLU 9.1 (two launches) -> 4.4.
//
// Every function returns the library's status (0: done), or kNotHandled before anything is launched: beam/_C.py then takes its
// general path, which also words the errors.  So nothing here has to be complete, and nothing here may differ from there.
// The interpreter's lock is released around the library's calls, as ctypes does.
#define PY_SSIZE_T_CLEAN
#include <Python.h>

#include <ATen/core/Tensor.h>
#include <c10/hip/HIPStream.h>
#include <torch/csrc/autograd/python_variable.h>

#include <climits>
#include <cstdint>

#include "../../include/beam_hip.h"

namespace {

constexpr long kNotHandled = -1;
constexpr long kFellBack = -2;  // gemmrc_ln: the call repeated itself as two passes

struct View {
  void* ptr;
  const int64_t* size;
  int64_t numel;
  int dims;
  int dtype;
};

// What _C._describe tells of a torch tensor; false: not an ordinary one.  (Subclasses, and wrappers without memory of their
// own, whose pointer throws, are the general path's.)
bool describe(PyObject* o, View* v) {
  if (!THPVariable_CheckExact(o)) return false;
  const at::Tensor& t = THPVariable_Unpack(o);
  if (!t.defined() || !t.is_cuda() || t.layout() != at::kStrided || !t.is_contiguous()) return false;
  const at::ScalarType s = t.scalar_type();
  if (s == at::kHalf) v->dtype = BEAM_F16;
  else if (s == at::kBFloat16) v->dtype = BEAM_BF16;
  else return false;
  v->ptr = t.data_ptr();
  v->size = t.sizes().data();
  v->dims = (int)t.dim();
  v->numel = t.numel();
  return true;
}

struct Problem {
  View a, b, c;
  int M, N, K;
  void* stream;
};

// [M, K] x [N, K] (or [K, N]) -> [M, N] of one type, and where a launch goes: the current device's current stream.
bool problem(PyObject* const* args, bool b_kmajor, Problem* q) {
  if (!describe(args[0], &q->a) || !describe(args[1], &q->b) || !describe(args[2], &q->c)) return false;
  if (q->a.dims != 2 || q->b.dims != 2 || q->c.dims != 2 || q->a.dtype != q->b.dtype || q->a.dtype != q->c.dtype) return false;
  const int64_t M = q->a.size[0], K = q->a.size[1], N = q->b.size[b_kmajor ? 1 : 0];
  if (q->b.size[b_kmajor ? 0 : 1] != K || q->c.size[0] != M || q->c.size[1] != N || M > INT_MAX || N > INT_MAX || K > INT_MAX) return false;
  q->M = (int)M;
  q->N = (int)N;
  q->K = (int)K;
  q->stream = c10::hip::getCurrentHIPStream().stream();
  return true;
}

// Runs f, which returns a status or kNotHandled, and hands its value on.  Whatever a tensor throws is left to the general path.
template <typename F>
PyObject* status_of(F f) {
  long s = kNotHandled;
  try {
    s = f();
  } catch (...) {
  }
  if (PyErr_Occurred()) PyErr_Clear();
  return PyLong_FromLong(s);
}

PyObject* gemmrc(PyObject*, PyObject* const* args, Py_ssize_t n) {
  return status_of([&]() -> long {
    Problem q;
    if (n != 3 || !problem(args, false, &q)) return kNotHandled;
    int rc;
    Py_BEGIN_ALLOW_THREADS;
    rc = beam_gemmrc(q.a.ptr, q.b.ptr, q.c.ptr, q.M, q.N, q.K, q.a.dtype, nullptr, q.stream);
    Py_END_ALLOW_THREADS;
    return rc;
  });
}

PyObject* matmul(PyObject*, PyObject* const* args, Py_ssize_t n) {
  return status_of([&]() -> long {
    Problem q;
    if (n != 3 || !problem(args, true, &q)) return kNotHandled;
    int rc;
    Py_BEGIN_ALLOW_THREADS;
    rc = beam_matmul_nn(q.a.ptr, q.b.ptr, q.c.ptr, q.M, q.N, q.K, q.a.dtype, nullptr, q.stream);
    Py_END_ALLOW_THREADS;
    return rc;
  });
}

// (a, b, c, workspace, its bytes): the library's choice of tile and slices
PyObject* gemmrc_splitk(PyObject*, PyObject* const* args, Py_ssize_t n) {
  return status_of([&]() -> long {
    Problem q;
    if (n != 5 || !problem(args, false, &q)) return kNotHandled;
    void* const ws = PyLong_AsVoidPtr(args[3]);
    const size_t ws_bytes = PyLong_AsSize_t(args[4]);
    if (PyErr_Occurred()) return kNotHandled;
    const int s = beam_splitk_effective(q.M, q.N, q.K, nullptr, 0);
    if (s < 0 || (s > 1 && beam_splitk_workspace_bytes(q.M, q.N, s) > ws_bytes)) return kNotHandled;
    int rc;
    Py_BEGIN_ALLOW_THREADS;
    rc = beam_gemmrc_splitk(q.a.ptr, q.b.ptr, q.c.ptr, q.M, q.N, q.K, q.a.dtype, nullptr, 0, s > 1 ? ws : nullptr, s > 1 ? ws_bytes : 0, q.stream);
    Py_END_ALLOW_THREADS;
    return rc;
  });
}

// (a, b, c, gamma, beta, eps, check, workspace, its bytes): BEAM_LN_AUTO
PyObject* gemmrc_ln(PyObject*, PyObject* const* args, Py_ssize_t n) {
  return status_of([&]() -> long {
    Problem q;
    View g, bt;
    if (n != 9 || !problem(args, false, &q) || !describe(args[3], &g) || !describe(args[4], &bt)) return kNotHandled;
    if (g.dims != 1 || bt.dims != 1 || g.size[0] != q.N || bt.size[0] != q.N || g.dtype != q.a.dtype || bt.dtype != q.a.dtype) return kNotHandled;
    const double eps = PyFloat_AsDouble(args[5]);
    const int check = PyObject_IsTrue(args[6]);
    void* const ws = PyLong_AsVoidPtr(args[7]);
    const size_t ws_bytes = PyLong_AsSize_t(args[8]);
    if (PyErr_Occurred()) return kNotHandled;
    const bool aligned = (((uintptr_t)q.a.ptr | (uintptr_t)q.b.ptr | (uintptr_t)q.c.ptr) & 15) == 0 && (((uintptr_t)g.ptr | (uintptr_t)bt.ptr) & 7) == 0;
    int rc, fell_back = 0;
    bool room;
    Py_BEGIN_ALLOW_THREADS;
    // (the query may be the first call of the process and set the device up)
    room = ws && ws_bytes >= (aligned ? beam_gemmrc_ln_workspace_bytes_for(q.M, q.N, q.K, nullptr, BEAM_LN_AUTO)
                                      : beam_gemmrc_ln_workspace_bytes_ex(q.M, q.N, nullptr, BEAM_LN_AUTO));
    rc = !room ? 0
         : check ? beam_gemmrc_ln_checked(q.a.ptr, q.b.ptr, g.ptr, bt.ptr, (float)eps, q.c.ptr, q.M, q.N, q.K, q.a.dtype, nullptr, ws, ws_bytes,
                                          q.stream, &fell_back)
                 : beam_gemmrc_ln_ex(q.a.ptr, q.b.ptr, g.ptr, bt.ptr, (float)eps, q.c.ptr, q.M, q.N, q.K, q.a.dtype, nullptr, BEAM_LN_AUTO, ws,
                                     ws_bytes, q.stream);
    Py_END_ALLOW_THREADS;
    return !room ? kNotHandled : rc == 0 && fell_back ? kFellBack : rc;
  });
}

// (a, b, c, x, y)
PyObject* parallel_gemmrc_silu(PyObject*, PyObject* const* args, Py_ssize_t n) {
  return status_of([&]() -> long {
    Problem q;
    View x, y;
    if (n != 5 || !problem(args, false, &q) || !describe(args[3], &x) || !describe(args[4], &y)) return kNotHandled;
    if (x.numel != y.numel || x.dtype != q.a.dtype || y.dtype != q.a.dtype) return kNotHandled;
    int rc;
    Py_BEGIN_ALLOW_THREADS;
    rc = beam_parallel_gemmrc_silu(q.a.ptr, q.b.ptr, q.c.ptr, q.M, q.N, q.K, x.ptr, y.ptr, x.numel, q.a.dtype, nullptr, q.stream);
    Py_END_ALLOW_THREADS;
    return rc;
  });
}

#define BEAM_METHOD(name) {#name, (PyCFunction)(void (*)(void))name, METH_FASTCALL, nullptr}
PyMethodDef kMethods[] = {BEAM_METHOD(gemmrc),    BEAM_METHOD(matmul),
                          BEAM_METHOD(gemmrc_splitk), BEAM_METHOD(gemmrc_ln),
                          BEAM_METHOD(parallel_gemmrc_silu), {nullptr, nullptr, 0, nullptr}};
PyModuleDef kModule = {PyModuleDef_HEAD_INIT, "_torch_binding", nullptr, -1, kMethods, nullptr, nullptr, nullptr, nullptr};

}  // namespace

PyMODINIT_FUNC PyInit__torch_binding() { return PyModule_Create(&kModule); }
