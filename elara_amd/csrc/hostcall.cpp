// Host side of the row ops' Python entry points: the argument checks and the C-ABI call of ops.gpu_adam,
// gpu_ops.init_rows and gpu_ops.replay_rows in one native call, for the arguments a training loop passes (plain
// contiguous GPU tensors of the expected types on the current device).  Everything else -- other types, strides or
// devices, arenas in host memory, wrapped tensors, errors -- is answered with NOT_TAKEN, and the Python path then
// converts, raises or runs as it always has, so the two accept and refuse the same calls.
//
// Why: at a few hundred rows a call is host time.  The Python checks and ctypes conversions of gpu_adam took 3.7 of its
// 7.5 us (600 rows of width 32), those of replay_rows 8 of 13.5 (5,000 rows); the calls here take 4.1 and 6.0 us.
//
// The library's entry points are handed over by address (bind), so this module calls the library that ctypes loaded.
#define PY_SSIZE_T_CLEAN
#include <Python.h>

#include <cstring>

#include <ATen/ops/empty.h>
#include <c10/core/DefaultDtype.h>
#include <c10/hip/HIPStream.h>
#include <torch/csrc/autograd/python_variable.h>

#include "../../include/elara_amd.h"

namespace {

using adam_scalars_t = decltype(&elr_adam_scalars);
using adam_rows_t = decltype(&elr_adam_rows);
using init_rows_t = decltype(&elr_init_rows);
using replay_rows_t = decltype(&elr_replay_rows);
adam_scalars_t f_scalars = nullptr;
adam_rows_t f_adam = nullptr;
init_rows_t f_init = nullptr;
replay_rows_t f_replay = nullptr;

constexpr int kNotTaken = -1000;

PyObject* not_taken() { return PyLong_FromLong(kNotTaken); }

// A plain dense GPU tensor: no subclass, no functorch or functional wrapper, no lazy negation or conjugation, strided
// and contiguous.
const at::Tensor* plain(PyObject* o) {
  if (!THPVariable_CheckExact(o)) return nullptr;
  const at::Tensor& t = THPVariable_Unpack(o);
  if (!t.defined() || !t.is_cuda() || t.layout() != at::kStrided || !t.has_storage()) return nullptr;
  constexpr c10::DispatchKeySet wrapped({c10::DispatchKey::FuncTorchBatched, c10::DispatchKey::FuncTorchGradWrapper,
                                         c10::DispatchKey::Functionalize, c10::DispatchKey::Python,
                                         c10::DispatchKey::Negative, c10::DispatchKey::Conjugate,
                                         c10::DispatchKey::ZeroTensor});
  if (t.key_set().has_any(wrapped) || !t.is_contiguous()) return nullptr;
  return &t;
}

bool real(PyObject* o, double& v) {
  v = PyFloat_AsDouble(o);
  if (v == -1.0 && PyErr_Occurred()) {
    PyErr_Clear();
    return false;
  }
  return true;
}

bool integer(PyObject* o, int64_t& v) {   // an int that fits (anything else is the Python path's to convert)
  if (!PyLong_CheckExact(o)) return false;
  int over = 0;
  v = PyLong_AsLongLongAndOverflow(o, &over);
  return !over;
}

// Other Python threads run while torch allocates and the library launches, as they do through torch and ctypes.  (The
// caller's frame keeps the arguments alive.)
struct NoGil {
  PyThreadState* s = PyEval_SaveThread();
  NoGil() = default;
  NoGil(const NoGil&) = delete;
  ~NoGil() { PyEval_RestoreThread(s); }
};

// The current stream of the current device, if that is t's device.
bool stream_on(const at::Tensor& t, void*& st) {
  const auto s = c10::hip::getCurrentHIPStream();   // of the current device
  if (s.device_index() != t.device().index()) return false;
  st = s.stream();
  return true;
}

PyObject* bind(PyObject*, PyObject* args) {
  unsigned long long a, b, c, d;
  if (!PyArg_ParseTuple(args, "KKKK", &a, &b, &c, &d)) return nullptr;
  f_scalars = reinterpret_cast<adam_scalars_t>(a);
  f_adam = reinterpret_cast<adam_rows_t>(b);
  f_init = reinterpret_cast<init_rows_t>(c);
  f_replay = reinterpret_cast<replay_rows_t>(d);
  Py_RETURN_NONE;
}

// adam(pool, slots, grad, lr, b1, b2, eps, step) -> return code, or NOT_TAKEN
PyObject* adam(PyObject*, PyObject* const* a, Py_ssize_t na) {
  if (na != 8 || !f_adam) return not_taken();
  const at::Tensor *pool = plain(a[0]), *slots = plain(a[1]), *grad = plain(a[2]);
  double lr, b1, b2, eps;
  int64_t step;
  if (!pool || !slots || !grad || !real(a[3], lr) || !real(a[4], b1) || !real(a[5], b2) || !real(a[6], eps) ||
      !integer(a[7], step))
    return not_taken();
  const auto it = slots->scalar_type();
  if (pool->scalar_type() != at::kFloat || pool->dim() != 3 || pool->size(1) != 3 ||
      (it != at::kInt && it != at::kLong) || grad->scalar_type() != at::kFloat || slots->device() != pool->device() ||
      grad->device() != pool->device())
    return not_taken();
  const int64_t n = slots->numel(), D = pool->size(2);
  if (n == 0 || D == 0 || grad->numel() != n * D) return not_taken();
  int rc = kNotTaken;
  try {
    NoGil g;
    void* st;
    if (stream_on(*pool, st)) {
      float sc[8];
      f_scalars(lr, b1, b2, eps, step, sc);
      rc = f_adam(static_cast<float*>(pool->data_ptr()), pool->size(0), slots->data_ptr(), it == at::kLong,
                  static_cast<const float*>(grad->data_ptr()), n, D, sc, st);
    }
  } catch (const std::exception&) {   // torch's own error comes from the Python path
    return not_taken();
  }
  return PyLong_FromLong(rc);
}

// The result [n, 3, D] on rows' device, as torch.empty(n, 3, D, device=...) makes it with the default type float32.
bool new_states(const at::Tensor& rows, int64_t D, at::Tensor& out) {
  if (c10::get_default_dtype_as_scalartype() != at::kFloat) return false;
  out = at::empty({rows.numel(), 3, D}, at::TensorOptions().dtype(at::kFloat).device(rows.device()));
  return true;
}

// init(rows, D, seed, bound) -> (return code, out), or NOT_TAKEN
PyObject* init(PyObject*, PyObject* const* a, Py_ssize_t na) {
  if (na != 4 || !f_init) return not_taken();
  const at::Tensor* rows = plain(a[0]);
  int64_t D, seed;
  double bound;
  if (!rows || rows->scalar_type() != at::kLong || !integer(a[1], D) || D < 1 || !integer(a[2], seed) ||
      !real(a[3], bound) || rows->numel() == 0)
    return not_taken();
  try {
    at::Tensor out;
    int rc = kNotTaken;
    {
      NoGil g;
      void* st;
      if (stream_on(*rows, st) && new_states(*rows, D, out))
        rc = f_init(static_cast<float*>(out.data_ptr()), static_cast<const int64_t*>(rows->data_ptr()),
                    rows->numel(), D, static_cast<uint32_t>(seed), static_cast<float>(bound), st);
    }
    if (rc == kNotTaken) return not_taken();
    return Py_BuildValue("(iN)", rc, THPVariable_Wrap(out));
  } catch (const std::exception&) {
    return not_taken();
  }
}

// replay(rows, logs, offs, steps, cnt, D, K, seed, bound, table, recip) -> (return code, out), or NOT_TAKEN
PyObject* replay(PyObject*, PyObject* const* a, Py_ssize_t na) {
  if (na != 11 || !f_replay) return not_taken();
  const at::Tensor* t[5];
  for (int i = 0; i < 5; ++i)
    if (!(t[i] = plain(a[i]))) return not_taken();
  const at::Tensor *table = plain(a[9]), *recip = plain(a[10]);
  const at::Tensor &rows = *t[0], &logs = *t[1], &offs = *t[2], &steps = *t[3], &cnt = *t[4];
  int64_t D, K, seed;
  double bound;
  if (!table || !recip || !integer(a[5], D) || D < 1 || !integer(a[6], K) || K < 1 || K > 8 || !integer(a[7], seed) ||
      !real(a[8], bound))
    return not_taken();
  const int64_t n = rows.numel();
  if (rows.scalar_type() != at::kLong || logs.scalar_type() != at::kFloat || offs.scalar_type() != at::kLong ||
      steps.scalar_type() != at::kInt || cnt.scalar_type() != at::kInt || table->scalar_type() != at::kFloat ||
      recip->scalar_type() != at::kDouble || n == 0 || offs.numel() != n || cnt.numel() != n ||
      steps.numel() != n * K || logs.numel() % D || table->dim() != 2 || table->size(1) != 8 || recip->dim() != 2 ||
      recip->size(0) != table->size(0) || recip->size(1) != 2)
    return not_taken();
  for (const at::Tensor* x : {&logs, &offs, &steps, &cnt, table, recip})
    if (x->device() != rows.device()) return not_taken();
  try {
    at::Tensor out;
    int rc = kNotTaken;
    {
      NoGil g;
      void* st;
      if (stream_on(rows, st) && new_states(rows, D, out))
        rc = f_replay(static_cast<float*>(out.data_ptr()), static_cast<const int64_t*>(rows.data_ptr()),
                      static_cast<const float*>(logs.data_ptr()), logs.numel() / D,
                      static_cast<const int64_t*>(offs.data_ptr()), static_cast<const int32_t*>(steps.data_ptr()),
                      static_cast<const int32_t*>(cnt.data_ptr()), n, D, static_cast<int>(K),
                      static_cast<uint32_t>(seed), static_cast<float>(bound),
                      static_cast<const float*>(table->data_ptr()), static_cast<const double*>(recip->data_ptr()),
                      table->size(0), st);
    }
    if (rc == kNotTaken) return not_taken();
    return Py_BuildValue("(iN)", rc, THPVariable_Wrap(out));
  } catch (const std::exception&) {
    return not_taken();
  }
}

#define ELR_STR1(x) #x
#define ELR_STR(x) ELR_STR1(x)
#define ELR_FAST(f) reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)()>(f))
PyMethodDef methods[] = {{"bind", bind, METH_VARARGS, "Addresses of the library's entry points."},
                         {"adam", ELR_FAST(adam), METH_FASTCALL, "elr_adam_rows with gpu_adam's checks."},
                         {"init", ELR_FAST(init), METH_FASTCALL, "elr_init_rows into a new tensor."},
                         {"replay", ELR_FAST(replay), METH_FASTCALL, "elr_replay_rows into a new tensor."},
                         {nullptr, nullptr, 0, nullptr}};
PyModuleDef module = {PyModuleDef_HEAD_INIT, "_hostcall", nullptr, -1, methods, nullptr, nullptr, nullptr, nullptr};

}  // namespace

// The file's name carries neither version, and another Python's or torch's objects are laid out differently: the former is
// refused here, the latter by the caller (elara_amd/_lib.py: host), both before any tensor is touched.
PyMODINIT_FUNC PyInit__hostcall() {
  constexpr const char built[] = ELR_STR(PY_MAJOR_VERSION) "." ELR_STR(PY_MINOR_VERSION) ".";
  if (std::strncmp(Py_GetVersion(), built, sizeof built - 1) != 0) {
    PyErr_Format(PyExc_ImportError, "_hostcall was built for Python %sx", built);
    return nullptr;
  }
  PyObject* m = PyModule_Create(&module);
  if (m) {
    PyModule_AddIntConstant(m, "NOT_TAKEN", kNotTaken);
    PyModule_AddStringConstant(m, "TORCH", ELR_TORCH_VERSION);
  }
  return m;
}
