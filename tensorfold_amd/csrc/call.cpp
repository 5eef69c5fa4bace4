// The launching entry points of include/tfmi.h as Python functions, for _lib.call: the arguments go from the interpreter to the
// library without ctypes, which converted each of a launch's 8 to 24 through an object of its own (2 to 3 us a launch; the decode
// layer of one row and the norm with q, k and v are bound by the host).  A pointer is a tensor, an int or None, a table of
// them a list, a whole number whatever has an __index__.  Raises what ctypes' caller raised: RuntimeError with the library's sentence; and what torch raises for the results that
// are made here: torch.OutOfMemoryError where a device is full.

#define PY_SSIZE_T_CLEAN
#include <Python.h>
#include <dlfcn.h>

#include <ATen/ops/empty.h>
#include <torch/csrc/Exceptions.h>
#include <torch/csrc/autograd/python_variable.h>

#include <cstdint>
#include <exception>
#include <optional>
#include <tuple>
#include <type_traits>
#include <utility>
#include <vector>

#include "../../include/tfmi.h"

#ifndef TF_CALL_ID
#define TF_CALL_ID "unknown"
#endif
#ifndef TF_CALL_FOR
#define TF_CALL_FOR "unknown"
#endif

namespace {

#define TF_ENTRIES(X)                                                                                                        \
  X(tf_qmm_pack) X(tf_qmm_unpack) X(tf_group_sums) X(tf_qmm) X(tf_qmm_own_sums) X(tf_qmm_static) X(tf_qmm_group)            \
  X(tf_qmm_prefill) X(tf_quantize_rows) X(tf_qmm_prefill8) X(tf_experts_pack) X(tf_experts_unpack) X(tf_experts_plan)       \
  X(tf_experts_run) X(tf_experts_run_desc) X(tf_experts_prefill) X(tf_moe_route_up) X(tf_moe_down_combine)                  \
  X(tf_moe_decode_sliced) X(tf_moe_route_decode) X(tf_moe_decode_experts) X(tf_moe_router) X(tf_moe_topk) X(tf_moe_combine) \
  X(tf_exl3x_rot_in) X(tf_exl3x_grouped) X(tf_exl3x_gateup_epilogue) X(tf_exl3x_down_combine) X(tf_exl3x_plan_rot_in)       \
  X(tf_add_norm) X(tf_exl3_rot_in) X(tf_exl3_linear) X(tf_exl3_rot_in_stacked) X(tf_exl3_linear_stacked) X(tf_exl3_gate_up) \
  X(tf_exl3_swiglu_rot_in) X(tf_exl3_unpack) X(tf_exl3_unpack_k8) X(tf_exl3_rot_in_unpack_k8) \
  X(tf_exl3_gemm)

struct Library {
  decltype(&::tf_last_error) tf_last_error;
#define TF_MEMBER(name) decltype(&::name) name;
  TF_ENTRIES(TF_MEMBER)
#undef TF_MEMBER
};
Library library;          // filled once by bind()

constexpr int TABLE = 8, TABLES = 12;          // entries of a list argument, lists of a call (tf_qmm_group has ten of up to four)

struct Tables {
  alignas(8) unsigned char at[TABLES][8 * TABLE];
  int used = 0;
};

// whatever stands for a whole number (an int, numpy's, a tensor's one), as ctypes takes it
uint64_t whole(PyObject* o) {
  if (PyLong_Check(o)) return PyLong_AsUnsignedLongLongMask(o);
  PyObject* index = PyNumber_Index(o);
  if (!index) return 0;
  const uint64_t value = PyLong_AsUnsignedLongLongMask(index);
  Py_DECREF(index);
  return value;
}

uint64_t address(PyObject* o) {
  if (o == Py_None) return 0;
  if (THPVariable_Check(o)) return (uint64_t)(uintptr_t)THPVariable_Unpack(o).data_ptr();
  if (PyLong_Check(o)) return PyLong_AsUnsignedLongLongMask(o);
  PyErr_SetString(PyExc_TypeError, "expected a tensor, an address or None");
  return 0;
}

template <class T>
T argument(PyObject* o, Tables& tables) {
  if constexpr (std::is_floating_point_v<T>) {
    return (T)PyFloat_AsDouble(o);
  } else if constexpr (std::is_pointer_v<T>) {
    if (!PyList_Check(o)) return reinterpret_cast<T>((uintptr_t)address(o));
    typedef std::remove_cv_t<std::remove_pointer_t<T>> Entry;
    if constexpr (std::is_void_v<Entry>) {
      PyErr_SetString(PyExc_TypeError, "a list where one address belongs");
      return nullptr;
    } else {
      const Py_ssize_t n = PyList_GET_SIZE(o);
      if (n > TABLE || tables.used == TABLES) {
        PyErr_SetString(PyExc_TypeError, "a longer list than any entry point takes");
        return nullptr;
      }
      Entry* table = reinterpret_cast<Entry*>(tables.at[tables.used++]);
      for (Py_ssize_t i = 0; i < n; ++i) {
        PyObject* item = PyList_GET_ITEM(o, i);
        if constexpr (std::is_pointer_v<Entry>) table[i] = reinterpret_cast<Entry>((uintptr_t)address(item));
        else table[i] = (Entry)whole(item);
      }
      return table;
    }
  } else {
    return (T)whole(o);
  }
}

template <class... A, size_t... I>
PyObject* run(int (*entry)(A...), PyObject* const* args, Py_ssize_t given, std::index_sequence<I...>) {
  if (given != (Py_ssize_t)sizeof...(A)) {
    PyErr_Format(PyExc_TypeError, "%zd arguments, the entry point takes %zd", given, (Py_ssize_t)sizeof...(A));
    return nullptr;
  }
  if (!entry) {
    PyErr_SetString(PyExc_RuntimeError, "tensorfold-amd: the library is not bound");
    return nullptr;
  }
  Tables tables;
  std::tuple<A...> values{argument<A>(args[I], tables)...};
  if (PyErr_Occurred()) return nullptr;
  int status;
  Py_BEGIN_ALLOW_THREADS;
  status = std::apply(entry, values);
  Py_END_ALLOW_THREADS;
  if (!status) Py_RETURN_NONE;
  PyErr_SetString(PyExc_RuntimeError, library.tf_last_error());
  return nullptr;
}

// no C++ exception (a tensor without storage, an allocation refused) leaves through the interpreter: it is raised as the type that
// torch's own functions raise it as
template <class F>
PyObject* caught(F&& f) {
  try {
    return f();
  } catch (...) {
    torch::translate_exception_to_python(std::current_exception());
    return nullptr;
  }
}

// The interpreter's lock let go for a scope: an allocation may wait for the device, and other threads go on meanwhile, as under
// torch's own functions.
struct Released {
  PyThreadState* state = PyEval_SaveThread();
  Released() = default;
  ~Released() { PyEval_RestoreThread(state); }
  Released(const Released&) = delete;
  Released& operator=(const Released&) = delete;
};

template <class... A>
PyObject* call(int (*entry)(A...), PyObject* const* args, Py_ssize_t given) {
  return run(entry, args, given, std::index_sequence_for<A...>());
}

#define TF_WRAP(name) \
  PyObject* call_##name(PyObject*, PyObject* const* args, Py_ssize_t given) { return caught([&] { return call(library.name, args, given); }); }
TF_ENTRIES(TF_WRAP)
#undef TF_WRAP

PyObject* listed(at::Tensor* tensors, size_t count) {
  PyObject* list = PyList_New(count);
  for (size_t i = 0; list && i < count; ++i) {
    PyObject* t = THPVariable_Wrap(std::move(tensors[i]));
    if (!t) {
      Py_DECREF(list);
      return nullptr;
    }
    PyList_SET_ITEM(list, i, t);
  }
  return list;
}

// empties(x, [(rows, columns, fp32?), ...]): uninitialised contiguous tensors on x's device, of its type or fp32
PyObject* empties(PyObject*, PyObject* const* args, Py_ssize_t given) {
  if (given != 2 || !THPVariable_Check(args[0]) || !PyList_Check(args[1])) {
    PyErr_SetString(PyExc_TypeError, "empties(x, [(rows, columns, fp32?), ...])");
    return nullptr;
  }
  return caught([&]() -> PyObject* {
    const auto same = at::TensorOptions().dtype(THPVariable_Unpack(args[0]).dtype()).device(THPVariable_Unpack(args[0]).device());
    const auto f32 = same.dtype(at::kFloat);
    struct Size {
      long long rows, columns;
      int wide;
    };
    std::vector<Size> sizes(PyList_GET_SIZE(args[1]));
    for (size_t i = 0; i < sizes.size(); ++i)
      if (!PyArg_ParseTuple(PyList_GET_ITEM(args[1], i), "LLp", &sizes[i].rows, &sizes[i].columns, &sizes[i].wide)) return nullptr;
    std::vector<at::Tensor> made;
    made.reserve(sizes.size());
    {
      const Released released;
      for (const Size& s : sizes) made.push_back(at::empty({s.rows, s.columns}, s.wide ? f32 : same));
    }
    return listed(made.data(), made.size());
  });
}

// ---- whole calls ---------------------------------------------------------------------------------------------------------------
//
// qmm.matmul, qmm.matmul_group, qmm.prefill_matmul and glue.add_rmsnorm where every argument is the ordinary one: results made here,
// then the launch.  What is not (a row layout that wants a copy, a buffer of the caller's, a wrong type) returns None and
// takes the caller's general way, which copies or raises.  The norm with q, k and v at one row: 26.2 us in Python with ctypes, 21.6
// with the launches above, 12.9 so (10 us on the GPU); a matmul of a few rows 15.9, 6.1.

PyObject *s_weight, *s_scales, *s_biases, *s_n, *s_k, *s_gs, *s_arith, *s_counters;          // attribute names, interned by bind

struct Owned {
  PyObject* o;
  explicit Owned(PyObject* p) : o(p) {}
  ~Owned() { Py_XDECREF(o); }
  Owned(const Owned&) = delete;
  Owned& operator=(const Owned&) = delete;
};

// a Q4's fields; `ok` is false where one is missing or not what pack makes
struct Weight {
  Owned w, s, b, c, n_, k_, gs_, a_;
  bool ok = false;
  long n = 0, k = 0, gs = 0, arith = 0;
  explicit Weight(PyObject* q)
      : w(PyObject_GetAttr(q, s_weight)), s(PyObject_GetAttr(q, s_scales)), b(PyObject_GetAttr(q, s_biases)),
        c(PyObject_GetAttr(q, s_counters)), n_(PyObject_GetAttr(q, s_n)), k_(PyObject_GetAttr(q, s_k)),
        gs_(PyObject_GetAttr(q, s_gs)), a_(PyObject_GetAttr(q, s_arith)) {
    if (!w.o || !s.o || !b.o || !c.o || !n_.o || !k_.o || !gs_.o || !a_.o) {
      PyErr_Clear();
      return;
    }
    if (!THPVariable_Check(w.o) || !THPVariable_Check(s.o) || !THPVariable_Check(b.o) || !PyLong_Check(n_.o) ||
        !PyLong_Check(k_.o) || !PyLong_Check(gs_.o) || !PyLong_Check(a_.o))
      return;
    n = PyLong_AsLong(n_.o), k = PyLong_AsLong(k_.o), gs = PyLong_AsLong(gs_.o), arith = PyLong_AsLong(a_.o);
    if (PyErr_Occurred()) {
      PyErr_Clear();
      return;
    }
    ok = n >= 1 && n <= INT32_MAX && k >= 1 && k <= INT32_MAX && (gs == 32 || gs == 64) && scales().dim() == 2;
  }
  const at::Tensor& weight() const { return THPVariable_Unpack(w.o); }
  const at::Tensor& scales() const { return THPVariable_Unpack(s.o); }
  const at::Tensor& biases() const { return THPVariable_Unpack(b.o); }
  bool counters_ok() const { return THPVariable_Check(c.o); }
  const at::Tensor& counters() const { return THPVariable_Unpack(c.o); }
};

// x: bf16 [m, k] on the GPU in rows the kernels read as they lie (a subclass's results are of its type: torch makes those)
bool ordinary_rows(PyObject* o, long k) {
  if (!THPVariable_CheckExact(o)) return false;
  const at::Tensor& x = THPVariable_Unpack(o);
  return x.dim() == 2 && x.scalar_type() == at::kBFloat16 && x.is_cuda() && x.size(1) == k && x.size(0) >= 1 &&
         x.size(0) <= INT32_MAX && x.stride(1) == 1 && (uintptr_t)x.data_ptr() % 16 == 0 && (x.size(0) == 1 || x.stride(0) % 8 == 0);
}

at::Tensor made(const at::Tensor& x, int64_t rows, int64_t columns, bool f32) {
  return at::empty({rows, columns}, at::TensorOptions().dtype(f32 ? at::kFloat : at::kBFloat16).device(x.device()));
}

bool launched(int status) {
  if (status) PyErr_SetString(PyExc_RuntimeError, library.tf_last_error());
  return !status;
}

int row_tile(int64_t m) { return m <= 16 ? 16 : m <= 32 ? 32 : 64; }
uint16_t* bits(const at::Tensor& t) { return static_cast<uint16_t*>(t.data_ptr()); }

// an int that a C int holds: what does not fit one is not cut down to it here
bool small(PyObject* o) {
  int over = 0;
  if (!PyLong_Check(o)) return false;
  const long value = PyLong_AsLongAndOverflow(o, &over);
  return !over && value >= INT32_MIN && value <= INT32_MAX;
}

// args[first ..]: small numbers, and the stream last
bool numbers(PyObject* const* args, Py_ssize_t given, Py_ssize_t wanted, Py_ssize_t first) {
  if (!library.tf_last_error || given != wanted || !PyLong_Check(args[given - 1])) return false;
  for (Py_ssize_t i = first; i < given - 1; ++i)
    if (!small(args[i])) return false;
  return true;
}

constexpr int COUNTER_ROWS = 8;          // rows up to which a call is given the weight's arrival counters

// matmul(x, q, slices, f32, stream)
PyObject* matmul(PyObject*, PyObject* const* args, Py_ssize_t given) {
  return caught([&]() -> PyObject* {
    if (!numbers(args, given, 5, 2)) Py_RETURN_NONE;
    const Weight q(args[1]);
    if (!q.ok || !ordinary_rows(args[0], q.k)) Py_RETURN_NONE;
    const at::Tensor& x = THPVariable_Unpack(args[0]);
    const int sk = (int)PyLong_AsLong(args[2]), f32 = PyLong_AsLong(args[3]) != 0;
    const int64_t m = x.size(0);
    const bool arrive = sk > 1 && m <= COUNTER_ROWS;
    if (sk < 1 || (arrive && !q.counters_ok())) Py_RETURN_NONE;
    const tf_stream_t stream = PyLong_AsVoidPtr(args[4]);
    at::Tensor out, part;
    int status;
    {
      const Released released;
      out = made(x, m, q.n, f32);
      if (sk > 1) part = made(x, sk * m, q.n, true);
      status = library.tf_qmm_own_sums(bits(x), x.stride(0), (const uint32_t*)q.weight().data_ptr(), bits(q.scales()), bits(q.biases()),
                                       q.scales().stride(0), out.data_ptr(), sk > 1 ? (float*)part.data_ptr() : nullptr,
                                       arrive ? (int32_t*)q.counters().data_ptr() : nullptr,
                                       arrive ? (int)(q.counters().numel() / TF_QMM_COUNTER_STRIDE) : 0, (int)m, (int)q.n, (int)q.k,
                                       sk, (int)q.gs, row_tile(m), f32, 1, stream);
    }
    return launched(status) ? THPVariable_Wrap(std::move(out)) : nullptr;
  });
}

// prefill_matmul(x, q, f32, tile, stream), the weight's own arithmetic
PyObject* prefill_matmul(PyObject*, PyObject* const* args, Py_ssize_t given) {
  return caught([&]() -> PyObject* {
    if (!numbers(args, given, 5, 2)) Py_RETURN_NONE;
    const Weight q(args[1]);
    if (!q.ok || !ordinary_rows(args[0], q.k) || !q.scales().is_contiguous() || !q.biases().is_contiguous()) Py_RETURN_NONE;
    const at::Tensor& x = THPVariable_Unpack(args[0]);
    const int f32 = PyLong_AsLong(args[2]) != 0, tile = (int)PyLong_AsLong(args[3]);
    const tf_stream_t stream = PyLong_AsVoidPtr(args[4]);
    at::Tensor out;
    int status;
    {
      const Released released;
      out = made(x, x.size(0), q.n, f32);
      status = library.tf_qmm_prefill(bits(x), x.stride(0), (const uint32_t*)q.weight().data_ptr(), bits(q.scales()), bits(q.biases()),
                                      out.data_ptr(), (int)x.size(0), (int)q.n, (int)q.k, (int)q.gs, f32, tile, (int)q.arith, stream);
    }
    return launched(status) ? THPVariable_Wrap(std::move(out)) : nullptr;
  });
}

// matmul_group(x, xs, [q, ...], [slices, ...], f32, stream)
PyObject* matmul_group(PyObject*, PyObject* const* args, Py_ssize_t given) {
  return caught([&]() -> PyObject* {
    constexpr int MOST = 4;
    if (!numbers(args, given, 6, 4) || !PyList_Check(args[2]) || !PyList_Check(args[3]) || !THPVariable_Check(args[1])) Py_RETURN_NONE;
    const int count = (int)PyList_GET_SIZE(args[2]), f32 = PyLong_AsLong(args[4]) != 0;
    if (count < 1 || count > MOST || PyList_GET_SIZE(args[3]) != count) Py_RETURN_NONE;
    std::optional<Weight> q[MOST];
    int sk[MOST], n[MOST], n_counters[MOST];
    for (int i = 0; i < count; ++i) {
      q[i].emplace(PyList_GET_ITEM(args[2], i));
      if (!q[i]->ok || q[i]->k != q[0]->k || q[i]->gs != q[0]->gs || !q[i]->counters_ok() || !small(PyList_GET_ITEM(args[3], i)))
        Py_RETURN_NONE;
      sk[i] = (int)PyLong_AsLong(PyList_GET_ITEM(args[3], i)), n[i] = (int)q[i]->n;
      if (sk[i] < 1) Py_RETURN_NONE;
      for (int j = 0; j < i; ++j)
        if (q[j]->c.o == q[i]->c.o) Py_RETURN_NONE;          // a weight given twice: refused by name
    }
    if (!ordinary_rows(args[0], q[0]->k)) Py_RETURN_NONE;
    const at::Tensor &x = THPVariable_Unpack(args[0]), &xs = THPVariable_Unpack(args[1]);
    const int64_t m = x.size(0), k = q[0]->k, gs = q[0]->gs;
    if (xs.scalar_type() != at::kFloat || xs.dim() != 2 || xs.size(0) != m || xs.size(1) != k / gs || !xs.is_contiguous() ||
        xs.device() != x.device())
      Py_RETURN_NONE;
    const uint32_t* w[MOST];
    const uint16_t *s[MOST], *b[MOST];
    int64_t stride[MOST], own = 0, place[MOST];
    float* part[MOST];
    int32_t* counters[MOST];
    void* to[MOST];
    at::Tensor out[MOST], parts;
    const tf_stream_t stream = PyLong_AsVoidPtr(args[5]);
    int status;
    {
      const Released released;
      for (int i = 0; i < count; ++i) {
        w[i] = (const uint32_t*)q[i]->weight().data_ptr(), s[i] = bits(q[i]->scales()), b[i] = bits(q[i]->biases());
        stride[i] = q[i]->scales().stride(0);
        out[i] = made(x, m, n[i], f32);
        to[i] = out[i].data_ptr();
        place[i] = own;                                      // the parts lie in one buffer, each on 256 bytes
        if (sk[i] > 1) own += (sk[i] * m * n[i] + 63) / 64 * 64;
        const bool arrive = sk[i] > 1 && m <= COUNTER_ROWS;
        counters[i] = arrive ? (int32_t*)q[i]->counters().data_ptr() : nullptr;
        n_counters[i] = arrive ? (int)(q[i]->counters().numel() / TF_QMM_COUNTER_STRIDE) : 0;
      }
      if (own) parts = made(x, 1, own, true);
      for (int i = 0; i < count; ++i) part[i] = sk[i] > 1 ? (float*)parts.data_ptr() + place[i] : nullptr;
      status = library.tf_qmm_group(bits(x), x.stride(0), (const float*)xs.data_ptr(), count, w, s, b, stride, to, part, counters,
                                    n_counters, n, sk, (int)m, (int)k, (int)gs, row_tile(m), f32, stream);
    }
    return launched(status) ? listed(out, count) : nullptr;
  });
}

// add_rmsnorm(x, r, w, eps, gs, stream) with a residual
PyObject* add_rmsnorm(PyObject*, PyObject* const* args, Py_ssize_t given) {
  return caught([&]() -> PyObject* {
    if (!numbers(args, given, 6, 4) || !PyFloat_Check(args[3]) || !THPVariable_CheckExact(args[0]) || !THPVariable_Check(args[1]) ||
        !THPVariable_Check(args[2]))
      Py_RETURN_NONE;
    const at::Tensor &x = THPVariable_Unpack(args[0]), &r = THPVariable_Unpack(args[1]), &w = THPVariable_Unpack(args[2]);
    const long gs = PyLong_AsLong(args[4]);
    auto plain = [](const at::Tensor& t, int64_t dims) {
      return t.dim() == dims && t.scalar_type() == at::kBFloat16 && t.is_cuda() && t.is_contiguous();
    };
    if (!plain(x, 2) || !plain(r, 2) || !plain(w, 1) || r.sizes() != x.sizes() || w.size(0) != x.size(1) ||
        (gs != 32 && gs != 64 && gs != 128))
      Py_RETURN_NONE;
    const int64_t rows = x.size(0), d = x.size(1);
    if (rows < 1 || rows > INT32_MAX || d < gs || d > 16384 || d % gs) Py_RETURN_NONE;
    const tf_stream_t stream = PyLong_AsVoidPtr(args[5]);
    const float eps = (float)PyFloat_AS_DOUBLE(args[3]);
    at::Tensor h, y, xs;
    int status;
    {
      const Released released;
      h = made(x, rows, d, false), y = made(x, rows, d, false), xs = made(x, rows, d / gs, true);
      status = library.tf_add_norm(bits(x), r.data_ptr(), 1, nullptr, 0, 0, bits(w), eps, bits(h), bits(y), (float*)xs.data_ptr(),
                                   (int)rows, (int)d, (int)gs, stream);
    }
    if (!launched(status)) return nullptr;
    Owned a(THPVariable_Wrap(std::move(h))), b(THPVariable_Wrap(std::move(y))), c(THPVariable_Wrap(std::move(xs)));
    if (!a.o || !b.o || !c.o) return nullptr;
    return PyTuple_Pack(3, a.o, b.o, c.o);
  });
}

// bind(path): take the entry points from the library file at `path` (already loaded, or loaded now)
PyObject* bind(PyObject*, PyObject* path) {
  const char* file = PyUnicode_AsUTF8(path);
  if (!file) return nullptr;
  void* handle = dlopen(file, RTLD_NOW | RTLD_LOCAL);
  if (!handle) {
    PyErr_SetString(PyExc_RuntimeError, dlerror());
    return nullptr;
  }
#define TF_FIND(name)                                                                       \
  library.name = reinterpret_cast<decltype(library.name)>(dlsym(handle, #name));            \
  if (!library.name) {                                                                      \
    PyErr_SetString(PyExc_RuntimeError, "tensorfold-amd: " #name " is not in the library"); \
    return nullptr;                                                                         \
  }
  TF_FIND(tf_last_error)
  TF_ENTRIES(TF_FIND)
  const std::pair<PyObject**, const char*> names[] = {{&s_weight, "weight"}, {&s_scales, "scales"}, {&s_biases, "biases"},
                                                      {&s_n, "n"},           {&s_k, "k"},           {&s_gs, "gs"},
                                                      {&s_arith, "arith"},   {&s_counters, "_counters"}};
  for (const auto& [at, name] : names)
    if (!(*at = PyUnicode_InternFromString(name))) return nullptr;
#undef TF_FIND
  Py_RETURN_NONE;
}

#define TF_METHOD(name) {#name, reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)()>(call_##name)), METH_FASTCALL, nullptr},
#define TF_WHOLE(name) {#name, reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)()>(name)), METH_FASTCALL, nullptr},
PyMethodDef methods[] = {{"bind", bind, METH_O, nullptr},
                         {"empties", reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)()>(empties)), METH_FASTCALL, nullptr},
                         TF_WHOLE(matmul) TF_WHOLE(matmul_group) TF_WHOLE(prefill_matmul) TF_WHOLE(add_rmsnorm)
                         TF_ENTRIES(TF_METHOD){nullptr, nullptr, 0, nullptr}};
#undef TF_METHOD
#undef TF_WHOLE

PyModuleDef module = {PyModuleDef_HEAD_INIT, "tfmi_call", nullptr, -1, methods, nullptr, nullptr, nullptr, nullptr};

}  // namespace

extern "C" __attribute__((used)) const char tf_call_id[] = "TFMI_CALL_ID=" TF_CALL_ID " TFMI_CALL_FOR=" TF_CALL_FOR;

PyMODINIT_FUNC PyInit_tfmi_call() { return PyModule_Create(&module); }
