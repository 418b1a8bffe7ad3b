// Host side of the per-layer calls (the CPython module logssms_amd._host):
//   * a typed entry for each hot C-ABI function, so that a call converts its
//     arguments in a loop over their C types (ctypes took 2.5 us for the 46
//     arguments of a decode step);
//   * conv_recurrent, the checks and the call of one decode or verify step
//     with tensors in hand.
// A decode step of one sequence is an 8 us kernel behind what the host does
// to launch it: 15.8 us in Python and ctypes, 5.8 us through this module.
#include <Python.h>
#include <dlfcn.h>

#include <utility>

#include <ATen/ATen.h>
#include <c10/hip/HIPStream.h>
#include <torch/csrc/Exceptions.h>
#include <torch/csrc/autograd/python_variable.h>

#include "../../include/gdn_mi355x.h"

namespace {

// ---------------------------------------------------------------- the library
// This module links no libgdn_mi355x.so: bind(handle) takes the functions from
// the one instance that the package has opened (whichever file that is), so
// that typed entries, ctypes calls and gdn_last_error share its state.
#define GDN_TYPED(X)                      \
  X(gdn_prefill_frontend)                 \
  X(gdn_prefill_qk)                       \
  X(gdn_prefill_fused)                    \
  X(gdn_prefill_split)                    \
  X(gdn_prefill_workspace_bytes)          \
  X(gdn_chunk_workspace_bytes)            \
  X(gdn_chunk_gated_delta_rule_ws)        \
  X(gdn_chunk_gated_delta_rule_logged_ws) \
  X(gdn_store_chunk_log)                  \
  X(gdn_conv_snapshots)                   \
  X(gdn_conv_windows_logstate)            \
  X(gdn_conv_decode)                      \
  X(gdn_conv_decode_logstate)             \
  X(gdn_recurrent_logstate)               \
  X(gdn_fused_recurrent)                  \
  X(gdn_fused_conv_recurrent)             \
  X(gdn_logstate_restore)                 \
  X(gdn_rms_norm_gated)
namespace lib {
#define GDN_POINTER(name) decltype(&::name) name = nullptr;
GDN_TYPED(GDN_POINTER)
GDN_POINTER(gdn_last_error)
}  // namespace lib

PyObject* bind(PyObject*, PyObject* handle) {
  void* opened = PyLong_AsVoidPtr(handle);
  if (!opened) {
    if (!PyErr_Occurred()) PyErr_SetString(PyExc_ValueError, "the handle of an opened library expected");
    return nullptr;
  }
  auto find = [&](auto& pointer, const char* name) {
    pointer = reinterpret_cast<std::decay_t<decltype(pointer)>>(dlsym(opened, name));
    if (!pointer) PyErr_Format(PyExc_RuntimeError, "%s is not in the library", name);
    return pointer != nullptr;
  };
#define GDN_FIND(name) && find(lib::name, #name)
  if (!(true GDN_TYPED(GDN_FIND) GDN_FIND(gdn_last_error))) return nullptr;
  Py_RETURN_NONE;
}

// ---------------------------------------------------------------- typed entries
// One Python argument as its C parameter; sets a Python error and returns
// false where it does not fit.
bool convert(PyObject* o, int64_t& v) {
  v = PyLong_AsLongLong(o);
  return v != -1 || !PyErr_Occurred();
}
bool convert(PyObject* o, int& v) {
  int64_t x;
  if (!convert(o, x)) return false;
  v = static_cast<int>(x);
  if (v == x) return true;
  PyErr_SetString(PyExc_OverflowError, "argument exceeds a C int");
  return false;
}
bool convert(PyObject* o, float& v) {
  const double x = PyFloat_AsDouble(o);
  v = static_cast<float>(x);
  return x != -1.0 || !PyErr_Occurred();
}
template <class T>
bool convert(PyObject* o, T*& v) {  // a device address, or None
  void* p = o == Py_None ? nullptr : PyLong_AsVoidPtr(o);
  if (!p && PyErr_Occurred()) return false;
  v = static_cast<T*>(p);
  return true;
}

// f(args...) without the interpreter lock, as ctypes calls: a launch that waits
// for a place in a full queue does not stop the process's other Python threads.
struct Unlocked {
  PyThreadState* state = PyEval_SaveThread();
  ~Unlocked() { PyEval_RestoreThread(state); }
};
template <class R, class... P, class... A>
R unlocked(R (*f)(P...), A... args) {
  const Unlocked scope;
  return f(args...);
}

bool bound(bool found) {
  if (!found) PyErr_SetString(PyExc_RuntimeError, "no library bound (logssms_amd._lib.host())");
  return found;
}

template <auto F> struct Entry;  // F: where bind() keeps the function
template <class R, class... A, R (**F)(A...)>
struct Entry<F> {
  template <size_t... I>
  static PyObject* invoke(PyObject* const* args, std::index_sequence<I...>) {
    std::tuple<A...> v{};
    if (!(convert(args[I], std::get<I>(v)) && ...)) return nullptr;
    return PyLong_FromLongLong(unlocked(*F, std::get<I>(v)...));
  }
  static PyObject* call(PyObject*, PyObject* const* args, Py_ssize_t n) {
    if (n != static_cast<Py_ssize_t>(sizeof...(A))) {
      PyErr_Format(PyExc_TypeError, "%zu arguments expected, %zd given", sizeof...(A), n);
      return nullptr;
    }
    if (!bound(*F != nullptr)) return nullptr;
    return invoke(args, std::index_sequence_for<A...>{});
  }
};

// ---------------------------------------------------------------- decode and verify
struct Failed {};  // a Python error is set

void require(bool ok, const char* what) {
  if (ok) return;
  PyErr_SetString(PyExc_AssertionError, what);
  throw Failed();
}

const at::Tensor& tensor(PyObject* o) {
  if (!THPVariable_Check(o)) {
    PyErr_Format(PyExc_TypeError, "a tensor expected, got %s", Py_TYPE(o)->tp_name);
    throw Failed();
  }
  return THPVariable_Unpack(o);
}
int64_t integer(PyObject* o) {
  int64_t v;
  if (!convert(o, v)) throw Failed();
  return v;
}
int dtype_code(const at::Tensor& t) {
  switch (t.scalar_type()) {
    case at::kFloat: return GDN_F32;
    case at::kBFloat16: return GDN_BF16;
    case at::kHalf: return GDN_F16;
    default:
      PyErr_Format(PyExc_TypeError, "unsupported dtype %s", c10::toString(t.scalar_type()));
      throw Failed();
  }
}
int index_code(const at::Tensor& t) {
  if (t.scalar_type() == at::kLong) return GDN_I64;
  if (t.scalar_type() == at::kInt) return GDN_I32;
  PyErr_Format(PyExc_TypeError, "index tensors must be int32 or int64, got %s", c10::toString(t.scalar_type()));
  throw Failed();
}

// conv_recurrent(mixed, row_index or None, gate, beta, conv_weight, A_log,
//   dt_bias, conv_state, recurrent_state, read_slots, write_slots, out or None,
//   num_k_heads, num_v_heads, head_k_dim, head_v_dim, conv_dim, state_len, layer)
// One decode step (write_slots [B]) or the T steps of a verify group
// (write_slots [B, T]); returns out ([rows, HV, dv], allocated when None).
PyObject* conv_recurrent(PyObject*, PyObject* const* args, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  try {
    require(n == 19, "conv_recurrent: 19 arguments expected");
    const at::Tensor &mixed = tensor(args[0]), &gate = tensor(args[2]), &beta = tensor(args[3]);
    const at::Tensor weight = tensor(args[4]).contiguous(), A_log = tensor(args[5]).contiguous(),
                     dt_bias = tensor(args[6]).contiguous();
    const at::Tensor &conv = tensor(args[7]), &state = tensor(args[8]), &reads = tensor(args[9]),
                     &writes = tensor(args[10]);
    const int64_t H = integer(args[12]), HV = integer(args[13]), dk = integer(args[14]), dv = integer(args[15]),
                  conv_dim = integer(args[16]), state_len = integer(args[17]), layer = integer(args[18]);
    const bool verify = writes.dim() == 2;
    require(mixed.dim() == 2 && mixed.size(1) == conv_dim, "mixed_qkv must be [rows, conv_dim]");
    require(verify || writes.dim() == 1, "write slots must be [B] or [B, T]");
    const int64_t B = writes.size(0), T = verify ? writes.size(1) : 1;
    require(reads.dim() == 1 && reads.size(0) == B && (verify || mixed.size(0) == B), "one read slot per sequence");
    require(T >= 1, "at least one step");
    require(conv.dim() == 4 && conv.size(2) == conv_dim && conv.size(3) == state_len && conv.stride(3) == 1 &&
                conv.stride(2) == state_len,
            "conv_state must be [slots, layers, conv_dim, state_len] with contiguous windows");
    require(state.dim() == 5 && state.size(2) == HV && state.size(3) == dk && state.size(4) == dv &&
                state.stride(4) == 1 && state.stride(3) == dv,
            "recurrent_state must be [slots, layers, HV, dk, dv] with contiguous rows");
    const at::Tensor* rows = nullptr;
    if (args[1] != Py_None) {
      rows = &tensor(args[1]);
      require(rows->dim() == 1 && rows->size(0) == B * T, "one row index per step");
    }
    at::Tensor out = args[11] == Py_None ? at::empty({B * T, HV, dv}, mixed.options()) : tensor(args[11]);
    require(out.is_contiguous() && out.dim() == 3 && out.size(1) == HV && out.size(2) == dv &&
                (verify || out.size(0) == B),
            "out must be a contiguous [rows, HV, dv]");
    if (B > 0) {
      if (!mixed.is_cuda()) {
        PyErr_SetString(PyExc_RuntimeError, "libgdn_mi355x kernels need tensors on a ROCm device");
        throw Failed();
      }
      if (!bound(lib::gdn_fused_conv_recurrent != nullptr)) throw Failed();
      const int rc = unlocked(
          lib::gdn_fused_conv_recurrent, mixed.data_ptr(), mixed.stride(0), mixed.stride(1), dtype_code(mixed),
          rows ? rows->data_ptr() : nullptr, rows ? index_code(*rows) : 0, weight.data_ptr(), nullptr,
          static_cast<int>(state_len + 1), gate.data_ptr(),
          gate.stride(0), gate.stride(1), dtype_code(gate), beta.data_ptr(), beta.stride(0), beta.stride(1),
          dtype_code(beta), A_log.data_ptr(), dtype_code(A_log), dt_bias.data_ptr(), dtype_code(dt_bias), B, T, H, HV,
          dk, dv, conv.data_ptr(), conv.stride(0), conv.stride(1), state.data_ptr(), dtype_code(state),
          state.stride(0), state.stride(1), state.stride(2), layer, reads.data_ptr(), reads.stride(0),
          index_code(reads), writes.data_ptr(), writes.stride(0), verify ? writes.stride(1) : 0, index_code(writes),
          out.data_ptr(), static_cast<float>(1.0 / std::sqrt(static_cast<double>(dk))),
          c10::hip::getCurrentHIPStream(mixed.device().index()).stream());
      if (rc != GDN_OK) {
        PyErr_Format(rc == GDN_ERR_UNSUPPORTED ? PyExc_NotImplementedError : PyExc_RuntimeError,
                     "gdn_fused_conv_recurrent failed (%d): %s", rc, lib::gdn_last_error());
        throw Failed();
      }
    }
    return THPVariable_Wrap(out);
  } catch (const Failed&) {
    return nullptr;
  }
  END_HANDLE_TH_ERRORS
}

#define GDN_METHOD(name) {#name, reinterpret_cast<PyCFunction>(&Entry<&lib::name>::call), METH_FASTCALL, nullptr},
PyMethodDef kMethods[] = {
    {"bind", &bind, METH_O, nullptr},
    {"conv_recurrent", reinterpret_cast<PyCFunction>(&conv_recurrent), METH_FASTCALL, nullptr},
    GDN_TYPED(GDN_METHOD)
    {nullptr, nullptr, 0, nullptr}};
PyModuleDef kModule = {PyModuleDef_HEAD_INIT, "_host", nullptr, -1, kMethods, nullptr, nullptr, nullptr, nullptr};

}  // namespace

PyMODINIT_FUNC PyInit__host() { return PyModule_Create(&kModule); }
