// The Python side's way into librtp_hip.so for the calls of a training step: a CPython extension over the C ABI of
// include/rtp_hip.h.  A layer's pass is a handful of 3 - 20 us launches, so what the host spends per launch decides the
// time of every call that is not huge: through ctypes a product cost 9 us of argument handling (45 descriptor fields set
// from Python, the stream object, the foreign call) around a 2.5 us launch; here it is under 1.5 us.
//
//   * every entry point that Python calls on the hot path, converted argument by argument from the C prototype itself
//     (`invoke`), the current stream put in front, a negative status raised as RtpError;
//   * `gemm`, and the products of the rotated linear layers, attention cores and experts on tensors, with their descriptors
//     filled and their operands checked here;
//   * GradBook: the parameters of a layer's shards and the slices of its gradient buffer, attached as .grad for a backward
//     pass in one call (one Python attribute access per parameter otherwise).
//
// The library itself stays free of torch and Python: it is opened by path and resolved by name (`bind`).
#include <Python.h>

#include <ATen/core/Tensor.h>
#include <c10/hip/HIPStream.h>
#include <dlfcn.h>
#include <torch/csrc/Dtype.h>
#include <torch/csrc/Exceptions.h>
#include <torch/csrc/autograd/python_variable.h>

#include <algorithm>
#include <chrono>
#include <cstring>
#include <exception>
#include <string>
#include <type_traits>
#include <utility>
#include <vector>

#include "rtp_hip.h"

namespace {

PyObject* g_error = nullptr;  // rtp_amd._lib.RtpError
decltype(&rtp_last_error) f_last_error = nullptr;

void* current_stream() { return (void*)c10::hip::getCurrentHIPStream().stream(); }

PyObject* raise_status(long rc) {
  PyErr_Format(g_error, "librtp_hip status %ld: %s", rc, f_last_error());
  return nullptr;
}

// A C++ exception may not cross into the interpreter, it would end the process: a tensor's data_ptr() throws for a sparse or
// a functorch tensor, its sizes for a nested one.  Every function Python can call is entered through here and such an
// exception raised as the Python one torch's own bindings make of it.
template <auto F>
struct Entry;
template <class... A, PyObject* (*F)(A...)>
struct Entry<F> {
  static PyObject* call(A... a) {
    try {
      return F(a...);
    } catch (const std::exception&) {
      torch::translate_exception_to_python(std::current_exception());
    }
    return nullptr;
  }
};

struct WithoutGil {
  PyThreadState* state = PyEval_SaveThread();
  ~WithoutGil() { PyEval_RestoreThread(state); }
};

// ---- one argument ----
template <class T>
bool from_py(PyObject* o, T& out) {
  if constexpr (std::is_pointer_v<T>) {
    if (o == Py_None) {
      out = nullptr;
    } else if (THPVariable_Check(o)) {
      out = (T)THPVariable_Unpack(o).data_ptr();
    } else {
      out = (T)PyLong_AsVoidPtr(o);
    }
  } else if constexpr (std::is_floating_point_v<T>) {
    out = (T)PyFloat_AsDouble(o);
  } else {
    out = (T)PyLong_AsLongLong(o);
  }
  return !(out == (T)0 || out == (T)-1) || !PyErr_Occurred();
}

template <bool STREAM, class R, class... A, size_t... I>
PyObject* invoke_at(R (*f)(A...), PyObject* const* args, std::index_sequence<I...>) {
  std::tuple<A...> v;
  if constexpr (STREAM) std::get<0>(v) = current_stream();
  constexpr size_t S = STREAM ? 1 : 0;
  bool ok = true;
  (void)std::initializer_list<int>{(ok = ok && (I < S || from_py(args[I < S ? 0 : I - S], std::get<I>(v))), 0)...};
  if (!ok) return nullptr;
  const R r = (WithoutGil(), std::apply(f, v));
  if constexpr (std::is_same_v<R, int>) {
    if (r < 0) return raise_status(r);
  }
  if constexpr (std::is_unsigned_v<R>) return PyLong_FromSize_t((size_t)r);
  return PyLong_FromLongLong((long long)r);
}
template <bool STREAM, class R, class... A>
PyObject* invoke(R (*f)(A...), const char* name, PyObject* const* args, Py_ssize_t n) {
  constexpr Py_ssize_t want = (Py_ssize_t)sizeof...(A) - (STREAM ? 1 : 0);
  if (n != want) return PyErr_Format(PyExc_TypeError, "%s takes %zd arguments, got %zd", name, want, n);
  return invoke_at<STREAM>(f, args, std::index_sequence_for<A...>{});
}

// X(name): the stream of the C prototype is the current one and not passed;  P(name): passed as declared
#define RTP_ENTRY_POINTS(X, P)                                                                                        \
  P(rtp_gemm_warm_next) P(rtp_colsum_workspace_bytes) X(rtp_colsum) X(rtp_shard_copy_async) X(rtp_zero_async)        \
  X(rtp_embedding_gather) X(rtp_embedding_gather_scale_pos) P(rtp_embedding_scatter_workspace_bytes)                  \
  X(rtp_embedding_sort_ids) X(rtp_embedding_scatter_add_det) X(rtp_embedding_scatter_add_scaled)                      \
  X(rtp_embedding_scatter_add_sgd) P(rtp_embedding_backward_supported) X(rtp_embedding_backward)                      \
  P(rtp_embedding_backward_grouped_supported) P(rtp_embedding_backward_grouped_workspace_bytes)                       \
  X(rtp_embedding_backward_grouped)                                                                                   \
  X(rtp_softmax_fwd_masks) X(rtp_softmax_bwd) P(rtp_attn_supported) X(rtp_attn_fwd) X(rtp_attn_bwd)                   \
  P(rtp_attn_flash_supported) X(rtp_attn_flash_fwd) X(rtp_attn_flash_bwd) P(rtp_attn_flash_kv_supported)              \
  X(rtp_attn_flash_kv_fwd) X(rtp_attn_flash_kv_bwd) P(rtp_layernorm_supported)                                        \
  X(rtp_add_layernorm_fwd) P(rtp_layernorm_bwd_workspace_bytes) X(rtp_layernorm_bwd) P(rtp_layernorm_bwd_blocks)      \
  X(rtp_layernorm_bwd_finalize) X(rtp_softmax_xent_fwd) X(rtp_softmax_xent_reduce) X(rtp_softmax_xent_bwd)            \
  P(rtp_top2_route_workspace_bytes) X(rtp_top2_route) X(rtp_top2_route_bwd) X(rtp_moe_dispatch) X(rtp_moe_combine)    \
  X(rtp_moe_combine_dweight) P(rtp_gate_supported) X(rtp_gate_fwd) X(rtp_gate_dgrad)                                  \
  P(rtp_gate_wgrad_workspace_bytes) X(rtp_gate_wgrad) X(rtp_conv2d_fwd) X(rtp_conv2d_wgrad)                           \
  P(rtp_conv2d_wgrad_workspace_bytes) X(rtp_conv2d_dgrad) X(rtp_sgd_step) X(rtp_sgd_step_multi) X(rtp_adam_step)      \
  X(rtp_adam_step_multi) X(rtp_cast)

#define DECLARE(name) decltype(&name) f_##name = nullptr;
RTP_ENTRY_POINTS(DECLARE, DECLARE)
#undef DECLARE
#define WRAP(name, stream)                                                     \
  PyObject* py_##name(PyObject*, PyObject* const* args, Py_ssize_t n) {        \
    return invoke<stream>(f_##name, #name, args, n);                           \
  }
#define WRAP_X(name) WRAP(name, true)
#define WRAP_P(name) WRAP(name, false)
RTP_ENTRY_POINTS(WRAP_X, WRAP_P)
#undef WRAP_X
#undef WRAP_P
#undef WRAP

decltype(&rtp_gemm) f_gemm = nullptr;
decltype(&rtp_gemm_workspace) f_gemm_workspace = nullptr;
decltype(&rtp_gemm_pair) f_gemm_pair = nullptr;
decltype(&rtp_gemm_rowsum_fused) f_rowsum_fused = nullptr;
decltype(&rtp_gemm_sgd_fused) f_sgd_fused = nullptr;
decltype(&rtp_rotated_linear_fwd) f_linear_fwd = nullptr;
decltype(&rtp_rotated_linear_bwd) f_linear_bwd = nullptr;

PyObject* py_bind(PyObject*, PyObject* args) {
  const char* path;
  PyObject* error;
  if (!PyArg_ParseTuple(args, "sO", &path, &error)) return nullptr;
  void* lib = dlopen(path, RTLD_NOW | RTLD_LOCAL);
  if (!lib) return PyErr_Format(PyExc_OSError, "%s", dlerror());
  Py_INCREF(error);
  g_error = error;
  auto get = [lib](const char* name, auto& f) {
    f = (std::remove_reference_t<decltype(f)>)dlsym(lib, name);
    if (!f) PyErr_Format(PyExc_OSError, "librtp_hip.so has no %s", name);
    return f != nullptr;
  };
  bool ok = get("rtp_last_error", f_last_error) && get("rtp_gemm", f_gemm) && get("rtp_gemm_workspace", f_gemm_workspace) &&
            get("rtp_gemm_pair", f_gemm_pair) &&
            get("rtp_gemm_rowsum_fused", f_rowsum_fused) && get("rtp_gemm_sgd_fused", f_sgd_fused) &&
            get("rtp_rotated_linear_fwd", f_linear_fwd) && get("rtp_rotated_linear_bwd", f_linear_bwd);
#define RESOLVE(name) ok = ok && get(#name, f_##name);
  RTP_ENTRY_POINTS(RESOLVE, RESOLVE)
#undef RESOLVE
  if (!ok) return nullptr;
  Py_RETURN_NONE;
}

// Scratch memory for the products launched while it lives, from torch's allocator on the current stream: given back with it, for what
// that stream runs afterwards.  (The allocator itself, not at::empty: no dispatch, and no Python under a mode of it.)
// Before the allocator refuses it waits for the device and gives all that it holds in reserve back, which costs a program near its memory's
// end more than the copies gain.  So a thread that was refused asks for as much on that device again only after a second.
struct Workspace {
  struct Refusal {
    std::chrono::steady_clock::time_point until;
    size_t bytes = 0;
    int device = -1;
  };
  static thread_local Refusal refused;
  std::vector<c10::DataPtr> held;
  Workspace() { f_gemm_workspace(&get, this); }
  ~Workspace() { f_gemm_workspace(nullptr, nullptr); }
  static void* get(void* self, size_t bytes) noexcept {
    int device = -1;
    try {
      device = c10::hip::getCurrentHIPStream().device_index();
      if (device == refused.device && bytes >= refused.bytes && std::chrono::steady_clock::now() < refused.until) return nullptr;
      auto& held = static_cast<Workspace*>(self)->held;
      held.push_back(c10::GetAllocator(c10::kCUDA)->allocate(bytes));
      return held.back().get();
    } catch (...) {  // no memory: the product does without
      refused = {std::chrono::steady_clock::now() + std::chrono::seconds(1), bytes, device};
      return nullptr;
    }
  }
};
thread_local Workspace::Refusal Workspace::refused;

int dtype_code(at::ScalarType t) {
  return t == at::kFloat ? (int)RTP_F32 : t == at::kBFloat16 ? (int)RTP_BF16 : -1;
}

PyObject* bad(const char* what) {
  PyErr_SetString(PyExc_ValueError, what);
  return nullptr;
}

// ---- gemm(dtype, *, a=, b=, ...): the keyword arguments of ops.gemm_raw ----
enum class K { ptr, i64, f32, flag, pair };
struct Field {
  const char* name;
  K kind;
  size_t at;  // offset in rtp_gemm_desc, or the flag's bit
  PyObject* key;
};
#define AT(f) offsetof(rtp_gemm_desc, f)
Field g_fields[] = {
    {"a", K::ptr, AT(a)}, {"b", K::ptr, AT(b)}, {"c_out", K::ptr, AT(c_out)}, {"m", K::i64, AT(m)}, {"n", K::i64, AT(n)},
    {"k", K::i64, AT(k)}, {"lda", K::i64, AT(lda)}, {"ldb", K::i64, AT(ldb)}, {"ldc", K::i64, AT(ldc)},
    {"a_kcontig", K::flag, 1u << 16}, {"b_kcontig", K::flag, 1u << 17}, {"c_in", K::ptr, AT(c_in)},
    {"ld_cin", K::i64, AT(ld_cin)}, {"bias", K::ptr, AT(bias)}, {"gate", K::ptr, AT(gate)},
    {"ld_gate", K::i64, AT(ld_gate)}, {"alpha", K::f32, AT(alpha)}, {"relu", K::flag, RTP_GEMM_RELU},
    {"out_f32", K::flag, RTP_GEMM_OUT_F32}, {"cin_f32", K::flag, RTP_GEMM_CIN_F32}, {"batch", K::i64, AT(batch)},
    {"zdiv", K::i64, AT(zdiv)}, {"a_s", K::pair, AT(a_so)}, {"b_s", K::pair, AT(b_so)}, {"c_s", K::pair, AT(c_so)},
    {"cin_s", K::pair, AT(cin_so)}, {"gate_s", K::pair, AT(gate_so)}, {"bias_s", K::pair, AT(bias_so)},
    {"groups", K::i64, AT(groups)}, {"a_sg", K::i64, AT(a_sg)}, {"b_sg", K::i64, AT(b_sg)}, {"c_sg", K::i64, AT(c_sg)},
    {"cin_sg", K::i64, AT(cin_sg)}, {"gate_sg", K::i64, AT(gate_sg)}, {"bias_sg", K::i64, AT(bias_sg)},
    {"ksegs", K::i64, AT(ksegs)}, {"a_sk", K::i64, AT(a_sk)}, {"b_sk", K::i64, AT(b_sk)}, {"bias_sk", K::i64, AT(bias_sk)},
    {"stream_out", K::flag, RTP_GEMM_STREAM_OUT}, {"rowsum", K::ptr, AT(a_rowsum)}, {"rowsum_sg", K::i64, AT(rowsum_sg)},
    {"rowsum_accum", K::flag, RTP_GEMM_ROWSUM_ACCUM}, {"sgd_master", K::ptr, AT(sgd_master)},
    {"sgd_weights", K::ptr, AT(sgd_weights)}, {"sgd_lr", K::f32, AT(sgd_lr)}, {"sgd_clip", K::f32, AT(sgd_clip)},
    {"sgd_skip_out", K::flag, RTP_GEMM_SGD_SKIP_OUT},
};
#undef AT
PyObject* g_field_index = nullptr;  // name -> index into g_fields

// Adds to `done` ROWSUM (1) if the row sums asked for will be produced, SGD (2) if the update will be applied: what the operands do not
// allow is left out of the launch and reported by its missing bit.
void settle_product(int dt, rtp_gemm_desc& d, uint32_t flags, int& done) {
  if (d.sgd_master) {
    void *const master = d.sgd_master, *const weights = d.sgd_weights;
    d.sgd_master = d.sgd_weights = nullptr;
    d.flags = (int32_t)(flags & 0xffff & ~(uint32_t)RTP_GEMM_SGD_SKIP_OUT);
    if (f_sgd_fused(dt, &d)) {
      d.sgd_master = master, d.sgd_weights = weights;
      done |= 2;
    } else {
      flags &= ~(uint32_t)RTP_GEMM_SGD_SKIP_OUT;
    }
  } else {
    flags &= ~(uint32_t)RTP_GEMM_SGD_SKIP_OUT;
  }
  d.flags = (int32_t)(flags & 0xffff);
  if (d.a_rowsum) {
    if (f_rowsum_fused(dt, &d))
      done |= 1;
    else
      d.a_rowsum = nullptr, d.rowsum_sg = 0;
  }
}
// Runs the product on the current stream.
bool launch_product(int dt, rtp_gemm_desc& d, uint32_t flags, int& done) {
  settle_product(dt, d, flags, done);
  void* st = current_stream();
  const int rc = (WithoutGil(), Workspace(), f_gemm(st, dt, &d));
  if (rc < 0) raise_status(rc);
  return rc >= 0;
}
PyObject* run_product(int dt, rtp_gemm_desc& d, uint32_t flags) {
  int done = 0;
  return launch_product(dt, d, flags, done) ? PyLong_FromLong(done) : nullptr;
}
rtp_gemm_desc product(int64_t m, int64_t n, int64_t k, bool a_kcontig, bool b_kcontig) {
  rtp_gemm_desc d;
  memset(&d, 0, sizeof(d));
  d.batch = d.zdiv = d.groups = d.ksegs = 1;
  d.alpha = 1.0f;
  d.m = m, d.n = n, d.k = k;
  d.a_kcontig = a_kcontig, d.b_kcontig = b_kcontig;
  return d;
}

PyObject* py_gemm(PyObject*, PyObject* const* args, Py_ssize_t nargs, PyObject* kwnames) {
  if (nargs != 1 || !THPDtype_Check(args[0])) return PyErr_Format(PyExc_TypeError, "gemm(dtype, *, ...)");
  const int dt = dtype_code(((THPDtype*)args[0])->scalar_type);
  if (dt < 0) return PyErr_Format(PyExc_TypeError, "rtp_amd kernels support float32 and bfloat16, got %R", args[0]);
  rtp_gemm_desc d = product(0, 0, 0, false, false);
  uint32_t flags = 0;
  const Py_ssize_t nk = kwnames ? PyTuple_GET_SIZE(kwnames) : 0;
  for (Py_ssize_t i = 0; i < nk; ++i) {
    PyObject *name = PyTuple_GET_ITEM(kwnames, i), *v = args[nargs + i];
    PyObject* idx = PyDict_GetItemWithError(g_field_index, name);
    if (!idx) return PyErr_Occurred() ? nullptr : PyErr_Format(PyExc_TypeError, "gemm: unknown argument %R", name);
    const Field& f = g_fields[PyLong_AsLong(idx)];
    char* at = (char*)&d + f.at;
    bool ok = true;
    switch (f.kind) {
      case K::ptr: ok = from_py(v, *(void**)at); break;
      case K::i64: ok = from_py(v, *(int64_t*)at); break;
      case K::f32: ok = from_py(v, *(float*)at); break;
      case K::pair:
        ok = PyTuple_Check(v) && PyTuple_GET_SIZE(v) == 2 && from_py(PyTuple_GET_ITEM(v, 0), ((int64_t*)at)[0]) &&
             from_py(PyTuple_GET_ITEM(v, 1), ((int64_t*)at)[1]);
        if (!ok && !PyErr_Occurred()) PyErr_Format(PyExc_TypeError, "gemm: %s takes a pair", f.name);
        break;
      case K::flag: {
        const int on = PyObject_IsTrue(v);
        ok = on >= 0;
        if (on) flags |= (uint32_t)f.at;
        break;
      }
    }
    if (!ok) return nullptr;
  }
  d.a_kcontig = (flags >> 16) & 1, d.b_kcontig = (flags >> 17) & 1;
  return run_product(dt, d, flags);
}
// ---- the rotated linear layer's products on tensors ----
struct Mat {
  char* p;
  int64_t rows, cols, ld;
};
// [rows, cols] with unit column stride; leading dimension as the C ABI wants it
bool as_mat(const at::Tensor& t, const char* what, Mat& m) {
  if (t.dim() != 2 || (t.size(1) > 1 && t.stride(1) != 1)) {
    PyErr_Format(PyExc_ValueError, "%s: need a 2-D tensor with unit column stride", what);
    return false;
  }
  m.p = (char*)t.data_ptr();
  m.rows = t.size(0), m.cols = t.size(1);
  m.ld = m.rows > 1 ? t.stride(0) : std::max<int64_t>(m.cols, 1);
  return true;
}
bool layer_of(const at::Tensor& home, int64_t w_off, PyObject* bias_off, int64_t n_s, int64_t k, rtp_rotated_linear& L,
              int& dt) {
  dt = dtype_code(home.scalar_type());
  if (home.dim() != 2 || !home.is_contiguous() || dt < 0) {
    PyErr_SetString(PyExc_ValueError,
                    "rotated_linear: home must be the contiguous fp32 / bf16 [shards, numel] buffer of the layer");
    return false;
  }
  if (!home.is_cuda()) {
    PyErr_SetString(g_error, "rtp_amd kernels run on the GPU only; got a CPU tensor (there is no CPU path)");
    return false;
  }
  L = rtp_rotated_linear{home.data_ptr(), home.size(1), home.size(0), w_off, -1, n_s, k};
  return bias_off == Py_None || from_py(bias_off, L.bias_off);
}
const at::Tensor* opt_tensor(PyObject* o) { return o == Py_None ? nullptr : &THPVariable_Unpack(o); }

// linear_fwd(x2, home, w_off, bias_off, n_s, k, y, col0, relu): y[:, col0 : col0 + shards*n_s] = x2 W_g^T + b_g
PyObject* py_linear_fwd(PyObject*, PyObject* const* a, Py_ssize_t n) {
  if (n != 9 || !THPVariable_Check(a[0]) || !THPVariable_Check(a[1]) || !THPVariable_Check(a[6]))
    return PyErr_Format(PyExc_TypeError, "linear_fwd(x2, home, w_off, bias_off, n_s, k, y, col0, relu)");
  const at::Tensor &x2 = THPVariable_Unpack(a[0]), &home = THPVariable_Unpack(a[1]), &y = THPVariable_Unpack(a[6]);
  int64_t w_off, n_s, k, col0;
  if (!from_py(a[2], w_off) || !from_py(a[4], n_s) || !from_py(a[5], k) || !from_py(a[7], col0)) return nullptr;
  rtp_rotated_linear L;
  int dt;
  Mat x, o;
  if (!layer_of(home, w_off, a[3], n_s, k, L, dt) || !as_mat(x2, "x", x) || !as_mat(y, "y", o)) return nullptr;
  const bool f32 = y.scalar_type() != home.scalar_type();
  if (x.cols != k || o.rows != x.rows || col0 < 0 || o.cols - col0 < n_s * L.shards ||
      x2.scalar_type() != home.scalar_type() || (f32 && y.scalar_type() != at::kFloat))
    return bad("rotated_linear_fwd: x [rows, k] in the shards' dtype, y [rows, >= shards * n_s] (or fp32)");
  const int flags = (PyObject_IsTrue(a[8]) ? RTP_GEMM_RELU : 0) | (f32 ? RTP_GEMM_OUT_F32 : 0);
  void* st = current_stream();
  // one row: any leading dimension that holds it
  const int64_t ldo = o.rows > 1 ? o.ld : std::max<int64_t>(o.cols, 1);
  char* out = o.p + col0 * (int64_t)y.element_size();
  const int rc = (WithoutGil(), Workspace(), f_linear_fwd(st, dt, &L, x.p, x.ld, x.rows, out, ldo, flags));
  if (rc < 0) return raise_status(rc);
  Py_RETURN_NONE;
}

// linear_bwd(dy2, col0, x2, home, w_off, bias_off, n_s, k, dx, dx_init, relu_gate, grads, accumulate,
//            sgd_master, sgd_weights, lr, clip, skip_store) -> done flags; see ops.rotated_linear_bwd
PyObject* py_linear_bwd(PyObject*, PyObject* const* a, Py_ssize_t n) {
  if (n != 18 || !THPVariable_Check(a[0]) || !THPVariable_Check(a[3]))
    return PyErr_Format(PyExc_TypeError, "linear_bwd: 18 arguments, got %zd", n);
  for (int i : {2, 8, 9, 10, 11})
    if (a[i] != Py_None && !THPVariable_Check(a[i])) return PyErr_Format(PyExc_TypeError, "linear_bwd: argument %d", i);
  const at::Tensor &dy2 = THPVariable_Unpack(a[0]), &home = THPVariable_Unpack(a[3]);
  int64_t col0, w_off, n_s, k;
  if (!from_py(a[1], col0) || !from_py(a[4], w_off) || !from_py(a[6], n_s) || !from_py(a[7], k)) return nullptr;
  rtp_rotated_linear L;
  int dt;
  Mat dy;
  if (!layer_of(home, w_off, a[5], n_s, k, L, dt) || !as_mat(dy2, "dy", dy)) return nullptr;
  if (col0 < 0 || dy.cols - col0 < n_s * L.shards || dy2.scalar_type() != home.scalar_type())
    return bad("rotated_linear_bwd: dy must be [rows, >= shards * n_s] in the shards' dtype");
  const at::Tensor *x2 = opt_tensor(a[2]), *dx = opt_tensor(a[8]), *init = opt_tensor(a[9]), *gate = opt_tensor(a[10]),
                   *grads = opt_tensor(a[11]);
  rtp_rotated_linear_bwd_args o;
  memset(&o, 0, sizeof(o));
  int32_t done = 0;
  o.done = &done;
  auto fits = [&](const at::Tensor& t, bool f32_ok) {
    return t.scalar_type() == home.scalar_type() || (f32_ok && t.scalar_type() == at::kFloat);
  };
  Mat m, x{nullptr, dy.rows, k, k};
  if (x2 && !as_mat(*x2, "x", x)) return nullptr;
  if (dx) {
    if (!as_mat(*dx, "dx", m)) return nullptr;
    if (m.rows != dy.rows || m.cols != k) return bad("rotated_linear_bwd: dx must be [rows, k]");
    if (!fits(*dx, true)) return PyErr_Format(PyExc_TypeError, "rotated_linear_bwd: dx must be in the shards' dtype or float32");
    o.dx = m.p, o.ld_dx = m.ld;
    o.dx_flags = dx->scalar_type() != home.scalar_type() ? RTP_GEMM_OUT_F32 : 0;
    if (init) {
      if (!as_mat(*init, "dx_init", m)) return nullptr;
      if (m.rows != dy.rows || m.cols != k) return bad("rotated_linear_bwd: dx_init must match dx");
      if (!fits(*init, true))
        return PyErr_Format(PyExc_TypeError, "rotated_linear_bwd: dx_init must be in the shards' dtype or float32");
      o.dx_init = m.p, o.ld_dx_init = m.ld;
      if (init->scalar_type() != home.scalar_type()) o.dx_flags |= RTP_GEMM_CIN_F32;
    }
    if (gate) {
      if (!as_mat(*gate, "relu_gate", m)) return nullptr;
      if (m.rows != dy.rows || m.cols != k) return bad("rotated_linear_bwd: relu_gate must match dx");
      if (!fits(*gate, false)) return PyErr_Format(PyExc_TypeError, "rotated_linear_bwd: relu_gate must be in the shards' dtype");
      o.relu_gate = m.p, o.ld_relu_gate = m.ld;
    }
  }
  if (grads) {
    if (grads->sizes() != home.sizes() || grads->scalar_type() != home.scalar_type() || !grads->is_contiguous() || !x2)
      return bad("rotated_linear_bwd: grads must be laid out like home, and the layer's input is needed");
    o.grads = grads->data_ptr();
    o.accumulate = PyObject_IsTrue(a[12]);
    if (!from_py(a[13], o.sgd_master) || !from_py(a[14], o.sgd_weights) || !from_py(a[15], o.sgd_lr) ||
        !from_py(a[16], o.sgd_clip))
      return nullptr;
    o.sgd_skip_grad_store = o.sgd_master ? PyObject_IsTrue(a[17]) : 0;
  }
  void* st = current_stream();
  const int64_t ldy = dy.rows > 1 ? dy.ld : std::max<int64_t>(dy.cols, 1);
  const char* in = dy.p + col0 * (int64_t)dy2.element_size();
  const int rc = (WithoutGil(), Workspace(), f_linear_bwd(st, dt, &L, in, ldy, x.p, x.ld, dy.rows, &o));
  if (rc < 0) return raise_status(rc);
  return PyLong_FromLong(done);
}

// ---- the products of a row-parallel layer, of an attention core and of a run of experts, on tensors ----
// The same launches as gemm() with the descriptor filled here instead of by some twenty keyword arguments and their lookup.
// Forward + backward of layers that the host bounds, in processes of the slower / faster kind (a backward pass wakes a thread):
// row-parallel Linear 254x176x2368 122 / 61 -> 95 / 48 us, attention over 80 x 3 positions 200 / 122 -> 177 / 107, 16 experts of
// 192x256 473 / 335 -> 424 / 299.

// every argument at one of `at` is a tensor
template <size_t N>
bool tensors_at(const char* who, PyObject* const* a, const int (&at)[N]) {
  for (int i : at)
    if (!THPVariable_Check(a[i])) {
      PyErr_Format(PyExc_TypeError, "%s: argument %d has to be a tensor", who, i);
      return false;
    }
  return true;
}
char* at_element(const at::Tensor& t, int64_t i) { return (char*)t.data_ptr() + i * (int64_t)t.element_size(); }

// row_fwd(x2, flat, w_off, bias_off, n, k_s, out, col0, c_in):
// out = (c_in +) sum_g x2[:, col0 + g*k_s : ...] W_g^T + sum_g b_g
PyObject* py_row_fwd(PyObject*, PyObject* const* a, Py_ssize_t nargs) {
  if (nargs != 9) return PyErr_Format(PyExc_TypeError, "row_fwd(x2, flat, w_off, bias_off, n, k_s, out, col0, c_in)");
  if (!tensors_at("row_fwd", a, {0, 1, 6})) return nullptr;
  if (a[8] != Py_None && !THPVariable_Check(a[8])) return PyErr_Format(PyExc_TypeError, "row_fwd: c_in");
  const at::Tensor &x2 = THPVariable_Unpack(a[0]), &flat = THPVariable_Unpack(a[1]), &out = THPVariable_Unpack(a[6]);
  const at::Tensor* c_in = opt_tensor(a[8]);
  int64_t w_off, n, k_s, col0;
  if (!from_py(a[2], w_off) || !from_py(a[4], n) || !from_py(a[5], k_s) || !from_py(a[7], col0)) return nullptr;
  rtp_rotated_linear L;
  int dt;
  Mat x, o, ci;
  if (!layer_of(flat, w_off, a[3], n, k_s, L, dt) || !as_mat(x2, "operand", x) || !as_mat(out, "operand", o)) return nullptr;
  uint32_t flags = 0;
  auto f32 = [&](const at::Tensor& t, const char* what, uint32_t flag) {
    if (t.scalar_type() == flat.scalar_type()) return true;
    flags |= flag;
    if (t.scalar_type() == at::kFloat) return true;
    PyErr_Format(PyExc_TypeError, "row_fwd: %s must be in the shards' dtype or float32", what);
    return false;
  };
  rtp_gemm_desc d = product(x.rows, n, k_s, true, true);
  if (!f32(out, "out", RTP_GEMM_OUT_F32)) return nullptr;
  if (c_in) {
    if (!as_mat(*c_in, "c_in", ci) || !f32(*c_in, "c_in", RTP_GEMM_CIN_F32)) return nullptr;
    if (ci.rows != o.rows || ci.cols != o.cols) return bad("row_fwd: c_in must have the output's shape");
    d.c_in = ci.p, d.ld_cin = ci.ld;
  }
  d.a = at_element(x2, col0), d.lda = x.ld;
  d.b = at_element(flat, w_off), d.ldb = k_s;
  d.c_out = o.p, d.ldc = o.ld;
  if (L.bias_off >= 0) d.bias = at_element(flat, L.bias_off);
  d.bias_sk = d.b_sk = L.numel, d.a_sk = k_s, d.ksegs = L.shards;
  return run_product(dt, d, flags);
}

// row_dgrad(dy2, flat, w_off, n, k_s, out, col0): out[:, col0 + g*k_s : ...] = dy2 W_g
PyObject* py_row_dgrad(PyObject*, PyObject* const* a, Py_ssize_t nargs) {
  if (nargs != 7) return PyErr_Format(PyExc_TypeError, "row_dgrad(dy2, flat, w_off, n, k_s, out, col0)");
  if (!tensors_at("row_dgrad", a, {0, 1, 5})) return nullptr;
  const at::Tensor &dy2 = THPVariable_Unpack(a[0]), &flat = THPVariable_Unpack(a[1]), &out = THPVariable_Unpack(a[5]);
  int64_t w_off, n, k_s, col0;
  if (!from_py(a[2], w_off) || !from_py(a[3], n) || !from_py(a[4], k_s) || !from_py(a[6], col0)) return nullptr;
  rtp_rotated_linear L;
  int dt;
  Mat dy, o;
  if (!layer_of(flat, w_off, Py_None, n, k_s, L, dt) || !as_mat(dy2, "operand", dy) || !as_mat(out, "operand", o)) return nullptr;
  rtp_gemm_desc d = product(dy.rows, k_s, n, true, false);
  d.a = dy.p, d.lda = dy.ld;
  d.b = at_element(flat, w_off), d.ldb = k_s, d.b_sg = L.numel;
  d.c_out = at_element(out, col0), d.ldc = o.ld, d.c_sg = k_s;
  d.groups = L.shards;
  return run_product(dt, d, 0);
}

// row_wgrad(dy2, x2, grads, first, w_off, bias_off, n, k_s, col0, cnt, accumulate, sgd_master, sgd_weights, lr, clip,
//           skip_store) -> done flags: grads[first+g, w_off : ...] (+)= dy2^T x2[:, col0 + g*k_s : ...], and the bias rows
PyObject* py_row_wgrad(PyObject*, PyObject* const* a, Py_ssize_t nargs) {
  if (nargs != 16) return PyErr_Format(PyExc_TypeError, "row_wgrad: 16 arguments, got %zd", nargs);
  if (!tensors_at("row_wgrad", a, {0, 1, 2})) return nullptr;
  const at::Tensor &dy2 = THPVariable_Unpack(a[0]), &x2 = THPVariable_Unpack(a[1]), &grads = THPVariable_Unpack(a[2]);
  int64_t first, w_off, n, k_s, col0, cnt;
  if (!from_py(a[3], first) || !from_py(a[4], w_off) || !from_py(a[6], n) || !from_py(a[7], k_s) || !from_py(a[8], col0) ||
      !from_py(a[9], cnt))
    return nullptr;
  rtp_rotated_linear L;
  int dt;
  Mat dy, x;
  if (!layer_of(grads, w_off, a[5], n, k_s, L, dt) || !as_mat(dy2, "operand", dy) || !as_mat(x2, "operand", x)) return nullptr;
  const bool accumulate = PyObject_IsTrue(a[10]);
  uint32_t flags = RTP_GEMM_STREAM_OUT;
  rtp_gemm_desc d = product(n, k_s, dy.rows, false, false);
  d.a = dy.p, d.lda = dy.ld;
  d.b = at_element(x2, col0), d.ldb = x.ld, d.b_sg = k_s;
  d.c_out = at_element(grads, first * L.numel + w_off), d.ldc = k_s, d.c_sg = L.numel;
  d.c_in = accumulate ? d.c_out : nullptr, d.ld_cin = k_s, d.cin_sg = L.numel;
  if (L.bias_off >= 0) d.a_rowsum = at_element(grads, first * L.numel + L.bias_off);
  d.rowsum_sg = L.numel;
  if (accumulate) flags |= RTP_GEMM_ROWSUM_ACCUM;
  d.groups = cnt;
  if (!from_py(a[11], d.sgd_master) || !from_py(a[12], d.sgd_weights) || !from_py(a[13], d.sgd_lr) ||
      !from_py(a[14], d.sgd_clip))
    return nullptr;
  if (PyObject_IsTrue(a[15])) flags |= RTP_GEMM_SGD_SKIP_OUT;
  return run_product(dt, d, flags);
}

// attention_wgrad(dout, o, dqkv, x, grads, first, cnt, accumulate, w_o, b_o, width, part, b_in, masters, weights, lr, clip, skip_store, apart) ->
// done flags, the in-projection's two bits up: the weight gradients of an attention layer whose shards hold W_in [3 part, width] at
// 0 and W_o [width, part] at w_o (biases at b_in, b_o or None) for the runs of `cnt` shards from `first` on, in one launch where that is
// faster and not `apart`: grads[first+g] (+)= dout^T o[:, block g] and dqkv[:, block g]^T x.  masters / weights: None, or the addresses of the
// fp32 parameters and their copies (W_o's, W_in's) as pairs.
PyObject* py_attention_wgrad(PyObject*, PyObject* const* a, Py_ssize_t nargs) {
  if (nargs != 19) return PyErr_Format(PyExc_TypeError, "attention_wgrad: 19 arguments, got %zd", nargs);
  if (!tensors_at("attention_wgrad", a, {0, 1, 2, 3, 4})) return nullptr;
  const at::Tensor &dout = THPVariable_Unpack(a[0]), &o = THPVariable_Unpack(a[1]), &dqkv = THPVariable_Unpack(a[2]),
                   &x = THPVariable_Unpack(a[3]), &grads = THPVariable_Unpack(a[4]);
  int64_t first, cnt, w_o, width, part;
  if (!from_py(a[5], first) || !from_py(a[6], cnt) || !from_py(a[8], w_o) || !from_py(a[10], width) || !from_py(a[11], part)) return nullptr;
  rtp_rotated_linear lo, li;
  int dt;
  Mat mdo, mo, mdq, mx;
  if (!layer_of(grads, w_o, a[9], width, part, lo, dt) || !layer_of(grads, 0, a[12], 3 * part, width, li, dt) || !as_mat(dout, "operand", mdo) ||
      !as_mat(o, "operand", mo) || !as_mat(dqkv, "operand", mdq) || !as_mat(x, "operand", mx))
    return nullptr;
  for (const at::Tensor* t : {&dout, &o, &dqkv, &x})
    if (t->scalar_type() != grads.scalar_type() || t->size(0) != dout.size(0) || !t->is_cuda())
      return bad("attention_wgrad: operands are matrices of as many rows in the gradients' dtype on the GPU");
  if (first < 0 || cnt < 1 || first + cnt > lo.shards || mdo.cols < width || mx.cols < width || mo.cols < (first + cnt) * part ||
      mdq.cols < (first + cnt) * 3 * part || w_o + width * part > lo.numel || 3 * part * width > lo.numel)
    return bad("attention_wgrad: operands do not fit the layer");
  const bool accumulate = PyObject_IsTrue(a[7]);
  const uint32_t flags = RTP_GEMM_STREAM_OUT | (accumulate ? (uint32_t)RTP_GEMM_ROWSUM_ACCUM : 0u) | (PyObject_IsTrue(a[17]) ? (uint32_t)RTP_GEMM_SGD_SKIP_OUT : 0u);
  void *masters[2] = {nullptr, nullptr}, *weights[2] = {nullptr, nullptr};
  float lr = 0.0f, clip = 0.0f;
  for (int side = 0; side < 2; ++side)
    if (PyObject* v = a[13 + side]; v != Py_None) {
      void** to = side ? weights : masters;
      if (!PyTuple_Check(v) || PyTuple_GET_SIZE(v) != 2 || !from_py(PyTuple_GET_ITEM(v, 0), to[0]) || !from_py(PyTuple_GET_ITEM(v, 1), to[1]))
        return PyErr_Occurred() ? nullptr : bad("attention_wgrad: a pair of addresses");
    }
  if (!from_py(a[15], lr) || !from_py(a[16], clip)) return nullptr;
  auto gradient = [&](const rtp_rotated_linear& L, const Mat& g, int64_t g_col, int64_t g_step, const Mat& in, int64_t in_col, int64_t in_step, int which) {
    const int64_t es = grads.element_size();
    rtp_gemm_desc d = product(L.n_s, L.k, g.rows, false, false);
    d.a = g.p + g_col * es, d.lda = g.ld, d.a_sg = g_step;
    d.b = in.p + in_col * es, d.ldb = in.ld, d.b_sg = in_step;
    d.c_out = at_element(grads, first * L.numel + L.w_off), d.ldc = L.k, d.c_sg = L.numel;
    d.c_in = accumulate ? d.c_out : nullptr, d.ld_cin = L.k, d.cin_sg = L.numel;
    if (L.bias_off >= 0) d.a_rowsum = at_element(grads, first * L.numel + L.bias_off);
    d.rowsum_sg = L.numel;
    d.groups = cnt;
    d.sgd_master = masters[which], d.sgd_weights = weights[which], d.sgd_lr = lr, d.sgd_clip = clip;
    return d;
  };
  rtp_gemm_desc d_o = gradient(lo, mdo, 0, 0, mo, first * part, part, 0);
  rtp_gemm_desc d_in = gradient(li, mdq, first * 3 * part, 3 * part, mx, 0, 0, 1);
  int done_o = 0, done_in = 0;
  settle_product(dt, d_o, flags, done_o);
  settle_product(dt, d_in, flags, done_in);
  void* st = current_stream();
  const bool apart = PyObject_IsTrue(a[18]);
  auto launch = [&] {
    if (!apart) return f_gemm_pair(st, dt, &d_o, &d_in);
    const int rc = f_gemm(st, dt, &d_o);
    return rc < 0 ? rc : f_gemm(st, dt, &d_in);
  };
  const int rc = (WithoutGil(), Workspace(), launch());
  if (rc < 0) return raise_status(rc);
  return PyLong_FromLong(done_o | done_in << 2);
}

// bmm(a, a_off, lda, a_kcontig, a_s, a_sg,  b, ... (as a),  c, c_off, ldc, c_s, c_sg,  m, n, k, batch, zdiv, groups):
// C = A B for every (group, outer, inner) problem, offsets and strides in elements, (outer, inner) strides as pairs; C in the
// operands' dtype or fp32
PyObject* py_bmm(PyObject*, PyObject* const* a, Py_ssize_t nargs) {
  if (nargs != 23) return PyErr_Format(PyExc_TypeError, "bmm: 23 arguments, got %zd", nargs);
  if (!tensors_at("bmm", a, {0, 6, 12})) return nullptr;
  const at::Tensor &A = THPVariable_Unpack(a[0]), &B = THPVariable_Unpack(a[6]), &C = THPVariable_Unpack(a[12]);
  const int dt = dtype_code(B.scalar_type());
  if (dt < 0 || A.scalar_type() != B.scalar_type() || (C.scalar_type() != B.scalar_type() && C.scalar_type() != at::kFloat))
    return bad("bmm: a and b fp32 or bf16, c in their dtype or fp32");
  if (!B.is_cuda()) {
    PyErr_SetString(g_error, "rtp_amd kernels run on the GPU only; got a CPU tensor (there is no CPU path)");
    return nullptr;
  }
  rtp_gemm_desc d = product(0, 0, 0, PyObject_IsTrue(a[3]), PyObject_IsTrue(a[9]));
  auto pair = [](PyObject* v, int64_t& so, int64_t& si) {
    if (!PyTuple_Check(v) || PyTuple_GET_SIZE(v) != 2) return PyErr_SetString(PyExc_TypeError, "bmm: a pair of strides"), false;
    return from_py(PyTuple_GET_ITEM(v, 0), so) && from_py(PyTuple_GET_ITEM(v, 1), si);
  };
  int64_t a_off, b_off, c_off;
  if (!from_py(a[1], a_off) || !from_py(a[2], d.lda) || !pair(a[4], d.a_so, d.a_si) || !from_py(a[5], d.a_sg) ||
      !from_py(a[7], b_off) || !from_py(a[8], d.ldb) || !pair(a[10], d.b_so, d.b_si) || !from_py(a[11], d.b_sg) ||
      !from_py(a[13], c_off) || !from_py(a[14], d.ldc) || !pair(a[15], d.c_so, d.c_si) || !from_py(a[16], d.c_sg) ||
      !from_py(a[17], d.m) || !from_py(a[18], d.n) || !from_py(a[19], d.k) || !from_py(a[20], d.batch) ||
      !from_py(a[21], d.zdiv) || !from_py(a[22], d.groups))
    return nullptr;
  d.a = at_element(A, a_off), d.b = at_element(B, b_off), d.c_out = at_element(C, c_off);
  return run_product(dt, d, C.scalar_type() != B.scalar_type() ? RTP_GEMM_OUT_F32 : 0);
}

// One local expert of every shard of a run: x, y [slots, m_dim] and h [slots, f_dim] contiguous, the expert's slab of
// `rows` slots starts at row r0 in the run's first shard and `row_step` rows further in each next one; w1, b1, w2, b2 are
// offsets inside a flat shard.
struct Experts {
  int dt;
  int64_t numel, shards, r0, row_step, rows, m_dim, f_dim, w1, b1, w2, b2;
  bool read(const char* who, const at::Tensor& flat, PyObject* const* a, const at::Tensor& narrow, const at::Tensor& wide) {
    dt = dtype_code(flat.scalar_type());
    if (flat.dim() != 2 || !flat.is_contiguous() || dt < 0) return bad("experts: flat must be a contiguous fp32 / bf16 matrix"), false;
    for (const at::Tensor* t : {&narrow, &wide})
      if (t->dim() != 2 || !t->is_contiguous() || t->scalar_type() != flat.scalar_type() || !t->is_cuda())
        return PyErr_Format(PyExc_ValueError, "%s: activations must be contiguous matrices in the shards' dtype on the GPU", who), false;
    numel = flat.size(1), shards = flat.size(0), m_dim = narrow.size(1), f_dim = wide.size(1);
    return from_py(a[0], r0) && from_py(a[1], row_step) && from_py(a[2], rows) && from_py(a[3], w1) && from_py(a[4], b1) &&
           from_py(a[5], w2) && from_py(a[6], b2);
  }
};
bool same_layout(const at::Tensor& t, const at::Tensor& like) {
  return t.sizes() == like.sizes() && t.is_contiguous() && t.scalar_type() == like.scalar_type();
}

// experts_fwd(flat, x, h, y, r0, row_step, rows, w1, b1, w2, b2): h = relu(x W1^T + b1), y = h W2^T + b2
PyObject* py_experts_fwd(PyObject*, PyObject* const* a, Py_ssize_t nargs) {
  if (nargs != 11) return PyErr_Format(PyExc_TypeError, "experts_fwd: 11 arguments, got %zd", nargs);
  if (!tensors_at("experts_fwd", a, {0, 1, 2, 3})) return nullptr;
  const at::Tensor &flat = THPVariable_Unpack(a[0]), &x = THPVariable_Unpack(a[1]), &h = THPVariable_Unpack(a[2]),
                   &y = THPVariable_Unpack(a[3]);
  Experts e;
  if (!e.read("experts_fwd", flat, a + 4, x, h)) return nullptr;
  if (!same_layout(y, x)) return bad("experts_fwd: y must be laid out like x");
  auto half = [&](const at::Tensor& in, const at::Tensor& out, int64_t w, int64_t b, int64_t n, int64_t k, uint32_t flags) {
    rtp_gemm_desc d = product(e.rows, n, k, true, true);
    d.a = at_element(in, e.r0 * k), d.lda = k, d.a_sg = e.row_step * k;
    d.b = at_element(flat, w), d.ldb = k, d.b_sg = e.numel;
    d.bias = at_element(flat, b), d.bias_sg = e.numel;
    d.c_out = at_element(out, e.r0 * n), d.ldc = n, d.c_sg = e.row_step * n;
    d.groups = e.shards;
    int done = 0;
    return launch_product(e.dt, d, flags, done);
  };
  if (!half(x, h, e.w1, e.b1, e.f_dim, e.m_dim, RTP_GEMM_RELU) || !half(h, y, e.w2, e.b2, e.m_dim, e.f_dim, 0)) return nullptr;
  Py_RETURN_NONE;
}

// experts_dgrad(flat, dy, h, dh, dx, r0, row_step, rows, w1, b1, w2, b2): dh = (dy W2) where h > 0, dx = dh W1
PyObject* py_experts_dgrad(PyObject*, PyObject* const* a, Py_ssize_t nargs) {
  if (nargs != 12) return PyErr_Format(PyExc_TypeError, "experts_dgrad: 12 arguments, got %zd", nargs);
  if (!tensors_at("experts_dgrad", a, {0, 1, 2, 3, 4})) return nullptr;
  const at::Tensor &flat = THPVariable_Unpack(a[0]), &dy = THPVariable_Unpack(a[1]), &h = THPVariable_Unpack(a[2]),
                   &dh = THPVariable_Unpack(a[3]), &dx = THPVariable_Unpack(a[4]);
  Experts e;
  if (!e.read("experts_dgrad", flat, a + 5, dy, h)) return nullptr;
  if (!same_layout(dh, h) || !same_layout(dx, dy)) return bad("experts_dgrad: dh and dx must be laid out like h and dy");
  auto half = [&](const at::Tensor& in, const at::Tensor& out, const at::Tensor* gate, int64_t w, int64_t n, int64_t k) {
    rtp_gemm_desc d = product(e.rows, n, k, true, false);
    d.a = at_element(in, e.r0 * k), d.lda = k, d.a_sg = e.row_step * k;
    d.b = at_element(flat, w), d.ldb = n, d.b_sg = e.numel;
    d.c_out = at_element(out, e.r0 * n), d.ldc = n, d.c_sg = e.row_step * n;
    if (gate) d.gate = at_element(*gate, e.r0 * n), d.ld_gate = n, d.gate_sg = e.row_step * n;
    d.groups = e.shards;
    int done = 0;
    return launch_product(e.dt, d, 0, done);
  };
  if (!half(dy, dh, &h, e.w2, e.f_dim, e.m_dim) || !half(dh, dx, nullptr, e.w1, e.m_dim, e.f_dim)) return nullptr;
  Py_RETURN_NONE;
}

// experts_wgrad(grads, dy, h, dh, x, r0, row_step, rows, w1, b1, w2, b2, first, cnt, accumulate) -> bit 0: the second layer's
// bias rows were produced, bit 1: the first layer's.  grads[first+g]: W2 (+)= dy^T h, W1 (+)= dh^T x over the slabs' rows, the
// bias gradients as the row sums of the first operands
PyObject* py_experts_wgrad(PyObject*, PyObject* const* a, Py_ssize_t nargs) {
  if (nargs != 15) return PyErr_Format(PyExc_TypeError, "experts_wgrad: 15 arguments, got %zd", nargs);
  if (!tensors_at("experts_wgrad", a, {0, 1, 2, 3, 4})) return nullptr;
  const at::Tensor &grads = THPVariable_Unpack(a[0]), &dy = THPVariable_Unpack(a[1]), &h = THPVariable_Unpack(a[2]),
                   &dh = THPVariable_Unpack(a[3]), &x = THPVariable_Unpack(a[4]);
  Experts e;
  if (!e.read("experts_wgrad", grads, a + 5, dy, h)) return nullptr;
  if (!same_layout(dh, h) || !same_layout(x, dy)) return bad("experts_wgrad: dh and x must be laid out like h and dy");
  int64_t first, cnt;
  if (!from_py(a[12], first) || !from_py(a[13], cnt)) return nullptr;
  const bool accumulate = PyObject_IsTrue(a[14]);
  // streamed stores: an expert's gradient (tens of MB per launch) is not read again before the optimiser, and written with
  // ordinary ones it evicts the launch's own operands from the caches (468 -> 338 us)
  const uint32_t flags = RTP_GEMM_STREAM_OUT | (accumulate ? (uint32_t)RTP_GEMM_ROWSUM_ACCUM : 0u);
  auto half = [&](const at::Tensor& g, const at::Tensor& in, int64_t w, int64_t b, int64_t m, int64_t n, int& done) {
    rtp_gemm_desc d = product(m, n, e.rows, false, false);
    d.a = at_element(g, e.r0 * m), d.lda = m, d.a_sg = e.row_step * m;
    d.b = at_element(in, e.r0 * n), d.ldb = n, d.b_sg = e.row_step * n;
    d.c_out = at_element(grads, first * e.numel + w), d.ldc = n, d.c_sg = e.numel;
    d.c_in = accumulate ? d.c_out : nullptr, d.ld_cin = n, d.cin_sg = e.numel;
    d.a_rowsum = at_element(grads, first * e.numel + b), d.rowsum_sg = e.numel;
    d.groups = cnt;
    return launch_product(e.dt, d, flags, done);
  };
  int done2 = 0, done1 = 0;
  if (!half(dy, h, e.w2, e.b2, e.m_dim, e.f_dim, done2) || !half(dh, x, e.w1, e.b1, e.f_dim, e.m_dim, done1)) return nullptr;
  return PyLong_FromLong((done2 & 1) | (done1 & 1) << 1);
}

// ---- GradBook ----
// The parameters of a layer, shard by shard, and their slices of the gradient buffer.  attach() is what a backward pass
// does before it writes the buffer (allign_grad of the reference, rtp/module/collectives.py:75-79), for all shards at once:
//   0  no parameter of some kind in every shard had a gradient: all slices attached, to be overwritten
//   1  every parameter holds its own slice: to be accumulated into
//  -1  anything else (shards that differ, a .grad somebody put there): nothing changed, the caller goes shard by shard
struct GradBook {
  PyObject_HEAD std::vector<std::vector<at::Tensor>>* params;
  std::vector<std::vector<at::Tensor>>* views;
};

bool tensor_lists(PyObject* o, std::vector<std::vector<at::Tensor>>& out) {
  PyObject* shards = PySequence_Fast(o, "GradBook: a list of lists of tensors");
  if (!shards) return false;
  bool ok = true;
  for (Py_ssize_t s = 0; ok && s < PySequence_Fast_GET_SIZE(shards); ++s) {
    PyObject* row = PySequence_Fast(PySequence_Fast_GET_ITEM(shards, s), "GradBook: a list of lists of tensors");
    if (!row) {
      ok = false;
      break;
    }
    out.emplace_back();
    for (Py_ssize_t i = 0; ok && i < PySequence_Fast_GET_SIZE(row); ++i) {
      PyObject* t = PySequence_Fast_GET_ITEM(row, i);
      if (!THPVariable_Check(t)) {
        PyErr_SetString(PyExc_TypeError, "GradBook: a list of lists of tensors");
        ok = false;
      } else {
        out.back().push_back(THPVariable_Unpack(t));
      }
    }
    Py_DECREF(row);
  }
  Py_DECREF(shards);
  return ok;
}

PyObject* book_new(PyTypeObject* type, PyObject* args, PyObject*) {
  PyObject *p, *v;
  if (!PyArg_ParseTuple(args, "OO", &p, &v)) return nullptr;
  GradBook* b = (GradBook*)type->tp_alloc(type, 0);
  if (!b) return nullptr;
  b->params = new std::vector<std::vector<at::Tensor>>();
  b->views = new std::vector<std::vector<at::Tensor>>();
  bool ok = tensor_lists(p, *b->params) && tensor_lists(v, *b->views);
  if (ok) {
    ok = b->params->size() == b->views->size();
    for (size_t s = 0; ok && s < b->params->size(); ++s) ok = (*b->params)[s].size() == (*b->views)[s].size();
    if (!ok) PyErr_SetString(PyExc_ValueError, "GradBook: one slice per parameter");
  }
  if (!ok) {
    Py_DECREF(b);
    return nullptr;
  }
  return (PyObject*)b;
}
void book_dealloc(PyObject* o) {
  GradBook* b = (GradBook*)o;
  delete b->params;
  delete b->views;
  Py_TYPE(o)->tp_free(o);
}
PyObject* book_attach(PyObject* o, PyObject*) {
  GradBook& b = *(GradBook*)o;
  size_t fresh = 0, full = 0;
  for (size_t s = 0; s < b.params->size(); ++s) {
    const auto& row = (*b.params)[s];
    const bool none = std::any_of(row.begin(), row.end(), [](const at::Tensor& p) { return !p.grad().defined(); });
    bool own = !none;
    for (size_t i = 0; own && i < row.size(); ++i) own = row[i].grad().data_ptr() == (*b.views)[s][i].data_ptr();
    fresh += none, full += own;
  }
  if (fresh == b.params->size()) {
    for (size_t s = 0; s < b.params->size(); ++s)
      for (size_t i = 0; i < (*b.params)[s].size(); ++i) (*b.params)[s][i].mutable_grad() = (*b.views)[s][i];
    return PyLong_FromLong(0);
  }
  return PyLong_FromLong(full == b.params->size() ? 1 : -1);
}
// every parameter has some gradient
PyObject* book_complete(PyObject* o, PyObject*) {
  for (const auto& row : *((GradBook*)o)->params)
    for (const at::Tensor& p : row)
      if (!p.grad().defined()) Py_RETURN_FALSE;
  Py_RETURN_TRUE;
}
// .grad = None for every parameter (zero_grad(set_to_none=True))
PyObject* book_drop(PyObject* o, PyObject*) {
  for (const auto& row : *((GradBook*)o)->params)
    for (const at::Tensor& p : row)
      if (p.grad().defined()) p.mutable_grad() = at::Tensor();
  Py_RETURN_NONE;
}

PyMethodDef book_methods[] = {{"attach", Entry<book_attach>::call, METH_NOARGS, nullptr},
                              {"complete", Entry<book_complete>::call, METH_NOARGS, nullptr},
                              {"drop", Entry<book_drop>::call, METH_NOARGS, nullptr},
                              {nullptr, nullptr, 0, nullptr}};
PyTypeObject g_book_type = {PyVarObject_HEAD_INIT(nullptr, 0)};

#define METHOD(name) {#name, (PyCFunction)(void*)Entry<py_##name>::call, METH_FASTCALL, nullptr},
PyMethodDef g_methods[] = {{"bind", Entry<py_bind>::call, METH_VARARGS, nullptr},
                           {"gemm", (PyCFunction)(void*)Entry<py_gemm>::call, METH_FASTCALL | METH_KEYWORDS, nullptr},
                           METHOD(linear_fwd) METHOD(linear_bwd) METHOD(row_fwd) METHOD(row_dgrad)
                           METHOD(row_wgrad) METHOD(attention_wgrad) METHOD(bmm) METHOD(experts_fwd)
                           METHOD(experts_dgrad) METHOD(experts_wgrad)
                           RTP_ENTRY_POINTS(METHOD, METHOD){nullptr, nullptr, 0, nullptr}};
#undef METHOD
PyModuleDef g_module = {PyModuleDef_HEAD_INIT, "_rtp_native", "librtp_hip.so for the calls of a training step", -1, g_methods};

}  // namespace

PyMODINIT_FUNC PyInit__rtp_native(void) {
  g_field_index = PyDict_New();
  for (size_t i = 0; i < sizeof(g_fields) / sizeof(g_fields[0]); ++i) {
    g_fields[i].key = PyUnicode_InternFromString(g_fields[i].name);
    PyObject* idx = PyLong_FromSize_t(i);
    PyDict_SetItem(g_field_index, g_fields[i].key, idx);
    Py_DECREF(idx);
  }
  g_book_type.tp_name = "_rtp_native.GradBook";
  g_book_type.tp_basicsize = sizeof(GradBook);
  g_book_type.tp_flags = Py_TPFLAGS_DEFAULT;
  g_book_type.tp_new = Entry<book_new>::call;
  g_book_type.tp_dealloc = book_dealloc;
  g_book_type.tp_methods = book_methods;
  if (PyType_Ready(&g_book_type) < 0) return nullptr;
  PyObject* m = PyModule_Create(&g_module);
  if (m) {
    Py_INCREF(&g_book_type);
    PyModule_AddObject(m, "GradBook", (PyObject*)&g_book_type);
  }
  return m;
}
