// CPython binding of the launching entry points: the entry's arguments are taken from the tensors here, and the calls that a
// program makes one at a time (the linear, the gated feed-forward, the attention over a cached prefix) are checked and given
// their output tensor here as well.
//
// Why not ctypes: a launch costs 3.3 us of host time; around it a linear's call spent 1.6 us converting 17 arguments, 2.1
// allocating the output through Python and 0.9 finding stream and workspace, more than most kernels of this size take.
// Calls in a row, us, ctypes against this: linear 1 x 720 -> 2048 7.4 -> 4.3 (the launch), gated feed-forward 50 x 720 x 2048
// 11.9 -> 10.5, attention 50 x (241 + 50) keys 10.2 -> 5.7 (both now the device's time); a SmolVLA request of two cameras
// without a recorded graph, whose prefix is 190 launches, 4610 -> 4420.
//
// Every C++ exception ends in a Python one (HANDLE_TH_ERRORS); the interpreter is let go of around the launch, as ctypes does.
#include <torch/csrc/Device.h>
#include <torch/csrc/Exceptions.h>
#include <torch/csrc/autograd/python_variable.h>

#include <ATen/ops/empty.h>
#include <c10/hip/HIPFunctions.h>
#include <c10/hip/HIPStream.h>

#include <array>
#include <tuple>
#include <type_traits>
#include <utility>

#include "../../include/tybok_hip.h"

namespace {

void* current_stream() { return (void*)c10::hip::getCurrentHIPStream().stream(); }

// An error that is already set as a Python exception.
[[noreturn]] void raised() { throw python_error(); }

template <class... A>
[[noreturn]] void raise(PyObject* type, const char* fmt, A... a) {
  PyErr_Format(type, fmt, a...);
  raised();
}

// ---------------------------------------------------------------- arguments
const at::Tensor& tensor(PyObject* o, const char* what) {
  if (!THPVariable_Check(o)) raise(PyExc_TypeError, "%s must be a tensor, got %s", what, Py_TYPE(o)->tp_name);
  return THPVariable_Unpack(o);
}

const at::Tensor* maybe_tensor(PyObject* o, const char* what) { return o == Py_None ? nullptr : &tensor(o, what); }

long long integer(PyObject* o) {
  const long long v = PyLong_AsLongLong(o);
  if (v == -1 && PyErr_Occurred()) raised();
  return v;
}

template <class T>
T arg(PyObject* o) {
  if constexpr (std::is_pointer_v<T>) {
    if (o == Py_None) return nullptr;
    if (THPVariable_Check(o)) return (T)THPVariable_Unpack(o).data_ptr();
    void* p = PyLong_AsVoidPtr(o);
    if (!p && PyErr_Occurred()) raised();
    return (T)p;
  } else if constexpr (std::is_floating_point_v<T>) {
    const double v = PyFloat_AsDouble(o);
    if (v == -1.0 && PyErr_Occurred()) raised();
    return (T)v;
  } else if constexpr (std::is_same_v<T, size_t>) {
    const size_t v = PyLong_AsSize_t(o);
    if (v == (size_t)-1 && PyErr_Occurred()) raised();
    return v;
  } else {
    const long long v = integer(o);
    if ((long long)(T)v != v) raise(PyExc_OverflowError, "an argument of %lld does not fit the entry point's type", v);
    return (T)v;
  }
}

// Calls f, the last of whose arguments is the stream, on torch's current one; a refusal becomes the RuntimeError of native.check.
template <class... P, class... A>
void launch(const char* name, int (*f)(P...), A... a) {
  void* stream = current_stream();
  int rc;
  {
    pybind11::gil_scoped_release free;
    rc = f(a..., stream);
  }
  if (rc != 0) {
    const char* msg = tk_last_error();
    raise(PyExc_RuntimeError, "%s failed (%d): %s", name, rc, msg ? msg : "unknown error");
  }
}

template <class... P, size_t... I>
void spread(const char* name, int (*f)(P...), PyObject* const* a, std::index_sequence<I...>) {
  using Types = std::tuple<P...>;
  // (braces: the conversions run in the order of the arguments)
  const std::tuple<std::tuple_element_t<I, Types>...> v{arg<std::tuple_element_t<I, Types>>(a[I])...};
  launch(name, f, std::get<I>(v)...);
}

template <class... P>
PyObject* entry(const char* name, int (*f)(P...), PyObject* const* a, Py_ssize_t n) {
  constexpr size_t want = sizeof...(P) - 1;  // all but the stream
  if ((size_t)n != want) raise(PyExc_TypeError, "%s takes %zu arguments, got %zd", name, want, n);
  spread(name, f, a, std::make_index_sequence<want>());
  Py_RETURN_NONE;
}

// ---------------------------------------------------------------- the workspace of a call
PyObject *s_buf, *s_nbytes;                          // interned attribute names
PyObject *g_default_ws = nullptr, *g_make_ws = nullptr;  // ops._default_ws and ops.default_workspace

struct Ws {
  void* ptr;
  size_t nbytes;
};

struct Ref {
  PyObject* o;
  explicit Ref(PyObject* p) : o(p) {
    if (!p) raised();
  }
  Ref(const Ref&) = delete;
  ~Ref() { Py_DECREF(o); }
};

// ws, or the default one of x's device (device_index >= 0).
Ws workspace(PyObject* ws, const at::Tensor& x) {
  if (ws == Py_None) {
    const Ref key(PyLong_FromLong(x.device().index()));
    PyObject* have = PyDict_GetItemWithError(g_default_ws, key.o);
    if (have) return workspace(have, x);
    if (PyErr_Occurred()) raised();
    const Ref dev(THPDevice_New(x.device()));
    const Ref made(PyObject_CallOneArg(g_make_ws, dev.o));
    return workspace(made.o, x);  // (the dictionary keeps it)
  }
  const Ref buf(PyObject_GetAttr(ws, s_buf)), nbytes(PyObject_GetAttr(ws, s_nbytes));
  return {arg<void*>(buf.o), arg<size_t>(nbytes.o)};
}

// ---------------------------------------------------------------- the checks of ops.py
struct Rows {
  int m, ld;
};

int fits(int64_t v) {
  if (v != (int)v) raise(PyExc_OverflowError, "a size or stride of %lld elements does not fit 32 bits", (long long)v);
  return (int)v;
}

Rows check_act(const at::Tensor& x, int64_t k) {
  if (x.scalar_type() != at::kBFloat16 || !x.is_cuda()) raise(PyExc_TypeError, "activations must be bf16 CUDA tensors");
  if (x.dim() != 2 || x.size(1) != k || x.stride(1) != 1) {
    const Ref shape(PyTuple_New(x.dim()));
    for (int64_t i = 0; i < x.dim(); ++i) PyTuple_SET_ITEM(shape.o, i, PyLong_FromLongLong(x.size(i)));
    raise(PyExc_ValueError, "activations must be [M, %lld] with unit inner stride, got %R", (long long)k, shape.o);
  }
  return {fits(x.size(0)), fits(x.stride(0))};
}

struct Resid {
  const void* p = nullptr;
  int ld = 0, dtype = TK_BF16;
};

Resid check_resid(const at::Tensor* r, int64_t m, int64_t n) {
  if (!r) return {};
  if (r->dim() != 2 || r->size(0) != m || r->size(1) != n || r->stride(1) != 1) raise(PyExc_ValueError, "residual must be [M, N] with unit inner stride");
  if (r->scalar_type() != at::kBFloat16 && r->scalar_type() != at::kFloat) raise(PyExc_TypeError, "residual must be bf16 or fp32");
  return {r->data_ptr(), fits(r->stride(0)), r->scalar_type() == at::kFloat ? TK_F32 : TK_BF16};
}

const void* check_vector(const at::Tensor* v, int64_t n, const char* what) {
  if (!v) return nullptr;
  if (v->scalar_type() != at::kBFloat16 || v->numel() != n || !v->is_contiguous())
    raise(PyExc_ValueError, "%s must be a contiguous bf16 tensor of %lld elements", what, (long long)n);
  return v->data_ptr();
}

const void* check_ada(PyObject* pair, int which, int64_t k) {
  const at::Tensor& t = tensor(PySequence_Fast_GET_ITEM(pair, which), "adaptive-norm scale / shift");
  if (t.scalar_type() != at::kFloat || t.numel() != k || t.dim() < 1 || t.stride(-1) != 1)
    raise(PyExc_ValueError, "adaptive-norm scale / shift must be fp32 vectors of %lld contiguous elements", (long long)k);
  return t.data_ptr();
}

at::Tensor output(PyObject* out, const at::Tensor& x, int64_t m, int64_t n) {
  return out == Py_None ? at::empty({m, n}, x.options().dtype(at::kBFloat16)) : tensor(out, "out");
}

// ---------------------------------------------------------------- whole calls
#define TK_ARGS(want)                                                                                       \
  if (n != want) raise(PyExc_TypeError, "%s takes %d arguments, got %zd", __func__, (int)want, n)

// fp8w_gemm(x, w, scale, n, k, resid, gate, out, split_k, ws)
PyObject* fp8w_gemm(PyObject*, PyObject* const* a, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  TK_ARGS(10);
  const at::Tensor& x = tensor(a[0], "activations");
  const int N = arg<int>(a[3]), K = arg<int>(a[4]);
  const Rows r = check_act(x, K);
  const at::Tensor out = output(a[7], x, r.m, N);
  const Resid res = check_resid(maybe_tensor(a[5], "residual"), r.m, N);
  const void* gate = check_vector(maybe_tensor(a[6], "gate"), N, "gate");
  const Ws ws = workspace(a[9], x);
  launch("tk_fp8w_gemm", tk_fp8w_gemm, x.data_ptr(), r.ld, arg<void*>(a[1]), arg<void*>(a[2]), out.data_ptr(), fits(out.stride(0)), res.p, res.ld,
         res.dtype, gate, r.m, N, K, arg<int>(a[8]), ws.ptr, ws.nbytes);
  return THPVariable_Wrap(out);
  END_HANDLE_TH_ERRORS
}

// fp8w_gated_ffn(x, wgu, scale_gate, scale_up, i, k, wd, scale_down, n, k of down, act, resid, gate, norm_w, eps, ada, out, ws)
PyObject* fp8w_gated_ffn(PyObject*, PyObject* const* a, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  TK_ARGS(18);
  const at::Tensor& x = tensor(a[0], "activations");
  const int I = arg<int>(a[4]), K = arg<int>(a[5]);
  const Rows r = check_act(x, K);
  if (integer(a[9]) != I || integer(a[8]) != K) raise(PyExc_ValueError, "down weight must be [K, I]");
  const at::Tensor out = output(a[16], x, r.m, K);
  const Resid res = check_resid(maybe_tensor(a[11], "residual"), r.m, K);
  const void* gate = check_vector(maybe_tensor(a[12], "gate"), K, "gate");
  const Ws ws = workspace(a[17], x);
  const int act = arg<int>(a[10]), ldy = fits(out.stride(0));
  if (a[13] != Py_None || a[15] != Py_None) {
    const void* norm = check_vector(maybe_tensor(a[13], "norm weight"), K, "norm weight");
    const void *scale = nullptr, *shift = nullptr;
    if (a[15] != Py_None) {
      const Ref pair(PySequence_Fast(a[15], "ada must be (scale, shift)"));
      if (PySequence_Fast_GET_SIZE(pair.o) != 2) raise(PyExc_ValueError, "ada must be (scale, shift)");
      scale = check_ada(pair.o, 0, K), shift = check_ada(pair.o, 1, K);
    }
    launch("tk_fp8w_norm_gated_ffn", tk_fp8w_norm_gated_ffn, x.data_ptr(), r.ld, norm, arg<float>(a[14]), scale, shift, arg<void*>(a[1]), arg<void*>(a[2]),
           arg<void*>(a[3]), arg<void*>(a[6]), arg<void*>(a[7]), out.data_ptr(), ldy, res.p, res.ld, res.dtype, gate, r.m, K, I, act, ws.ptr, ws.nbytes);
  } else {
    launch("tk_fp8w_gated_ffn", tk_fp8w_gated_ffn, x.data_ptr(), r.ld, arg<void*>(a[1]), arg<void*>(a[2]), arg<void*>(a[3]), arg<void*>(a[6]),
           arg<void*>(a[7]), out.data_ptr(), ldy, res.p, res.ld, res.dtype, gate, r.m, K, I, act, ws.ptr, ws.nbytes);
  }
  return THPVariable_Wrap(out);
  END_HANDLE_TH_ERRORS
}

// One side of the keys: K [L, G, D] and V^T [G, D, >= L rounded up to 32].  A dimension of one element never advances: its
// stride is passed as 0, whatever the tensor records for it.
struct Keys {
  const void *k = nullptr, *vt = nullptr;
  int len = 0, heads = 0, sl = 0, sh = 0, vt_sd = 0, vt_sh = 0;
};

Keys check_keys(const at::Tensor& k, const at::Tensor& vt, int64_t d, const char* refusal) {
  const auto padded = [](int64_t len) { return (len + 31) / 32 * 32; };
  if (k.dim() != 3 || k.scalar_type() != at::kBFloat16 || k.size(2) != d || k.stride(2) != 1 || vt.scalar_type() != at::kBFloat16 || vt.dim() != 3 ||
      vt.size(0) != k.size(1) || vt.size(1) != d || vt.stride(2) != 1 || vt.size(2) < padded(k.size(0)))
    raise(PyExc_ValueError, "%s", refusal);
  Keys r;
  r.len = fits(k.size(0)), r.heads = fits(k.size(1));
  r.sl = r.len > 1 ? fits(k.stride(0)) : 0, r.sh = r.heads > 1 ? fits(k.stride(1)) : 0;
  r.vt_sh = r.heads > 1 ? fits(vt.stride(0)) : 0, r.vt_sd = fits(vt.stride(1));
  r.k = k.data_ptr(), r.vt = vt.data_ptr();
  return r;
}

bool is_mask(const at::Tensor& t) { return t.scalar_type() == at::kByte || t.scalar_type() == at::kBool; }

// expert_attn(q, prefix k, vt, k_lo, vt_lo, suffix k, vt, prefix_pad, mask_mode, mask2d, logits_bf16, out, ws)
PyObject* expert_attn(PyObject*, PyObject* const* a, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  TK_ARGS(13);
  const at::Tensor& q = tensor(a[0], "q");
  if (q.scalar_type() != at::kBFloat16 || q.dim() != 3 || q.stride(2) != 1) raise(PyExc_TypeError, "q must be bf16 [M, H, D] with a contiguous head dim");
  const int64_t m = q.size(0), h = q.size(1), d = q.size(2);
  Keys pre, suf;
  const void *k_lo = nullptr, *vt_lo = nullptr;
  int heads = 0;
  if (a[1] != Py_None) {
    const at::Tensor &k = tensor(a[1], "prefix K"), &vt = tensor(a[2], "prefix V^T");
    pre = check_keys(k, vt, d, "prefix must hold bf16 K [P, G, D] and V^T [G, D, >= P rounded up to 32]");
    heads = pre.heads;
    if (a[3] != Py_None) {
      const at::Tensor* lo = maybe_tensor(a[4], "the low plane of V^T");
      const at::Tensor& kl = tensor(a[3], "the low plane of K");
      if (!lo || kl.strides() != k.strides() || lo->strides() != vt.strides()) raise(PyExc_ValueError, "low planes must mirror the high planes' layout");
      k_lo = kl.data_ptr(), vt_lo = lo->data_ptr();
    }
  }
  if (a[5] != Py_None) {
    const at::Tensor& k = tensor(a[5], "suffix K");
    if (a[1] != Py_None && k.dim() == 3 && k.size(1) != heads) raise(PyExc_ValueError, "prefix and suffix must have the same number of kv heads");
    suf = check_keys(k, tensor(a[6], "suffix V^T"), d, "suffix must hold bf16 K [S, G, D] and V^T [G, D, >= S rounded up to 32]");
    heads = suf.heads;
  }
  const void* pad = nullptr;
  if (const at::Tensor* t = maybe_tensor(a[7], "prefix_pad")) {
    // (bool and uint8 are one byte each)
    if (!is_mask(*t) || t->numel() != pre.len || !t->is_contiguous()) raise(PyExc_ValueError, "prefix_pad must be a contiguous uint8/bool [P]");
    pad = t->data_ptr();
  }
  const void* mask2d = nullptr;
  int mask_ld = 0;
  if (const at::Tensor* t = maybe_tensor(a[9], "mask2d")) {
    if (!is_mask(*t) || t->dim() != 2 || t->size(0) != m || t->stride(1) != 1 || t->size(1) < (pre.len + 31) / 32 * 32)
      raise(PyExc_ValueError, "mask2d must be uint8/bool [M, >= P rounded up to 32] with unit inner stride");
    mask2d = t->data_ptr(), mask_ld = fits(t->stride(0));
  }
  const at::Tensor out = output(a[11], q, m, h * d);
  const Ws ws = workspace(a[12], q);
  launch("tk_expert_attn", tk_expert_attn, q.data_ptr(), fits(q.stride(0)), fits(q.stride(1)), pre.k, k_lo, pre.sl, pre.sh, pre.vt, vt_lo, pre.vt_sd,
         pre.vt_sh, suf.k, suf.sl, suf.sh, suf.vt, suf.vt_sd, suf.vt_sh, pad, mask2d, mask_ld, out.data_ptr(), fits(out.stride(0)), fits(m), pre.len,
         suf.len, fits(h), heads > 1 ? heads : 1, fits(d), arg<int>(a[8]), arg<int>(a[10]), ws.ptr, ws.nbytes);
  return THPVariable_Wrap(out);
  END_HANDLE_TH_ERRORS
}

// empty_bf16(like, m, n): bf16 [m, n] on like's device
PyObject* empty_bf16(PyObject*, PyObject* const* a, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  TK_ARGS(3);
  return THPVariable_Wrap(at::empty({integer(a[1]), integer(a[2])}, tensor(a[0], "like").options().dtype(at::kBFloat16)));
  END_HANDLE_TH_ERRORS
}

// set_workspaces(dictionary device index -> Workspace, function device -> Workspace)
PyObject* set_workspaces(PyObject*, PyObject* const* a, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  TK_ARGS(2);
  if (!PyDict_Check(a[0])) raise(PyExc_TypeError, "set_workspaces: a dictionary and a function");
  Py_INCREF(a[0]), Py_INCREF(a[1]);
  Py_XDECREF(g_default_ws), Py_XDECREF(g_make_ws);
  g_default_ws = a[0], g_make_ws = a[1];
  Py_RETURN_NONE;
  END_HANDLE_TH_ERRORS
}

#define TK_ENTRY(f)                                                            \
  PyObject* call_##f(PyObject*, PyObject* const* a, Py_ssize_t n) {            \
    HANDLE_TH_ERRORS                                                           \
    return entry(#f, f, a, n);                                                 \
    END_HANDLE_TH_ERRORS                                                       \
  }
#define TK_ENTRIES(X)                                                                                                          \
  X(tk_quant_act_rows) X(tk_w8a8_gemm) X(tk_w8a8_gated_ffn) X(tk_bf16w_dense) X(tk_f16w_dense) X(tk_bf16w_dense_rope)          \
  X(tk_bf16w_dense_vt) X(tk_bf16w_linear) X(tk_attn_prepare_kv) X(tk_expert_kv_project) X(tk_expert_cross_attn_fused)          \
  X(tk_batched_attn) X(tk_batched_transpose_v) X(tk_expert_tail) X(tk_expert_tail_embed) X(tk_layer_norm) X(tk_layer_norm_f16) \
  X(tk_add_layer_norm) X(tk_add_layer_norm_f16) X(tk_add_layer_norm_rows) X(tk_rms_norm_rows) X(tk_rope_rows) X(tk_prefix_meta) \
  X(tk_patchify_images) X(tk_patchify_images_f32) X(tk_prefix_rows)
TK_ENTRIES(TK_ENTRY)

#define TK_METHOD(f) {#f, (PyCFunction)(void (*)(void))call_##f, METH_FASTCALL, nullptr},
#define TK_WHOLE(f) {#f, (PyCFunction)(void (*)(void))f, METH_FASTCALL, nullptr},
PyMethodDef methods[] = {TK_WHOLE(fp8w_gemm) TK_WHOLE(fp8w_gated_ffn) TK_WHOLE(expert_attn) TK_WHOLE(empty_bf16) TK_WHOLE(set_workspaces)
                             TK_ENTRIES(TK_METHOD){nullptr, nullptr, 0, nullptr}};

PyModuleDef module = {PyModuleDef_HEAD_INIT, "tk_calls", "Launches of libtybok_hip.so on torch tensors.", -1, methods, nullptr, nullptr, nullptr, nullptr};

}  // namespace

PyMODINIT_FUNC PyInit_tk_calls() {
  s_buf = PyUnicode_InternFromString("buf");
  s_nbytes = PyUnicode_InternFromString("nbytes");
  if (!s_buf || !s_nbytes) return nullptr;
  return PyModule_Create(&module);
}
