// The host path of the public entry points: argument checks, buffers, autograd and the C-ABI calls, as one Python module.
//
// A call of a small problem lasts a few microseconds on the GPU, and what surrounds it decides: a Python
// autograd.Function takes 4-5 us per call on the way forward and, because the engine runs the backward on a thread of its own
// that has to take the interpreter lock from the waiting caller, 60-90 us on the way back.  Here the whole path is
// native: the functions take their arguments without a signature object (METH_FASTCALL), a call that needs no gradient
// creates no graph node, and the backward never touches the interpreter.
#include <Python.h>
#include <ATen/ATen.h>
#include <c10/core/DeviceGuard.h>
#include <c10/hip/HIPStream.h>
#include <torch/csrc/Exceptions.h>
#include <torch/csrc/autograd/custom_function.h>
#include <torch/csrc/autograd/python_variable.h>

#include "../../include/adasplash_hip.h"

namespace {
using at::Tensor;
using torch::autograd::AutogradContext;
using torch::autograd::variable_list;

// An assertion of the reference's entry points: becomes Python's AssertionError.
struct ArgumentAssertion {
  std::string what;
};
template <typename... A> void require(bool ok, const A&... parts) {
  if (!ok) throw ArgumentAssertion{c10::str(parts...)};
}

int dtype_code(const Tensor& t) {
  switch (t.scalar_type()) {
    case at::kFloat: return ADSP_F32;
    case at::kBFloat16: return ADSP_BF16;
    case at::kHalf: return ADSP_F16;
    default: C10_THROW_ERROR(TypeError, c10::str("unsupported dtype ", t.scalar_type(), "; expected float32, bfloat16 or float16"));
  }
}
void require_device(const Tensor& t) {
  TORCH_CHECK(!t.defined() || t.is_cuda(), "adasplash_amd kernels run on a ROCm device only; got a CPU tensor");
}
void check(int status, const char* what) {
  TORCH_CHECK(status == ADSP_OK, what, " failed: ", adsp_status_string(status), " (status ", status, ")");
}
void* stream_of(const Tensor& t) { return (void*)c10::hip::getCurrentHIPStream(t.get_device()).stream(); }
void* data(const Tensor& t) { return t.defined() ? t.data_ptr() : nullptr; }
size_t align256(size_t n) { return (n + 255) / 256 * 256; }
Tensor bytes(size_t n, const Tensor& like) {
  return at::empty({(int64_t)n}, like.options().dtype(at::kByte).requires_grad(false));
}

// ---- entmax rows ----------------------------------------------------------------------------------------------------
Tensor rows_forward(const Tensor& x, double alpha, int64_t n_iter, bool use_histogram, bool fast_math) {
  Tensor y = at::empty_like(x);  // (the kernel writes every element, zeros included)
  const int64_t cols = x.size(-1);
  const c10::DeviceGuard guard(x.device());
  check(adsp_entmax_rows_fwd(x.data_ptr(), y.data_ptr(), cols > 0 ? x.numel() / cols : 0, cols, dtype_code(x), alpha,
                             (int)n_iter, use_histogram, fast_math, stream_of(x)),
        "adsp_entmax_rows_fwd");
  return y;
}

struct RowsFunction : torch::autograd::Function<RowsFunction> {
  static Tensor forward(AutogradContext* ctx, const Tensor& x, double alpha, int64_t n_iter, bool use_histogram, bool fast_math) {
    Tensor y = rows_forward(x, alpha, n_iter, use_histogram, fast_math);
    ctx->save_for_backward({y});
    ctx->saved_data["alpha"] = alpha;
    return y;
  }
  static variable_list backward(AutogradContext* ctx, variable_list grads) {
    const Tensor y = ctx->get_saved_variables()[0];
    Tensor dy = grads[0];
    if (!dy.is_contiguous()) dy = dy.contiguous();
    if (dy.scalar_type() != y.scalar_type()) dy = dy.to(y.scalar_type());
    Tensor dx = at::empty_like(dy);
    const int64_t cols = y.size(-1);
    const c10::DeviceGuard guard(y.device());
    check(adsp_entmax_rows_bwd(y.data_ptr(), dy.data_ptr(), dx.data_ptr(), cols > 0 ? y.numel() / cols : 0, cols, dtype_code(y),
                               ctx->saved_data["alpha"].toDouble(), stream_of(y)),
          "adsp_entmax_rows_bwd");
    return {dx, Tensor(), Tensor(), Tensor(), Tensor()};
  }
};

// ---- attention ------------------------------------------------------------------------------------------------------
struct AttnCall {
  int version;  // 1: block-mask entry point, 2: causal alpha = 1.5
  double alpha;
  bool causal;
  int niter;
  Tensor varlen;
  int varlen_bits() const { return !varlen.defined() ? 0 : (varlen.scalar_type() == at::kLong ? 64 : 32); }
};
enum KeepMode { KEEP_NEVER = 0, KEEP_ALWAYS = 1, KEEP_AUTO = 2 };

// One allocation holds what the backward reads besides q, k and v: thresholds [B, Hq, N] fp32, the tile mask, and the supports
// the forward keeps (none when `supports` is 0).
struct SavedLayout {
  size_t bmask_off, supports_off, total, supports;
  SavedLayout(const Tensor& q, size_t supports_bytes) : supports(supports_bytes) {
    const int64_t B = q.size(0), Hq = q.size(1), N = q.size(2);
    bmask_off = align256((size_t)(B * Hq * N) * 4);
    supports_off = align256(bmask_off + (size_t)(B * Hq) * adsp_attn_bmask_words((int)N) * 4);
    total = supports_off + supports;
  }
};

// out, and in `saved` what a later backward needs.  Without one (`keep` is false) thresholds and tile mask share the
// workspace's allocation.
Tensor attn_forward(const Tensor& q, const Tensor& k, const Tensor& v, const AttnCall& c, bool keep, int keep_mode, Tensor* saved,
                    size_t* supports_bytes, bool* has_mask = nullptr) {
  const int B = (int)q.size(0), Hq = (int)q.size(1), N = (int)q.size(2), D = (int)q.size(3), Hkv = (int)k.size(1);
  const int dt = dtype_code(q);
  require(k.scalar_type() == q.scalar_type() && v.scalar_type() == q.scalar_type(), "q, k and v must share a dtype");
  // (a caller that asked for supports gets the route that keeps them)
  const bool mask = keep && ((keep_mode == KEEP_ALWAYS && dt != ADSP_F32) || adsp_attn_bwd_reads_bmask(B, Hq, Hkv, N, D, dt, c.alpha, c.causal));
  size_t sup = 0;
  if (mask && keep_mode != KEEP_NEVER) {
    sup = adsp_attn_supports_bytes(B, Hq, Hkv, N, D, dt);
    // "auto": at most twice the bytes of q, or 256 MiB
    const size_t most = std::max((size_t)2 * q.numel() * q.element_size(), (size_t)256 << 20);
    if (keep_mode == KEEP_AUTO && sup > most) sup = 0;
  }
  const c10::DeviceGuard guard(q.device());
  const SavedLayout l(q, sup);
  const size_t ws_bytes = adsp_attn_workspace_bytes(B, Hq, Hkv, N, D, dt);
  Tensor out = at::empty_like(q);
  Tensor kept, ws;
  char *kp, *wp;
  if (keep) {
    kept = bytes(l.total, q);
    kp = (char*)kept.data_ptr();
    if (ws_bytes) ws = bytes(ws_bytes, q);
    wp = (char*)data(ws);
  } else {
    kept = bytes(align256(l.total) + ws_bytes, q);
    kp = (char*)kept.data_ptr();
    wp = ws_bytes ? kp + align256(l.total) : nullptr;
  }
  float* taus = (float*)kp;
  int32_t* bmask = mask ? (int32_t*)(kp + l.bmask_off) : nullptr;
  void* supports = sup ? kp + l.supports_off : nullptr;
  void* stream = stream_of(q);
  if (c.version == 2) {
    const int st = sup ? adsp_attn_v2_fwd_keep(q.data_ptr(), k.data_ptr(), v.data_ptr(), out.data_ptr(), taus, bmask, data(c.varlen),
                                               c.varlen_bits(), B, Hq, Hkv, N, D, dt, c.niter, wp, ws_bytes, supports, sup, stream)
                       : adsp_attn_v2_fwd(q.data_ptr(), k.data_ptr(), v.data_ptr(), out.data_ptr(), taus, bmask, data(c.varlen),
                                          c.varlen_bits(), B, Hq, Hkv, N, D, dt, c.niter, wp, ws_bytes, stream);
    check(st, sup ? "adsp_attn_v2_fwd_keep" : "adsp_attn_v2_fwd");
  } else {
    const int st = sup ? adsp_attn_v1_fwd_keep(q.data_ptr(), k.data_ptr(), v.data_ptr(), out.data_ptr(), taus, bmask, data(c.varlen),
                                               c.varlen_bits(), B, Hq, N, D, dt, c.alpha, c.causal, c.niter, wp, ws_bytes, supports,
                                               sup, stream)
                       : adsp_attn_v1_fwd(q.data_ptr(), k.data_ptr(), v.data_ptr(), out.data_ptr(), taus, bmask, data(c.varlen),
                                          c.varlen_bits(), B, Hq, N, D, dt, c.alpha, c.causal, c.niter, wp, ws_bytes, nullptr, stream);
    check(st, sup ? "adsp_attn_v1_fwd_keep" : "adsp_attn_v1_fwd");
  }
  if (saved) *saved = kept;
  if (supports_bytes) *supports_bytes = sup;
  if (has_mask) *has_mask = mask;
  return out;
}

struct AttnFunction : torch::autograd::Function<AttnFunction> {
  static Tensor forward(AutogradContext* ctx, const Tensor& q, const Tensor& k, const Tensor& v, const AttnCall& c, int keep_mode) {
    Tensor saved;
    size_t sup = 0;
    bool mask = false;
    Tensor out = attn_forward(q, k, v, c, true, keep_mode, &saved, &sup, &mask);
    ctx->save_for_backward({q, k, v, saved});
    ctx->saved_data["alpha"] = c.alpha;
    ctx->saved_data["causal"] = c.causal;
    ctx->saved_data["supports"] = (int64_t)sup;
    ctx->saved_data["bmask"] = mask;
    if (c.varlen.defined()) ctx->saved_data["varlen"] = c.varlen;
    return out;
  }
  static variable_list backward(AutogradContext* ctx, variable_list grads) {
    const variable_list sv = ctx->get_saved_variables();
    const Tensor &q = sv[0], &k = sv[1], &v = sv[2], &saved = sv[3];
    const Tensor dout = grads[0].to(q.scalar_type()).contiguous();
    const int B = (int)q.size(0), Hq = (int)q.size(1), N = (int)q.size(2), D = (int)q.size(3), Hkv = (int)k.size(1);
    const int dt = dtype_code(q);
    const double alpha = ctx->saved_data["alpha"].toDouble();
    const bool causal = ctx->saved_data["causal"].toBool();
    AttnCall c{0, alpha, causal, 0, Tensor()};
    const auto it = ctx->saved_data.find("varlen");
    if (it != ctx->saved_data.end()) c.varlen = it->second.toTensor();
    const SavedLayout l(q, (size_t)ctx->saved_data["supports"].toInt());
    const c10::DeviceGuard guard(q.device());
    Tensor dq = at::empty_like(q), dk = at::empty_like(k), dv = at::empty_like(v);
    const size_t per_row = align256((size_t)B * Hq * N * 4);  // delta and 1 / sum p in front of the workspace
    const size_t ws_bytes = adsp_attn_bwd_workspace_bytes_causal(B, Hq, Hkv, N, D, dt, causal);
    Tensor scratch = bytes(2 * per_row + ws_bytes, q);
    char* const sp = (char*)scratch.data_ptr();
    char* const kp = (char*)saved.data_ptr();
    void* const ws = ws_bytes ? sp + 2 * per_row : nullptr;
    int32_t* const bmask = ctx->saved_data["bmask"].toBool() ? (int32_t*)(kp + l.bmask_off) : nullptr;
    void* const stream = stream_of(q);
    const int st =
        l.supports ? adsp_attn_bwd_kept(q.data_ptr(), k.data_ptr(), v.data_ptr(), dout.data_ptr(), (float*)kp, bmask,
                                        data(c.varlen), c.varlen_bits(), dq.data_ptr(), dk.data_ptr(), dv.data_ptr(), (float*)sp,
                                        (float*)(sp + per_row), B, Hq, Hkv, N, D, dt, alpha, causal, ws, ws_bytes,
                                        kp + l.supports_off, l.supports, stream)
                   : adsp_attn_bwd(q.data_ptr(), k.data_ptr(), v.data_ptr(), dout.data_ptr(), (float*)kp, bmask,
                                   data(c.varlen), c.varlen_bits(), dq.data_ptr(), dk.data_ptr(), dv.data_ptr(), (float*)sp,
                                   (float*)(sp + per_row), B, Hq, Hkv, N, D, dt, alpha, causal, ws, ws_bytes, stream);
    check(st, l.supports ? "adsp_attn_bwd_kept" : "adsp_attn_bwd");
    return {dq, dk, dv, Tensor(), Tensor()};
  }
};

// The checks of the reference's entry points (adasplash/adasplash_v2.py:1248-1276, adasplash/adasplash_block_mask.py:926-960).
void check_attention(const Tensor& q, const Tensor& k, const Tensor& v, AttnCall& c) {
  if (q.dim() != 4) C10_THROW_ERROR(ValueError, c10::str("q must have shape (batch, heads, sequence, head_dim); got ", q.sizes()));
  require(k.dim() == 4 && v.dim() == 4, "k and v must have shape (batch, heads, sequence, head_dim).");
  const int64_t B = q.size(0), Hq = q.size(1), N = q.size(2), D = q.size(3);
  require(D == 16 || D == 32 || D == 64 || D == 128 || D == 256, "head_dim must be 16, 32, 64, 128 or 256; got ", D, ".");
  const bool pow2 = (N & (N - 1)) == 0;
  if (c.version == 2) {
    require(k.sizes() == v.sizes(), "K and V must share shape; got k.shape=", k.sizes(), " v.shape=", v.sizes());
    const int64_t Hkv = k.size(1);
    require(Hkv >= 1 && Hq % Hkv == 0, "N_H (", Hq, ") must be a positive multiple of N_KV_H (", Hkv, ").");
    require(k.size(0) == B && k.size(2) == N && k.size(3) == D, "K/V must have shape (B=", B, ", N_KV_H, N_CTX=", N, ", H_DIM=", D,
            "); got ", k.sizes(), ".");
    require(N >= 64, "N_CTX=", N, " must be at least BMASK_TILE=64.");
    if (!c.varlen.defined()) {
      require(pow2, "If varlen is None, N_CTX must be a power of two.");
    } else {
      require(c.varlen.dim() == 1 && c.varlen.size(0) == B, "varlen must be a 1-D tensor of shape (B=", B, ",); got ", c.varlen.sizes(), ".");
      require(c.varlen.scalar_type() == at::kInt || c.varlen.scalar_type() == at::kLong, "varlen must be int32/int64; got ",
              c.varlen.scalar_type(), ".");
      require(c.varlen.device() == q.device(), "varlen must be on the same device as q.");
      require(c.varlen.is_contiguous(), "varlen must be contiguous.");
    }
  } else {
    if (!c.varlen.defined()) {
      require(N > 0 && pow2, "If varlen is not used, the context length must be a power of two.");
    } else {
      require(c.varlen.dim() == 1, "varlen must be a one-dimensional tensor.");
      require(c.varlen.size(0) == B, "varlen must have one entry per batch item (B=", B, ").");
    }
    require(k.sizes() == q.sizes() && v.sizes() == q.sizes(), "q, k and v must share one shape (no GQA in v1).");
  }
  require(q.is_contiguous() && k.is_contiguous() && v.is_contiguous(), "Q, K and/or V are not contiguous.");
  if (c.varlen.defined() && !c.varlen.is_contiguous()) c.varlen = c.varlen.contiguous();
  require_device(q);
  require_device(k);
  require_device(v);
  require_device(c.varlen);
  require(!c.varlen.defined() || c.varlen.scalar_type() == at::kInt || c.varlen.scalar_type() == at::kLong,
          "varlen must be int32/int64; got ", c.varlen.defined() ? c.varlen.scalar_type() : at::kInt, ".");
}

// ---- a few queries against a cache of keys --------------------------------------------------------------------------
// What stands between a tensor and its data: batches of vmap, wrappers of functorch's gradients, subclasses with a dispatch of
// their own, a sign that a view carries.  Torch's operators honour it; the data pointer does not.
bool is_plain(const Tensor& t) {
  static const c10::DispatchKeySet behind{c10::DispatchKey::FuncTorchBatched, c10::DispatchKey::FuncTorchGradWrapper, c10::DispatchKey::Python,
                                          c10::DispatchKey::Negative, c10::DispatchKey::ZeroTensor};
  return !t.defined() || !t.key_set().has_any(behind);
}

// Undefined where adsp_attn_decode_fwd does not take the call: a gradient is asked for, many queries, other head dims or types, an
// inner stride, tensors that are more than their data.
Tensor decode_forward(const Tensor& q, const Tensor& k, const Tensor& v, double alpha, const Tensor& varlen, bool causal, bool left,
                      const Tensor& slopes) {
  const int64_t B = q.size(0), H = q.size(1), q_len = q.size(2), D = q.size(3), k_len = k.size(2);
  const auto t = q.scalar_type();
  if (!is_plain(q) || !is_plain(k) || !is_plain(v) || !is_plain(varlen) || !is_plain(slopes)) return Tensor();
  if (!q.is_cuda() || !k.is_cuda() || !v.is_cuda() || k.device() != q.device() || v.device() != q.device()) return Tensor();
  if ((t != at::kFloat && t != at::kBFloat16 && t != at::kHalf) || k.scalar_type() != t || v.scalar_type() != t) return Tensor();
  if (q_len < 1 || q_len > 16 || (D != 32 && D != 64 && D != 128 && D != 256) || k_len < 1 || k_len > (1 << 24)) return Tensor();
  if (B < 1 || H < 1 || B * H > 65535 || !(alpha > 1.0)) return Tensor();
  if (varlen.defined() && (q_len == k_len || (varlen.scalar_type() != at::kInt && varlen.scalar_type() != at::kLong))) return Tensor();
  const int64_t per16 = 16 / q.element_size();
  for (const Tensor* x : {&k, &v}) {
    if (x->stride(3) != 1 || x->stride(0) % per16 || x->stride(1) % per16 || x->stride(2) % per16 || (uintptr_t)x->data_ptr() % 16)
      return Tensor();
  }
  const c10::DeviceGuard guard(q.device());
  Tensor qc = q.contiguous();
  if ((uintptr_t)qc.data_ptr() % 16) qc = qc.clone();
  Tensor vl = varlen, sl = slopes;
  if (vl.defined()) vl = vl.to(q.device()).contiguous();
  if (sl.defined()) sl = sl.to(q.device(), at::kFloat).contiguous();
  Tensor out = at::empty(q.sizes(), v.options());
  const size_t ws_bytes = adsp_attn_decode_workspace_bytes((int)B, (int)H, (int)q_len, (int)k_len);
  Tensor ws = bytes(ws_bytes, q);
  check(adsp_attn_decode_fwd(qc.data_ptr(), k.data_ptr(), v.data_ptr(), out.data_ptr(), data(vl),
                             !vl.defined() ? 0 : (vl.scalar_type() == at::kLong ? 64 : 32), left, (const float*)data(sl), (int)B, (int)H,
                             (int)q_len, (int)k_len, (int)D, k.stride(0), k.stride(1), k.stride(2), v.stride(0), v.stride(1), v.stride(2),
                             dtype_code(q), alpha, causal, ws.data_ptr(), ws_bytes, stream_of(q)),
        "adsp_attn_decode_fwd");
  return out;
}

bool wants_grad(const Tensor& t) { return t.requires_grad(); }
// A dual tensor of forward-mode differentiation need not ask for a gradient; the kernels have no forward derivative, with or
// without a graph and whatever the grad mode is.
bool has_tangent(const Tensor& t) { return t.defined() && t._fw_grad(0).defined(); }
void refuse_tangent(std::initializer_list<const Tensor*> inputs) {
  for (const Tensor* t : inputs)
    if (has_tangent(*t)) C10_THROW_ERROR(NotImplementedError, "forward-mode differentiation (jvp) of the entmax kernels is not implemented");
}

// ---- Python side ----------------------------------------------------------------------------------------------------
const Tensor& tensor_arg(PyObject* o, const char* what) {
  if (!THPVariable_Check(o)) C10_THROW_ERROR(TypeError, c10::str(what, " must be a tensor; got ", Py_TYPE(o)->tp_name));
  return THPVariable_Unpack(o);
}
double double_arg(PyObject* o) {
  const double v = PyFloat_AsDouble(o);
  if (v == -1.0 && PyErr_Occurred()) throw python_error();
  return v;
}
long long_arg(PyObject* o) {
  PyObject* i = PyNumber_Long(o);
  if (!i) throw python_error();
  const long v = PyLong_AsLong(i);
  Py_DECREF(i);
  if (v == -1 && PyErr_Occurred()) throw python_error();
  return v;
}
bool bool_arg(PyObject* o) {
  const int v = PyObject_IsTrue(o);
  if (v < 0) throw python_error();
  return v != 0;
}
void expect_args(Py_ssize_t n, Py_ssize_t want) {
  if (n != want) C10_THROW_ERROR(TypeError, c10::str("expected ", want, " arguments; got ", n));
}
template <typename F> PyObject* guarded(F f) {
  HANDLE_TH_ERRORS
  try {
    return THPVariable_Wrap(f());
  } catch (const ArgumentAssertion& e) {
    PyErr_SetString(PyExc_AssertionError, e.what.c_str());
    return nullptr;
  }
  END_HANDLE_TH_ERRORS
}

// entmax_rows(x, alpha, n_iter, use_histogram, fast_math)
PyObject* py_entmax_rows(PyObject*, PyObject* const* a, Py_ssize_t n) {
  return guarded([&] {
    expect_args(n, 5);
    const Tensor& x = tensor_arg(a[0], "x");
    const double alpha = double_arg(a[1]);
    const int64_t n_iter = long_arg(a[2]);
    const bool hist = bool_arg(a[3]), fast = bool_arg(a[4]);
    require(x.dim() > 0, "x must have at least one dimension");
    require(x.is_contiguous(), "x must be contiguous");
    require_device(x);
    refuse_tangent({&x});
    const bool grad = at::GradMode::is_enabled() && wants_grad(x);
    pybind11::gil_scoped_release no_gil;
    return grad ? RowsFunction::apply(x, alpha, n_iter, hist, fast) : rows_forward(x, alpha, n_iter, hist, fast);
  });
}

// attention(q, k, v, version, alpha, is_causal, niter, varlen, keep_mode)
PyObject* py_attention(PyObject*, PyObject* const* a, Py_ssize_t n) {
  return guarded([&] {
    expect_args(n, 9);
    const Tensor &q = tensor_arg(a[0], "q"), &k = tensor_arg(a[1], "k"), &v = tensor_arg(a[2], "v");
    AttnCall c{(int)long_arg(a[3]), double_arg(a[4]), bool_arg(a[5]), (int)long_arg(a[6]), Tensor()};
    if (a[7] != Py_None) c.varlen = tensor_arg(a[7], "varlen");
    const int keep_mode = (int)long_arg(a[8]);
    check_attention(q, k, v, c);
    refuse_tangent({&q, &k, &v});
    const bool grad = at::GradMode::is_enabled() && (wants_grad(q) || wants_grad(k) || wants_grad(v));
    pybind11::gil_scoped_release no_gil;
    return grad ? AttnFunction::apply(q, k, v, c, keep_mode) : attn_forward(q, k, v, c, false, KEEP_NEVER, nullptr, nullptr);
  });
}

// decode_attention(q, k, v, alpha, varlen, is_causal, left_padding, slopes) -> tensor, or None where the kernels do not take the call
PyObject* py_decode_attention(PyObject*, PyObject* const* a, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  expect_args(n, 8);
  const Tensor &q = tensor_arg(a[0], "q"), &k = tensor_arg(a[1], "k"), &v = tensor_arg(a[2], "v");
  const double alpha = double_arg(a[3]);
  Tensor varlen, slopes;
  if (a[4] != Py_None) varlen = tensor_arg(a[4], "varlen");
  const bool causal = bool_arg(a[5]), left = bool_arg(a[6]);
  if (a[7] != Py_None) slopes = tensor_arg(a[7], "alibi_slopes");
  if (at::GradMode::is_enabled() && (wants_grad(q) || wants_grad(k) || wants_grad(v) || (slopes.defined() && wants_grad(slopes))))
    Py_RETURN_NONE;
  if (has_tangent(q) || has_tangent(k) || has_tangent(v) || has_tangent(slopes)) Py_RETURN_NONE;  // (the dense path says what it can do)
  Tensor out;
  {
    pybind11::gil_scoped_release no_gil;
    out = decode_forward(q, k, v, alpha, varlen, causal, left, slopes);
  }
  if (!out.defined()) Py_RETURN_NONE;
  return THPVariable_Wrap(out);
  END_HANDLE_TH_ERRORS
}

PyMethodDef methods[] = {
    {"entmax_rows", (PyCFunction)(void (*)(void))py_entmax_rows, METH_FASTCALL, "alpha-entmax of the last dimension, with autograd"},
    {"attention", (PyCFunction)(void (*)(void))py_attention, METH_FASTCALL, "sparse entmax attention, with autograd"},
    {"decode_attention", (PyCFunction)(void (*)(void))py_decode_attention, METH_FASTCALL, "a few queries against a cache of keys"},
    {nullptr, nullptr, 0, nullptr}};
PyModuleDef module_def = {PyModuleDef_HEAD_INIT, "_adsp_torch", nullptr, -1, methods};
}  // namespace

PyMODINIT_FUNC PyInit__adsp_torch(void) {
  PyObject* m = PyModule_Create(&module_def);
  if (m && PyModule_AddStringConstant(m, "build_id", ADSP_BINDING_ID) != 0) {
    Py_DECREF(m);
    return nullptr;
  }
  return m;
}
