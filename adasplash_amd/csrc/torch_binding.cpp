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
// "auto": supports of at most twice the bytes of q, or 256 MiB
bool keeps_supports(int mode, size_t supports, size_t q_bytes) {
  if (mode == KEEP_NEVER || supports == 0) return false;
  return mode == KEEP_ALWAYS || supports <= std::max(2 * q_bytes, (size_t)256 << 20);
}

// What a forward leaves behind besides its output, in one allocation: thresholds [B, Hq, N] fp32, the tile mask, and the
// supports it keeps (none when `supports` is 0).
struct Kept {
  Tensor buffer;
  bool mask = false;
  size_t supports = 0, bmask_off = 0, supports_off = 0;
  int64_t rows = 0, mask_words = 0;
  size_t layout(const Tensor& q) {
    const int64_t B = q.size(0), Hq = q.size(1), N = q.size(2);
    rows = B * Hq * N;
    mask_words = B * Hq * (int64_t)adsp_attn_bmask_words((int)N);
    bmask_off = align256((size_t)rows * 4);
    supports_off = align256(bmask_off + (size_t)mask_words * 4);
    return supports_off + supports;
  }
  char* base() const { return (char*)buffer.data_ptr(); }
  float* taus() const { return (float*)base(); }
  int32_t* bmask() const { return mask ? (int32_t*)(base() + bmask_off) : nullptr; }
  void* kept_supports() const { return supports ? base() + supports_off : nullptr; }
};

// What the caller wants of a forward besides its output.
struct Wants {
  bool backward = false;         // what the backward reads: the tile mask where it does, and supports as the mode says
  int keep_mode = KEEP_NEVER;
  bool mask = false;             // the tile mask in any case
  bool outlives = false;         // what the forward leaves outlives the call
  unsigned long long* tile_counts = nullptr;
};

Tensor attn_forward(const Tensor& q, const Tensor& k, const Tensor& v, const AttnCall& c, const Wants& w, Kept& kept) {
  const int B = (int)q.size(0), Hq = (int)q.size(1), N = (int)q.size(2), D = (int)q.size(3), Hkv = (int)k.size(1);
  const int dt = dtype_code(q);
  require(k.scalar_type() == q.scalar_type() && v.scalar_type() == q.scalar_type(), "q, k and v must share a dtype");
  // (a caller that asked for supports gets the route that keeps them)
  kept.mask = w.mask || (w.backward && ((w.keep_mode == KEEP_ALWAYS && dt != ADSP_F32) ||
                                        adsp_attn_bwd_reads_bmask(B, Hq, Hkv, N, D, dt, c.alpha, c.causal)));
  if (kept.mask && w.backward && !w.tile_counts) {
    const size_t sup = adsp_attn_supports_bytes(B, Hq, Hkv, N, D, dt);
    if (keeps_supports(w.keep_mode, sup, q.numel() * q.element_size())) kept.supports = sup;
  }
  const c10::DeviceGuard guard(q.device());
  const size_t keep_bytes = kept.layout(q), ws_bytes = adsp_attn_workspace_bytes(B, Hq, Hkv, N, D, dt);
  Tensor out = at::empty_like(q);
  Tensor ws;
  void* wp = nullptr;
  if (w.outlives) {
    kept.buffer = bytes(keep_bytes, q);
    if (ws_bytes) ws = bytes(ws_bytes, q);
    wp = data(ws);
  } else {  // nothing outlives the call: one allocation for all of it
    kept.buffer = bytes(align256(keep_bytes) + ws_bytes, q);
    if (ws_bytes) wp = kept.base() + align256(keep_bytes);
  }
  const size_t sup = kept.supports;
  float* const taus = w.outlives ? kept.taus() : nullptr;  // (nobody reads the thresholds of a call without a gradient)
  void* const stream = stream_of(q);
  if (c.version == 2) {
    const int st = sup ? adsp_attn_v2_fwd_keep(q.data_ptr(), k.data_ptr(), v.data_ptr(), out.data_ptr(), taus, kept.bmask(),
                                               data(c.varlen), c.varlen_bits(), B, Hq, Hkv, N, D, dt, c.niter, wp, ws_bytes,
                                               kept.kept_supports(), sup, stream)
                       : adsp_attn_v2_fwd(q.data_ptr(), k.data_ptr(), v.data_ptr(), out.data_ptr(), taus, kept.bmask(),
                                          data(c.varlen), c.varlen_bits(), B, Hq, Hkv, N, D, dt, c.niter, wp, ws_bytes, stream);
    check(st, sup ? "adsp_attn_v2_fwd_keep" : "adsp_attn_v2_fwd");
  } else {
    const int st = sup ? adsp_attn_v1_fwd_keep(q.data_ptr(), k.data_ptr(), v.data_ptr(), out.data_ptr(), taus, kept.bmask(),
                                               data(c.varlen), c.varlen_bits(), B, Hq, N, D, dt, c.alpha, c.causal, c.niter, wp,
                                               ws_bytes, kept.kept_supports(), sup, stream)
                       : adsp_attn_v1_fwd(q.data_ptr(), k.data_ptr(), v.data_ptr(), out.data_ptr(), taus, kept.bmask(),
                                          data(c.varlen), c.varlen_bits(), B, Hq, N, D, dt, c.alpha, c.causal, c.niter, wp, ws_bytes,
                                          w.tile_counts, stream);
    check(st, sup ? "adsp_attn_v1_fwd_keep" : "adsp_attn_v1_fwd");
  }
  return out;
}

// dq, dk, dv from what the forward left (`bmask` and `supports` may be null)
variable_list attn_backward(const Tensor& q, const Tensor& k, const Tensor& v, const Tensor& upstream, const float* taus,
                            const int32_t* bmask, const void* supports, size_t supports_bytes, const AttnCall& c) {
  const Tensor dout = upstream.to(q.scalar_type()).contiguous();
  const int B = (int)q.size(0), Hq = (int)q.size(1), N = (int)q.size(2), D = (int)q.size(3), Hkv = (int)k.size(1);
  const int dt = dtype_code(q);
  const c10::DeviceGuard guard(q.device());
  Tensor dq = at::empty_like(q), dk = at::empty_like(k), dv = at::empty_like(v);
  const size_t per_row = align256((size_t)B * Hq * N * 4);  // delta and 1 / sum p in front of the workspace
  const size_t ws_bytes = adsp_attn_bwd_workspace_bytes_causal(B, Hq, Hkv, N, D, dt, c.causal);
  Tensor scratch = bytes(2 * per_row + ws_bytes, q);
  char* const sp = (char*)scratch.data_ptr();
  void* const ws = ws_bytes ? sp + 2 * per_row : nullptr;
  void* const stream = stream_of(q);
  const int st = supports_bytes
                     ? adsp_attn_bwd_kept(q.data_ptr(), k.data_ptr(), v.data_ptr(), dout.data_ptr(), taus, bmask, data(c.varlen),
                                          c.varlen_bits(), dq.data_ptr(), dk.data_ptr(), dv.data_ptr(), (float*)sp,
                                          (float*)(sp + per_row), B, Hq, Hkv, N, D, dt, c.alpha, c.causal, ws, ws_bytes, supports,
                                          supports_bytes, stream)
                     : adsp_attn_bwd(q.data_ptr(), k.data_ptr(), v.data_ptr(), dout.data_ptr(), taus, bmask, data(c.varlen),
                                     c.varlen_bits(), dq.data_ptr(), dk.data_ptr(), dv.data_ptr(), (float*)sp, (float*)(sp + per_row),
                                     B, Hq, Hkv, N, D, dt, c.alpha, c.causal, ws, ws_bytes, stream);
  check(st, supports_bytes ? "adsp_attn_bwd_kept" : "adsp_attn_bwd");
  return {dq, dk, dv};
}

struct AttnFunction : torch::autograd::Function<AttnFunction> {
  static Tensor forward(AutogradContext* ctx, const Tensor& q, const Tensor& k, const Tensor& v, const AttnCall& c, int keep_mode) {
    Kept kept;
    Wants wants;
    wants.backward = wants.outlives = true;
    wants.keep_mode = keep_mode;
    Tensor out = attn_forward(q, k, v, c, wants, kept);
    ctx->save_for_backward({q, k, v, kept.buffer});
    ctx->saved_data["alpha"] = c.alpha;
    ctx->saved_data["causal"] = c.causal;
    ctx->saved_data["supports"] = (int64_t)kept.supports;
    ctx->saved_data["bmask"] = kept.mask;
    if (c.varlen.defined()) ctx->saved_data["varlen"] = c.varlen;
    return out;
  }
  static variable_list backward(AutogradContext* ctx, variable_list grads) {
    const variable_list sv = ctx->get_saved_variables();
    const Tensor &q = sv[0], &k = sv[1], &v = sv[2];
    AttnCall c{0, ctx->saved_data["alpha"].toDouble(), ctx->saved_data["causal"].toBool(), 0, Tensor()};
    const auto it = ctx->saved_data.find("varlen");
    if (it != ctx->saved_data.end()) c.varlen = it->second.toTensor();
    Kept kept;
    kept.mask = ctx->saved_data["bmask"].toBool();
    kept.supports = (size_t)ctx->saved_data["supports"].toInt();
    kept.layout(q);
    kept.buffer = sv[3];
    variable_list d = attn_backward(q, k, v, grads[0], kept.taus(), kept.bmask(), kept.kept_supports(), kept.supports, c);
    d.resize(5);  // (no gradients of the call's description and the mode)
    return d;
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
    if (grad) return AttnFunction::apply(q, k, v, c, keep_mode);
    Kept kept;
    return attn_forward(q, k, v, c, Wants(), kept);
  });
}

// The forward and the backward as plain functions, for measurements and tests: what they leave and take is in the caller's hands.
// Shapes and types of q, k and v are the caller's business beyond what keeps the kernels inside the tensors.
void check_plain(const Tensor& q, const Tensor& k, const Tensor& v, const AttnCall& c) {
  require(q.dim() == 4 && k.dim() == 4 && k.sizes() == v.sizes(), "q, k and v must have shape (batch, heads, sequence, head_dim).");
  require(k.size(0) == q.size(0) && k.size(2) == q.size(2) && k.size(3) == q.size(3) && (c.version == 2 || k.size(1) == q.size(1)),
          "q and k do not fit each other: ", q.sizes(), " and ", k.sizes());
  require(q.is_contiguous() && k.is_contiguous() && v.is_contiguous(), "Q, K and/or V are not contiguous.");
  require(!c.varlen.defined() || ((c.varlen.scalar_type() == at::kInt || c.varlen.scalar_type() == at::kLong) && c.varlen.is_contiguous() &&
                                  c.varlen.numel() == q.size(0)),
          "varlen must be int32/int64, one entry per batch item");
  for (const Tensor* t : {&q, &k, &v, &c.varlen}) require_device(*t);
}

// attention_forward(q, k, v, version, alpha, is_causal, niter, varlen, keep_mode or None, tile_mask, tile_counts)
//   -> (out, taus, bmask or None, supports or None); keep_mode None: nothing is kept for a backward
PyObject* py_attention_forward(PyObject*, PyObject* const* a, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  try {
    expect_args(n, 11);
    const Tensor &q = tensor_arg(a[0], "q"), &k = tensor_arg(a[1], "k"), &v = tensor_arg(a[2], "v");
    AttnCall c{(int)long_arg(a[3]), double_arg(a[4]), bool_arg(a[5]), (int)long_arg(a[6]), Tensor()};
    if (a[7] != Py_None) c.varlen = tensor_arg(a[7], "varlen");
    Wants wants;
    wants.outlives = true;
    wants.backward = a[8] != Py_None;
    if (wants.backward) wants.keep_mode = (int)long_arg(a[8]);
    wants.mask = bool_arg(a[9]);
    check_plain(q, k, v, c);
    if (a[10] != Py_None) {
      const Tensor& counts = tensor_arg(a[10], "tile_counts");
      require_device(counts);
      require(c.version == 1 && counts.scalar_type() == at::kLong && counts.numel() == 2 && counts.is_contiguous(),
              "tile_counts must be two int64, with the block-mask variant");
      wants.tile_counts = (unsigned long long*)counts.data_ptr();
    }
    Kept kept;
    Tensor out, taus, bmask, supports;
    {
      pybind11::gil_scoped_release no_gil;
      out = attn_forward(q, k, v, c, wants, kept);
      const auto part = [&](size_t off, int64_t len, at::ScalarType t) { return kept.buffer.narrow(0, (int64_t)off, len).view(t); };
      taus = part(0, kept.rows * 4, at::kFloat).view({q.size(0), q.size(1), q.size(2)});
      if (kept.mask) bmask = part(kept.bmask_off, kept.mask_words * 4, at::kInt).view({q.size(0), q.size(1), -1});
      if (kept.supports) supports = part(kept.supports_off, (int64_t)kept.supports, at::kByte);
    }
    PyObject* tuple = PyTuple_New(4);
    if (!tuple) throw python_error();
    Tensor* const parts[4] = {&out, &taus, &bmask, &supports};
    for (int i = 0; i < 4; ++i) PyTuple_SET_ITEM(tuple, i, THPVariable_Wrap(*parts[i]));  // (an undefined tensor becomes None)
    return tuple;
  } catch (const ArgumentAssertion& e) {
    PyErr_SetString(PyExc_AssertionError, e.what.c_str());
    return nullptr;
  }
  END_HANDLE_TH_ERRORS
}

// attention_backward(q, k, v, dout, taus, bmask or None, alpha, is_causal, varlen, supports or None) -> (dq, dk, dv)
PyObject* py_attention_backward(PyObject*, PyObject* const* a, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  try {
    expect_args(n, 10);
    const Tensor &q = tensor_arg(a[0], "q"), &k = tensor_arg(a[1], "k"), &v = tensor_arg(a[2], "v"), &dout = tensor_arg(a[3], "dout"),
                 &taus = tensor_arg(a[4], "taus");
    AttnCall c{2, double_arg(a[6]), bool_arg(a[7]), 0, Tensor()};
    if (a[8] != Py_None) c.varlen = tensor_arg(a[8], "varlen");
    Tensor bmask, supports;
    if (a[5] != Py_None) bmask = tensor_arg(a[5], "bmask");
    if (a[9] != Py_None) supports = tensor_arg(a[9], "supports");
    check_plain(q, k, v, c);
    for (const Tensor* t : std::initializer_list<const Tensor*>{&dout, &taus, &bmask, &supports}) require_device(*t);
    require(k.scalar_type() == q.scalar_type() && v.scalar_type() == q.scalar_type(), "q, k and v must share a dtype");
    require(dout.sizes() == q.sizes(), "dout must have q's shape");
    const int64_t heads = q.size(0) * q.size(1);
    require(taus.scalar_type() == at::kFloat && taus.is_contiguous() && taus.numel() == heads * q.size(2), "taus must be what the forward returned");
    require(!bmask.defined() || (bmask.scalar_type() == at::kInt && bmask.is_contiguous() &&
                                 bmask.numel() == heads * (int64_t)adsp_attn_bmask_words((int)q.size(2))),
            "bmask must be what the forward returned");
    require(!supports.defined() || (supports.scalar_type() == at::kByte && supports.is_contiguous()), "supports must be what the forward returned");
    variable_list d;
    {
      pybind11::gil_scoped_release no_gil;
      d = attn_backward(q, k, v, dout, (const float*)taus.data_ptr(), (const int32_t*)data(bmask), data(supports),
                        supports.defined() ? (size_t)supports.numel() : 0, c);
    }
    PyObject* tuple = PyTuple_New(3);
    if (!tuple) throw python_error();
    for (int i = 0; i < 3; ++i) PyTuple_SET_ITEM(tuple, i, THPVariable_Wrap(d[i]));
    return tuple;
  } catch (const ArgumentAssertion& e) {
    PyErr_SetString(PyExc_AssertionError, e.what.c_str());
    return nullptr;
  }
  END_HANDLE_TH_ERRORS
}

// keeps_supports(mode, supports_bytes, q_bytes): whether a forward keeps supports of that size for its backward
PyObject* py_keeps_supports(PyObject*, PyObject* const* a, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  expect_args(n, 3);
  return PyBool_FromLong(keeps_supports((int)long_arg(a[0]), (size_t)long_arg(a[1]), (size_t)long_arg(a[2])));
  END_HANDLE_TH_ERRORS
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
    {"attention_forward", (PyCFunction)(void (*)(void))py_attention_forward, METH_FASTCALL, "the attention forward, with what it leaves behind"},
    {"attention_backward", (PyCFunction)(void (*)(void))py_attention_backward, METH_FASTCALL, "the attention backward from what the forward left"},
    {"keeps_supports", (PyCFunction)(void (*)(void))py_keeps_supports, METH_FASTCALL, "whether supports of a size are kept"},
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
