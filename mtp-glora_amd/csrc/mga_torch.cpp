// The package's per-layer calls for torch tensors, as one native call each:
// argument checks, output and workspace allocation, the C ABI call and the
// autograd node. The Python forms spend 20-50 us of interpreter time on each,
// more than the kernels take at small sizes. Forward and backward together,
// Python form -> native: norm + RoPE staging 152-190 -> 90 us (5120 rows, kernels
// 46 us), fp32 attention with its cache update 213 -> 103 us (320 queries),
// soft cross-entropy of 52 rows 117 -> 55 us, a 1387-row gated LoRA layer
// 176 -> 157 us, a chunk's cache bookkeeping 309 -> 270 us.
//
// Every entry returns None when the call is not of its plain form (a tensor
// that is not a dense GPU tensor, strides or types that need a copy or an error
// message, functorch transforms, forward-mode tangents, dispatch modes,
// tracing): the caller then takes the Python form, which handles or refuses it.
// Nothing has been launched or changed in that case. Apart from what the graph
// saves for a backward, nothing is kept from one call to the next.
//
// The C ABI is reached through function pointers that bind() receives, so both
// forms use the one library that the package has loaded; its errors are raised
// by the package's own Python function, with the same exception types.
#include <c10/core/impl/LocalDispatchKeySet.h>
#include <c10/core/impl/TorchDispatchModeTLS.h>
#include <c10/hip/HIPStream.h>
#include <torch/csrc/Exceptions.h>
#include <torch/csrc/jit/frontend/tracer.h>
#include <torch/extension.h>

#include "../../include/mtp_glora_amd.h"

namespace {

using at::Tensor;
using torch::autograd::AutogradContext;
using torch::autograd::Function;
using torch::autograd::variable_list;

#define MGA_API(X)                                                                                    \
  X(mga_header_hash) X(mga_kv_append) X(mga_attn_workspace_bytes) X(mga_attn_fwd_ws) X(mga_attn_bwd_ws) \
  X(mga_qk_norm_rope_stage_fwd) X(mga_qk_norm_rope_bwd) X(mga_gated_lora_workspace_bytes)             \
  X(mga_gated_lora_fwd) X(mga_gated_lora_bwd) X(mga_soft_ce_workspace_floats) X(mga_soft_ce_loss)     \
  X(mga_soft_ce_bwd)
struct Api {
#define X(f) decltype(&::f) f = nullptr;
  MGA_API(X)
#undef X
} g;

PyObject *g_raise = nullptr;   // raise(function name, code): owned for the life of the process

void bind_api(const std::map<std::string, int64_t> &addr, const py::object &raise) {
  // argument lists are compiled in: a library of another header must not be called
  const auto at = addr.find("mga_header_hash");
  if (at == addr.end() || reinterpret_cast<decltype(&::mga_header_hash)>(at->second)() != MGA_HEADER_HASH)
    throw std::runtime_error("_mga_torch.so and libmtp_glora_amd.so were built from different headers: build both "
                             "with `python __graft_entry__.py`");
#define X(f) g.f = reinterpret_cast<decltype(&::f)>(addr.at(#f));
  MGA_API(X)
#undef X
  Py_XDECREF(g_raise);
  g_raise = raise.inc_ref().ptr();
}

void check_rc(const char *fn, int rc) {
  if (rc == MGA_OK) return;
  py::gil_scoped_acquire gil;
  Py_XDECREF(PyObject_CallFunction(g_raise, "si", fn, rc));
  python_error e;
  e.persist();
  throw e;
}

// No transform, mode or trace is watching the calls.
bool eager() {
  return !c10::impl::tls_is_dispatch_key_included(c10::DispatchKey::FuncTorchDynamicLayerFrontMode) &&
         !c10::impl::TorchDispatchModeTLS::any_modes_set() && !torch::jit::tracer::isTracing();
}

bool plain(const Tensor &t) {
  static const c10::DispatchKeySet wrapped{c10::DispatchKey::Python,        c10::DispatchKey::FuncTorchBatched,
                                           c10::DispatchKey::FuncTorchGradWrapper, c10::DispatchKey::Functionalize,
                                           c10::DispatchKey::Conjugate,     c10::DispatchKey::Negative,
                                           c10::DispatchKey::ZeroTensor};
  return t.defined() && t.is_cuda() && t.layout() == at::kStrided && !t.key_set().has_any(wrapped) &&
         !t._fw_grad(0).defined();
}

int dtype_code(at::ScalarType t) {
  return t == at::kBFloat16 ? MGA_DTYPE_BF16 : t == at::kHalf ? MGA_DTYPE_F16 : t == at::kFloat ? MGA_DTYPE_F32 : -1;
}

bool same(const Tensor &a, const Tensor &b) { return a.scalar_type() == b.scalar_type() && a.device() == b.device(); }

void *stream(const Tensor &t) { return c10::hip::getCurrentHIPStream(t.device().index()).stream(); }

bool aligned16(const Tensor &t) { return reinterpret_cast<uintptr_t>(t.data_ptr()) % 16 == 0; }

// [1, H, S, D] with unit stride on D and 16-byte aligned rows
bool rows4(const Tensor &t) {
  const int64_t eb = t.element_size();
  return t.dim() == 4 && t.size(0) == 1 && t.stride(3) == 1 && t.stride(1) * eb % 16 == 0 && t.stride(2) * eb % 16 == 0 &&
         t.stride(1) >= 0 && t.stride(2) > 0 && t.stride(2) < (int64_t(1) << 23) && t.numel() > 0 && aligned16(t);
}

bool int32_on(const Tensor &t, const Tensor &like) {
  return plain(t) && t.scalar_type() == at::kInt && t.is_contiguous() && t.device() == like.device();
}

Tensor bytes(int64_t n, const Tensor &like) { return at::empty({n}, like.options().dtype(at::kByte)); }

// ---- cache rows --------------------------------------------------------------

bool kv_append(const Tensor &sk, const Tensor &sv, const Tensor &dk, const Tensor &dv, int64_t off,
               const std::optional<Tensor> &idx, std::optional<int64_t> n_rows) {
  if (!eager() || !plain(sk) || !plain(sv) || !plain(dk) || !plain(dv) || !rows4(sk) || !rows4(sv)) return false;
  if (!same(sk, sv) || !same(sk, dk) || !same(sk, dv) || sk.sizes() != sv.sizes() || sk.strides() != sv.strides())
    return false;
  if (dk.dim() != 3 || dk.sizes() != dv.sizes() || dk.strides() != dv.strides() || dk.stride(2) != 1 ||
      dk.size(0) != sk.size(1) || dk.size(2) != sk.size(3) || dtype_code(sk.scalar_type()) < 0)
    return false;
  if (idx && !int32_on(*idx, sk)) return false;
  const int64_t rows = n_rows ? *n_rows : idx ? idx->numel() : sk.size(2);
  if (rows < 0 || off < 0 || off + rows > dk.size(1) || (!idx && rows > sk.size(2))) return false;
  const at::DeviceGuard guard(sk.device());
  return g.mga_kv_append(sk.data_ptr(), sv.data_ptr(), sk.stride(1), sk.stride(2), sk.size(2),
                         idx ? idx->data_ptr<int32_t>() : nullptr, (int32_t)rows, dk.data_ptr(), dv.data_ptr(),
                         dk.stride(0), dk.stride(1), off, dk.size(1), (int32_t)dk.size(0), (int32_t)dk.size(2),
                         dtype_code(sk.scalar_type()), stream(sk)) == MGA_OK;
}

// Identity on the staged buffer view whose backward routes the rows of the
// chunk (the last ones) to the chunk's K or V and drops the detached prefix.
struct StageKV : public Function<StageKV> {
  static Tensor forward(AutogradContext *ctx, const Tensor &cur, const Tensor &full) {
    ctx->saved_data["P"] = full.size(2) - cur.size(2);
    return full.view_as(full);
  }
  static variable_list backward(AutogradContext *ctx, const variable_list &grad) {
    return {grad[0].slice(2, ctx->saved_data["P"].toInt()), Tensor()};
  }
};

bool at_row(const Tensor &t, const Tensor &buf, int64_t P) {
  return P < buf.size(1) && t.size(1) == buf.size(0) && t.stride(1) == buf.stride(0) && t.stride(2) == buf.stride(1) &&
         t.stride(3) == buf.stride(2) &&
         t.data_ptr() == static_cast<char *>(buf.data_ptr()) + P * buf.stride(1) * buf.element_size();
}

// The cache update's device side: the chunk's rows behind the prefix, unless
// they are there already (restage: the caller can write them again), and the
// views of prefix and chunk. (k, v, were there)
std::optional<std::tuple<Tensor, Tensor, bool>> update_kv(const Tensor &k, const Tensor &v, const Tensor &kb,
                                                          const Tensor &vb, int64_t P, bool restage) {
  if (!eager() || !plain(k) || !plain(v) || !plain(kb) || !plain(vb) || k.dim() != 4 || v.sizes() != k.sizes() ||
      !same(k, kb) || !same(v, vb) || kb.dim() != 3 || vb.sizes() != kb.sizes() ||
      kb.is_inference() || vb.is_inference())
    return std::nullopt;
  const bool in_place = at_row(k, kb, P);
  if (at_row(v, vb, P) != in_place || (in_place && !restage) ||
      (!in_place && !kv_append(k, v, kb, vb, P, std::nullopt, std::nullopt)))
    return std::nullopt;
  kb.unsafeGetTensorImpl()->bump_version();   // before the views: they record the version
  vb.unsafeGetTensorImpl()->bump_version();
  const int64_t L = P + k.size(2);
  Tensor kf = kb.unsqueeze(0).slice(2, 0, L), vf = vb.unsqueeze(0).slice(2, 0, L);
  if (k.requires_grad()) kf = StageKV::apply(k, kf);
  if (v.requires_grad()) vf = StageKV::apply(v, vf);
  return std::make_tuple(kf, vf, in_place);
}

// ---- attention ----------------------------------------------------------------

struct Mask {   // code, then the eight BlockMask tensors in the C ABI's order
  std::vector<Tensor> t;
  int64_t P;
  double scale;
  int64_t grad_start;
};

struct Attention : public Function<Attention> {
  // k_src, v_src receive the gradients of the rows from grad_start on
  static variable_list forward(AutogradContext *ctx, const Tensor &q, const Tensor &k_src, const Tensor &v_src,
                               const Tensor &k, const Tensor &v, const Mask &m) {
    const int64_t Hq = q.size(1), S = q.size(2), D = q.size(3), Hkv = k.size(1), L = k.size(2);
    const int dt = dtype_code(q.scalar_type());
    Tensor o = at::empty({1, S, Hq, D}, q.options().requires_grad(false));
    Tensor lse = at::empty({1, Hq, S}, q.options().requires_grad(false).dtype(at::kFloat));
    const int64_t wn = g.mga_attn_workspace_bytes((int32_t)S, (int32_t)L, (int32_t)Hq, (int32_t)Hkv, (int32_t)D, dt, 0, 0);
    Tensor ws;
    if (wn > 0) ws = bytes(wn, q);
    auto p = [&](int i) { return m.t[i].data_ptr<int32_t>(); };
    check_rc("mga_attn_fwd_ws",
             g.mga_attn_fwd_ws(q.data_ptr(), q.stride(1), q.stride(2), k.data_ptr(), k.stride(1), k.stride(2),
                               v.data_ptr(), v.stride(1), v.stride(2), o.data_ptr(), D, Hq * D, lse.data_ptr<float>(),
                               p(0), p(1), p(2), p(3), p(4), (int32_t)S, (int32_t)L, (int32_t)m.P, (int32_t)Hq,
                               (int32_t)Hkv, (int32_t)D, dt, (float)m.scale, wn > 0 ? ws.data_ptr() : nullptr, wn,
                               stream(q)));
    ctx->set_materialize_grads(false);
    ctx->save_for_backward({q, k, v, o, lse});
    ctx->saved_data["mask"] = m.t;
    ctx->saved_data["P"] = m.P;
    ctx->saved_data["scale"] = m.scale;
    ctx->saved_data["grad_start"] = m.grad_start;
    return {o, lse};
  }

  static variable_list backward(AutogradContext *ctx, const variable_list &grad) {
    TORCH_CHECK_NOT_IMPLEMENTED(!grad[1].defined(),
                                "gradient through the attention LSE is not supported (the decoder layers discard it)");
    variable_list out(6);
    if (!grad[0].defined()) return out;
    const auto saved = ctx->get_saved_variables();
    const Tensor &q = saved[0], &k = saved[1], &v = saved[2], &o = saved[3], &lse = saved[4];
    const auto mask = ctx->saved_data["mask"].toTensorVector();
    const int64_t P = ctx->saved_data["P"].toInt();
    const double scale = ctx->saved_data["scale"].toDouble();
    const int64_t Hq = q.size(1), S = q.size(2), D = q.size(3), Hkv = k.size(1), L = k.size(2);
    const int dt = dtype_code(q.scalar_type());
    const at::DeviceGuard guard(q.device());
    const bool need_kv = ctx->needs_input_grad(1) || ctx->needs_input_grad(2);
    const int64_t gs = need_kv ? ctx->saved_data["grad_start"].toInt() : L, Lg = L - gs;
    Tensor d = grad[0];
    TORCH_CHECK(d.sizes() == o.sizes(), "grad_output shape ", d.sizes(), " != output shape ", o.sizes());
    if (d.scalar_type() != q.scalar_type()) d = d.to(q.scalar_type());
    const int64_t eb = d.element_size();
    // rows that the kernels do not read where they are: one row expanded, or rows too far apart
    if (d.stride(3) != 1 || d.stride(1) * eb % 16 || d.stride(2) * eb % 16 || d.stride(1) <= 0 ||
        d.stride(1) >= (int64_t(1) << 23) || !aligned16(d))
      d = d.clone(at::MemoryFormat::Contiguous);
    const auto opt = q.options().requires_grad(false);
    Tensor dq = at::empty({1, S, Hq, D}, opt), dk, dv;
    if (Lg > 0) {
      dk = at::empty({1, Lg, Hkv, D}, opt);
      dv = at::empty({1, Lg, Hkv, D}, opt);
    }
    Tensor delta = at::empty({MGA_BWD_WS_WORDS_PER_ROW * Hq * S}, opt.dtype(at::kFloat));
    const int64_t wn = g.mga_attn_workspace_bytes((int32_t)S, (int32_t)L, (int32_t)Hq, (int32_t)Hkv, (int32_t)D, dt, 1,
                                                  (int32_t)gs);
    Tensor ws;
    if (wn > 0) ws = bytes(wn, q);
    auto p = [&](int i) { return mask[i].data_ptr<int32_t>(); };
    check_rc("mga_attn_bwd_ws",
             g.mga_attn_bwd_ws(q.data_ptr(), q.stride(1), q.stride(2), k.data_ptr(), k.stride(1), k.stride(2),
                               v.data_ptr(), v.stride(1), v.stride(2), o.data_ptr(), o.stride(2), o.stride(1),
                               d.data_ptr(), d.stride(2), d.stride(1), lse.data_ptr<float>(), delta.data_ptr<float>(),
                               dq.data_ptr(), D, Hq * D, Lg > 0 ? dk.data_ptr() : nullptr, D, Hkv * D,
                               Lg > 0 ? dv.data_ptr() : nullptr, D, Hkv * D, (int32_t)gs, p(0), p(1), p(2), p(3), p(4),
                               p(5), p(6), p(7), p(8), (int32_t)S, (int32_t)L, (int32_t)P, (int32_t)Hq, (int32_t)Hkv,
                               (int32_t)D, dt, (float)scale, MGA_BWD_DQ | (need_kv ? MGA_BWD_DKDV : 0),
                               wn > 0 ? ws.data_ptr() : nullptr, wn, stream(q)));
    if (ctx->needs_input_grad(0)) out[0] = dq.transpose(1, 2);
    if (Lg > 0 && ctx->needs_input_grad(1)) out[1] = dk.transpose(1, 2);
    if (Lg > 0 && ctx->needs_input_grad(2)) out[2] = dv.transpose(1, 2);
    return out;
  }
};

// mask: code and the eight BlockMask tensors; (o [1, S, Hq, D], lse [1, Hq, S])
std::optional<std::tuple<Tensor, Tensor>> attention(const Tensor &q, const Tensor &k_src, const Tensor &v_src,
                                                    const Tensor &k, const Tensor &v, std::vector<Tensor> mask,
                                                    int64_t P, double scale, int64_t grad_start) {
  if (!eager() || !plain(q) || !plain(k_src) || !plain(v_src) || !plain(k) || !plain(v)) return std::nullopt;
  if (!rows4(q) || !rows4(k) || !rows4(v) || !same(q, k) || !same(q, v) || k.sizes() != v.sizes()) return std::nullopt;
  const int64_t D = q.size(3), Hkv = k.size(1);
  if (dtype_code(q.scalar_type()) < 0 || (D != 64 && D != 128) || k.size(3) != D || q.size(1) % Hkv ||
      k.size(2) != P + q.size(2) || P < 0 || !(scale > 0) || !std::isfinite((float)scale) || (float)scale <= 0.f ||
      grad_start < 0 || grad_start > k.size(2))
    return std::nullopt;
  if (mask.size() != 9 || k_src.size(2) != k.size(2) - grad_start) return std::nullopt;
  for (const auto &t : mask)
    if (!int32_on(t, q)) return std::nullopt;
  const at::DeviceGuard guard(q.device());
  const auto r = Attention::apply(q, k_src, v_src, k.detach(), v.detach(), Mask{std::move(mask), P, scale, grad_start});
  return std::make_tuple(r[0], r[1]);
}

// ---- q/k norm + RoPE into the cache rows --------------------------------------

// [1, S, H, D] with unit stride on D
bool heads4(const Tensor &t) { return t.dim() == 4 && t.size(0) == 1 && t.stride(3) == 1 && t.numel() > 0; }

// cos / sin [1, S, D] or [S, D]: row stride, or -1
int64_t table_stride(const Tensor &t, int64_t S, int64_t D) {
  const int64_t n = t.dim();
  if ((n != 2 && n != 3) || (n == 3 && t.size(0) != 1) || t.size(n - 2) != S || t.size(n - 1) != D || t.stride(n - 1) != 1)
    return -1;
  return t.stride(n - 2);
}

// a tensor on t's memory that is not an autograd view of it
Tensor rows_alias(const Tensor &t) {
  return at::empty({0}, t.options().requires_grad(false)).set_(t.storage(), t.storage_offset(), t.sizes(), t.strides());
}

struct NormRopeStage : public Function<NormRopeStage> {
  static variable_list forward(AutogradContext *ctx, const Tensor &q, const Tensor &k, const Tensor &v,
                               const Tensor &qw, const Tensor &kw, const Tensor &cos, const Tensor &sin, double eps,
                               const Tensor &kd, const Tensor &vd) {
    const int64_t S = q.size(1), Hq = q.size(2), D = q.size(3), Hkv = k.size(2);
    const auto opt = q.options().requires_grad(false);
    Tensor qo = at::empty({1, S, Hq, D}, opt);
    Tensor rstd = at::empty({S, Hq + Hkv}, opt.dtype(at::kFloat));
    check_rc("mga_qk_norm_rope_stage_fwd",
             g.mga_qk_norm_rope_stage_fwd(
                 q.data_ptr(), q.stride(1), q.stride(2), k.data_ptr(), k.stride(1), k.stride(2), v.data_ptr(),
                 v.stride(1), v.stride(2), qw.data_ptr(), kw.data_ptr(), cos.data_ptr(), sin.data_ptr(),
                 table_stride(cos, S, D), (float)eps, nullptr, 0, (int32_t)S, (int32_t)Hq, (int32_t)Hkv, (int32_t)D,
                 dtype_code(q.scalar_type()), qo.data_ptr(), qo.stride(1), qo.stride(2), kd.data_ptr(), kd.stride(2),
                 kd.stride(1), vd.data_ptr(), vd.stride(2), vd.stride(1), rstd.data_ptr<float>(), stream(q)));
    ctx->save_for_backward({q, k, qw, kw, cos, sin, rstd});
    return {qo.transpose(1, 2), rows_alias(kd), rows_alias(vd)};
  }

  static variable_list backward(AutogradContext *ctx, const variable_list &grad) {
    const auto s = ctx->get_saved_variables();
    const Tensor &q = s[0], &k = s[1], &qw = s[2], &kw = s[3], &cos = s[4], &sin = s[5], &rstd = s[6];
    const int64_t S = q.size(1), Hq = q.size(2), D = q.size(3), Hkv = k.size(2);
    const at::DeviceGuard guard(q.device());
    auto heads = [&](Tensor t) {
      t = t.to(q.scalar_type()).transpose(1, 2);
      return t.stride(3) == 1 ? t : t.contiguous();
    };
    variable_list out(10);
    if (ctx->needs_input_grad(0) || ctx->needs_input_grad(1)) {
      const Tensor gq = heads(grad[0]), gk = heads(grad[1]);
      const auto opt = q.options().requires_grad(false);
      Tensor dq = at::empty({1, S, Hq, D}, opt), dk = at::empty({1, S, Hkv, D}, opt);
      check_rc("mga_qk_norm_rope_bwd",
               g.mga_qk_norm_rope_bwd(q.data_ptr(), q.stride(1), q.stride(2), k.data_ptr(), k.stride(1), k.stride(2),
                                      qw.data_ptr(), kw.data_ptr(), cos.data_ptr(), sin.data_ptr(),
                                      table_stride(cos, S, D), rstd.data_ptr<float>(), (int32_t)S, (int32_t)Hq,
                                      (int32_t)Hkv, (int32_t)D, dtype_code(q.scalar_type()), gq.data_ptr(),
                                      gq.stride(1), gq.stride(2), gk.data_ptr(), gk.stride(1), gk.stride(2),
                                      dq.data_ptr(), dq.stride(1), dq.stride(2), dk.data_ptr(), dk.stride(1),
                                      dk.stride(2), stream(q)));
      if (ctx->needs_input_grad(0)) out[0] = dq;
      if (ctx->needs_input_grad(1)) out[1] = dk;
    }
    if (ctx->needs_input_grad(2)) out[2] = grad[2].transpose(1, 2);
    return out;
  }
};

std::optional<std::tuple<Tensor, Tensor, Tensor>> norm_rope_stage(const Tensor &q, const Tensor &k, const Tensor &v,
                                                                  const Tensor &qw, const Tensor &kw,
                                                                  const Tensor &cos, const Tensor &sin, double eps,
                                                                  const Tensor &kd, const Tensor &vd) {
  if (!eager()) return std::nullopt;
  for (const Tensor *t : {&q, &k, &v, &qw, &kw, &cos, &sin, &kd, &vd})
    if (!plain(*t) || !same(*t, q)) return std::nullopt;
  if (!heads4(q) || !heads4(k) || !heads4(v) || dtype_code(q.scalar_type()) < 0) return std::nullopt;
  const int64_t S = q.size(1), D = q.size(3), Hkv = k.size(2);
  if (k.size(1) != S || k.size(3) != D || v.sizes() != k.sizes() || D > 128 || D % 2) return std::nullopt;
  for (const Tensor *w : {&qw, &kw})
    if (w->dim() != 1 || w->size(0) != D || w->stride(0) != 1) return std::nullopt;
  if (table_stride(cos, S, D) < 0 || table_stride(cos, S, D) != table_stride(sin, S, D)) return std::nullopt;
  for (const Tensor *d : {&kd, &vd})
    if (d->dim() != 4 || d->size(0) != 1 || d->size(1) != Hkv || d->size(2) != S || d->size(3) != D || d->stride(3) != 1)
      return std::nullopt;
  const at::DeviceGuard guard(q.device());
  const auto r = NormRopeStage::apply(q, k, v, qw, kw, cos, sin, eps, kd, vd);
  return std::make_tuple(r[0], r[1], r[2]);
}

// ---- gated LoRA -----------------------------------------------------------------

// a [rows, cols] view that 16-byte vectors can read
bool rows2(const Tensor &t, int64_t cols) {
  return t.dim() == 2 && t.size(1) == cols && t.size(0) > 0 && t.stride(1) == 1 && t.stride(0) >= cols &&
         t.stride(0) % 8 == 0 && aligned16(t);
}

struct GatedLora : public Function<GatedLora> {
  static Tensor forward(AutogradContext *ctx, const Tensor &x, const Tensor &w, const Tensor &a, const Tensor &b,
                        const std::optional<Tensor> &gate, double scaling, double p, int64_t seed) {
    const int64_t N = w.size(0), K = w.size(1), rank = a.size(0), rp = (rank + 31) / 32 * 32;
    const Tensor x2 = x.detach().view({-1, K});
    const int64_t S = x2.size(0);
    const int dt = dtype_code(w.scalar_type());
    const auto opt = w.options().requires_grad(false);
    Tensor y = at::empty({S, N}, opt), t = at::empty({S, rp}, opt), h;
    if (p > 0 && (K % 128 || dt != MGA_DTYPE_BF16)) h = at::empty({S, K}, opt);
    const int64_t wn = g.mga_gated_lora_workspace_bytes((int32_t)S, (int32_t)K, (int32_t)N, (int32_t)rank);
    Tensor ws = bytes(wn, w);
    check_rc("mga_gated_lora_fwd",
             g.mga_gated_lora_fwd(x2.data_ptr(), x2.stride(0), w.data_ptr(), w.stride(0), a.data_ptr(), a.stride(0),
                                  b.data_ptr(), b.stride(0), gate ? gate->data_ptr<float>() : nullptr, (float)scaling, p, (uint64_t)seed, (int32_t)S, (int32_t)K, (int32_t)N, (int32_t)rank,
                                  y.data_ptr(), y.stride(0), t.data_ptr(), t.stride(0),
                                  h.defined() ? h.data_ptr() : nullptr, h.defined() ? h.stride(0) : 0, ws.data_ptr(),
                                  wn, dt, stream(w)));
    ctx->save_for_backward({x2, h, t, w, a, b, gate ? *gate : Tensor()});
    ctx->saved_data["scaling"] = scaling;
    ctx->saved_data["p"] = p;
    ctx->saved_data["seed"] = seed;
    ctx->saved_data["shape"] = x.sizes().vec();
    auto shape = x.sizes().vec();
    shape.back() = N;
    return y.view(shape);
  }

  static variable_list backward(AutogradContext *ctx, const variable_list &grad) {
    const auto s = ctx->get_saved_variables();
    const Tensor &x = s[0], &h = s[1], &t = s[2], &w = s[3], &a = s[4], &b = s[5], &gate = s[6];
    const int64_t N = w.size(0), K = w.size(1), rank = a.size(0), S = x.size(0);
    const int dt = dtype_code(w.scalar_type());
    const at::DeviceGuard guard(w.device());
    Tensor gy = grad[0].to(w.scalar_type()).reshape({-1, N});
    if (!rows2(gy, N)) gy = gy.contiguous();
    const auto opt = w.options().requires_grad(false);
    Tensor gx, ga, gb;
    if (ctx->needs_input_grad(0)) gx = at::empty({S, K}, opt);
    if (ctx->needs_input_grad(2)) ga = at::empty({rank, K}, opt);
    if (ctx->needs_input_grad(3)) gb = at::empty({N, rank}, opt);
    const int64_t wn = g.mga_gated_lora_workspace_bytes((int32_t)S, (int32_t)K, (int32_t)N, (int32_t)rank);
    Tensor ws = bytes(wn, w);
    auto ptr = [](const Tensor &v) { return v.defined() ? v.data_ptr() : nullptr; };
    auto rs = [](const Tensor &v) { return v.defined() ? v.stride(0) : 0; };
    check_rc("mga_gated_lora_bwd",
             g.mga_gated_lora_bwd(gy.data_ptr(), gy.stride(0), x.data_ptr(), x.stride(0), ptr(h), rs(h), w.data_ptr(),
                                  w.stride(0), a.data_ptr(), a.stride(0), b.data_ptr(), b.stride(0), t.data_ptr(),
                                  t.stride(0), gate.defined() ? gate.data_ptr<float>() : nullptr,
                                  (float)ctx->saved_data["scaling"].toDouble(), ctx->saved_data["p"].toDouble(),
                                  (uint64_t)ctx->saved_data["seed"].toInt(), (int32_t)S, (int32_t)K, (int32_t)N,
                                  (int32_t)rank, ptr(gx), rs(gx), ptr(ga), rs(ga), ptr(gb), rs(gb), ws.data_ptr(), wn,
                                  dt, stream(w)));
    variable_list out(8);
    if (gx.defined()) out[0] = gx.view(ctx->saved_data["shape"].toIntVector());
    out[2] = ga;
    out[3] = gb;
    return out;
  }
};

std::optional<Tensor> gated_lora(const Tensor &x, const Tensor &w, const Tensor &a, const Tensor &b,
                                 const std::optional<Tensor> &gate_mask, double scaling, double p, int64_t seed) {
  if (!eager()) return std::nullopt;
  for (const Tensor *t : {&x, &w, &a, &b})
    if (!plain(*t) || !same(*t, w)) return std::nullopt;
  if (gate_mask && (!plain(*gate_mask) || gate_mask->device() != w.device() || gate_mask->requires_grad()))
    return std::nullopt;
  if (dtype_code(w.scalar_type()) < 0 || w.dim() != 2 || a.dim() != 2 || b.dim() != 2 || !w.is_contiguous() ||
      !a.is_contiguous() || !b.is_contiguous() || x.dim() < 1 || x.numel() == 0 || w.numel() == 0 || a.numel() == 0)
    return std::nullopt;
  const int64_t K = w.size(1), N = w.size(0);
  if (x.size(-1) != K || a.size(1) != K || b.size(0) != N || b.size(1) != a.size(0) || K % 16 || !(p >= 0 && p < 1) ||
      !aligned16(a))
    return std::nullopt;
  const int64_t S = x.numel() / K;
  if (!x.is_contiguous() && x.dim() != 2) return std::nullopt;
  if (!rows2(x.detach().view({S, K}), K)) return std::nullopt;
  const at::DeviceGuard guard(w.device());
  std::optional<Tensor> gate;
  if (gate_mask) {
    if (gate_mask->numel() != S) return std::nullopt;
    gate = gate_mask->reshape({-1}).to(at::kFloat).contiguous();
  }
  return GatedLora::apply(x, w, a, b, gate, scaling, p, seed);
}

// ---- soft cross-entropy ------------------------------------------------------------

struct SoftCE : public Function<SoftCE> {
  static Tensor forward(AutogradContext *ctx, const Tensor &x, const Tensor &t) {
    const int32_t N = (int32_t)x.size(1), V = (int32_t)x.size(2);
    const auto opt = x.options().requires_grad(false).dtype(at::kFloat);
    Tensor loss = at::empty({N}, opt), stats = at::empty({4, N}, opt), total = at::empty({}, opt);
    Tensor ws = at::empty({g.mga_soft_ce_workspace_floats(N, V)}, opt);
    check_rc("mga_soft_ce_loss",
             g.mga_soft_ce_loss(x.data_ptr(), x.stride(1), t.data_ptr(), t.stride(1), N, V,
                                dtype_code(x.scalar_type()), loss.data_ptr<float>(), stats.data_ptr<float>(),
                                total.data_ptr<float>(), ws.data_ptr<float>(), stream(x)));
    ctx->save_for_backward({x.detach(), t.detach(), stats});
    return total;
  }
  static variable_list backward(AutogradContext *ctx, const variable_list &grad) {
    const auto s = ctx->get_saved_variables();
    const Tensor &x = s[0], &t = s[1], &stats = s[2];
    const at::DeviceGuard guard(x.device());
    const Tensor go = grad[0].detach().reshape({1}).to(x.device(), at::kFloat).contiguous();
    Tensor gx = at::empty(x.sizes(), x.options());
    check_rc("mga_soft_ce_bwd",
             g.mga_soft_ce_bwd(x.data_ptr(), x.stride(1), t.data_ptr(), t.stride(1), (int32_t)x.size(1),
                               (int32_t)x.size(2), dtype_code(x.scalar_type()), go.data_ptr<float>(),
                               stats.data_ptr<float>(), gx.data_ptr(), gx.stride(1), stream(x)));
    return {gx, Tensor()};
  }
};

std::optional<Tensor> soft_ce(const Tensor &x, const Tensor &t) {
  if (!eager() || !plain(x) || !plain(t) || !same(x, t) || dtype_code(x.scalar_type()) < 0) return std::nullopt;
  if (x.dim() != 3 || x.sizes() != t.sizes() || x.size(0) != 1 || x.numel() == 0 || x.stride(2) != 1 ||
      t.stride(2) != 1 || x.stride(1) < x.size(2) || t.stride(1) < x.size(2))
    return std::nullopt;
  const at::DeviceGuard guard(x.device());
  return SoftCE::apply(x, t);
}

}  // namespace

#define MGA_DEF(f) m.def(#f, torch::wrap_pybind_function_no_gil(f))
PYBIND11_MODULE(_mga_torch, m) {
  m.def("bind", &bind_api);
  MGA_DEF(kv_append);
  MGA_DEF(update_kv);
  MGA_DEF(attention);
  MGA_DEF(norm_rope_stage);
  MGA_DEF(gated_lora);
  MGA_DEF(soft_ce);
}
