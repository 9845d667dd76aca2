// Eager host path of the attention in native code: what fa2.py's
// _forward_impl / _backward_impl do for operands the kernels take as they lie in
// memory -- plan, outputs and workspaces from torch's allocator, parameter
// blocks, launches on torch's current stream -- with the autograd node (the
// reference's Function, python/fa2.py:437-558) in C++.  A training step at B1
// T256 Hq4 D64 spends 50 us on the GPU; its host side through the Python custom
// ops and ctypes took 300 us.
//
// Everything else -- operands to be copied or padded, mask / score conversions,
// errors, double backward, the event log, a dS limit -- is handed back to the
// general Python path, which stays the one definition of what those do:
// attention() returns None, the node's backward calls `general_backward`.
#include <torch/extension.h>

#include <ATen/PythonTorchFunctionTLS.h>
#include <ATen/record_function.h>
#include <c10/core/DeviceGuard.h>
#include <c10/core/impl/LocalDispatchKeySet.h>
#include <c10/core/impl/TorchDispatchModeTLS.h>
#include <c10/hip/HIPStream.h>

#include <algorithm>
#include <cstdint>
#include <cstdlib>
#include <optional>

#include "fa2_4d_mask.h"

namespace {

using at::Tensor;

// Entry points of libfa2_4d_mask.so as the Python loader resolved them, and
// the Python side: general_backward(...), and the module whose settings send a
// backward there.
struct Api {
  int (*fwd_plan)(const FaFwdParams*, FaFwdPlan*);
  int (*fwd)(const FaFwdParams*);
  int (*mask_plan)(const FaMaskParams*, int64_t*);
  int (*mask_prepare)(const FaMaskParams*);
  int (*bwd_plan)(const FaBwdParams*, FaBwdPlan*);
  int (*bwd_preprocess)(const FaBwdParams*);
  int (*bwd)(const FaBwdParams*);
  int (*bwd_finalize)(const FaBwdParams*);
};
Api g_api{};
PyObject* g_general_backward = nullptr;   // callable, held for good
PyObject* g_settings = nullptr;           // module fa2: _event_log, DS_LIMIT_BYTES
int64_t g_ds_limit = 0;                   // the default limit

// A dense device tensor that is its own memory: no batched, wrapped, negated,
// all-zero or subclass tensor (batched gradients reach a backward as such), whose
// data pointer is missing or means something else.
bool plain(const Tensor& x) {
  using K = c10::DispatchKey;
  constexpr c10::DispatchKeySet wrapped({K::Python, K::Negative, K::Conjugate, K::ZeroTensor, K::Batched, K::FuncTorchBatched,
                                         K::FuncTorchGradWrapper, K::Functionalize});
  const c10::DispatchKeySet keys = x.key_set();
  return keys.has(K::CUDA) && !keys.has_any(wrapped);
}

// The logical [B, T, H, D] view of a tensor given as [B, H, T, D] (bhsd) or
// [B, T, H, D]: sizes, and strides with those of size-1 axes 0.
struct Operand {
  int64_t B, T, H, D, sb, st, sh;
  const void* p;
};
Operand operand(const Tensor& x, bool bhsd) {
  const int t = bhsd ? 2 : 1, h = bhsd ? 1 : 2;
  auto st = [&](int i) { return x.size(i) == 1 ? (int64_t)0 : x.stride(i); };
  return {x.size(0), x.size(t), x.size(h), x.size(3), st(0), st(t), st(h), x.const_data_ptr()};
}
// Columns contiguous, rows 16-byte aligned (fa2.py _kernel_operand).
bool in_place(const Tensor& x, const Operand& o) {
  return (x.size(3) == 1 || x.stride(3) == 1) && o.sb % 8 == 0 && o.st % 8 == 0 && o.sh % 8 == 0 && (uintptr_t)o.p % 16 == 0;
}
int kernel_head_dim(int64_t D) { return D <= 64 ? 64 : (D <= 128 ? 128 : 256); }

// A mask / score the kernels read as it is (fa2.py _kernel_side).
bool side_ok(const Tensor& x, at::ScalarType dtype, const Tensor& q, int64_t B, int64_t Hq, int64_t Tq, int64_t Tk) {
  return x.dim() == 4 && x.scalar_type() == dtype && x.device() == q.device() && x.size(2) == Tq && x.size(3) == Tk &&
         (x.size(0) == 1 || x.size(0) == B) && (x.size(1) == 1 || x.size(1) == Hq) && (Tk == 1 || x.stride(3) == 1);
}
int64_t side_stride(const Tensor& x, int i) { return x.size(i) == 1 ? 0 : x.stride(i); }

int dtype_code(const Tensor& q) { return q.scalar_type() == at::kBFloat16 ? FA_DTYPE_BF16 : FA_DTYPE_FP16; }

void* stream_of(const Tensor& q) { return (void*)c10::hip::getCurrentHIPStream(q.device().index()).stream(); }

// The mask of a forward's or backward's problem, to prepare.
template <typename P> FaMaskParams mask_params(const P& p) {
  FaMaskParams m{};
  m.mask = p.mask;
  m.mask_stride_b = p.mask_stride_b; m.mask_stride_h = p.mask_stride_h; m.mask_stride_q = p.mask_stride_q;
  m.batch = p.batch; m.seqlen_q = p.seqlen_q; m.seqlen_k = p.seqlen_k; m.heads_q = p.heads_q;
  m.is_causal = p.is_causal;
  m.stream = p.stream;
  return m;
}

struct Forward {
  Tensor out, lse, mask_ws, o_lo;   // out in the caller's layout; the last two undefined where not made
  Tensor mask, score;               // as given, undefined where not
};

// False: not for this path (nothing launched that matters).
bool forward(const Tensor& q, const Tensor& k, const Tensor& v, const Tensor& mask, const Tensor& score, double scale,
             bool causal, bool bhsd, bool residual, Forward* f) {
  const Operand oq = operand(q, bhsd), ok = operand(k, bhsd), ov = operand(v, bhsd);
  if (ok.B != oq.B || ov.B != oq.B || ok.T != ov.T || ok.H != ov.H || ok.D != oq.D || ov.D != oq.D || ok.H == 0 ||
      oq.H % ok.H != 0 || oq.D % 16 != 0 || oq.D > 256 || oq.D == 0 || oq.B * oq.T * oq.H * ok.T == 0)
    return false;
  if (!in_place(q, oq) || !in_place(k, ok) || !in_place(v, ov)) return false;
  if (mask.defined() && !side_ok(mask, at::kBool, q, oq.B, oq.H, oq.T, ok.T)) return false;
  if (score.defined() && !side_ok(score, at::kFloat, q, oq.B, oq.H, oq.T, ok.T)) return false;

  const c10::DeviceGuard on_device(q.device());
  FaFwdParams p{};
  p.q = oq.p; p.k = ok.p; p.v = ov.p;
  p.q_stride_b = oq.sb; p.q_stride_t = oq.st; p.q_stride_h = oq.sh;
  p.k_stride_b = ok.sb; p.k_stride_t = ok.st; p.k_stride_h = ok.sh;
  p.v_stride_b = ov.sb; p.v_stride_t = ov.st; p.v_stride_h = ov.sh;
  p.batch = (int32_t)oq.B; p.seqlen_q = (int32_t)oq.T; p.seqlen_k = (int32_t)ok.T;
  p.heads_q = (int32_t)oq.H; p.heads_k = (int32_t)ok.H;
  p.head_dim = kernel_head_dim(oq.D);
  p.head_dim_in = (int32_t)oq.D;
  p.scale = (float)scale;
  p.is_causal = causal;
  p.dtype = dtype_code(q);
  p.stream = stream_of(q);
  if (mask.defined()) {
    p.mask = (const uint8_t*)mask.const_data_ptr();
    p.mask_stride_b = side_stride(mask, 0); p.mask_stride_h = side_stride(mask, 1); p.mask_stride_q = side_stride(mask, 2);
  }
  if (score.defined()) {
    p.score = (const float*)score.const_data_ptr();
    p.score_stride_b = side_stride(score, 0); p.score_stride_h = side_stride(score, 1); p.score_stride_q = side_stride(score, 2);
  }
  FaFwdPlan plan{};
  if (residual) p.mask_ws = p.mask;   // (for the plan: it will be prepared, the backward reads it)
  if (g_api.fwd_plan(&p, &plan) != FA_OK) return false;
  p.mask_ws = nullptr;
  RECORD_FUNCTION("tilelang_fa2_4d_mask::fwd", c10::ArrayRef<const c10::IValue>());   // (the custom op's name in a profile)

  const auto bytes = q.options().dtype(at::kByte);
  const Tensor O = at::empty({oq.B, oq.T, oq.H, oq.D}, q.options());
  f->out = bhsd ? O.transpose(1, 2) : O;
  f->lse = at::empty({oq.B, oq.H, oq.T}, q.options().dtype(at::kFloat));
  const Operand oo = operand(f->out, bhsd);
  p.o = const_cast<void*>(oo.p);
  p.o_stride_b = oo.sb; p.o_stride_t = oo.st; p.o_stride_h = oo.sh;
  p.lse = f->lse.data_ptr<float>();
  if (residual && (mask.defined() || score.defined())) {
    f->o_lo = at::empty({oq.B, oq.T, oq.H, oq.D}, q.options());
    const Operand ol = operand(f->o_lo, false);
    p.o_lo = const_cast<void*>(ol.p);
    p.o_lo_stride_b = ol.sb; p.o_lo_stride_t = ol.st; p.o_lo_stride_h = ol.sh;
  }
  Tensor ws;
  if (plan.workspace_bytes) {
    ws = at::empty({plan.workspace_bytes}, bytes);
    p.workspace = ws.data_ptr();
    p.workspace_bytes = plan.workspace_bytes;
  }
  if (mask.defined() && (residual || plan.needs_mask_ws)) {
    FaMaskParams m = mask_params(p);
    int64_t n = 0;
    if (g_api.mask_plan(&m, &n) != FA_OK) return false;
    f->mask_ws = at::empty({n}, bytes);
    m.workspace = f->mask_ws.data_ptr();
    if (g_api.mask_prepare(&m) != FA_OK) return false;
    p.mask_ws = m.workspace;
  }
  return g_api.fwd(&p) == FA_OK;
}

struct Gradients {
  Tensor dq, dk, dv;   // in the caller's layout
};

bool backward(const Tensor& dout, const Tensor& q, const Tensor& k, const Tensor& v, const Tensor& out, const Tensor& lse,
              const Tensor& mask, const Tensor& score, const Tensor& mask_ws, const Tensor& o_lo, double scale, bool causal,
              bool atomic, bool bhsd, Gradients* g) {
  // saved tensors come back through hooks: as the forward saw them, or not here
  const at::ScalarType dt = q.scalar_type();
  auto as_saved = [&](const Tensor& x, at::ScalarType t) { return plain(x) && x.device() == q.device() && x.scalar_type() == t; };
  if ((dt != at::kBFloat16 && dt != at::kHalf) || !as_saved(q, dt) || !as_saved(k, dt) || !as_saved(v, dt) ||
      !as_saved(out, dt) || !as_saved(lse, at::kFloat) || (o_lo.defined() && !as_saved(o_lo, dt)) || q.dim() != 4 ||
      k.dim() != 4 || !v.sizes().equals(k.sizes()) || !out.sizes().equals(q.sizes()) || !dout.sizes().equals(q.sizes()) ||
      !lse.is_contiguous())
    return false;
  const Operand oq = operand(q, bhsd), ok = operand(k, bhsd), ov = operand(v, bhsd), oo = operand(out, bhsd);
  if (ok.B != oq.B || ok.D != oq.D || ok.H == 0 || oq.H % ok.H != 0 || lse.numel() != oq.B * oq.H * oq.T ||
      (o_lo.defined() && !o_lo.sizes().equals({oq.B, oq.T, oq.H, oq.D})))
    return false;
  Tensor d = dout.scalar_type() == dt ? dout : dout.to(dt);
  Operand od = operand(d, bhsd);
  if (!in_place(d, od)) {
    d = bhsd ? d.transpose(1, 2).contiguous().transpose(1, 2) : d.contiguous();
    od = operand(d, bhsd);
  }
  if (!in_place(q, oq) || !in_place(k, ok) || !in_place(v, ov) || !in_place(out, oo) || !in_place(d, od)) return false;
  if (mask.defined() && (!mask_ws.defined() || !as_saved(mask_ws, at::kByte) || !mask_ws.is_contiguous() || !plain(mask) ||
                         !side_ok(mask, at::kBool, q, oq.B, oq.H, oq.T, ok.T)))
    return false;
  if (score.defined() && (!plain(score) || !side_ok(score, at::kFloat, q, oq.B, oq.H, oq.T, ok.T))) return false;
  // rows the kernels reach with 32-bit byte offsets (fa2.py _rows_reachable);
  // half as far where columns are missing
  const int64_t far = (oq.T + 32) * 2 * std::max({std::abs(oq.st), std::abs(od.st), oq.D * oq.H});
  if (far >= ((int64_t)1 << (oq.D == kernel_head_dim(oq.D) ? 32 : 31))) return false;

  const c10::DeviceGuard on_device(q.device());
  FaBwdParams p{};
  p.q = oq.p; p.k = ok.p; p.v = ov.p; p.o = oo.p; p.dout = od.p;
  p.q_stride_b = oq.sb; p.q_stride_t = oq.st; p.q_stride_h = oq.sh;
  p.k_stride_b = ok.sb; p.k_stride_t = ok.st; p.k_stride_h = ok.sh;
  p.v_stride_b = ov.sb; p.v_stride_t = ov.st; p.v_stride_h = ov.sh;
  p.o_stride_b = oo.sb; p.o_stride_t = oo.st; p.o_stride_h = oo.sh;
  p.do_stride_b = od.sb; p.do_stride_t = od.st; p.do_stride_h = od.sh;
  p.batch = (int32_t)oq.B; p.seqlen_q = (int32_t)oq.T; p.seqlen_k = (int32_t)ok.T;
  p.heads_q = (int32_t)oq.H; p.heads_k = (int32_t)ok.H;
  p.head_dim = kernel_head_dim(oq.D);
  p.head_dim_in = (int32_t)oq.D;
  p.scale = (float)scale;
  p.is_causal = causal;
  p.atomic_dq = atomic;
  p.dtype = dtype_code(q);
  p.stream = stream_of(q);
  p.ds_limit_bytes = g_ds_limit;
  if (mask.defined()) {
    p.mask = (const uint8_t*)mask.const_data_ptr();
    p.mask_stride_b = side_stride(mask, 0); p.mask_stride_h = side_stride(mask, 1); p.mask_stride_q = side_stride(mask, 2);
    p.mask_ws = mask_ws.const_data_ptr();
    // (prepared for the broadcast axes of the mask as it was: a hook that copies a
    // broadcast mask gives back one with more planes than the workspace has)
    const FaMaskParams m = mask_params(p);
    int64_t n = 0;
    if (g_api.mask_plan(&m, &n) != FA_OK || n != mask_ws.numel()) return false;
  }
  if (score.defined()) {
    p.score = (const float*)score.const_data_ptr();
    p.score_stride_b = side_stride(score, 0); p.score_stride_h = side_stride(score, 1); p.score_stride_q = side_stride(score, 2);
  }
  Operand ol{};
  if (o_lo.defined()) {
    ol = operand(o_lo, false);
    if (!in_place(o_lo, ol)) return false;
    p.o_lo = ol.p;
    p.o_lo_stride_b = ol.sb; p.o_lo_stride_t = ol.st; p.o_lo_stride_h = ol.sh;
  }
  FaBwdPlan plan{};
  if (g_api.bwd_plan(&p, &plan) != FA_OK) return false;
  RECORD_FUNCTION("tilelang_fa2_4d_mask::bwd", c10::ArrayRef<const c10::IValue>());
  p.kv_split = plan.kv_split;

  const auto f32 = q.options().dtype(at::kFloat);
  const Tensor dQ = at::empty({oq.B, oq.T, oq.H, oq.D}, q.options());
  const Tensor dK = at::empty({ok.B, ok.T, ok.H, ok.D}, q.options());
  const Tensor dV = at::empty({ok.B, ok.T, ok.H, ok.D}, q.options());
  const Tensor delta = at::empty({2, oq.B, oq.H, oq.T}, f32);   // Delta, backward LSE
  const Tensor dead = at::zeros({oq.B * ok.H}, q.options().dtype(at::kInt));
  Tensor dq_acc, dk_acc, dv_acc, ds;
  if (plan.needs_dq_accum) dq_acc = at::empty({plan.dq_accum_elems}, f32);
  if (plan.dkv_accum_elems > 0) {
    dk_acc = at::empty({plan.dkv_accum_elems}, f32);
    dv_acc = at::empty({plan.dkv_accum_elems}, f32);
    p.dk_accum = dk_acc.data_ptr<float>();
    p.dv_accum = dv_acc.data_ptr<float>();
  }
  if (plan.needs_dq_accum) p.dq_accum = dq_acc.data_ptr<float>();
  if (plan.ds_elems) {
    ds = at::empty({plan.ds_elems}, q.options());
    p.ds_tiles = ds.data_ptr();
  }
  p.ds_tiles_elems = plan.ds_elems;
  p.lse = lse.const_data_ptr<float>();
  p.delta = delta.data_ptr<float>();
  p.dead_flags = dead.data_ptr<int32_t>();
  const Operand gq = operand(dQ, false), gk = operand(dK, false), gv = operand(dV, false);
  p.dq = dQ.data_ptr(); p.dk = dK.data_ptr(); p.dv = dV.data_ptr();
  p.dq_stride_b = gq.sb; p.dq_stride_t = gq.st; p.dq_stride_h = gq.sh;
  p.dk_stride_b = gk.sb; p.dk_stride_t = gk.st; p.dk_stride_h = gk.sh;
  p.dv_stride_b = gv.sb; p.dv_stride_t = gv.st; p.dv_stride_h = gv.sh;
  if (g_api.bwd_preprocess(&p) != FA_OK || g_api.bwd(&p) != FA_OK || g_api.bwd_finalize(&p) != FA_OK) return false;
  g->dq = bhsd ? dQ.transpose(1, 2) : dQ;
  g->dk = bhsd ? dK.transpose(1, 2) : dK;
  g->dv = bhsd ? dV.transpose(1, 2) : dV;
  return true;
}

// The Python path's gradients, for what the native one does not take.
Gradients general_backward(const Tensor& dout, const Tensor& q, const Tensor& k, const Tensor& v, const Tensor& out,
                           const Tensor& lse, const Tensor& mask, const Tensor& score, const Tensor& mask_ws,
                           const Tensor& o_lo, double scale, bool causal, bool atomic, bool bhsd) {
  pybind11::gil_scoped_acquire gil;
  auto opt = [](const Tensor& t) { return t.defined() ? std::optional<Tensor>(t) : std::nullopt; };
  const auto r = pybind11::handle(g_general_backward)(dout, q, k, v, out, lse, opt(mask), opt(score), opt(mask_ws),
                                                      opt(o_lo), scale, causal, atomic, bhsd)
                     .cast<std::tuple<Tensor, Tensor, Tensor>>();
  return {std::get<0>(r), std::get<1>(r), std::get<2>(r)};
}

// A backward that nothing traces, transforms or intercepts, and no setting that only
// the Python host path honours (fa2.py _plain_eager, without its Python calls: through
// them a small step took 6 us longer).
bool plain_backward(const Tensor& dout) {
  using K = c10::DispatchKey;
  const auto* meta = torch::autograd::impl::get_autograd_meta(dout);
  if (!plain(dout) || (meta && meta->fw_grad_) || at::GradMode::is_enabled() ||
      c10::impl::TorchDispatchModeTLS::any_modes_set() || at::impl::PythonTorchFunctionTLS::stack_len() > 0 ||
      c10::impl::tls_is_dispatch_key_included(K::FuncTorchDynamicLayerFrontMode) ||
      c10::impl::tls_is_dispatch_key_included(K::Tracer) || c10::impl::tls_is_dispatch_key_included(K::PythonDispatcher))
    return false;
  pybind11::gil_scoped_acquire gil;
  const pybind11::handle m(g_settings);
  const pybind11::object log = m.attr("_event_log"), limit = m.attr("DS_LIMIT_BYTES");
  return log.is_none() && limit.equal(pybind11::int_(0));
}

struct Attention : torch::autograd::Function<Attention> {
  // `done`: the forward's results, made before (so that what is not for this
  // path leaves no node behind)
  static Tensor forward(torch::autograd::AutogradContext* ctx, const Tensor& q, const Tensor& k, const Tensor& v,
                        const Forward& done, double scale, bool causal, bool atomic, bool bhsd) {
    // out itself is saved (not another view of its memory): a change of it in
    // place before the backward is then noticed
    ctx->save_for_backward({q, k, v, done.out, done.lse, done.mask, done.score, done.mask_ws, done.o_lo});
    ctx->saved_data["scale"] = scale;
    ctx->saved_data["flags"] = (int64_t)(causal | atomic << 1 | bhsd << 2);
    ctx->set_materialize_grads(false);
    return done.out;
  }
  static torch::autograd::variable_list backward(torch::autograd::AutogradContext* ctx, torch::autograd::variable_list grads) {
    torch::autograd::variable_list none(8);
    if (!grads[0].defined()) return none;   // the output does not reach the loss
    const auto s = ctx->get_saved_variables();
    const double scale = ctx->saved_data["scale"].toDouble();
    const int64_t flags = ctx->saved_data["flags"].toInt();
    const bool causal = flags & 1, atomic = flags >> 1 & 1, bhsd = flags >> 2 & 1;
    Gradients g;
    bool done = false;
    if (plain_backward(grads[0])) {
      at::AutoDispatchBelowADInplaceOrView below;
      done = ::backward(grads[0], s[0], s[1], s[2], s[3], s[4], s[5], s[6], s[7], s[8], scale, causal, atomic, bhsd, &g);
    }
    if (!done)
      g = general_backward(grads[0], s[0], s[1], s[2], s[3], s[4], s[5], s[6], s[7], s[8], scale, causal, atomic, bhsd);
    none[0] = g.dq;
    none[1] = g.dk;
    none[2] = g.dv;
    return none;
  }
};

// O in the caller's layout, or None: not for this path.
std::optional<Tensor> attention(const Tensor& q, const Tensor& k, const Tensor& v, const std::optional<Tensor>& mask_,
                                const std::optional<Tensor>& score_, double scale, bool causal, bool atomic, bool bhsd) {
  const Tensor mask = mask_.value_or(Tensor()), score = score_.value_or(Tensor());
  if (!q.is_cuda() || k.device() != q.device() || v.device() != q.device() || q.dim() != 4 || k.dim() != 4 || v.dim() != 4 ||
      (q.scalar_type() != at::kBFloat16 && q.scalar_type() != at::kHalf) || k.scalar_type() != q.scalar_type() ||
      v.scalar_type() != q.scalar_type())
    return std::nullopt;
  if (!plain(q) || !plain(k) || !plain(v) || (mask.defined() && !plain(mask)) || (score.defined() && !plain(score)))
    return std::nullopt;
  const bool grad = at::GradMode::is_enabled() && (q.requires_grad() || k.requires_grad() || v.requires_grad());
  // a score alone that wants a gradient (it gets none): the custom op's node
  if (!grad && at::GradMode::is_enabled() && score.defined() && score.requires_grad()) return std::nullopt;
  Forward f;
  {
    at::AutoDispatchBelowADInplaceOrView below;
    if (!forward(q, k, v, mask, score, scale, causal, bhsd, grad, &f)) return std::nullopt;
  }
  if (!grad) return f.out;
  f.mask = mask;
  f.score = score;
  return Attention::apply(q, k, v, f, scale, causal, atomic, bhsd);
}

void init(const std::vector<uintptr_t>& fn, pybind11::object general, pybind11::object settings, int64_t ds_limit) {
  TORCH_CHECK(fn.size() == 8, "eight entry points expected");
  g_api = Api{(decltype(Api::fwd_plan))fn[0],     (decltype(Api::fwd))fn[1],  (decltype(Api::mask_plan))fn[2],
              (decltype(Api::mask_prepare))fn[3], (decltype(Api::bwd_plan))fn[4], (decltype(Api::bwd_preprocess))fn[5],
              (decltype(Api::bwd))fn[6],          (decltype(Api::bwd_finalize))fn[7]};
  g_general_backward = general.release().ptr();
  g_settings = settings.release().ptr();
  g_ds_limit = ds_limit;
}

}  // namespace

PYBIND11_MODULE(_fa2_host, m) {
  m.def("init", &init);
  m.def("attention", &attention, pybind11::call_guard<pybind11::gil_scoped_release>());
  m.attr("ABI_VERSION") = FA_ABI_VERSION;
}
