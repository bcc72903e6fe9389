// The host path of an eager call, above the C ABI (include/jvpfa.h): tensors in, tensors out.
//
// A short call is bound by the host: at B2 H12 L128 D64 the forward kernel takes 10 us, and unpacking dual tensors,
// filling the argument block through ctypes, allocating, and two autograd Functions took 48 us of Python; a step with
// its backward paid the interpreter again on autograd's device thread.  Everything between the Python signature and the
// launch is therefore here: forward and backward as library calls on freshly allocated outputs, and the autograd node
// that joins them.  Measured (eager, per call): dual forward B2 H12 L128 D64 47.8 -> 17.5 us, forward + backward
// B8 H6 L197 D64 260 -> 97 - 120 us (it depends on the cores that the two threads get; primal_of has what came off since).
#include <ATen/ATen.h>
#include <ATen/core/grad_mode.h>
#include <c10/core/DeviceGuard.h>
#include <c10/hip/HIPException.h>
#include <c10/hip/HIPStream.h>
#include <torch/csrc/autograd/custom_function.h>
#include <torch/csrc/autograd/functions/basic_ops.h>
#include <torch/csrc/autograd/variable.h>
#include <torch/extension.h>

#include <atomic>
#include <cmath>
#include <optional>
#include <string>
#include <tuple>
#include <utility>
#include <vector>

#include "../../include/jvpfa.h"

namespace {

using at::Tensor;
using OptTensor = std::optional<Tensor>;
using torch::autograd::AutogradContext;
using torch::autograd::variable_list;

// What a call is besides its tensors; the same in the forward and the backward.
struct Call {
  OptTensor mask, key_limit, tiles_q, tiles_k, bits_k, bits_q;
  int64_t mask_kind = JVPFA_MASK_NONE;
  bool causal = false;
  double scale = 1.0, dropout_p = 0.0;
  uint64_t seed = 0;
  bool split = true;
};

constexpr int64_t PADDED_HEAD_DIM = 16;  // runs on the kernels for 32 with zero columns appended

void check(int status) { TORCH_CHECK(status == JVPFA_OK, "libjvpfa: ", jvpfa_error_string(status), " (status ", status, ")"); }

void require_gpu(std::initializer_list<const Tensor *> tensors) {
  for (const Tensor *t : tensors)
    TORCH_CHECK(!t->defined() || t->is_cuda(), "jvp_flash_attention_amd runs on an AMD GPU only (HIP kernels); got a tensor on ",
                t->device(), ".  There is no CPU path.");
}

const void *in(const Tensor &t) { return t.defined() ? t.const_data_ptr() : nullptr; }
void *out(const Tensor &t) { return t.defined() ? t.mutable_data_ptr() : nullptr; }
template <typename P> const P *in(const OptTensor &t) { return t ? static_cast<const P *>(t->const_data_ptr()) : nullptr; }

Tensor given(const OptTensor &t) { return t ? *t : Tensor(); }
OptTensor maybe(const Tensor &t) { return t.defined() ? OptTensor(t) : std::nullopt; }

Tensor like(const Tensor &t) { return at::empty(t.sizes(), t.options().requires_grad(false)); }
Tensor pad(const Tensor &t) { return t.defined() ? at::constant_pad_nd(t, {0, 32 - PADDED_HEAD_DIM}, 0) : t; }
Tensor cut(const Tensor &t) { return t.defined() ? t.narrow(-1, 0, PADDED_HEAD_DIM).contiguous() : t; }
Tensor dense(const Tensor &t) { return t.defined() ? t.contiguous() : t; }

jvpfa_problem problem(const Tensor &q, const Call &c) {
  jvpfa_problem p = {};
  p.Z = static_cast<int32_t>(q.size(0));
  p.H = static_cast<int32_t>(q.size(1));
  p.L = static_cast<int32_t>(q.size(2));
  p.D = static_cast<int32_t>(q.size(3));
  p.dtype = q.scalar_type() == at::kBFloat16 ? JVPFA_BF16 : q.scalar_type() == at::kHalf ? JVPFA_FP16 : JVPFA_FP32;
  p.causal = c.causal ? 1 : 0;
  p.mask_kind = static_cast<int32_t>(c.mask_kind);
  p.sm_scale = static_cast<float>(c.scale);
  p.dropout_p = static_cast<float>(c.dropout_p);
  p.dropout_seed = c.seed;
  if (c.mask_kind != JVPFA_MASK_NONE) {
    p.mask = c.mask->const_data_ptr();
    // a size-1 axis broadcasts, whatever stride torch reports for it
    for (int i = 0; i < 4; ++i) p.mask_stride[i] = c.mask->size(i) == 1 ? 0 : c.mask->stride(i);
  }
  return p;
}

// (o, ot, M, mu); ot and mu are undefined without tangents.
std::tuple<Tensor, Tensor, Tensor, Tensor> forward(const Tensor &q, const Tensor &k, const Tensor &v, const Tensor &qt,
                                                   const Tensor &kt, const Tensor &vt, const Call &c) {
  require_gpu({&q, &k, &v, &qt, &kt, &vt});
  if (q.size(3) == PADDED_HEAD_DIM) {
    // zero columns change neither Q K^T nor the columns of P V that are kept
    auto [o, ot, M, mu] = forward(pad(q), pad(k), pad(v), pad(qt), pad(kt), pad(vt), c);
    return {cut(o), cut(ot), M, mu};
  }
  const c10::DeviceGuard guard(q.device());
  const bool dual = qt.defined();
  Tensor o = like(q), ot, mu;
  const auto stat = q.options().dtype(at::kFloat).requires_grad(false);
  Tensor M = at::empty({q.size(0), q.size(1), q.size(2)}, stat);
  if (dual) {
    ot = like(q);
    mu = at::empty({q.size(0), q.size(1), q.size(2)}, stat);
  }
  jvpfa_fwd_args a = {};
  a.struct_size = sizeof(a);
  a.p = problem(q, c);
  a.q = in(q), a.k = in(k), a.v = in(v);
  a.qt = in(qt), a.kt = in(kt), a.vt = in(vt);
  a.o = out(o), a.ot = out(ot);
  a.M = static_cast<float *>(out(M)), a.mu = static_cast<float *>(out(mu));
  a.key_limit = in<int32_t>(c.key_limit), a.tiles_q = in<int32_t>(c.tiles_q), a.mask_bits_q = in<uint32_t>(c.bits_q);
  a.Hk = static_cast<int32_t>(k.size(1)), a.Lk = static_cast<int32_t>(k.size(2));  // may differ from q's
  Tensor workspace;
  if (c.split) {
    a.split_workspace_bytes = jvpfa_fwd_split_needed(&a);
    if (a.split_workspace_bytes) {
      workspace = at::empty({static_cast<int64_t>(a.split_workspace_bytes)}, q.options().dtype(at::kByte).requires_grad(false));
      a.split_workspace = out(workspace);
    }
  }
  check(jvpfa_fwd(&a, c10::hip::getCurrentHIPStream(q.device().index()).stream()));
  return {o, ot, M, mu};
}

// dq, dk, dv and, when asked for, dq', dk', dv' (undefined otherwise).
std::vector<Tensor> backward(const Tensor &q, const Tensor &k, const Tensor &v, const Tensor &qt, const Tensor &kt,
                             const Tensor &vt, const Tensor &o, const Tensor &ot, const Tensor &M, const Tensor &mu,
                             const Tensor &go, const Tensor &gt, const Call &c, bool want_tangent_grads) {
  require_gpu({&q, &k, &v, &qt, &kt, &vt, &o, &ot, &M, &mu, &go, &gt});
  if (q.size(3) == PADDED_HEAD_DIM) {
    auto g = backward(pad(q), pad(k), pad(v), pad(qt), pad(kt), pad(vt), pad(o), pad(ot), M, mu, pad(go), pad(gt), c, want_tangent_grads);
    for (Tensor &t : g) t = cut(t);
    return g;
  }
  const c10::DeviceGuard guard(q.device());
  std::vector<Tensor> g = {like(q), like(k), like(v), Tensor(), Tensor(), Tensor()};
  if (want_tangent_grads) g[3] = like(q), g[4] = like(k), g[5] = like(v);
  jvpfa_bwd_args a = {};
  a.struct_size = sizeof(a);
  a.p = problem(q, c);
  a.q = in(q), a.k = in(k), a.v = in(v);
  a.qt = in(qt), a.kt = in(kt), a.vt = in(vt);
  a.o = in(o), a.ot = in(ot);
  a.M = static_cast<const float *>(in(M)), a.mu = static_cast<const float *>(in(mu));
  a.go = in(go), a.gt = in(gt);
  a.dq = out(g[0]), a.dk = out(g[1]), a.dv = out(g[2]);
  a.dqt = out(g[3]), a.dkt = out(g[4]), a.dvt = out(g[5]);
  const auto bytes = static_cast<int64_t>(jvpfa_bwd_workspace_bytes(a.p.Z, a.p.H, a.p.L));
  Tensor workspace = at::empty({bytes}, q.options().dtype(at::kByte).requires_grad(false));
  a.workspace = out(workspace);
  a.key_limit = in<int32_t>(c.key_limit), a.tiles_q = in<int32_t>(c.tiles_q), a.tiles_k = in<int32_t>(c.tiles_k);
  a.mask_bits = in<uint32_t>(c.bits_k), a.mask_bits_q = in<uint32_t>(c.bits_q);
  a.Hk = static_cast<int32_t>(k.size(1)), a.Lk = static_cast<int32_t>(k.size(2));
  Tensor shares;
  if (c.split) {
    a.split_workspace_bytes = jvpfa_bwd_split_needed(&a);
    if (a.split_workspace_bytes) {
      shares = at::empty({static_cast<int64_t>(a.split_workspace_bytes)}, q.options().dtype(at::kByte).requires_grad(false));
      a.split_workspace = out(shares);
    }
  }
  check(jvpfa_bwd(&a, c10::hip::getCurrentHIPStream(q.device().index()).stream()));
  return g;
}

bool any_requires_grad(std::initializer_list<const Tensor *> tensors) {
  if (!at::GradMode::is_enabled()) return false;
  for (const Tensor *t : tensors)
    if (t->defined() && t->requires_grad()) return true;
  return false;
}

// The current stream of a device, and the id of the graph capture under way on it (0: none).
std::pair<uintptr_t, uint64_t> stream_state(int64_t device) {
  const hipStream_t stream = c10::hip::getCurrentHIPStream(static_cast<c10::DeviceIndex>(device)).stream();
  hipStreamCaptureStatus status = hipStreamCaptureStatusNone;
  unsigned long long id = 0;
  if (stream) C10_HIP_CHECK(hipStreamGetCaptureInfo(stream, &status, &id));  // (the default stream cannot be captured)
  return {reinterpret_cast<uintptr_t>(stream), status == hipStreamCaptureStatusActive ? id : 0};
}

std::atomic<int64_t> masks_forgotten{0};  // calls of forget_mask, which stand for writes that no version counter shows

// What a call derived from its mask holds for another call if nothing here has changed; a mask without a version counter
// never compares equal.
struct MaskState {
  int64_t version = -1, forgotten = 0, stream = 0, capture = 0;
  bool holds_for(const MaskState &o) const {
    return version >= 0 && version == o.version && forgotten == o.forgotten && stream == o.stream && capture == o.capture;
  }
};
MaskState mask_state(const Tensor &mask, const Tensor &q) {
  const auto [stream, capture] = stream_state(q.device().index());
  return {mask.is_inference() ? -1 : static_cast<int64_t>(mask._version()), masks_forgotten.load(), static_cast<int64_t>(stream),
          static_cast<int64_t>(capture)};
}

// A backward uses what its forward derived from the mask, or looks it up again where the mask may have changed.
void renew_hints(Call &c, const MaskState &then, const Tensor &q, int64_t Lk) {
  if (c.mask_kind == JVPFA_MASK_NONE || then.holds_for(mask_state(*c.mask, q))) return;
  const py::gil_scoped_acquire gil;
  const py::object hints = py::module_::import("jvp_flash_attention_amd._lib").attr("mask_hints")(q, *c.mask, c.mask_kind, Lk, true, c.dropout_p > 0.0);
  std::tie(c.key_limit, c.tiles_q, c.tiles_k, c.bits_k, c.bits_q) = hints.cast<std::tuple<OptTensor, OptTensor, OptTensor, OptTensor, OptTensor>>();
}

// ---- autograd ------------------------------------------------------------------------------------
// (q, k, v[, q', k', v']) -> (O[, O']), differentiable in every tensor input.  A gradient that does not arrive stays
// absent: without one for O' the first-order backward runs (the tangent inputs then have zero gradients).
struct Attention : public torch::autograd::Function<Attention> {
  // (the tangents as optionals: the node takes no undefined tensors)
  static variable_list forward(AutogradContext *ctx, const Tensor &q, const Tensor &k, const Tensor &v, const OptTensor &qt_,
                               const OptTensor &kt_, const OptTensor &vt_, const Call &c) {
    const Tensor qt = given(qt_), kt = given(kt_), vt = given(vt_);
    auto [o, ot, M, mu] = ::forward(q, k, v, qt, kt, vt, c);
    ctx->set_materialize_grads(false);
    ctx->save_for_backward({q, k, v, qt, kt, vt, o, ot, M, mu});
    // (the mask is kept as it is and may be refilled: see renew_hints)
    ctx->saved_data["c"] = c10::IValue(std::make_tuple(c.mask, c.mask_kind, c.causal, c.scale, c.dropout_p, static_cast<int64_t>(c.seed), c.split));
    if (c.mask) {
      const MaskState m = mask_state(*c.mask, q);
      ctx->saved_data["hints"] = c10::IValue(std::make_tuple(c.key_limit, c.tiles_q, c.tiles_k, c.bits_k, c.bits_q, m.version, m.forgotten,
                                                             m.stream, m.capture));
    }
    if (qt.defined()) return {o, ot};
    return {o};
  }

  static variable_list backward(AutogradContext *ctx, const variable_list &grads) {
    const auto s = ctx->get_saved_variables();
    Call c;
    const auto e = ctx->saved_data["c"].toTuple()->elements();
    c.mask = e[0].toOptional<Tensor>(), c.mask_kind = e[1].toInt(), c.causal = e[2].toBool(), c.scale = e[3].toDouble();
    c.dropout_p = e[4].toDouble(), c.seed = static_cast<uint64_t>(e[5].toInt()), c.split = e[6].toBool();
    const bool dual = s[3].defined();
    const Tensor go = dense(grads[0]), gt = dual ? dense(grads[1]) : Tensor();
    const bool want_t = dual && (ctx->needs_input_grad(3) || ctx->needs_input_grad(4) || ctx->needs_input_grad(5));
    variable_list g;
    {
      const at::AutoGradMode off(false);
      if (c.mask) {
        const auto h = ctx->saved_data["hints"].toTuple()->elements();
        c.key_limit = h[0].toOptional<Tensor>(), c.tiles_q = h[1].toOptional<Tensor>(), c.tiles_k = h[2].toOptional<Tensor>();
        c.bits_k = h[3].toOptional<Tensor>(), c.bits_q = h[4].toOptional<Tensor>();
        renew_hints(c, {h[5].toInt(), h[6].toInt(), h[7].toInt(), h[8].toInt()}, s[0], s[1].size(2));
      }
      if (gt.defined()) {
        g = ::backward(s[0], s[1], s[2], s[3], s[4], s[5], s[6], s[7], s[8], s[9], go, gt, c, want_t);
      } else {
        if (go.defined()) g = ::backward(s[0], s[1], s[2], {}, {}, {}, s[6], {}, s[8], {}, go, {}, c, false);
        else g = {at::zeros_like(s[0]), at::zeros_like(s[1]), at::zeros_like(s[2]), {}, {}, {}};
        if (want_t) g[3] = at::zeros_like(s[0]), g[4] = at::zeros_like(s[1]), g[5] = at::zeros_like(s[2]);
      }
    }
    // create_graph, and an arriving gradient that depends on something: the gradients carry a node that says what is
    // missing (as behind torch's once_differentiable; gradients of constants are constants)
    if (any_requires_grad({&go, &gt})) {
      for (Tensor &t : g) {
        if (!t.defined()) continue;
        auto error = std::make_shared<torch::autograd::DelayedError>(
            "trying to differentiate twice a function that was marked with @once_differentiable", 1);
        t = (*error)({t.detach().requires_grad_()})[0];
      }
    }
    g.emplace_back();  // the call
    return g;
  }
};

// A dual tensor's primal as an input of the node: the storage and the version counter of t, none of its tangents, and the edge
// that gradients of t take.  A differentiable view (_fw_primal) puts a node of its own between the two, and joining O and O' by
// _make_dual another one behind the output; autograd's device thread then ran four nodes more in every backward.  Measured,
// bf16, forward + backward: B8 H6 L197 D64 118 -> 104 us, B1 H16 L1024 D128 causal 115 -> 106 us; forward alone B2 H12 L128 D64
// 17.3 -> 16.9 us.
Tensor primal_of(const Tensor &t) {
  const auto version = torch::autograd::impl::version_counter(t);
  const Tensor p(t.unsafeGetTensorImpl()->shallow_copy_and_detach(version, false));
  if (at::GradMode::is_enabled() && t.requires_grad()) torch::autograd::impl::set_gradient_edge(p, torch::autograd::impl::gradient_edge(t));
  return p;
}

// The argument checks of a call without a mask, as one yes or no; the caller words the error.
bool acceptable(const Tensor &q, const Tensor &k, const Tensor &v, double dropout_p) {
  if (!(dropout_p >= 0.0 && dropout_p < 1.0) || q.dim() != 4 || k.dim() != 4 || v.dim() != 4) return false;
  const int64_t d = q.size(3);
  if (d != 16 && d != 32 && d != 64 && d != 128 && d != 256) return false;
  if (k.sizes() != v.sizes() || k.size(3) != d || k.size(0) != q.size(0)) return false;
  if (k.size(1) < 1 || q.size(1) % k.size(1) != 0 || q.size(2) < 1) return false;
  const auto t = q.scalar_type();
  return (t == at::kBFloat16 || t == at::kHalf || t == at::kFloat) && k.scalar_type() == t && v.scalar_type() == t;
}

// Attention of q, k, v, which may be dual tensors of `level` (negative: no forward-mode level is open); the result is
// then one, too.  None when the arguments are not acceptable.
OptTensor attend(const Tensor &q, const Tensor &k, const Tensor &v, int64_t level, std::optional<double> scale, Call c) {
  if (!acceptable(q, k, v, c.dropout_p)) return std::nullopt;
  c.scale = scale ? *scale : 1.0 / std::sqrt(static_cast<double>(q.size(3)));
  Tensor qp = q, kp = k, vp = v, qt, kt, vt;
  if (level >= 0) {
    auto take = [level](Tensor &primal, Tensor &tangent) {
      tangent = primal._fw_grad(level);
      if (tangent.defined()) primal = primal_of(primal);
    };
    take(qp, qt), take(kp, kt), take(vp, vt);
    if (qt.defined() || kt.defined() || vt.defined()) {
      qt = qt.defined() ? dense(qt) : at::zeros(qp.sizes(), qp.options());
      kt = kt.defined() ? dense(kt) : at::zeros(kp.sizes(), kp.options());
      vt = vt.defined() ? dense(vt) : at::zeros(vp.sizes(), vp.options());
    }
  }
  qp = dense(qp), kp = dense(kp), vp = dense(vp);
  Tensor o, ot;
  if (any_requires_grad({&qp, &kp, &vp, &qt, &kt, &vt})) {
    const variable_list r = Attention::apply(qp, kp, vp, maybe(qt), maybe(kt), maybe(vt), c);
    o = r[0];
    if (qt.defined()) {
      ot = r[1];
      o._set_fw_grad(ot, level, /*is_inplace_op=*/false);  // (as the operators of torch hand out their tangents)
    }
    return o;
  }
  std::tie(o, ot, std::ignore, std::ignore) = forward(qp, kp, vp, qt, kt, vt, c);
  return ot.defined() ? at::_make_dual(o, ot, level) : o;
}

Call make_call(OptTensor mask, int64_t mask_kind, bool causal, double dropout_p, uint64_t seed, OptTensor key_limit,
               OptTensor tiles_q, OptTensor tiles_k, OptTensor bits_k, OptTensor bits_q, bool split) {
  Call c;
  if (mask_kind != JVPFA_MASK_NONE) c.mask = std::move(mask);
  c.mask_kind = mask_kind, c.causal = causal, c.dropout_p = dropout_p, c.seed = seed;
  c.key_limit = std::move(key_limit), c.tiles_q = std::move(tiles_q), c.tiles_k = std::move(tiles_k);
  c.bits_k = std::move(bits_k), c.bits_q = std::move(bits_q);
  c.split = split;
  return c;
}

}  // namespace

PYBIND11_MODULE(_torch_binding, m) {
  m.def("attend", [](const Tensor &q, const Tensor &k, const Tensor &v, int64_t level, std::optional<double> scale, bool causal,
                     double dropout_p, uint64_t seed, bool split, OptTensor mask, int64_t mask_kind, OptTensor key_limit,
                     OptTensor tiles_q, OptTensor tiles_k, OptTensor bits_k, OptTensor bits_q) {
    const py::gil_scoped_release released;
    return attend(q, k, v, level, scale, make_call(mask, mask_kind, causal, dropout_p, seed, key_limit, tiles_q, tiles_k, bits_k, bits_q, split));
  });
  m.def("stream_state", &stream_state);
  m.def("forget_masks", [] { ++masks_forgotten; });
  m.def("fwd", [](const Tensor &q, const Tensor &k, const Tensor &v, const OptTensor &qt, const OptTensor &kt, const OptTensor &vt,
                  double scale, bool causal, double dropout_p, uint64_t seed, bool split, OptTensor mask, int64_t mask_kind,
                  OptTensor key_limit, OptTensor tiles_q, OptTensor bits_q) {
    Call c = make_call(mask, mask_kind, causal, dropout_p, seed, key_limit, tiles_q, {}, {}, bits_q, split);
    c.scale = scale;
    auto [o, ot, M, mu] = forward(q, k, v, given(qt), given(kt), given(vt), c);
    return std::make_tuple(o, maybe(ot), M, maybe(mu));
  });
  m.def("bwd", [](const Tensor &q, const Tensor &k, const Tensor &v, const OptTensor &qt, const OptTensor &kt, const OptTensor &vt,
                  const Tensor &o, const OptTensor &ot, const Tensor &M, const OptTensor &mu, const OptTensor &go, const OptTensor &gt,
                  double scale, bool causal, bool want_tangent_grads, double dropout_p, uint64_t seed, bool split, OptTensor mask,
                  int64_t mask_kind, OptTensor key_limit, OptTensor tiles_q, OptTensor tiles_k, OptTensor bits_k, OptTensor bits_q) {
    Call c = make_call(mask, mask_kind, causal, dropout_p, seed, key_limit, tiles_q, tiles_k, bits_k, bits_q, split);
    c.scale = scale;
    std::vector<OptTensor> r;
    for (const Tensor &t : backward(q, k, v, given(qt), given(kt), given(vt), o, given(ot), M, given(mu), given(go), given(gt), c, want_tangent_grads))
      r.push_back(maybe(t));
    return r;
  });
}
