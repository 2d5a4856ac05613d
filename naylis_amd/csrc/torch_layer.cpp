// Host side of the fused MoM layer node (model.py:189-276) in C++: a torch
// extension over the C ABI of libnaylis_mom.so.  layer_fwd / layer_bwd run
// the forward and the backward of mom_kernels.hip_layer.MomLayerFunction --
// router, bank K/V, q projection, token order, gated read, o projection with
// the folded ReZero gate, and their gradients -- as one call each from
// Python instead of about fifteen ctypes and torch calls.  They make the same
// library calls in the same order, with the same allocations and products
// (linear_fwd, linear_dgrad, library_wgrad: the library's GEMM, or hipBLASLt
// through at::mm / at::linear on torch's current stream), which the Python node
// takes from here, so their results are bitwise those of the Python node.
//
// MomLayerNode is the same node as a C++ autograd function: its forward
// calls layer_fwd and saves what the Python node saves, its backward calls
// layer_bwd, so the autograd engine runs the backward without Python.
//
// The library's symbols are not linked here: libnaylis_mom.so is loaded with
// global visibility before this module (naylis_amd/_lib.py), so these calls
// bind to that one instance (its timing state and scratch arrays included).
#include "torch_common.h"

using namespace naylis_ext;

namespace {

void* opt_ptr(const c10::optional<at::Tensor>& t) { return t.has_value() && t->defined() ? t->data_ptr() : nullptr; }

// The read's inputs and what its backward takes: bank K / V (from the caller,
// or projected from the bank's slots), queries, token order, output, the pair
// path's side buffer and the log-sum-exp.  A gradient-checkpointed layer runs
// this again in its backward (no random numbers: the same bits).
struct ReadState {
  at::Tensor slots, k, v, q, order, out, side, lse;
};

ReadState read_part(const at::Tensor& x, const c10::optional<at::Tensor>& m_blocks, const at::Tensor& w_q,
                    const at::Tensor& w_k, const at::Tensor& w_v, const c10::optional<at::Tensor>& k_ext,
                    const c10::optional<at::Tensor>& v_ext, const at::Tensor& top_idx, const at::Tensor& gates,
                    int64_t n_heads, int64_t num_blocks, int64_t block_size, int64_t top_k, void* st) {
  const int64_t B = x.size(0), T = x.size(1), D = x.size(2), H = n_heads, HD = D / n_heads;
  ReadState r;
  // ---- bank K/V (model.py:253-256), unless the caller projected the bank
  if (!k_ext.has_value()) {
    r.slots = m_blocks->reshape({-1, D}).to(at::kBFloat16).contiguous();
    const int64_t L = r.slots.size(0);
    r.k = at::empty({L, D}, x.options().dtype(at::kBFloat16));
    r.v = at::empty({L, D}, x.options().dtype(at::kBFloat16));
    check(naylis_mom_bank_kv_fwd(r.slots.data_ptr(), w_k.data_ptr(), w_v.data_ptr(), r.k.data_ptr(), r.v.data_ptr(), L, D,
                                 D, st));
  } else {
    r.k = *k_ext;
    r.v = *v_ext;
  }
  // ---- q projection, token order, gated read (model.py:251, 258-276)
  r.q = linear_fwd(x, {w_q}, at::kBFloat16, st)[0];
  const int64_t words = naylis_mom_read_order_words(B, T, num_blocks, top_k);
  if (words <= 0) check(NAYLIS_ERR_ARG);
  r.order = at::empty({words}, x.options().dtype(at::kInt));
  {
    at::Tensor ows = workspace(naylis_mom_read_order_workspace_bytes(B, T, num_blocks, top_k), x);
    check(naylis_mom_read_order(top_idx.data_ptr<int32_t>(), r.order.data_ptr<int32_t>(), ows.data_ptr(), ows.numel(),
                                B, T, num_blocks, top_k, st));
  }
  r.out = at::empty_like(r.q);
  const size_t side_bytes = naylis_mom_read_side_bytes(B, T, H, HD, num_blocks, block_size, top_k);
  if (side_bytes > 0) r.side = at::empty({(int64_t)side_bytes}, x.options().dtype(at::kByte));
  r.lse = at::empty({H, B, T}, x.options().dtype(at::kFloat));
  check(naylis_mom_read_fwd(r.q.data_ptr(), r.k.data_ptr(), r.v.data_ptr(), top_idx.data_ptr<int32_t>(),
                            gates.data_ptr<float>(), r.order.data_ptr<int32_t>(), r.out.data_ptr(),
                            ptr(r.side), r.lse.data_ptr<float>(), nullptr, 0, B, T, H, HD,
                            num_blocks, block_size, top_k, st));
  return r;
}

// layer_fwd; without `gate` y and w_os stay undefined.
std::vector<at::Tensor> forward_parts(at::Tensor x, const c10::optional<at::Tensor>& m_blocks, const at::Tensor& w_down,
                                      const at::Tensor& w_up, const at::Tensor& w_q, const at::Tensor& w_k,
                                      const at::Tensor& w_v, const at::Tensor& w_o, const at::Tensor& scale,
                                      const c10::optional<at::Tensor>& noise, double noise_scale, int64_t n_heads,
                                      int64_t num_blocks, int64_t block_size, int64_t top_k, int64_t noise_kind,
                                      const c10::optional<at::Tensor>& k_ext, const c10::optional<at::Tensor>& v_ext,
                                      bool gate, int64_t stream) {
  at::DeviceGuard guard(x.device());
  void* st = reinterpret_cast<void*>(stream);
  x = x.contiguous();
  const int64_t B = x.size(0), T = x.size(1), D = x.size(2);
  const int64_t R = w_down.size(0), E = w_up.size(0);
  const auto f32 = x.options().dtype(at::kFloat);
  // ---- router (model.py:169-220)
  at::Tensor logits = at::empty({B, T, E}, f32), probs = at::empty({B, T, E}, f32);
  at::Tensor top_idx = at::empty({B, T, top_k}, x.options().dtype(at::kInt));
  at::Tensor gates = at::empty({B, T, top_k}, f32), act = at::empty({B, T, R}, f32);
  {
    at::Tensor rws = workspace(naylis_mom_router_workspace_bytes(B, T, D, R, E, top_k), x);
    check(naylis_mom_router_fwd(x.data_ptr(), kBF16, w_down.data_ptr<float>(), w_up.data_ptr<float>(),
                                static_cast<const float*>(opt_ptr(noise)), (int)noise_kind, (float)noise_scale,
                                logits.data_ptr<float>(), probs.data_ptr<float>(), top_idx.data_ptr<int32_t>(),
                                gates.data_ptr<float>(), act.data_ptr<float>(), nullptr, rws.data_ptr(), rws.numel(),
                                B, T, D, R, E, top_k, st));
  }
  // ---- bank K/V, q projection, token order, gated read
  const ReadState rd = read_part(x, m_blocks, w_q, w_k, w_v, k_ext, v_ext, top_idx, gates, n_heads, num_blocks,
                                 block_size, top_k, st);
  // ---- o projection with the ReZero gate folded into the weight (model.py:251, 239)
  at::Tensor y, w_os;
  if (gate) {
    std::tie(y, w_os) = gated_linear_forward(rd.out.view({B * T, D}), w_o, scale, st);
    y = y.view({B, T, D});
  }
  return {y, probs, top_idx, act, gates, rd.slots, rd.k, rd.v, rd.q, rd.order, rd.out, rd.side, rd.lse, w_os};
}

// layer_bwd; without `gate` the incoming gradient is that of the read's output.
std::vector<at::Tensor> backward_parts(
    const c10::optional<at::Tensor>& dy, const c10::optional<at::Tensor>& d_probs, const at::Tensor& x,
    const c10::optional<at::Tensor>& slots, const at::Tensor& w_down, const at::Tensor& w_up, const at::Tensor& w_q,
    const at::Tensor& w_k, const at::Tensor& w_v, const at::Tensor& w_o, const at::Tensor& scale,
    const at::Tensor& act, const at::Tensor& probs, const at::Tensor& top_idx, const at::Tensor& gates,
    const at::Tensor& k, const at::Tensor& v, const at::Tensor& q, const at::Tensor& order, const at::Tensor& out,
    const c10::optional<at::Tensor>& side, const at::Tensor& lse, const at::Tensor& w_os, int64_t n_heads,
    int64_t num_blocks, int64_t block_size, int64_t top_k, bool external_bank, const std::vector<int64_t>& m_shape,
    bool m_bf16, bool gate, int64_t stream) {
  const NoAutocast no_autocast;
  at::DeviceGuard guard(x.device());
  void* st = reinterpret_cast<void*>(stream);
  const int64_t B = x.size(0), T = x.size(1), D = x.size(2);
  const int64_t R = w_down.size(0), E = w_up.size(0), H = n_heads, HD = D / n_heads, L = k.size(0), N = B * T;
  const auto f32 = x.options().dtype(at::kFloat);
  // ---- o projection with the folded gate: d out, dW_o, ds
  at::Tensor dy_t = dy.has_value() && dy->defined() ? *dy : at::zeros({B, T, D}, x.options().dtype(at::kBFloat16));
  GatedGrads go;
  if (gate)
    go = gated_linear_backward(dy_t.reshape({N, D}), out.view({N, D}), w_o, w_os, scale, st);
  else
    go.dout2 = dy_t.to(at::kBFloat16).contiguous();
  // ---- gated read
  at::Tensor dq = at::empty_like(q), dk = at::empty_like(k), dv = at::empty_like(v), dgates = at::empty_like(gates);
  {
    const size_t nbytes = naylis_mom_read_workspace_bytes(B, T, H, HD, num_blocks, block_size, top_k);
    if (nbytes == 0) check(NAYLIS_ERR_ARG);
    at::Tensor rws = workspace(nbytes, x);
    check(naylis_mom_read_bwd(q.data_ptr(), k.data_ptr(), v.data_ptr(), top_idx.data_ptr<int32_t>(),
                              gates.data_ptr<float>(), order.data_ptr<int32_t>(), out.data_ptr(), opt_ptr(side),
                              lse.data_ptr<float>(), go.dout2.data_ptr(), dq.data_ptr(), dk.data_ptr(), dv.data_ptr(),
                              dgates.data_ptr<float>(), rws.data_ptr(), rws.numel(), B, T, H, HD, num_blocks,
                              block_size, top_k, st));
  }
  go.dout2 = at::Tensor();
  // ---- bank K/V (the caller's grouped node takes dK, dV when it projected the bank)
  at::Tensor d_m, dw_k, dw_v, dk_ext, dv_ext;
  if (external_bank) {
    dk_ext = dk;
    dv_ext = dv;
  } else {
    at::Tensor d_slots = at::empty({L, D}, x.options().dtype(m_bf16 ? at::kBFloat16 : at::kFloat));
    dw_k = at::empty_like(w_k);
    dw_v = at::empty_like(w_v);
    check(naylis_mom_bank_kv_bwd(slots->data_ptr(), w_k.data_ptr(), w_v.data_ptr(), dk.data_ptr(), dv.data_ptr(),
                                 d_slots.data_ptr(), m_bf16 ? kBF16 : kF32, dw_k.data_ptr(), dw_v.data_ptr(), kBF16,
                                 L, D, D, st));
    d_m = d_slots.view(m_shape);
  }
  // ---- q projection: dx = dq W_q (the router adds its part below), dW_q = dq^T x
  at::Tensor dq2 = dq.view({N, D});
  at::Tensor dx = linear_dgrad(dq2, w_q, st).view({B, T, D});
  at::Tensor dw_q = library_wgrad(x.view({N, D}), dq2, w_q.scalar_type(), st);
  // ---- router, accumulating into dx; d_probs as one row with stride 0 when it
  // is an expanded row, else dense (the hip_router.d_probs_arg rule)
  const ProbsGrad dp = probs_grad(d_probs.has_value() ? *d_probs : at::Tensor(), E);
  at::Tensor dw_down = at::empty({R, D}, f32), dw_up = at::empty({E, R}, f32);
  {
    at::Tensor rws = workspace(naylis_mom_router_workspace_bytes(B, T, D, R, E, top_k), x);
    check(naylis_mom_router_bwd(x.data_ptr(), kBF16, w_down.data_ptr<float>(), w_up.data_ptr<float>(),
                                act.data_ptr<float>(), probs.data_ptr<float>(), top_idx.data_ptr<int32_t>(),
                                gates.data_ptr<float>(), dgates.data_ptr<float>(),
                                static_cast<const float*>(ptr(dp.t)), dp.stride, nullptr, dx.data_ptr(), 1,
                                dw_down.data_ptr<float>(), dw_up.data_ptr<float>(), rws.data_ptr(), rws.numel(), B,
                                T, D, R, E, top_k, st));
  }
  return {dx, d_m, dw_down, dw_up, dw_q, dw_k, dw_v, go.dw_o, go.ds, dk_ext, dv_ext};
}

}  // namespace

// Returns [y, probs, top_idx, act, gates, slots, k, v, q, order, out, side,
// lse, w_os]; slots is undefined (None) with an external bank, side when the
// read keeps no side buffer.
std::vector<at::Tensor> layer_fwd(at::Tensor x, c10::optional<at::Tensor> m_blocks, at::Tensor w_down,
                                  at::Tensor w_up, at::Tensor w_q, at::Tensor w_k, at::Tensor w_v, at::Tensor w_o,
                                  at::Tensor scale, c10::optional<at::Tensor> noise, double noise_scale,
                                  int64_t n_heads, int64_t num_blocks, int64_t block_size, int64_t top_k,
                                  int64_t noise_kind, c10::optional<at::Tensor> k_ext,
                                  c10::optional<at::Tensor> v_ext, int64_t stream) {
  return forward_parts(x, m_blocks, w_down, w_up, w_q, w_k, w_v, w_o, scale, noise, noise_scale, n_heads, num_blocks,
                       block_size, top_k, noise_kind, k_ext, v_ext, true, stream);
}

// Returns [dx, d_m, dw_down, dw_up, dw_q, dw_k, dw_v, dw_o, ds, dk_ext,
// dv_ext]; with an external bank d_m, dw_k, dw_v are undefined and dk_ext,
// dv_ext the bank's K / V gradients, else the reverse.
std::vector<at::Tensor> layer_bwd(c10::optional<at::Tensor> dy, c10::optional<at::Tensor> d_probs, at::Tensor x,
                                  c10::optional<at::Tensor> slots, at::Tensor w_down, at::Tensor w_up,
                                  at::Tensor w_q, at::Tensor w_k, at::Tensor w_v, at::Tensor w_o, at::Tensor scale,
                                  at::Tensor act, at::Tensor probs, at::Tensor top_idx, at::Tensor gates,
                                  at::Tensor k, at::Tensor v, at::Tensor q, at::Tensor order, at::Tensor out,
                                  c10::optional<at::Tensor> side, at::Tensor lse, at::Tensor w_os, int64_t n_heads,
                                  int64_t num_blocks, int64_t block_size, int64_t top_k, bool external_bank,
                                  std::vector<int64_t> m_shape, bool m_bf16, int64_t stream) {
  return backward_parts(dy, d_probs, x, slots, w_down, w_up, w_q, w_k, w_v, w_o, scale, act, probs, top_idx, gates, k,
                        v, q, order, out, side, lse, w_os, n_heads, num_blocks, block_size, top_k, external_bank,
                        m_shape, m_bf16, true, stream);
}

namespace {

c10::optional<at::Tensor> opt(const at::Tensor& t) {
  return t.defined() ? c10::optional<at::Tensor>(t) : c10::nullopt;
}

// Inputs as MomLayerFunction.forward takes them; the autograd function takes
// only defined tensors, so an absent noise draw is passed as x with
// has_noise false, and the bank (m_blocks) or the external K / V that the
// call does not use likewise (external tells which); no gradient flows to
// those placeholders.  Outputs y (without `gate` the read's output), probs, top_idx.
struct MomLayerNode : public torch::autograd::Function<MomLayerNode> {
  static torch::autograd::variable_list forward(torch::autograd::AutogradContext* ctx, at::Tensor x,
                                                at::Tensor m_blocks, at::Tensor w_down, at::Tensor w_up,
                                                at::Tensor w_q, at::Tensor w_k, at::Tensor w_v, at::Tensor w_o,
                                                at::Tensor scale, at::Tensor noise, bool has_noise,
                                                double noise_scale, int64_t n_heads, int64_t num_blocks,
                                                int64_t block_size, int64_t top_k, int64_t noise_kind,
                                                at::Tensor k_ext, at::Tensor v_ext, bool external, bool ckpt,
                                                bool gate, int64_t stream) {
    const at::Tensor none;
    x = x.contiguous();
    std::vector<at::Tensor> r = forward_parts(
        x, external ? c10::nullopt : opt(m_blocks), w_down, w_up, w_q, w_k, w_v, w_o, scale,
        has_noise ? opt(noise) : c10::nullopt, noise_scale, n_heads, num_blocks, block_size, top_k, noise_kind,
        external ? opt(k_ext) : c10::nullopt, external ? opt(v_ext) : c10::nullopt, gate, stream);
    // r: y, probs, top_idx, act, gates, slots, k, v, q, order, out, side, lse, w_os
    if (ckpt)  // the read's inputs only: its backward runs read_part again
      ctx->save_for_backward({x, external ? none : m_blocks, w_down, w_up, w_q, w_k, w_v, w_o, scale, r[3], r[1],
                              r[2], r[4], external ? k_ext : none, external ? v_ext : none, none, none, none, none,
                              none, r[13]});
    else
      ctx->save_for_backward({x, r[5], w_down, w_up, w_q, w_k, w_v, w_o, scale, r[3], r[1], r[2], r[4], r[6], r[7],
                              r[8], r[9], r[10], r[11], r[12], r[13]});
    ctx->saved_data["ckpt"] = ckpt;
    ctx->saved_data["gate"] = gate;
    ctx->saved_data["geom"] = std::vector<int64_t>{n_heads, num_blocks, block_size, top_k};
    ctx->saved_data["external"] = external;
    ctx->saved_data["m_shape"] = external ? std::vector<int64_t>{} : m_blocks.sizes().vec();
    ctx->saved_data["m_bf16"] = !external && m_blocks.scalar_type() == at::kBFloat16;
    ctx->mark_non_differentiable({r[2]});
    ctx->set_materialize_grads(false);
    return {gate ? r[0] : r[10], r[1], r[2]};
  }

  static torch::autograd::variable_list backward(torch::autograd::AutogradContext* ctx,
                                                 torch::autograd::variable_list grads) {
    torch::autograd::variable_list s = ctx->get_saved_variables();
    const std::vector<int64_t> geom = ctx->saved_data["geom"].toIntVector();
    const bool external = ctx->saved_data["external"].toBool();
    std::vector<int64_t> m_shape = ctx->saved_data["m_shape"].toIntVector();
    const bool m_bf16 = ctx->saved_data["m_bf16"].toBool();
    // s: x, slots, w_down, w_up, w_q, w_k, w_v, w_o, scale, act, probs, top_idx, gates, k, v, q, order,
    // out, side, lse, w_os
    if (ctx->saved_data["ckpt"].toBool()) {  // s[1] is the bank
      const NoAutocast no_autocast;
      at::DeviceGuard guard(s[0].device());
      const ReadState rd = read_part(s[0], opt(s[1]), s[4], s[5], s[6], opt(s[13]), opt(s[14]), s[11], s[12], geom[0],
                                     geom[1], geom[2], geom[3], current_stream(s[0]));
      s[1] = rd.slots;
      s[13] = rd.k;
      s[14] = rd.v;
      s[15] = rd.q;
      s[16] = rd.order;
      s[17] = rd.out;
      s[18] = rd.side;
      s[19] = rd.lse;
    }
    const bool gate = ctx->saved_data["gate"].toBool();
    std::vector<at::Tensor> r =
        backward_parts(opt(grads[0]), opt(grads[1]), s[0], opt(s[1]), s[2], s[3], s[4], s[5], s[6], s[7], s[8], s[9],
                       s[10], s[11], s[12], s[13], s[14], s[15], s[16], s[17], opt(s[18]), s[19], s[20], geom[0],
                       geom[1], geom[2], geom[3], external, m_shape, m_bf16, gate,
                       reinterpret_cast<int64_t>(current_stream(s[0])));
    // r: dx, d_m, dw_down, dw_up, dw_q, dw_k, dw_v, dw_o, ds, dk_ext, dv_ext
    const at::Tensor none;
    if (gate) r[8] = r[8].view(s[8].sizes());
    return {r[0], r[1], r[2], r[3], r[4], r[5], r[6], r[7], r[8], none, none, none,
            none, none, none, none, none, r[9], r[10], none, none, none, none};
  }
};

std::vector<at::Tensor> mom_layer_node(at::Tensor x, c10::optional<at::Tensor> m_blocks, at::Tensor w_down,
                                       at::Tensor w_up, at::Tensor w_q, at::Tensor w_k, at::Tensor w_v,
                                       at::Tensor w_o, at::Tensor scale, c10::optional<at::Tensor> noise,
                                       double noise_scale, int64_t n_heads, int64_t num_blocks, int64_t block_size,
                                       int64_t top_k, int64_t noise_kind, c10::optional<at::Tensor> k_ext,
                                       c10::optional<at::Tensor> v_ext, bool ckpt, int64_t stream) {
  const bool external = k_ext.has_value() && k_ext->defined();
  const bool has_noise = noise.has_value() && noise->defined();
  TORCH_CHECK(external || (m_blocks.has_value() && m_blocks->defined()), "mom_layer: no bank and no external K / V");
  TORCH_CHECK(!external || (v_ext.has_value() && v_ext->defined()), "mom_layer: external K without V");
  // the kernels take every size from x and the geometry
  TORCH_CHECK(x.dim() == 3 && n_heads > 0 && num_blocks > 0 && block_size > 0 && x.size(2) % n_heads == 0,
              "mom_layer: x must be (B, T, D) with D a multiple of the heads");
  const int64_t D = x.size(2), L = num_blocks * block_size;
  if (external) {
    TORCH_CHECK(k_ext->sizes() == at::IntArrayRef({L, D}) && v_ext->sizes() == k_ext->sizes(),
                "mom_layer: bank K / V must be (", L, ", ", D, "), got ", k_ext->sizes(), " / ", v_ext->sizes());
  } else {
    TORCH_CHECK(m_blocks->numel() == L * D, "mom_layer: bank of ", m_blocks->numel(), " values, the layer expects ", L,
                " slots of ", D);
  }
  for (const at::Tensor* w : {&w_q, &w_k, &w_v, &w_o})
    TORCH_CHECK(w->sizes() == at::IntArrayRef({D, D}), "mom_layer: projection weights must be (", D, ", ", D, "), got ",
                w->sizes());
  TORCH_CHECK(w_down.dim() == 2 && w_down.size(1) == D &&
                  w_up.sizes() == at::IntArrayRef({num_blocks, w_down.size(0)}),
              "mom_layer: router weights must be (R, ", D, ") and (", num_blocks, ", R), got ", w_down.sizes(), " and ",
              w_up.sizes());
  TORCH_CHECK(!has_noise || noise->numel() == x.size(0) * x.size(1) * num_blocks, "mom_layer: noise must be (B, T, ",
              num_blocks, "), got ", noise->sizes());
  // A checkpointed layer at a token count without the gated weight gradient
  // (naylis_mom_gated_wgrad) has the o projection and gate in their own node:
  // gradients of W_o and the gate taken with create_graph then keep the read's
  // output, and through it the layer, in their graph.
  const bool gate = !ckpt || x.numel() / x.size(-1) % 8 == 0;
  std::vector<at::Tensor> r =
      MomLayerNode::apply(x, external ? x : *m_blocks, w_down, w_up, w_q, w_k, w_v, w_o, scale, has_noise ? *noise : x,
                          has_noise, noise_scale, n_heads, num_blocks, block_size, top_k, noise_kind,
                          external ? *k_ext : x, external ? *v_ext : x, external, ckpt, gate, stream);
  if (!gate) r[0] = gated_linear(r[0], w_o, scale, stream);
  return r;
}

}  // namespace

PYBIND11_MODULE(TORCH_EXTENSION_NAME, m) {
  m.doc() = "Autograd nodes over the C ABI of libnaylis_mom.so";
  bind_nodes(m);
  m.def("layer_fwd", &layer_fwd, "MoM layer forward (router, bank K/V, q projection, read, o projection)");
  m.def("layer_bwd", &layer_bwd, "MoM layer backward (the forward's gradients in one fixed order)");
  m.def("mom_layer", &mom_layer_node,
        "The fused layer node as a C++ autograd function: returns (y, probs, top_idx) with its backward attached");
}
