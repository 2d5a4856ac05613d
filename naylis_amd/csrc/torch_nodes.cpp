// The library's single operations as C++ autograd functions, and the decode
// step: what the Python modules of mom_kernels/ call.  Each node allocates its
// outputs, makes its C-ABI calls on the caller's current stream (a backward on
// the one current then) and saves its tensors; the autograd engine runs the
// backward without Python.
// Argument checks and dispatch rules stay in the Python wrappers.
//
// A Python autograd function over ctypes costs 15 - 30 us of host time per
// call and direction, a node here about 6.  Host time to enqueue a pass, with
// Python functions and now (fewer launches included): one decode step 16.7 and
// 8.6 us, the checkpointed layer (3885 tokens, forward and backward, its
// recompute in the layer's node) 1222 and 295, the decoder's MLP half 596 and
// 367 and attention half 793 and 531, eight layers' evaluation 3770 and 1826.
#include <ATen/autocast_mode.h>
#include <c10/hip/HIPStream.h>

#include "torch_common.h"

namespace naylis_ext {

using torch::autograd::AutogradContext;
using torch::autograd::Function;
using torch::autograd::variable_list;

namespace {

bool plain_bf16(const at::Tensor& t) {
  return t.scalar_type() == at::kBFloat16 && t.is_contiguous() && (uintptr_t)t.data_ptr() % 16 == 0;
}

// Autocast to another type than bf16 makes torch's products cast their operands.
bool bf16_products() {
  return !at::autocast::is_autocast_enabled(at::kCUDA) ||
         at::autocast::get_autocast_dtype(at::kCUDA) == at::kBFloat16;
}

// A product of more 128 x 128 tiles than CUs and too few 256 x 128 ones for
// theirs: on the library's GEMM it runs with padded tiles and one stage ahead,
// 1.3 to 2 times hipBLASLt's time (K 1024, 1533 x 2816: 23.1 us against 14.5, as
// an input gradient 30.9 against 22.2; K 2816, 4221 x 1024: 49 / 29, 67 / 35).
bool between_tiles(int64_t rows, int64_t cols) {
  const int64_t n = (cols + 127) / 128;
  return (rows + 127) / 128 * n > 256 && (rows + 255) / 256 * n < 144;
}

// Where the library's GEMM takes a forward product (whole 128-column tiles).
// One product up to 6 M outputs: from 1000 rows on its kernel is level with
// hipBLASLt's or ahead (2042 x 1024 over 1024: 9.5 against 10.3 us, x 2816 17.9
// against 20.9), below that behind on the device and ahead where the host sets
// the pace, with a call of 6 us against 18 (64 rows, 1024 over 1024: kernels 7.2
// against 6.7 us, calls back to back 7.1 against 17.7; over 2816 13.8 against 6.9
// and 13.6 against 17.8; 1 row over 2816: 15.9 / 6.3 and 16.1 / 17.8).  Longer K
// leaves it behind everywhere (over 4096, 2042 x 1024 25.8 against 25.4, 512 rows
// 19.4 against 14.3; over 5632, 2042 x 2048 53.6 against 49.5).  Two or three of
// one input up to 768 tiles of 128 x 128, in one launch: q/k/v of 2042 tokens at
// d 1024 18.6 us against 31.4, of 64 7.4 / 19.4; gate/up 1024 -> 2816 27.6 / 41.8.
// Past that hipBLASLt's tiles win (two of 3885 x 1024 -> 2816, 1335 tiles: 50
// against 47).
bool own_fwd(int64_t n, int64_t N, int64_t D_in, int64_t D_out) {
  return N > 0 && D_in % 64 == 0 && D_out % 128 == 0 && D_in <= 2816 &&
         (n == 1 ? N * D_out <= 6 << 20 && !between_tiles(N, D_out) : n * N * D_out <= 12 << 20);
}

// ... and an input gradient: ahead of hipBLASLt's kernel from 64 rows to 6 M
// outputs (1021 x 1024 over 1024 7.6 against 9.5 us, 2042 rows 9.9 / 12.0, 2042 x
// 2048 over 2048 22.2 / 25.6, 1021 x 2816 over 1024 12.3 / 17.0).  Past it neither
// is ahead by a rule of size: over 2048 and 5632, 8192 to 16384 rows, hipBLASLt by
// 2 - 9 %, 16384 x 2816 over 1024 the library (97 against 111).
bool own_dgrad(int64_t N, int64_t D_in, int64_t D_out) {
  return N >= 64 && D_in % 128 == 0 && D_out % 64 == 0 && D_out <= 2816 && N * D_in <= 6 << 20 &&
         !between_tiles(N, D_in);
}

}  // namespace

void raise_status(int rc) {
  const char* msg = naylis_mom_last_error();
  namespace py = pybind11;
  py::gil_scoped_acquire gil;
  const py::object type = py::module_::import("naylis_amd._lib").attr("NaylisError");
  PyErr_SetObject(type.ptr(), type(rc, msg ? msg : "unknown error").ptr());
  python_error e;
  e.persist();
  throw e;
}

void* current_stream(const at::Tensor& t) { return c10::hip::getCurrentHIPStream(t.get_device()).stream(); }

std::vector<at::Tensor> linear_fwd(const at::Tensor& x, const std::vector<at::Tensor>& w, at::ScalarType dtype,
                                   void* st) {
  const int64_t D_out = w[0].size(0), D_in = w[0].size(1), N = x.numel() / std::max<int64_t>(D_in, 1), n = w.size();
  bool own = x.size(-1) == D_in && own_fwd(n, N, D_in, D_out) && x.scalar_type() == at::kBFloat16 && bf16_products();
  for (const at::Tensor& t : w) own = own && plain_bf16(t) && t.sizes() == w[0].sizes();
  std::vector<at::Tensor> y;
  const at::Tensor xc = own ? x.contiguous() : x;
  if (!own || !plain_bf16(xc)) {
    for (const at::Tensor& t : w)
      y.push_back(dtype == at::kFloat ? at::mm(x.reshape({-1, D_in}), t.t(), at::kFloat) : at::linear(x, t));
    return y;
  }
  std::vector<int64_t> shape = x.sizes().vec();
  if (dtype == at::kFloat)
    shape = {N, D_out};
  else
    shape.back() = D_out;
  const void* wp[3];
  void* yp[3];
  for (int64_t i = 0; i < n; ++i) {
    y.push_back(at::empty(shape, x.options().dtype(dtype)));
    wp[i] = w[i].data_ptr();
    yp[i] = y[i].data_ptr();
  }
  check(naylis_mom_linear_fwd(xc.data_ptr(), wp, yp, (int)n, dtype == at::kFloat ? kF32 : kBF16, N, D_in, D_out, st));
  return y;
}

at::Tensor linear_dgrad(const at::Tensor& dy, const at::Tensor& w, void* st) {
  const int64_t N = dy.size(0), D_out = w.size(0), D_in = w.size(1);
  // in grad mode (a backward with create_graph) the product itself is differentiated
  if (!own_dgrad(N, D_in, D_out) || !plain_bf16(dy) || !plain_bf16(w) || !bf16_products() || at::GradMode::is_enabled())
    return at::mm(dy, w);
  at::Tensor dx = at::empty({N, D_in}, dy.options());
  check(naylis_mom_linear_dgrad(dy.data_ptr(), w.data_ptr(), dx.data_ptr(), N, D_in, D_out, st));
  return dx;
}

at::Tensor library_wgrad(const at::Tensor& xin, const at::Tensor& dy, at::ScalarType dtype, void* st) {
  const int64_t N = xin.size(0), D_in = xin.size(1), D_out = dy.size(1);
  const auto grad = [&] { return at::empty({D_out, D_in}, xin.options().dtype(dtype)); };
  const int code = dtype == at::kBFloat16 ? kBF16 : kF32;
  if (N % 8 || D_in % 8 || D_out % 8) {
    if (N % 8 && D_in % 8 == 0 && D_out % 8 == 0 && N * std::max(D_in, D_out) < 1 << 29 && plain_bf16(xin) &&
        plain_bf16(dy) && bf16_products() && !at::GradMode::is_enabled()) {
      at::Tensor ws = workspace(naylis_mom_linear_wgrad_rows_workspace_bytes(N, D_in, D_out), xin), dw = grad();
      check(naylis_mom_linear_wgrad_rows(xin.data_ptr(), dy.data_ptr(), dw.data_ptr(), code, ws.data_ptr(), ws.numel(),
                                         N, D_in, D_out, st));
      return dw;
    }
    if (dtype == at::kFloat) return at::mm(dy.t(), xin, at::kFloat);
    return at::mm(dy.t(), xin).to(dtype);
  }
  at::Tensor ws = workspace(naylis_mom_linear_wgrad_workspace_bytes(N, D_in, D_out), xin);
  at::Tensor dw = grad();
  check(naylis_mom_linear_wgrad(xin.data_ptr(), dy.data_ptr(), dw.data_ptr(), code, ws.data_ptr(), ws.numel(), N, D_in,
                                D_out, st));
  return dw;
}

std::pair<at::Tensor, at::Tensor> gated_linear_forward(const at::Tensor& out2, const at::Tensor& w_o,
                                                       const at::Tensor& s, void* st) {
  at::Tensor w_os = at::empty_like(w_o);
  check(naylis_mom_rezero_scale(w_o.data_ptr(), dtype_code(w_o), s.data_ptr<float>(), w_os.data_ptr(),
                                dtype_code(w_os), w_o.numel(), st));
  return {linear_fwd(out2, {w_os}, at::kFloat, st)[0], w_os};
}

GatedGrads gated_linear_backward(const at::Tensor& dy, const at::Tensor& out2, const at::Tensor& w_o,
                                 const at::Tensor& w_os, const at::Tensor& s, void* st) {
  const int64_t N = out2.size(0), D_in = out2.size(1), D_out = dy.size(1);
  GatedGrads g;
  at::Tensor dy2;
  if (N % 8 == 0) {
    dy2 = dy.to(at::kBFloat16).contiguous();
    g.dout2 = linear_dgrad(dy2, w_os, st);
  } else {  // d out from bf16(s dy) and W_o, one rounding less than from bf16(dy) and bf16(s W_o)
    const at::Tensor d = dy.contiguous();
    at::Tensor dz = at::empty({N, D_out}, d.options().dtype(at::kBFloat16));
    const bool cast = d.scalar_type() != at::kBFloat16;
    dy2 = cast ? at::empty_like(dz) : d;
    check(naylis_mom_rezero_round(d.data_ptr(), dtype_code(d), s.data_ptr<float>(), cast ? dy2.data_ptr() : nullptr,
                                  dz.data_ptr(), d.numel(), st));
    g.dout2 = linear_dgrad(dz, w_o, st);
  }
  g.dw_o = at::empty_like(w_o);
  g.ds = at::empty({1}, out2.options().dtype(at::kFloat));
  if (out2.scalar_type() == at::kBFloat16 && w_o.scalar_type() == at::kBFloat16 && w_o.is_contiguous() &&
      out2.is_contiguous() && N % 8 == 0 && D_in % 8 == 0 && D_out % 8 == 0) {
    // dW' = dy^T out stays inside the split-K reduction, whose epilogue writes
    // dW_o = s dW' and the partials of ds = sum(dW' W_o)
    at::Tensor ws = workspace(naylis_mom_gated_wgrad_workspace_bytes(N, D_in, D_out), out2);
    check(naylis_mom_gated_wgrad(out2.data_ptr(), dy2.data_ptr(), w_o.data_ptr(), s.data_ptr<float>(),
                                 g.dw_o.data_ptr(), g.ds.data_ptr<float>(), ws.data_ptr(), ws.numel(), N, D_in, D_out,
                                 st));
    return g;
  }
  at::Tensor dw_s = library_wgrad(out2, dy2, at::kFloat, st);
  at::Tensor ws = workspace(naylis_mom_rezero_workspace_bytes(w_o.numel()), out2);
  check(naylis_mom_rezero_bwd(dw_s.data_ptr(), dtype_code(dw_s), w_o.data_ptr(), dtype_code(w_o), s.data_ptr<float>(),
                              g.dw_o.data_ptr(), g.ds.data_ptr<float>(), ws.data_ptr(), ws.numel(), w_o.numel(), st));
  return g;
}

ProbsGrad probs_grad(const at::Tensor& g, int64_t E) {
  if (!g.defined()) return {g, E};
  bool row = g.scalar_type() == at::kFloat && g.stride(-1) == 1;
  for (int64_t i = 0; row && i + 1 < g.dim(); ++i) row = g.stride(i) == 0;
  if (row) return {g, 0};
  return {g.to(at::kFloat).contiguous(), E};
}

namespace {

at::Tensor f32_or_none(const at::Tensor& t) { return t.defined() ? t.to(at::kFloat).contiguous() : t; }

at::TensorOptions f32_of(const at::Tensor& t) { return t.options().dtype(at::kFloat); }

// ---- RMSNorm, with and without the residual add in front --------------------

struct RmsNorm : public Function<RmsNorm> {
  static at::Tensor forward(AutogradContext* ctx, at::Tensor x, at::Tensor w, double eps, int64_t st) {
    at::DeviceGuard guard(x.device());
    const int64_t D = x.size(-1);
    const at::Tensor x2 = x.contiguous().view({-1, D});
    const int64_t N = x2.size(0);
    at::Tensor y = at::empty_like(x2), rstd = at::empty({N}, f32_of(x));
    check(naylis_mom_rmsnorm_fwd(x2.data_ptr(), dtype_code(x), w.data_ptr(), y.data_ptr(), rstd.data_ptr<float>(), N,
                                 D, (float)eps, stream_ptr(st)));
    ctx->save_for_backward({x2, w, rstd});
    ctx->saved_data["shape"] = x.sizes().vec();
    return y.view(x.sizes());
  }
  static variable_list backward(AutogradContext* ctx, variable_list grads) {
    const variable_list s = ctx->get_saved_variables();
    const at::Tensor &x2 = s[0], &w = s[1], &rstd = s[2];
    at::DeviceGuard guard(x2.device());
    const int64_t N = x2.size(0), D = x2.size(1);
    const at::Tensor dy = grads[0].to(x2.scalar_type()).contiguous();
    at::Tensor dx = at::empty_like(x2), dw = at::empty_like(w);
    at::Tensor ws = workspace(naylis_mom_rmsnorm_workspace_bytes(N, D), x2);
    check(naylis_mom_rmsnorm_bwd(x2.data_ptr(), dtype_code(x2), w.data_ptr(), rstd.data_ptr<float>(), dy.data_ptr(),
                                 dx.data_ptr(), dw.data_ptr(), ws.data_ptr(), ws.numel(), N, D,
                                 current_stream(x2)));
    return {dx.view(ctx->saved_data["shape"].toIntVector()), dw, at::Tensor(), at::Tensor()};
  }
};

struct AddRmsNorm : public Function<AddRmsNorm> {
  static variable_list forward(AutogradContext* ctx, at::Tensor x, at::Tensor a, at::Tensor w, double eps,
                               int64_t st) {
    at::DeviceGuard guard(x.device());
    const int64_t D = x.size(-1);
    const at::Tensor x2 = x.contiguous().view({-1, D}), a2 = a.contiguous().view({-1, D});
    const int64_t N = x2.size(0);
    at::Tensor s = at::empty_like(x2), y = at::empty_like(x2), rstd = at::empty({N}, f32_of(x));
    check(naylis_mom_add_rmsnorm_fwd(x2.data_ptr(), a2.data_ptr(), dtype_code(a2), w.data_ptr(), s.data_ptr(),
                                     y.data_ptr(), rstd.data_ptr<float>(), dtype_code(x2), N, D, (float)eps,
                                     stream_ptr(st)));
    ctx->save_for_backward({s, w, rstd});
    ctx->saved_data["shape"] = x.sizes().vec();
    ctx->set_materialize_grads(false);
    return {s.view(x.sizes()), y.view(x.sizes())};
  }
  static variable_list backward(AutogradContext* ctx, variable_list grads) {
    const variable_list v = ctx->get_saved_variables();
    const at::Tensor &s = v[0], &w = v[1], &rstd = v[2];
    at::DeviceGuard guard(s.device());
    const int64_t N = s.size(0), D = s.size(1);
    const at::Tensor dy = grads[1].defined() ? grads[1].to(s.scalar_type()).contiguous() : at::zeros_like(s);
    const at::Tensor dres = grads[0].defined() ? grads[0].to(s.scalar_type()).contiguous() : grads[0];
    at::Tensor ds = at::empty_like(s), dw = at::empty_like(w);
    at::Tensor ws = workspace(naylis_mom_rmsnorm_workspace_bytes(N, D), s);
    check(naylis_mom_add_rmsnorm_bwd(s.data_ptr(), w.data_ptr(), rstd.data_ptr<float>(), dy.data_ptr(), ptr(dres),
                                     ds.data_ptr(), dw.data_ptr(), ws.data_ptr(), ws.numel(), dtype_code(s), N, D,
                                     current_stream(s)));
    ds = ds.view(ctx->saved_data["shape"].toIntVector());
    return {ds, ds, dw, at::Tensor(), at::Tensor()};
  }
};

// ---- rotary embedding, causal attention, SwiGLU -----------------------------

variable_list rope_call(const at::Tensor& q_in, const at::Tensor& k_in, const at::Tensor& cs, const at::Tensor& sn,
                        bool backward, void* st) {
  at::DeviceGuard guard(q_in.device());
  const at::Tensor q = q_in.contiguous(), k = k_in.contiguous(), c = cs.contiguous(), s = sn.contiguous();
  at::Tensor qo = at::empty_like(q), ko = at::empty_like(k);
  check(naylis_mom_rope(q.data_ptr(), k.data_ptr(), c.data_ptr(), s.data_ptr(), qo.data_ptr(), ko.data_ptr(),
                        dtype_code(q), backward, q.size(0), q.size(1), q.size(2), q.size(3), c.size(0), st));
  return {qo, ko};
}

struct Rope : public Function<Rope> {
  static variable_list forward(AutogradContext* ctx, at::Tensor q, at::Tensor k, at::Tensor cs, at::Tensor sn,
                               int64_t st) {
    ctx->save_for_backward({cs, sn});
    return rope_call(q, k, cs, sn, false, stream_ptr(st));
  }
  static variable_list backward(AutogradContext* ctx, variable_list grads) {
    const variable_list s = ctx->get_saved_variables();
    const variable_list g = rope_call(grads[0], grads[1], s[0], s[1], true, current_stream(grads[0]));
    return {g[0], g[1], at::Tensor(), at::Tensor(), at::Tensor()};
  }
};

// Contiguous at an address that the kernels' 16-byte loads take.
at::Tensor aligned(const at::Tensor& t) {
  const at::Tensor c = t.contiguous();
  return (uintptr_t)c.data_ptr() % 16 == 0 ? c : c.clone();
}

variable_list attention_grads(const at::Tensor& q, const at::Tensor& k, const at::Tensor& v, const at::Tensor& out,
                              const at::Tensor& lse, const at::Tensor& grad, double scale) {
  at::DeviceGuard guard(q.device());
  const at::Tensor dout = aligned(grad.to(q.scalar_type()));
  at::Tensor dq = at::empty_like(q), dk = at::empty_like(k), dv = at::empty_like(v), delta = at::empty_like(lse);
  check(naylis_mom_attn_bwd(q.data_ptr(), k.data_ptr(), v.data_ptr(), out.data_ptr(), lse.data_ptr<float>(),
                            dout.data_ptr(), dq.data_ptr(), dk.data_ptr(), dv.data_ptr(), delta.data_ptr<float>(),
                            (float)scale, q.size(0), q.size(1), q.size(2), q.size(3), current_stream(q)));
  return {dq, dk, dv};
}

// The gradients as a node of their own, for a backward with create_graph: they
// depend on q, k, v and the incoming gradient, and a second derivative raises
// (as torch's flash attention does) instead of leaving this part out.
struct CausalAttentionGrad : public Function<CausalAttentionGrad> {
  static variable_list forward(AutogradContext*, at::Tensor q, at::Tensor k, at::Tensor v, at::Tensor out,
                               at::Tensor lse, at::Tensor dout, double scale) {
    return attention_grads(q, k, v, out, lse, dout, scale);
  }
  static variable_list backward(AutogradContext*, variable_list) {
    TORCH_CHECK(false, "causal_attention: the derivative of its backward is not implemented");
  }
};

struct CausalAttention : public Function<CausalAttention> {
  static at::Tensor forward(AutogradContext* ctx, at::Tensor q, at::Tensor k, at::Tensor v, double scale,
                            int64_t st) {
    at::DeviceGuard guard(q.device());
    const int64_t B = q.size(0), S = q.size(1), H = q.size(2), hd = q.size(3);
    q = aligned(q);
    k = aligned(k);
    v = aligned(v);
    at::Tensor out = at::empty_like(q), lse = at::empty({B, H, S}, f32_of(q));
    check(naylis_mom_attn_fwd(q.data_ptr(), k.data_ptr(), v.data_ptr(), out.data_ptr(), lse.data_ptr<float>(),
                              (float)scale, B, S, H, hd, stream_ptr(st)));
    ctx->save_for_backward({q, k, v, out, lse});
    ctx->saved_data["scale"] = scale;
    return out;
  }
  static variable_list backward(AutogradContext* ctx, variable_list grads) {
    const variable_list s = ctx->get_saved_variables();
    const double scale = ctx->saved_data["scale"].toDouble();
    variable_list g = at::GradMode::is_enabled()
                          ? CausalAttentionGrad::apply(s[0], s[1], s[2], s[3], s[4], grads[0], scale)
                          : attention_grads(s[0], s[1], s[2], s[3], s[4], grads[0], scale);
    g.resize(5);
    return g;
  }
};

struct SwiGLU : public Function<SwiGLU> {
  static at::Tensor forward(AutogradContext* ctx, at::Tensor g, at::Tensor u, int64_t st) {
    at::DeviceGuard guard(g.device());
    g = g.contiguous();
    u = u.contiguous();
    at::Tensor h = at::empty_like(g);
    check(naylis_mom_swiglu_fwd(g.data_ptr(), u.data_ptr(), h.data_ptr(), dtype_code(g), g.numel(), stream_ptr(st)));
    ctx->save_for_backward({g, u});
    return h;
  }
  static variable_list backward(AutogradContext* ctx, variable_list grads) {
    const variable_list s = ctx->get_saved_variables();
    const at::Tensor &g = s[0], &u = s[1];
    at::DeviceGuard guard(g.device());
    const at::Tensor dh = grads[0].to(g.scalar_type()).contiguous();
    at::Tensor dg = at::empty_like(g), du = at::empty_like(u);
    check(naylis_mom_swiglu_bwd(g.data_ptr(), u.data_ptr(), dh.data_ptr(), dg.data_ptr(), du.data_ptr(),
                                dtype_code(g), g.numel(), current_stream(g)));
    return {dg, du, at::Tensor()};
  }
};

// ---- bias-free projections of one input -------------------------------------

// y_i = x W_i^T for n <= 3 weights (w_i past n repeat w_0 and get no gradient);
// the input gradients accumulate in the products' epilogues.
struct SharedLinear : public Function<SharedLinear> {
  static variable_list forward(AutogradContext* ctx, at::Tensor x, at::Tensor w0, at::Tensor w1, at::Tensor w2,
                               int64_t n, int64_t st) {
    at::DeviceGuard guard(x.device());
    std::vector<at::Tensor> w = {w0, w1, w2};
    w.resize(n);
    variable_list saved = w;
    saved.push_back(x);
    ctx->save_for_backward(saved);
    return linear_fwd(x, w, x.scalar_type(), stream_ptr(st));
  }
  static variable_list backward(AutogradContext* ctx, variable_list grads) {
    const variable_list s = ctx->get_saved_variables();
    const at::Tensor& x = s.back();
    at::DeviceGuard guard(x.device());
    void* st = current_stream(x);
    const size_t n = s.size() - 1;
    const at::Tensor x2 = x.reshape({-1, x.size(-1)}).contiguous();
    variable_list r(6);
    for (size_t i = 0; i < n; ++i) {
      const at::Tensor& w = s[i];
      const at::Tensor dy = grads[i].reshape({-1, w.size(0)}).contiguous();
      if (ctx->needs_input_grad(0)) {
        if (i == 0)
          r[0] = linear_dgrad(dy, w, st);
        else
          r[0].addmm_(dy, w);
      }
      if (ctx->needs_input_grad(1 + i)) r[1 + i] = library_wgrad(x2, dy, w.scalar_type(), st);
    }
    if (r[0].defined()) r[0] = r[0].view(x.sizes());
    return r;
  }
};

// ---- the MoM layer's parts --------------------------------------------------

struct Route : public Function<Route> {
  static variable_list forward(AutogradContext* ctx, at::Tensor x, at::Tensor w_down, at::Tensor w_up,
                               at::Tensor noise, bool has_noise, double noise_scale, int64_t top_k, bool want_h,
                               int64_t noise_kind, int64_t st) {
    at::DeviceGuard guard(x.device());
    const int64_t B = x.size(0), T = x.size(1), D = x.size(2), R = w_down.size(0), E = w_up.size(0);
    const auto f32 = f32_of(x);
    at::Tensor logits = at::empty({B, T, E}, f32), probs = at::empty({B, T, E}, f32);
    at::Tensor idx = at::empty({B, T, top_k}, x.options().dtype(at::kInt)), gates = at::empty({B, T, top_k}, f32);
    at::Tensor act = at::empty({B, T, R}, f32), h;
    if (want_h) h = at::empty({B, T, D}, f32);
    at::Tensor ws = workspace(need(naylis_mom_router_workspace_bytes(B, T, D, R, E, top_k)), x);
    check(naylis_mom_router_fwd(x.data_ptr(), dtype_code(x), w_down.data_ptr<float>(), w_up.data_ptr<float>(),
                                has_noise ? noise.data_ptr<float>() : nullptr, (int)noise_kind, (float)noise_scale,
                                logits.data_ptr<float>(), probs.data_ptr<float>(), idx.data_ptr<int32_t>(),
                                gates.data_ptr<float>(), act.data_ptr<float>(),
                                want_h ? h.data_ptr<float>() : nullptr, ws.data_ptr(), ws.numel(), B, T, D, R, E,
                                top_k, stream_ptr(st)));
    ctx->save_for_backward({x, w_down, w_up, act, probs, idx, gates});
    ctx->set_materialize_grads(false);
    if (want_h) {
      ctx->mark_non_differentiable({idx, h});
      return {logits, probs, idx, gates, h};
    }
    ctx->mark_non_differentiable({idx});
    return {logits, probs, idx, gates};
  }
  static variable_list backward(AutogradContext* ctx, variable_list grads) {
    const variable_list s = ctx->get_saved_variables();
    const at::Tensor &x = s[0], &w_down = s[1], &w_up = s[2], &act = s[3], &probs = s[4], &idx = s[5], &gates = s[6];
    at::DeviceGuard guard(x.device());
    const int64_t B = x.size(0), T = x.size(1), D = x.size(2), R = w_down.size(0), E = w_up.size(0),
                  k = idx.size(2);
    const at::Tensor d_logits = f32_or_none(grads[0]), d_gates = f32_or_none(grads[3]);
    const ProbsGrad dp = probs_grad(grads[1], E);
    at::Tensor dx = at::empty_like(x), dw_down = at::empty({R, D}, f32_of(x)), dw_up = at::empty({E, R}, f32_of(x));
    at::Tensor ws = workspace(naylis_mom_router_workspace_bytes(B, T, D, R, E, k), x);
    check(naylis_mom_router_bwd(x.data_ptr(), dtype_code(x), w_down.data_ptr<float>(), w_up.data_ptr<float>(),
                                act.data_ptr<float>(), probs.data_ptr<float>(), idx.data_ptr<int32_t>(),
                                gates.data_ptr<float>(), static_cast<const float*>(ptr(d_gates)),
                                static_cast<const float*>(ptr(dp.t)), dp.stride,
                                static_cast<const float*>(ptr(d_logits)), dx.data_ptr(), 0, dw_down.data_ptr<float>(),
                                dw_up.data_ptr<float>(), ws.data_ptr(), ws.numel(), B, T, D, R, E, k,
                                current_stream(x)));
    variable_list r(10);
    r[0] = dx;
    r[1] = dw_down;
    r[2] = dw_up;
    return r;
  }
};

struct RouterStats : public Function<RouterStats> {
  static at::Tensor forward(AutogradContext* ctx, at::Tensor probs, at::Tensor idx, int64_t st) {
    at::DeviceGuard guard(probs.device());
    const int64_t E = probs.size(-1), N = probs.numel() / std::max<int64_t>(E, 1);
    at::Tensor stats = at::empty({2 * E + 3}, probs.options());
    at::Tensor ws = workspace(need(naylis_mom_router_stats_workspace_bytes(N, E)), probs);
    check(naylis_mom_router_stats(probs.data_ptr<float>(), idx.data_ptr<int32_t>(), stats.data_ptr<float>(),
                                  ws.data_ptr(), ws.numel(), N, E, idx.size(-1), stream_ptr(st)));
    ctx->save_for_backward({stats});
    ctx->saved_data["shape"] = probs.sizes().vec();
    return stats;
  }
  static variable_list backward(AutogradContext* ctx, variable_list grads) {
    const at::Tensor stats = ctx->get_saved_variables()[0];
    const std::vector<int64_t> shape = ctx->saved_data["shape"].toIntVector();
    const int64_t E = shape.back();
    int64_t N = 1;
    for (size_t i = 0; i + 1 < shape.size(); ++i) N *= shape[i];
    // d mean_prob_e = d_stats[e] + d_aux E frac_e; every token gets 1 / N of it
    const at::Tensor& d = grads[0];
    const at::Tensor row = (d.narrow(0, 0, E) + d.select(0, 2 * E) * E * stats.narrow(0, E, E)) / N;
    return {row.expand(shape), at::Tensor(), at::Tensor()};
  }
};

struct Read : public Function<Read> {
  static at::Tensor forward(AutogradContext* ctx, at::Tensor q, at::Tensor k, at::Tensor v, at::Tensor idx,
                            at::Tensor gates, int64_t num_blocks, int64_t block_size, int64_t st) {
    at::DeviceGuard guard(q.device());
    const int64_t B = q.size(0), S = q.size(1), H = q.size(2), HD = q.size(3), top_k = idx.size(-1);
    at::Tensor out = at::empty_like(q), side;
    const size_t side_bytes = naylis_mom_read_side_bytes(B, S, H, HD, num_blocks, block_size, top_k);
    if (side_bytes > 0) side = workspace(side_bytes, q);
    at::Tensor lse = at::empty({H, B, S}, f32_of(q));
    const int64_t words = naylis_mom_read_order_words(B, S, num_blocks, top_k);
    if (words <= 0) check(NAYLIS_ERR_ARG);
    at::Tensor order = at::empty({words}, idx.options());
    at::Tensor ows = workspace(naylis_mom_read_order_workspace_bytes(B, S, num_blocks, top_k), q);
    check(naylis_mom_read_order(idx.data_ptr<int32_t>(), order.data_ptr<int32_t>(), ows.data_ptr(), ows.numel(), B, S,
                                num_blocks, top_k, stream_ptr(st)));
    check(naylis_mom_read_fwd(q.data_ptr(), k.data_ptr(), v.data_ptr(), idx.data_ptr<int32_t>(),
                              gates.data_ptr<float>(), order.data_ptr<int32_t>(), out.data_ptr(), ptr(side),
                              lse.data_ptr<float>(), nullptr, 0, B, S, H, HD, num_blocks, block_size, top_k,
                              stream_ptr(st)));
    ctx->save_for_backward({q, k, v, idx, gates, order, out, side, lse});
    ctx->saved_data["geom"] = std::vector<int64_t>{num_blocks, block_size};
    return out;
  }
  static variable_list backward(AutogradContext* ctx, variable_list grads) {
    const variable_list s = ctx->get_saved_variables();
    const at::Tensor &q = s[0], &k = s[1], &v = s[2], &idx = s[3], &gates = s[4], &order = s[5], &out = s[6],
                     &side = s[7], &lse = s[8];
    const std::vector<int64_t> geom = ctx->saved_data["geom"].toIntVector();
    at::DeviceGuard guard(q.device());
    const int64_t B = q.size(0), S = q.size(1), H = q.size(2), HD = q.size(3), top_k = idx.size(-1);
    const at::Tensor dout = grads[0].contiguous().to(q.scalar_type());
    at::Tensor dq = at::empty_like(q), dk = at::empty_like(k), dv = at::empty_like(v), dg = at::empty_like(gates);
    at::Tensor ws = workspace(need(naylis_mom_read_workspace_bytes(B, S, H, HD, geom[0], geom[1], top_k)), q);
    check(naylis_mom_read_bwd(q.data_ptr(), k.data_ptr(), v.data_ptr(), idx.data_ptr<int32_t>(),
                              gates.data_ptr<float>(), order.data_ptr<int32_t>(), out.data_ptr(), ptr(side),
                              lse.data_ptr<float>(), dout.data_ptr(), dq.data_ptr(), dk.data_ptr(), dv.data_ptr(),
                              dg.data_ptr<float>(), ws.data_ptr(), ws.numel(), B, S, H, HD, geom[0], geom[1], top_k,
                              current_stream(q)));
    return {dq, dk, dv, at::Tensor(), dg, at::Tensor(), at::Tensor(), at::Tensor()};
  }
};

struct GatedLinear : public Function<GatedLinear> {
  static at::Tensor forward(AutogradContext* ctx, at::Tensor out, at::Tensor w_o, at::Tensor s, int64_t st) {
    at::DeviceGuard guard(out.device());
    const auto [y2, w_os] = gated_linear_forward(out.reshape({-1, w_o.size(1)}), w_o, s, stream_ptr(st));
    ctx->save_for_backward({out, w_o, w_os, s});
    std::vector<int64_t> shape = out.sizes().vec();
    shape.back() = w_o.size(0);
    return y2.view(shape);
  }
  static variable_list backward(AutogradContext* ctx, variable_list grads) {
    const variable_list v = ctx->get_saved_variables();
    const at::Tensor &out = v[0], &w_o = v[1], &w_os = v[2], &s = v[3];
    const NoAutocast no_autocast;
    at::DeviceGuard guard(out.device());
    if (at::GradMode::is_enabled()) {  // create_graph: s * (out W_o^T) in products that autograd knows
      const at::Tensor dy = grads[0].reshape({-1, w_o.size(0)}), o = out.reshape({-1, w_o.size(1)});
      const at::Tensor dz = (dy * s).to(o.scalar_type());
      return {at::mm(dz, w_o).view(out.sizes()), at::mm(dz.t(), o), (dy * at::mm(o, w_o.t())).sum().view(s.sizes()),
              at::Tensor()};
    }
    const GatedGrads g = gated_linear_backward(grads[0].reshape({-1, w_o.size(0)}), out.reshape({-1, w_o.size(1)}),
                                               w_o, w_os, s, current_stream(out));
    return {g.dout2.view(out.sizes()), g.dw_o, g.ds.view(s.sizes()), at::Tensor()};
  }
};

}  // namespace

at::Tensor gated_linear(const at::Tensor& out, const at::Tensor& w_o, const at::Tensor& s, int64_t st) {
  return GatedLinear::apply(out, w_o, s, st);
}

namespace {

// ---- LM loss ----------------------------------------------------------------

struct Xent : public Function<Xent> {
  static at::Tensor forward(AutogradContext* ctx, at::Tensor logits, at::Tensor labels, int64_t ignore_index,
                            int64_t st) {
    at::DeviceGuard guard(logits.device());
    logits = logits.contiguous();
    labels = labels.to(at::kLong).contiguous();
    const int64_t N = logits.size(0), V = logits.size(1);
    at::Tensor loss = at::empty({N}, f32_of(logits)), lse = at::empty({N}, f32_of(logits));
    check(naylis_mom_xent_fwd(logits.data_ptr(), labels.data_ptr<int64_t>(), loss.data_ptr<float>(),
                              lse.data_ptr<float>(), N, V, ignore_index, stream_ptr(st)));
    ctx->save_for_backward({logits, labels, lse});
    ctx->saved_data["ignore_index"] = ignore_index;
    return loss;
  }
  static variable_list backward(AutogradContext* ctx, variable_list grads) {
    const variable_list s = ctx->get_saved_variables();
    const at::Tensor &logits = s[0], &labels = s[1], &lse = s[2];
    const int64_t ignore_index = ctx->saved_data["ignore_index"].toInt();
    at::DeviceGuard guard(logits.device());
    const int64_t N = logits.size(0), V = logits.size(1);
    at::Tensor g = grads[0].to(at::kFloat);
    const bool one = g.dim() == 1 && g.stride(0) == 0;  // one gradient for every row (the sum's backward)
    if (!one) g = g.contiguous();
    at::Tensor dlogits = at::empty_like(logits);
    check(naylis_mom_xent_bwd(logits.data_ptr(), labels.data_ptr<int64_t>(), lse.data_ptr<float>(),
                              g.data_ptr<float>(), one ? 0 : 1, dlogits.data_ptr(), N, V, ignore_index,
                              current_stream(logits)));
    return {dlogits, at::Tensor(), at::Tensor(), at::Tensor()};
  }
};

// ---- decode -----------------------------------------------------------------

void require(bool ok, const char* what) {
  if (!ok) throw std::runtime_error(what);
}

std::vector<at::Tensor> decode_step(at::Tensor sum_state, at::Tensor t_prev, at::Tensor x_new, at::Tensor w_down,
                                    at::Tensor w_up, int64_t top_k, at::Tensor q_new, const at::Tensor& k8,
                                    const at::Tensor& v8, const at::Tensor& k_scale, const at::Tensor& v_scale,
                                    int64_t num_blocks, int64_t block_size, c10::optional<at::Tensor> out_state,
                                    int64_t st) {
  require(x_new.dim() == 2 && q_new.dim() == 3, "decode_step: x_new must be (B, D) and q_new (B, H, head_dim)");
  const int64_t B = x_new.size(0), D = x_new.size(1), H = q_new.size(1), R = w_down.size(0), E = w_up.size(0);
  if (E != num_blocks)
    throw std::runtime_error("decode_step: the router has " + std::to_string(E) + " experts but the bank " +
                             std::to_string(num_blocks) + " blocks");
  require(q_new.size(0) == B && H > 0 && q_new.size(2) == D / H && q_new.scalar_type() == at::kBFloat16,
          "decode_step: q_new must be (B, H, D / H) bf16");
  require(x_new.scalar_type() == at::kBFloat16 || x_new.scalar_type() == at::kFloat,
          "decode_step: x_new must be bf16 or fp32");
  require(k8.dim() == 2 && k8.size(0) == num_blocks * block_size && k8.size(1) == D,
          "decode_step: the bank's shape does not match num_blocks * block_size x D");
  sum_state = sum_state.to(at::kDouble).contiguous();
  t_prev = t_prev.to(x_new.device(), at::kInt).contiguous();
  at::Tensor state;
  if (out_state.has_value()) {
    state = *out_state;
    require(state.data_ptr() != sum_state.data_ptr() && state.scalar_type() == at::kDouble,
            "decode_step: out_state must be a separate fp64 buffer");
  } else {
    state = at::empty_like(sum_state);
  }
  x_new = x_new.contiguous();
  q_new = q_new.contiguous();
  w_down = w_down.to(at::kFloat).contiguous();
  w_up = w_up.to(at::kFloat).contiguous();
  at::DeviceGuard guard(x_new.device());
  at::Tensor out = at::empty({B, H, D / H}, x_new.options().dtype(at::kBFloat16));
  at::Tensor idx = at::empty({B, top_k}, x_new.options().dtype(at::kInt));
  at::Tensor gates = at::empty({B, top_k}, f32_of(x_new));
  check(naylis_mom_decode_step(sum_state.data_ptr<double>(), state.data_ptr<double>(), t_prev.data_ptr<int32_t>(),
                               x_new.data_ptr(), dtype_code(x_new), w_down.data_ptr<float>(),
                               w_up.data_ptr<float>(), q_new.data_ptr(), static_cast<const uint8_t*>(k8.data_ptr()),
                               static_cast<const uint8_t*>(v8.data_ptr()), k_scale.data_ptr<float>(),
                               v_scale.data_ptr<float>(), out.data_ptr(), idx.data_ptr<int32_t>(),
                               gates.data_ptr<float>(), B, D, H, R, E, block_size, top_k, stream_ptr(st)));
  return {out, state, idx, gates};
}

}  // namespace

void bind_nodes(pybind11::module_& m) {
  namespace py = pybind11;
  py::register_exception_translator([](std::exception_ptr p) {
    try {
      if (p) std::rethrow_exception(p);
    } catch (python_error& e) {
      e.restore();
    }
  });
  using at::Tensor;
  m.def("rms_norm", [](Tensor x, Tensor w, double eps, int64_t st) { return RmsNorm::apply(x, w, eps, st); });
  m.def("add_rms_norm",
        [](Tensor x, Tensor a, Tensor w, double eps, int64_t st) { return AddRmsNorm::apply(x, a, w, eps, st); });
  m.def("rope", [](Tensor q, Tensor k, Tensor c, Tensor s, int64_t st) { return Rope::apply(q, k, c, s, st); });
  m.def("causal_attention",
        [](Tensor q, Tensor k, Tensor v, double scale, int64_t st) { return CausalAttention::apply(q, k, v, scale, st); });
  m.def("swiglu", [](Tensor g, Tensor u, int64_t st) { return SwiGLU::apply(g, u, st); });
  m.def("shared_linear", [](Tensor x, std::vector<Tensor> w, int64_t st) {
    TORCH_CHECK(!w.empty() && w.size() <= 3, "shared_linear: one to three weights");
    return SharedLinear::apply(x, w[0], w[w.size() > 1 ? 1 : 0], w[w.size() > 2 ? 2 : 0], (int64_t)w.size(), st);
  });
  m.def("linear", [](Tensor x, std::vector<Tensor> w, bool f32, int64_t st) {  // the products alone, no graph
    at::NoGradGuard no_grad;
    at::DeviceGuard guard(x.device());
    return linear_fwd(x, w, f32 ? at::kFloat : x.scalar_type(), stream_ptr(st));
  });
  m.def("linear_dgrad", [](Tensor dy, Tensor w, int64_t st) {
    at::NoGradGuard no_grad;
    at::DeviceGuard guard(dy.device());
    return linear_dgrad(dy, w, stream_ptr(st));
  });
  m.def("linear_wgrad", [](Tensor xin, Tensor dy, bool f32, int64_t st) {
    at::NoGradGuard no_grad;
    at::DeviceGuard guard(xin.device());
    return library_wgrad(xin, dy, f32 ? at::kFloat : at::kBFloat16, stream_ptr(st));
  });
  m.def("route", [](Tensor x, Tensor wd, Tensor wu, c10::optional<Tensor> noise, double noise_scale, int64_t top_k,
                    bool want_h, int64_t kind, int64_t st) {
    return Route::apply(x, wd, wu, noise.has_value() ? *noise : x, noise.has_value(), noise_scale, top_k, want_h, kind,
                        st);
  });
  m.def("router_stats", [](Tensor probs, Tensor idx, int64_t st) { return RouterStats::apply(probs, idx, st); });
  m.def("read", [](Tensor q, Tensor k, Tensor v, Tensor idx, Tensor gates, int64_t nb, int64_t bs, int64_t st) {
    return Read::apply(q, k, v, idx, gates, nb, bs, st);
  });
  m.def("gated_linear", [](Tensor out, Tensor w, Tensor s, int64_t st) { return GatedLinear::apply(out, w, s, st); });
  m.def("xent", [](Tensor logits, Tensor labels, int64_t ignore, int64_t st) {
    return Xent::apply(logits, labels, ignore, st);
  });
  m.def("decode_step", &decode_step);
}

}  // namespace naylis_ext
