// Shared by the torch extension's sources: status checks, workspaces and the
// weight-gradient call over the C ABI of libnaylis_mom.so.
#pragma once
#include <torch/extension.h>

#include <algorithm>
#include <stdexcept>
#include <string>
#include <vector>

#include "../../include/naylis_mom.h"

namespace naylis_ext {

constexpr int kF32 = 0, kBF16 = 1;

// A non-zero status of a C-ABI call raises naylis_amd._lib.NaylisError: as a
// Python error, which the autograd engine carries out of a backward's thread.
[[noreturn]] void raise_status(int rc);

inline void check(int rc) {
  if (rc != NAYLIS_OK) raise_status(rc);
}

// A workspace query's answer (0: the shape is not supported, with a message).
inline size_t need(size_t nbytes) {
  if (nbytes == 0) check(NAYLIS_ERR_ARG);
  return nbytes;
}

inline at::Tensor workspace(size_t nbytes, const at::Tensor& like) {
  return at::empty({(int64_t)std::max<size_t>(nbytes, 1)}, like.options().dtype(at::kByte));
}

inline int dtype_code(const at::Tensor& t) { return t.scalar_type() == at::kBFloat16 ? kBF16 : kF32; }

inline void* ptr(const at::Tensor& t) { return t.defined() ? t.data_ptr() : nullptr; }

inline void* stream_ptr(int64_t st) { return reinterpret_cast<void*>(st); }

// torch's current stream on t's device
void* current_stream(const at::Tensor& t);

// The kernels read the products' results by their pointers, as bf16: a backward
// that the caller runs under autocast must not make them another type.
struct NoAutocast {
  c10::impl::ExcludeDispatchKeyGuard guard{c10::autocast_dispatch_keyset};
};

// y_i = x W_i^T for one to three weights (x (..., D_in), y_i (..., D_out) in
// `dtype`), and dx = dy W (dy (N, D_out)): the library's GEMM where the rules
// in torch_nodes.cpp say so, else torch's (hipBLASLt).
std::vector<at::Tensor> linear_fwd(const at::Tensor& x, const std::vector<at::Tensor>& w, at::ScalarType dtype,
                                   void* st);
at::Tensor linear_dgrad(const at::Tensor& dy, const at::Tensor& w, void* st);

// dW = dy^T xin over all rows: the library's GEMM when N, D_in, D_out are
// multiples of 8 (any row count of plain bf16 operands), else torch's product
at::Tensor library_wgrad(const at::Tensor& xin, const at::Tensor& dy, at::ScalarType dtype, void* st);

// y2 = out2 (s W_o)^T in fp32 and the scaled weight; its backward (d out2, dW_o, ds)
std::pair<at::Tensor, at::Tensor> gated_linear_forward(const at::Tensor& out2, const at::Tensor& w_o,
                                                       const at::Tensor& s, void* st);
struct GatedGrads {
  at::Tensor dout2, dw_o, ds;
};
GatedGrads gated_linear_backward(const at::Tensor& dy2, const at::Tensor& out2, const at::Tensor& w_o,
                                 const at::Tensor& w_os, const at::Tensor& s, void* st);

// y = out (s W_o)^T, fp32, as a node
at::Tensor gated_linear(const at::Tensor& out, const at::Tensor& w_o, const at::Tensor& s, int64_t st);

// The router backward's d_probs: an fp32 gradient expanded from one row goes in
// as that row with stride 0, anything else as a dense fp32 copy with stride E.
struct ProbsGrad {
  at::Tensor t;
  int64_t stride;
};
ProbsGrad probs_grad(const at::Tensor& g, int64_t E);

void bind_nodes(pybind11::module_& m);

}  // namespace naylis_ext
