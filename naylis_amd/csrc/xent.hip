// Next-token cross-entropy of the decoder's LM head, fused: the reference
// computes F.cross_entropy(shift_logits.float(), labels, reduction="sum")
// (model.py:536-545): an fp32 copy of the (N, V) logits, log_softmax and the
// label pick forward, and as many full passes backward.  Here the forward
// reads the bf16 logits once per row (max, sum of exp, the label's logit) and
// writes the row's loss and log-sum-exp; the backward reads them once more and
// writes the bf16 gradient (softmax - one_hot) * g_row.  Rows whose label is
// ignore_index have loss 0 and gradient 0.
#include "common.h"
#include "timing.h"

namespace naylis {

// 16 bytes that the kernel does not read again (kept out of the caches' way)
__device__ __forceinline__ uint4 load_once(const bf16_t* p) {
  return __builtin_bit_cast(uint4, __builtin_nontemporal_load(reinterpret_cast<const f32x4*>(p)));
}

// One workgroup per row; V = 2048 nch.  A thread holds U chunks of 8 values in
// registers, all their loads in flight at once, and reads them once: its own
// maximum, then the sum of exp2 against that maximum, rescaled when a later
// tile raises it.  The 256 threads' (maximum, sum) pairs meet in one exchange
// at the end, so no barrier stands between the maximum and the sum.  x - m is
// exact for bf16 values of similar size, so one product with log2 e and
// v_exp_f32 replace expf; values over 87 below their thread's maximum add 0.
// Bound by HBM (the logits once).  16376 x 32768: 308 - 358 us (each row read
// twice, one load in flight per wave, a full expf per value) -> 156 us, 6.8
// TB/s (178 us with temporal loads).
template <int U>
__global__ __launch_bounds__(256) void xent_fwd_kernel(const bf16_t* __restrict__ logits,
                                                       const int64_t* __restrict__ labels, float* __restrict__ loss,
                                                       float* __restrict__ lse_out, int V, long ignore_index) {
  __shared__ float red[8];
  const long row = blockIdx.x;
  const bf16_t* x = logits + row * (long)V;
  const int nch = V >> 11;
  const long lab = labels[row];
  // a label that is neither ignore_index nor a class gives a NaN loss (the
  // reference's F.cross_entropy raises on it): bad data cannot pass silently
  const bool in_range = lab >= 0 && lab < V;
  const float xl = bf16_to_f32(x[in_range ? lab : 0]);
  float m = -INFINITY, s = 0.f;
  for (int c0 = 0; c0 < nch; c0 += U) {
    uint4 u[U];
#pragma unroll
    for (int i = 0; i < U; ++i)  // chunks past the row's end read its last one and are masked below
      u[i] = load_once(x + min(c0 + i, nch - 1) * 2048 + threadIdx.x * 8);
    if (c0 + U > nch) {
#pragma unroll
      for (int i = 0; i < U; ++i)
        if (c0 + i >= nch) u[i] = make_uint4(0xff80ff80u, 0xff80ff80u, 0xff80ff80u, 0xff80ff80u);  // -inf
    }
    float mt = m;
#pragma unroll
    for (int i = 0; i < U; ++i) {
      const uint32_t w[4] = {u[i].x, u[i].y, u[i].z, u[i].w};
#pragma unroll
      for (int e = 0; e < 4; ++e)
        mt = fmaxf(mt, fmaxf(__uint_as_float(w[e] << 16), __uint_as_float(w[e] & 0xffff0000u)));
    }
    // a thread whose values are all -inf so far sums against 0, so that its sum stays 0
    const float ref = mt == -INFINITY ? 0.f : mt;
    float t[4] = {0.f, 0.f, 0.f, 0.f};  // independent chains
#pragma unroll
    for (int i = 0; i < U; ++i) {
      const uint32_t w[4] = {u[i].x, u[i].y, u[i].z, u[i].w};
#pragma unroll
      for (int e = 0; e < 4; ++e)
        t[e] += __builtin_amdgcn_exp2f((__uint_as_float(w[e] << 16) - ref) * kLog2e) +
                __builtin_amdgcn_exp2f((__uint_as_float(w[e] & 0xffff0000u) - ref) * kLog2e);
    }
    if (c0 > 0) s *= __builtin_amdgcn_exp2f((m - ref) * kLog2e);
    s += (t[0] + t[1]) + (t[2] + t[3]);
    m = mt;
  }
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const float mw = wave_allmax(m);
  const float sw = wave_allsum(m == -INFINITY ? s : s * __builtin_amdgcn_exp2f((m - mw) * kLog2e));
  if (lane == 0) {
    red[wave] = mw;
    red[4 + wave] = sw;
  }
  __syncthreads();
  if (threadIdx.x == 0) {
    const float mx = fmaxf(fmaxf(red[0], red[1]), fmaxf(red[2], red[3]));
    float sum = 0.f;  // NaN where the whole row is -inf (-inf less itself), as log_softmax gives
#pragma unroll
    for (int w = 0; w < 4; ++w) sum += red[4 + w] * __builtin_amdgcn_exp2f((red[w] - mx) * kLog2e);
    const float lse = mx + logf(sum);
    loss[row] = lab == ignore_index ? 0.f : in_range ? lse - xl : __builtin_nanf("");
    lse_out[row] = lse;
  }
}

// e^d to about an ulp, tiny results included: with d log2 e = n + r, n whole,
// 2^r 2^n. v_exp_f32 of the rounded product alone is off by up to |d| 2^-24 of
// the result, and 0 under 2^-126: at logits of deviation 60 (V 2048) 6.3e-3 of the
// bf16 gradients then are not the correctly rounded ones, 1.5e-5 with this
// (deviation 12, V 32768: 1.4e-3 and 2.1e-4), for 16376 x 32768 in 401 us against
// 399 and 512 x 32768, from the caches, in 13.5 against 12.3 (expf 407 and 14.8).
// d is kept from -inf, where r is NaN.
__device__ __forceinline__ float exp_full(float d) {
  constexpr float kLog2eLo = 1.92596299e-8f;  // log2 e - kLog2e
  d = d < -200.f ? -200.f : d;                // (a NaN stays)
  const float n = rintf(d * kLog2e);
  const float r = fmaf(d, kLog2eLo, fmaf(d, kLog2e, -n));
  return ldexpf(__builtin_amdgcn_exp2f(r), (int)n);
}

// The stores bypass the caches: the gradient of a training batch exceeds them.
// 4096 x 24576: 81 -> 78 us; 16376 x 32768: 409 -> 401 us (5.4 TB/s).
// d logits[r, j] = (exp(x - lse) - [j == label]) * g[r * g_stride]
__global__ __launch_bounds__(256) void xent_bwd_kernel(const bf16_t* __restrict__ logits,
                                                       const int64_t* __restrict__ labels,
                                                       const float* __restrict__ lse, const float* __restrict__ g,
                                                       long g_stride, bf16_t* __restrict__ dlogits, int V,
                                                       long ignore_index) {
  const long row = blockIdx.x;
  const bf16_t* x = logits + row * (long)V;
  bf16_t* dx = dlogits + row * (long)V;
  const long lab = labels[row];
  // ignore_index rows get a zero gradient, out-of-range labels a NaN one
  const float gr = lab == ignore_index ? 0.f : (lab >= 0 && lab < V) ? g[row * g_stride] : __builtin_nanf("");
  const float l = lse[row];
  for (int j = threadIdx.x * 8; j < V; j += 2048) {
    const uint4 u = *reinterpret_cast<const uint4*>(x + j);
    const uint32_t w[4] = {u.x, u.y, u.z, u.w};
    bf16x8 r;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const float a = __uint_as_float(w[i] << 16), b = __uint_as_float(w[i] & 0xffff0000u);
      const float pa = exp_full(a - l) - (j + 2 * i == lab ? 1.f : 0.f);
      const float pb = exp_full(b - l) - (j + 2 * i + 1 == lab ? 1.f : 0.f);
      r[2 * i] = (__bf16)(pa * gr);
      r[2 * i + 1] = (__bf16)(pb * gr);
    }
    __builtin_nontemporal_store(__builtin_bit_cast(f32x4, r), reinterpret_cast<f32x4*>(dx + j));
  }
}

hipError_t launch_xent(const void* logits, const int64_t* labels, float* loss, float* lse, const float* g,
                       long g_stride, void* dlogits, bool bwd, long N, int V, long ignore_index, hipStream_t st) {
  if (N == 0) return hipSuccess;
  if (!bwd) {
    // 8 chunks a tile (16 chunks, the whole row at V 32768, take 138 registers
    // and 182 us against 178); short rows take the tile that holds them
    // (16384 rows of 2048: 16.1 us against 29.8 in a tile of 4, of 4096: 23.1
    // against 33.3)
    auto fwd = [&](auto kernel) {
      NAYLIS_TIMED("xent_fwd", st, hipLaunchKernelGGL(kernel, dim3((unsigned)N), dim3(256), 0, st,
                                                      (const bf16_t*)logits, labels, loss, lse, V, ignore_index));
    };
    if (V > 4 * 2048)
      fwd(xent_fwd_kernel<8>);
    else if (V > 2 * 2048)
      fwd(xent_fwd_kernel<4>);
    else if (V > 2048)
      fwd(xent_fwd_kernel<2>);
    else
      fwd(xent_fwd_kernel<1>);
  } else {
    NAYLIS_TIMED("xent_bwd", st, hipLaunchKernelGGL(xent_bwd_kernel, dim3((unsigned)N), dim3(256), 0, st,
                                                    (const bf16_t*)logits, labels, lse, g, g_stride,
                                                    (bf16_t*)dlogits, V, ignore_index));
  }
  return hipGetLastError();
}

}  // namespace naylis
