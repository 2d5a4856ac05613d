// Causal attention of the decoder's Llama attention (model.py:279-345), head
// dimension 64, bf16 operands with fp32 sums and softmax:
//   o = softmax(scale q k^T, k <= q) v
// q, k, v, o (B, S, H, 64) row-major, as the projections write and read them,
// so no operand is transposed in memory.
//
// Products run on v_mfma_f32_32x32x16_bf16 (fragment layouts in common.h).
// The forward and the dQ kernel form S^T = K Q^T: a lane owns one query, its
// softmax state is one register, and P^T / dS^T leave the accumulators as the
// B operand of the next product.  The dK/dV kernel forms S = Q K^T, where a
// lane owns one key and P / dS feed dV^T = dO^T P and dK^T = Q^T dS the same
// way.  K / V (or Q / dO) pass through LDS in stages of 64 rows, double
// buffered with one barrier a stage; a workgroup's other operands stay in
// registers.  Backward recomputes P from the forward's log-sum-exp in both
// kernels (7 products of the causal triangle): dQ, dK and dV are each summed
// in one workgroup in a fixed order, with no atomics.
//
// Bound by the vector units: per 32 x 32 tile a forward wave issues 8 MFMAs
// (256 cycles) and about 16 exp2, 16 fma, 16 adds, 8 max3 and 8 packs.
// B 8, S 2048, H 16: forward 219 -> 108 us, backward 955 -> 280 us (dQ 115, dK/dV
// 165 - 176) against torch's scaled_dot_product_attention.
#include "common.h"
#include "launch.h"
#include "timing.h"

namespace naylis {

namespace {

constexpr int kAttnHd = 64;
constexpr int kStageRows = 64;
constexpr int kBlockRows = 128;  // queries (or keys) of a workgroup
constexpr int kStageBytes = kStageRows * 128;

// LDS rows are 128 bytes without padding; 16-byte chunk c of row r sits in
// slot c ^ swz(r).  16 consecutive rows' chunk c then cover 256 bytes (row
// fragments), and so do 4 consecutive rows' 64-byte halves (transposing reads).
__device__ __forceinline__ int swz(int r) { return ((r & 2) << 1) | ((r >> 2) & 1) | ((r >> 2) & 2); }

// Fragment of rows row0 .. row0 + 31 (row0 a multiple of 32): lane l gets
// X(row0 + l % 32, 16 ks + 8 (l / 32) + e).
struct RowFrag {
  int off[4];
  __device__ __forceinline__ RowFrag(int lane) {
    const int r = lane & 31, g = lane >> 5;
#pragma unroll
    for (int ks = 0; ks < 4; ++ks) off[ks] = r * 128 + (((2 * ks + g) ^ swz(r)) << 4);
  }
  __device__ __forceinline__ bf16x8 get(const uint8_t* tile, int row0, int ks) const {
    return *reinterpret_cast<const bf16x8*>(tile + row0 * 128 + off[ks]);
  }
};

// A fragment of X^T, features 32 t .. 32 t + 31, over rows k0 .. k0 + 15 (k0
// a multiple of 16): lds_frag_T<true, true> of common.h on the swizzled rows.
struct TransFrag {
  int lo[2], hi[2];
  __device__ __forceinline__ TransFrag(int lane) {
    const int q = lane >> 4, j = lane & 15, g = q >> 1, mq = q & 1, c = j & 3;
    const int r0 = (j >> 2) + 4 * g, r1 = r0 + 8, ch = 2 * (c & 1) + mq, b = 8 * (c >> 1);
#pragma unroll
    for (int t = 0; t < 2; ++t) {
      lo[t] = r0 * 128 + (((4 * t + ch) ^ swz(r0)) << 4) + b;
      hi[t] = r1 * 128 + (((4 * t + ch) ^ swz(r1)) << 4) + b;
    }
  }
  __device__ __forceinline__ bf16x8 get(const uint8_t* tile, int k0, int t) const {
    const v4i16 a = lds_read_tr16(reinterpret_cast<const bf16_t*>(tile + k0 * 128 + lo[t]));
    const v4i16 b = lds_read_tr16(reinterpret_cast<const bf16_t*>(tile + k0 * 128 + hi[t]));
    typedef short v8i16 __attribute__((ext_vector_type(8)));
    const v8i16 v = __builtin_shufflevector(a, b, 0, 1, 2, 3, 4, 5, 6, 7);
    return __builtin_bit_cast(bf16x8, v);
  }
};

// A thread's share (two 16-byte chunks) of a 64-row stage of one operand,
// loaded through a resource that ends with the sequence: rows past it are 0.
struct StageCopy {
  int voff[2], lds;
  __device__ __forceinline__ StageCopy(int tid, int ld) {
    const int r = tid >> 3, c = tid & 7;
    voff[0] = (r * ld + c * 8) * 2;
    voff[1] = ((r + 32) * ld + c * 8) * 2;
    lds = r * 128 + ((c ^ swz(r)) << 4);
  }
  __device__ __forceinline__ void load(uint4 (&x)[2], __amdgpu_buffer_rsrc_t rs, int soff) const {
    x[0] = __builtin_bit_cast(uint4, __builtin_amdgcn_raw_buffer_load_b128(rs, voff[0], soff, 0));
    x[1] = __builtin_bit_cast(uint4, __builtin_amdgcn_raw_buffer_load_b128(rs, voff[1], soff, 0));
  }
  __device__ __forceinline__ void store(const uint4 (&x)[2], uint8_t* tile) const {
    *reinterpret_cast<uint4*>(tile + lds) = x[0];
    *reinterpret_cast<uint4*>(tile + lds + 32 * 128) = x[1];
  }
};

// B operand fragments of 32 rows straight from memory: lane l gets row
// row0 + l % 32, features 16 ks + 8 (l / 32) + e (zeros past the sequence).
__device__ __forceinline__ void load_rows(bf16x8 (&f)[4], __amdgpu_buffer_rsrc_t rs, int row0, int ld, int lane) {
  const int off = ((row0 + (lane & 31)) * ld + 8 * (lane >> 5)) * 2;
#pragma unroll
  for (int ks = 0; ks < 4; ++ks)
    f[ks] = __builtin_bit_cast(bf16x8, __builtin_amdgcn_raw_buffer_load_b128(rs, off + 32 * ks, 0, 0));
}

// Transposed accumulators (lane = row, registers = features 32 t + 16 g + v)
// times x to row `row` of a (., ld) bf16 tensor.
__device__ __forceinline__ void store_row(bf16_t* p, const f32x16 (&a)[2], float x, int g) {
#pragma unroll
  for (int t = 0; t < 2; ++t) {
    f32x16 s;
#pragma unroll
    for (int v = 0; v < 16; ++v) s[v] = a[t][v] * x;
    *reinterpret_cast<bf16x8*>(p + 32 * t + 16 * g) = pack8(s, 0);
    *reinterpret_cast<bf16x8*>(p + 32 * t + 16 * g + 8) = pack8(s, 8);
  }
}

struct AttnDims {
  int S, H, BH, ld;  // ld = H * 64, row stride in elements
};

}  // namespace

// Forward: 4 waves of 32 queries (64 a wave, which halve the LDS reads, keep
// 200 registers and two waves a SIMD: 98 against 87 us at B 8, S 2048, H 16,
// and twice the time where they leave CUs idle).  Workgroups run longest first (a query
// block's work grows with its position), heads innermost so that an XCD keeps
// its heads' K and V in its L2.  The running reference m is the largest score so
// far, so that the largest weight is exactly 1 in bf16: a reference that moves
// only by factors over 2^8 rescales less (95 against 108 us) but rounds that
// weight too, and the output's error (2-norm, fp64) is 2.08e-3 against 1.99e-3 on
// normal scores of 1021 keys, 2.13e-3 against 1.75e-3 on scores three times that
// (torch's flash attention 2.00e-3 and 1.76e-3).
__global__ __launch_bounds__(256, 4) void attn_fwd_kernel(const bf16_t* __restrict__ q, const bf16_t* __restrict__ k,
                                                          const bf16_t* __restrict__ v, bf16_t* __restrict__ o,
                                                          float* __restrict__ lse, AttnDims d, int nqb, float c) {
  __shared__ __align__(16) uint8_t kt[2][kStageBytes];
  __shared__ __align__(16) uint8_t vt[2][kStageBytes];
  const int tid = threadIdx.x, lane = tid & 63, g = lane >> 5, col = lane & 31;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int qb = nqb - 1 - blockIdx.x / d.BH, bh = blockIdx.x % d.BH;
  const long base = (long)(bh / d.H) * d.S * d.ld + (bh % d.H) * kAttnHd;
  const uint32_t bytes = ((uint32_t)(d.S - 1) * d.ld + kAttnHd) * 2;
  const __amdgpu_buffer_rsrc_t rk = make_rsrc(k + base, bytes), rv = make_rsrc(v + base, bytes);
  const int q0 = qb * kBlockRows + wave * 32, row = q0 + col;  // the wave's first query, the lane's

  bf16x8 qf[4];
  load_rows(qf, make_rsrc(q + base, bytes), q0, d.ld, lane);
  const StageCopy cp(tid, d.ld);
  const RowFrag rf(lane);
  const TransFrag tf(lane);
  f32x16 acc[2];
  acc[0] = acc[1] = f32x16{};
  float m = kNegBig, l = 0.f;
  const int nst = (min(d.S, (qb + 1) * kBlockRows) + kStageRows - 1) / kStageRows;
  const int step = kStageRows * d.ld * 2;
  uint4 xk[2], xv[2];
  cp.load(xk, rk, 0);
  cp.load(xv, rv, 0);
  cp.store(xk, kt[0]);
  cp.store(xv, vt[0]);
  lds_barrier();
  for (int st = 0; st < nst; ++st) {
    const int nx = min(st + 1, nst - 1) * step;  // past the last stage: loaded again, not read
    cp.load(xk, rk, nx);
    cp.load(xv, rv, nx);
    const uint8_t* kb = kt[st & 1];
    const uint8_t* vb = vt[st & 1];
#pragma unroll
    for (int sub = 0; sub < 2; ++sub) {
      const int kv0 = st * kStageRows + 32 * sub;
      if (kv0 > q0) continue;  // above the diagonal (wave-uniform)
      f32x16 s = f32x16{};
#pragma unroll
      for (int ks = 0; ks < 4; ++ks) s = mfma32(rf.get(kb, 32 * sub, ks), qf[ks], s);
      if (kv0 == q0) {
#pragma unroll
        for (int i = 0; i < 16; ++i)
          if (acc_row(g, i) > col) s[i] = -INFINITY;
      }
      float mx = s[0];
#pragma unroll
      for (int i = 1; i < 16; ++i) mx = fmaxf(mx, s[i]);
      if (__any(mx * c > m)) {
        // per query, so that a row's result does not depend on its neighbours'
        const float mr = xor32_f32(mx, [](float a, float b) { return fmaxf(a, b); }) * c;
        const float mn = fmaxf(m, mr);
        const float al = __builtin_amdgcn_exp2f(m - mn);
        m = mn;
        l *= al;
#pragma unroll
        for (int i = 0; i < 16; ++i) {
          acc[0][i] *= al;
          acc[1][i] *= al;
        }
      }
      float ls = 0.f;
#pragma unroll
      for (int i = 0; i < 16; ++i) {
        s[i] = __builtin_amdgcn_exp2f(fmaf(s[i], c, -m));
        ls += s[i];
      }
      l += ls;
      const bf16x8 pf[2] = {pack8(s, 0), pack8(s, 8)};
#pragma unroll
      for (int h = 0; h < 2; ++h)
#pragma unroll
        for (int t = 0; t < 2; ++t) acc[t] = mfma32(tf.get(vb, 32 * sub + 16 * h, t), pf[h], acc[t]);
    }
    cp.store(xk, kt[(st + 1) & 1]);
    cp.store(xv, vt[(st + 1) & 1]);
    lds_barrier();
  }
  const float ls = xor32_f32(l, [](float a, float b) { return a + b; });
  if (row < d.S) {
    store_row(o + base + (long)row * d.ld, acc, 1.f / ls, g);
    if (g == 0) lse[(long)bh * d.S + row] = m + log2f(ls);
  }
}

// dQ (and delta = rowsum(dO o), which the dK/dV kernel reads): the forward's
// walk with P from the log-sum-exp.
__global__ __launch_bounds__(256, 3) void attn_bwd_dq_kernel(
    const bf16_t* __restrict__ q, const bf16_t* __restrict__ k, const bf16_t* __restrict__ v,
    const bf16_t* __restrict__ o, const float* __restrict__ lse, const bf16_t* __restrict__ dout,
    bf16_t* __restrict__ dq, float* __restrict__ delta, AttnDims d, int nqb, float scale) {
  __shared__ __align__(16) uint8_t kt[2][kStageBytes];
  __shared__ __align__(16) uint8_t vt[2][kStageBytes];
  const int tid = threadIdx.x, lane = tid & 63, g = lane >> 5, col = lane & 31;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int qb = nqb - 1 - blockIdx.x / d.BH, bh = blockIdx.x % d.BH;
  const long base = (long)(bh / d.H) * d.S * d.ld + (bh % d.H) * kAttnHd;
  const uint32_t bytes = ((uint32_t)(d.S - 1) * d.ld + kAttnHd) * 2;
  const __amdgpu_buffer_rsrc_t rk = make_rsrc(k + base, bytes), rv = make_rsrc(v + base, bytes);
  const int q0 = qb * kBlockRows + wave * 32, row = q0 + col;
  const float c = scale * kLog2e;

  bf16x8 qf[4], df[4];
  load_rows(qf, make_rsrc(q + base, bytes), q0, d.ld, lane);
  load_rows(df, make_rsrc(dout + base, bytes), q0, d.ld, lane);
  const float ml = -lse[(long)bh * d.S + min(row, d.S - 1)];
  float md = 0.f;  // -delta of the lane's query
  {
    bf16x8 of[4];
    load_rows(of, make_rsrc(o + base, bytes), q0, d.ld, lane);
#pragma unroll
    for (int ks = 0; ks < 4; ++ks)
#pragma unroll
      for (int e = 0; e < 8; ++e) md = fmaf(-(float)df[ks][e], (float)of[ks][e], md);
    md = xor32_f32(md, [](float a, float b) { return a + b; });
    if (g == 0 && row < d.S) delta[(long)bh * d.S + row] = -md;
  }
  const StageCopy cp(tid, d.ld);
  const RowFrag rf(lane);
  const TransFrag tf(lane);
  f32x16 acc[2];
  acc[0] = acc[1] = f32x16{};
  const int nst = (min(d.S, (qb + 1) * kBlockRows) + kStageRows - 1) / kStageRows;
  const int step = kStageRows * d.ld * 2;
  uint4 xk[2], xv[2];
  cp.load(xk, rk, 0);
  cp.load(xv, rv, 0);
  cp.store(xk, kt[0]);
  cp.store(xv, vt[0]);
  lds_barrier();
  for (int st = 0; st < nst; ++st) {
    const int nx = min(st + 1, nst - 1) * step;
    cp.load(xk, rk, nx);
    cp.load(xv, rv, nx);
    const uint8_t* kb = kt[st & 1];
    const uint8_t* vb = vt[st & 1];
#pragma unroll
    for (int sub = 0; sub < 2; ++sub) {
      const int kv0 = st * kStageRows + 32 * sub;
      if (kv0 > q0) continue;
      f32x16 s = f32x16{}, dp;
#pragma unroll
      for (int i = 0; i < 16; ++i) dp[i] = md;
#pragma unroll
      for (int ks = 0; ks < 4; ++ks) {
        s = mfma32(rf.get(kb, 32 * sub, ks), qf[ks], s);
        dp = mfma32(rf.get(vb, 32 * sub, ks), df[ks], dp);
      }
      if (kv0 == q0) {
#pragma unroll
        for (int i = 0; i < 16; ++i)
          if (acc_row(g, i) > col) s[i] = -INFINITY;
      }
#pragma unroll
      for (int i = 0; i < 16; ++i) s[i] = __builtin_amdgcn_exp2f(fmaf(s[i], c, ml)) * dp[i];
      const bf16x8 sf[2] = {pack8(s, 0), pack8(s, 8)};
#pragma unroll
      for (int h = 0; h < 2; ++h)
#pragma unroll
        for (int t = 0; t < 2; ++t) acc[t] = mfma32(tf.get(kb, 32 * sub + 16 * h, t), sf[h], acc[t]);
    }
    cp.store(xk, kt[(st + 1) & 1]);
    cp.store(xv, vt[(st + 1) & 1]);
    lds_barrier();
  }
  if (row < d.S) store_row(dq + base + (long)row * d.ld, acc, scale, g);
}

// dK, dV: 4 waves of 32 keys, whose K and V rows stay in registers; the
// queries from the diagonal to the end pass through LDS with their -lse / c
// and -delta, which start the accumulators of S and dP.  Queries past the
// sequence get -inf there, so their P is 0.  193 registers, two waves a SIMD;
// held to 168 for three it spills 31 and takes 346 us for 176.
__global__ __launch_bounds__(256, 2) void attn_bwd_dkdv_kernel(
    const bf16_t* __restrict__ q, const bf16_t* __restrict__ k, const bf16_t* __restrict__ v,
    const float* __restrict__ lse, const bf16_t* __restrict__ dout, const float* __restrict__ delta,
    bf16_t* __restrict__ dk, bf16_t* __restrict__ dv, AttnDims d, float scale) {
  __shared__ __align__(16) uint8_t qt[2][kStageBytes];
  __shared__ __align__(16) uint8_t dt[2][kStageBytes];
  __shared__ __align__(16) float rows[2][2][kStageRows];  // [buffer][-lse / c, -delta][query]
  const int tid = threadIdx.x, lane = tid & 63, g = lane >> 5, col = lane & 31;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int kb = blockIdx.x / d.BH, bh = blockIdx.x % d.BH;
  const long base = (long)(bh / d.H) * d.S * d.ld + (bh % d.H) * kAttnHd;
  const uint32_t bytes = ((uint32_t)(d.S - 1) * d.ld + kAttnHd) * 2;
  const __amdgpu_buffer_rsrc_t rq = make_rsrc(q + base, bytes), rd = make_rsrc(dout + base, bytes);
  const int kv0 = kb * kBlockRows + wave * 32;
  const float c = scale * kLog2e, rc = 1.f / c;

  bf16x8 kf[4], vf[4];
  load_rows(kf, make_rsrc(k + base, bytes), kv0, d.ld, lane);
  load_rows(vf, make_rsrc(v + base, bytes), kv0, d.ld, lane);
  const StageCopy cp(tid, d.ld);
  const RowFrag rf(lane);
  const TransFrag tf(lane);
  f32x16 ak[2], av[2];
  ak[0] = ak[1] = av[0] = av[1] = f32x16{};
  const int st0 = kb * (kBlockRows / kStageRows), nst = (d.S + kStageRows - 1) / kStageRows;
  const int step = kStageRows * d.ld * 2;
  // threads 0 .. 63 carry -lse / c, 64 .. 127 -delta of the stage's queries
  auto load_stat = [&](int st) {
    const int row = st * kStageRows + (tid & 63);
    const long i = (long)bh * d.S + min(row, d.S - 1);
    if (tid < 64) return row < d.S ? -lse[i] * rc : -INFINITY;
    return tid < 128 && row < d.S ? -delta[i] : 0.f;
  };
  uint4 xq[2], xd[2];
  cp.load(xq, rq, st0 * step);
  cp.load(xd, rd, st0 * step);
  float xs = load_stat(st0);
  cp.store(xq, qt[0]);
  cp.store(xd, dt[0]);
  if (tid < 128) rows[0][tid >> 6][tid & 63] = xs;
  lds_barrier();
  for (int st = st0; st < nst; ++st) {
    const int nx = min(st + 1, nst - 1), buf = (st - st0) & 1;
    cp.load(xq, rq, nx * step);
    cp.load(xd, rd, nx * step);
    xs = load_stat(nx);
#pragma unroll
    for (int sub = 0; sub < 2; ++sub) {
      const int q0 = st * kStageRows + 32 * sub;
      if (q0 < kv0) continue;  // above the diagonal
      f32x16 s, dp;
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const f32x4 a = *reinterpret_cast<const f32x4*>(&rows[buf][0][32 * sub + 8 * i + 4 * g]);
        const f32x4 b = *reinterpret_cast<const f32x4*>(&rows[buf][1][32 * sub + 8 * i + 4 * g]);
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          s[4 * i + e] = a[e];
          dp[4 * i + e] = b[e];
        }
      }
#pragma unroll
      for (int ks = 0; ks < 4; ++ks) {
        s = mfma32(rf.get(qt[buf], 32 * sub, ks), kf[ks], s);
        dp = mfma32(rf.get(dt[buf], 32 * sub, ks), vf[ks], dp);
      }
#pragma unroll
      for (int i = 0; i < 16; ++i) s[i] = __builtin_amdgcn_exp2f(s[i] * c);
      if (q0 == kv0) {
#pragma unroll
        for (int i = 0; i < 16; ++i)
          if (acc_row(g, i) < col) s[i] = 0.f;
      }
      const bf16x8 pf[2] = {pack8(s, 0), pack8(s, 8)};
#pragma unroll
      for (int i = 0; i < 16; ++i) s[i] *= dp[i];
      const bf16x8 sf[2] = {pack8(s, 0), pack8(s, 8)};
#pragma unroll
      for (int h = 0; h < 2; ++h)
#pragma unroll
        for (int ft = 0; ft < 2; ++ft) {
          av[ft] = mfma32(tf.get(dt[buf], 32 * sub + 16 * h, ft), pf[h], av[ft]);
          ak[ft] = mfma32(tf.get(qt[buf], 32 * sub + 16 * h, ft), sf[h], ak[ft]);
        }
    }
    cp.store(xq, qt[buf ^ 1]);
    cp.store(xd, dt[buf ^ 1]);
    if (tid < 128) rows[buf ^ 1][tid >> 6][tid & 63] = xs;
    lds_barrier();
  }
  const int row = kv0 + col;
  if (row < d.S) {
    store_row(dk + base + (long)row * d.ld, ak, scale, g);
    store_row(dv + base + (long)row * d.ld, av, 1.f, g);
  }
}

// Byte offsets inside one sequence stay below 2^31, the 64 rows that a stage
// may lie past its end included.
bool attn_supported(long B, long S, long H) {
  return B > 0 && S > 0 && H > 0 && B * H <= (1 << 20) && (S + 512) * H * kAttnHd * 2 < 0x7fffffffL &&
         (S + kBlockRows - 1) / kBlockRows * B * H < (1L << 31);
}

hipError_t launch_attn_fwd(const void* q, const void* k, const void* v, void* o, float* lse, float scale, long B,
                           long S, long H, hipStream_t st) {
  const AttnDims d{(int)S, (int)H, (int)(B * H), (int)(H * kAttnHd)};
  const int nqb = (int)((S + kBlockRows - 1) / kBlockRows);
  NAYLIS_TIMED("attn_fwd", st,
               hipLaunchKernelGGL(attn_fwd_kernel, dim3((unsigned)(nqb * d.BH)), dim3(256), 0, st, (const bf16_t*)q,
                                  (const bf16_t*)k, (const bf16_t*)v, (bf16_t*)o, lse, d, nqb, scale * kLog2e));
  return hipGetLastError();
}

hipError_t launch_attn_bwd(const void* q, const void* k, const void* v, const void* o, const float* lse,
                           const void* dout, void* dq, void* dk, void* dv, float* delta, float scale, long B, long S,
                           long H, hipStream_t st) {
  const AttnDims d{(int)S, (int)H, (int)(B * H), (int)(H * kAttnHd)};
  const int nb = (int)((S + kBlockRows - 1) / kBlockRows);
  const dim3 grid((unsigned)(nb * d.BH));
  NAYLIS_TIMED("attn_bwd_dq", st,
               hipLaunchKernelGGL(attn_bwd_dq_kernel, grid, dim3(256), 0, st, (const bf16_t*)q, (const bf16_t*)k,
                                  (const bf16_t*)v, (const bf16_t*)o, lse, (const bf16_t*)dout, (bf16_t*)dq, delta, d,
                                  nb, scale));
  hipError_t e = hipGetLastError();
  if (e != hipSuccess) return e;
  NAYLIS_TIMED("attn_bwd_dkdv", st,
               hipLaunchKernelGGL(attn_bwd_dkdv_kernel, grid, dim3(256), 0, st, (const bf16_t*)q, (const bf16_t*)k,
                                  (const bf16_t*)v, lse, (const bf16_t*)dout, delta, (bf16_t*)dk, (bf16_t*)dv, d,
                                  scale));
  return hipGetLastError();
}

}  // namespace naylis
