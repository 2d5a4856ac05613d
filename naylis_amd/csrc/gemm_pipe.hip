// Pipelined bf16 GEMM (gfx950, v_mfma_f32_32x32x16_bf16, fp32 sums): the
// products of gemm.hip whose grid fills the chip with 256 x 128 tiles, those
// that fit it once with smaller ones, and the weight gradients, whose K (all
// tokens) is cut into equal ranges of the (tile, K step) list so that every CU
// works to the end.
//
// 8 waves (4 x 2) of 64 x 64 per 256 x 128 tile, K steps of 64.  Stages go from
// memory to LDS directly (buffer loads with an LDS destination, no staging
// registers), through a ring of 3 x 48 KB: at step s the loads of stage s + 2
// are issued while stage s + 1 is in flight.  One barrier a step, before its
// last 16-wide slice: fragments are read a slice ahead, the last slice's before
// the barrier and those of the next stage's first slice after it, so LDS
// latency lies under the products of the slice before.  Steps of 32 in a ring
// of 6 hold as many bytes in flight but pay twice the barriers: 2042 x 2816 over
// K 1024 19.1 us against 17.0, 4096 x 1536 over 1536 27.1 against 22.6; weight
// gradients over 16384 tokens 3 - 5 % slower.
//
// Direct loads write LDS in lane order, so the tiles cannot be padded; 64-byte
// groups (row-contiguous operands, [k][row]) or 16-byte chunks (K-contiguous
// ones, [row][k]) are permuted by XOR on the source address instead, which
// leaves both fragment reads (ds_read_b64_tr_b16, ds_read_b128) free of bank
// conflicts.
//
// Large products are bound by the matrix units at the clock that the card holds
// under them: operands of zeros run 15 - 20 % faster.  Against gemm.hip (kernel
// and reduction, 16384 tokens, launches back to back): 1024 x 1024 48.5 -> 42.7
// us (39.4 + 7.4 in the layer's backward, operands out of the caches), 1024 x
// 2816 127 -> 97 (0.97 PFLOP/s), 1536 x 1536 107 -> 82, 2048 x 2048 149 -> 134;
// whole tiles, 5632 x 2048 over 4096: 117 -> 86 (1.10 PFLOP/s).
#include "common.h"
#include "launch_gemm.h"
#include "timing.h"

#include <algorithm>
#include <numeric>

namespace naylis {

namespace {

// WAVES waves, WM of them along M, each with TM x TN tiles of 32 x 32; K steps
// of BK, RING stages of them in LDS.
template <int WAVES_, int WM_, int TM_, int TN_, int BK_, int RING_>
struct PipeCfg {
  static constexpr int WAVES = WAVES_, WM = WM_, TM = TM_, TN = TN_, BK = BK_, RING = RING_, NT = 64 * WAVES;
  static constexpr int BM = WM * TM * 32, BN = WAVES / WM * TN * 32;
  static constexpr int ABYTES = BM * BK * 2, STAGE = ABYTES + BN * BK * 2;
  // 1 KB pieces of A and B that a wave loads of each stage
  static constexpr int NA = ABYTES / 1024 / WAVES, NB = (STAGE - ABYTES) / 1024 / WAVES;
  static constexpr bool A_ROWS = (BM & (BM - 1)) == 0;  // the XOR of row-contiguous A needs it
  static constexpr int FLIGHT = (RING - 2) * (NA + NB);  // loads in flight past the stage waited for
  static_assert(NA * WAVES * 1024 == ABYTES && NB * WAVES * 1024 == STAGE - ABYTES && RING * STAGE <= 160 * 1024);
};
using Cfg128 = PipeCfg<8, 4, 2, 2, 64, 3>;     // 256 x 128
using Cfg128K32 = PipeCfg<8, 4, 2, 2, 32, 6>;  // ... for an odd number of 32s of K
using Cfg256 = PipeCfg<8, 2, 4, 2, 32, 5>;     // 256 x 256
using Cfg192 = PipeCfg<8, 2, 3, 2, 64, 2>;     // 192 x 256, K-contiguous A only
// Products of at most one of these per CU.  They are bound by latency (one
// step: a barrier, an LDS read and 4 dependent products) and by what one CU
// draws from L2, so stages are deep (6 - 8 of 16 - 24 KB) and 128 x 128 and 64 x
// 128 take 8 waves, two per SIMD: with 4 waves the former is 10 - 15 % slower.
using CfgS128 = PipeCfg<8, 4, 1, 2, 64, 4>;  // 128 x 128
using CfgS64 = PipeCfg<8, 2, 1, 1, 64, 6>;   // 64 x 128
using CfgS32 = PipeCfg<4, 2, 1, 1, 64, 8>;   // 64 x 64

typedef int i32x4 __attribute__((ext_vector_type(4)));

// Buffer resource words over [base, base + bytes) (make_rsrc of common.h).
__device__ __forceinline__ i32x4 rsrc_words(const void* base, uint32_t bytes) {
  const uint64_t a = (uint64_t)base;
  return i32x4{(int)(uint32_t)a, (int)((a >> 32) & 0xffff), (int)bytes, 0x00020000};
}

// 64 lanes x 16 bytes from the resource at voff + soff to LDS at byte `lds`
// plus 16 lane.  Written in assembly because the compiler, which cannot tell
// ring slots apart, would wait for every such load before the next
// transposing LDS read; it has no register output, and the waits on vmcnt
// before the barriers below are the ones that its readers need.
__device__ __forceinline__ void load_to_lds(i32x4 rs, int voff, int soff, uint32_t lds) {
  asm volatile(
      "s_mov_b32 m0, %0\n\t"
      "s_nop 0\n\t"
      "buffer_load_dwordx4 %1, %2, %3 offen lds" ::"s"(lds),
      "v"(voff), "s"(rs), "s"(soff)
      : "memory", "m0");
}

struct PipeOp {
  const bf16_t* p1;
  const bf16_t* p2;
  long ld;
};
struct PipeJob {
  PipeOp a, b;
  void* c;
  long ldc;
};
struct PipeJobs {
  PipeJob j[kGemmMaxJobs];
};

// One operand's tile of a stage (ROWS rows, BK k).
template <bool KC, int ROWS, int BK>
struct Operand {
  static constexpr int RB = KC ? BK * 2 : ROWS * 2;  // bytes of an LDS row
  static constexpr int CPR = RB / 16;                // its 16-byte chunks
  // XOR applied to the chunk index of LDS row i: 16 rows' equal chunks (KC) or
  // four rows' 64-byte groups then cover 256 bytes
  static __device__ __forceinline__ int swz(int i) {
    if constexpr (KC) return RB == 64 ? (i >> 2) & 3 : (i >> 1) & 7;
    return RB == 128 ? (i & 2) << 1 : (i & 3) << 2;
  }
  i32x4 r1, r2;
  long ld;

  // Resources from the tile's first row (or column), sized to each K segment.
  __device__ __forceinline__ void init(const PipeOp& op, int row0, int nrows, int K1, int K) {
    ld = op.ld;
    auto rsrc = [&](const bf16_t* p, int kseg) {
      const long ext = KC ? (long)(nrows - row0 - 1) * ld + kseg : (long)(kseg - 1) * ld + (nrows - row0);
      return rsrc_words(KC ? p + (long)row0 * ld : p + row0, (uint32_t)(kseg > 0 && ext > 0 ? ext * 2 : 0));
    };
    r1 = rsrc(op.p1, K1);
    r2 = rsrc(op.p2, K - K1);
  }
  // Byte offset of this lane's chunk of 1 KB piece `u` of a stage; rows past
  // the operand's end read its last ones (their products are not stored).
  __device__ __forceinline__ int voff(int u, int row0, int nrows, int lane) const {
    const int i = u * (64 / CPR) + lane / CPR, c = lane % CPR;  // LDS row, chunk
    if constexpr (KC) {
      const int r = min(row0 + i, nrows - 1) - row0;
      return (int)((long)r * ld * 2) + ((c ^ swz(i)) << 4);
    } else {
      const int r = min(row0 + ((c ^ swz(i)) << 3), nrows - 8) - row0;
      return (int)(((long)i * ld + r) * 2);
    }
  }
  __device__ __forceinline__ int soff(int k) const { return (int)(KC ? (long)k * 2 : (long)k * ld * 2); }
};

// Fragments (A layout of common.h) of rows m0 + 32 i, i < T, K slice h of 16.
template <bool KC, int ROWS, int T, int BK>
struct Frags {
  using Op = Operand<KC, ROWS, BK>;
  static constexpr int RB = Op::RB;
  int off[KC ? BK / 16 : T];
  __device__ __forceinline__ Frags(int m0, int lane) {
    if constexpr (KC) {
      const int r = lane & 31, g = lane >> 5;
#pragma unroll
      for (int h = 0; h < BK / 16; ++h) off[h] = (m0 + r) * RB + (((2 * h + g) ^ Op::swz(r)) << 4);
    } else {  // lds_frag_T<false, false> of common.h
      const int q = lane >> 4, j = lane & 15, x = j >> 2;
#pragma unroll
      for (int i = 0; i < T; ++i)
        off[i] = (8 * (q >> 1) + x) * RB + (((m0 / 32 + i) ^ (Op::swz(x) >> 2)) << 6) + 32 * (q & 1) + 8 * (j & 3);
    }
  }
  __device__ __forceinline__ void get(bf16x8 (&f)[T], const uint8_t* tile, int h) const {
#pragma unroll
    for (int i = 0; i < T; ++i) {
      if constexpr (KC) {
        f[i] = *reinterpret_cast<const bf16x8*>(tile + off[h] + 32 * i * RB);
      } else {
        const uint8_t* p = tile + off[i] + 16 * h * RB;
        const v4i16 lo = lds_read_tr16(reinterpret_cast<const bf16_t*>(p));
        const v4i16 hi = lds_read_tr16(reinterpret_cast<const bf16_t*>(p + 4 * RB));
        typedef short v8i16 __attribute__((ext_vector_type(8)));
        const v8i16 v = __builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7);
        f[i] = __builtin_bit_cast(bf16x8, v);
      }
    }
  }
};

}  // namespace

// Tile (m, n) of rank r and back: columns in bands of 4, row by row inside a
// band, so that the tiles of consecutive ranks share operand panels.
struct TileGrid {
  int tiles_m, tiles_n;
  __host__ __device__ void tile_of(int r, int& m, int& n) const {
    const int band = r / (tiles_m * 4), rest = tiles_n - band * 4, width = rest < 4 ? rest : 4;
    const int i = r - band * tiles_m * 4;
    m = i / width;
    n = band * 4 + i % width;
  }
  __host__ __device__ int rank_of(int m, int n) const {
    const int band = n / 4, rest = tiles_n - band * 4, width = rest < 4 ? rest : 4;
    return band * tiles_m * 4 + m * width + n % 4;
  }
};

// K ranges: workgroup w takes steps [w per, (w + 1) per) of the list (tile, K
// step), nk steps a tile (the last ones empty where K has fewer).  Workgroups
// whose ranges start at the same K step walk the same rows of K together; they
// are nk / gcd(per, nk) apart, on one XCD where that is a multiple of 8, and
// their tiles `stride` = per / gcd(per, nk) apart in the list.  The list therefore holds the tiles of ranks 0, 1, 2, .. `stride`
// places apart: those workgroups' tiles share panels.  2816 x 1024 over 16384
// tokens: 160 us for the kernel with the tiles listed row by row, 92 so.
struct Ranges {
  int per, stride, nk;
  __host__ __device__ int rank_of(int t, int tiles) const {  // of the list's tile t
    const int r = t % stride, extra = tiles % stride;
    return r * (tiles / stride) + (r < extra ? r : extra) + t / stride;
  }
  __host__ __device__ int tile_at(int q, int tiles) const {  // rank q's place in the list
    const int base = tiles / stride, extra = tiles % stride, big = extra * (base + 1);
    return q < big ? q % (base + 1) * stride + q / (base + 1)
                   : (q - big) % base * stride + extra + (q - big) / base;
  }
};

// OUT: 0 = fp32 C, 1 = bf16 C, one tile of one job per workgroup; 2 = fp32
// partials over Ranges: workgroup w's sum over its share of the list's tile t
// goes to partial w + t (unique: a later workgroup never holds an earlier
// tile).
template <class C, bool AKC, bool BKC, int OUT>
__global__ __launch_bounds__(C::NT, C::WAVES == 8 ? 2 : 1) void gemm_pipe_kernel(PipeJobs jobs, int M, int N, int K, int K1, int tiles_m,
                                                           int tiles_n, Ranges rg, float* __restrict__ ws) {
  __shared__ __align__(1024) uint8_t ring[C::RING * C::STAGE];
  const uint32_t ring0 = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) void*)ring;  // LDS byte address
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int wm = wave % C::WM * (32 * C::TM), wn = wave / C::WM * (32 * C::TN);
  constexpr int BK = C::BK;
  // where both operands are row-contiguous, rows of K past the last one are out of their resources and read as zeros
  const int nk = (K + BK - 1) / BK, tiles = tiles_m * tiles_n;
  const Frags<AKC, C::BM, C::TM, BK> fa(wm, lane);
  const Frags<BKC, C::BN, C::TN, BK> fb(wn, lane);

  int w = blockIdx.x, pos, end;  // this workgroup's steps: pos .. end
  const PipeJob* job = &jobs.j[0];
  if constexpr (OUT == 2) {
    pos = w * rg.per;
    end = min(pos + rg.per, tiles * rg.nk);
  } else {
    w = xcd_remap(w, gridDim.x);
    job = &jobs.j[w / tiles];
    pos = w % tiles * nk;
    end = pos + nk;
  }
  while (pos < end) {
    const int len = OUT == 2 ? rg.nk : nk;
    const int t = pos / len, kb = pos - t * len, share = min(len - kb, end - pos);
    const int n = OUT == 2 ? min(share, nk - kb) : share;  // steps that K has (none: a partial of zeros)
    int tm, tn;
    TileGrid{tiles_m, tiles_n}.tile_of(OUT == 2 ? rg.rank_of(t, tiles) : t, tm, tn);
    const int m0 = tm * C::BM, n0 = tn * C::BN;
    Operand<AKC, C::BM, BK> A;
    Operand<BKC, C::BN, BK> B;
    A.init(job->a, m0, M, K1, K);
    B.init(job->b, n0, N, K1, K);
    int va[C::NA], vb[C::NB];
#pragma unroll
    for (int i = 0; i < C::NA; ++i) va[i] = A.voff(wave + C::WAVES * i, m0, M, lane);
#pragma unroll
    for (int i = 0; i < C::NB; ++i) vb[i] = B.voff(wave + C::WAVES * i, n0, N, lane);
    const i32x4 none = rsrc_words(jobs.j[0].a.p1, 0);
    f32x16 acc[C::TM][C::TN];
#pragma unroll
    for (int i = 0; i < C::TM; ++i)
#pragma unroll
      for (int j = 0; j < C::TN; ++j) acc[i][j] = f32x16{};

    // stage s of this part into ring slot `slot`; past the last one an empty
    // resource keeps the number of loads in flight the same
    auto load = [&](int s, int slot) {
      const int k = (kb + s) * BK;
      const bool live = s < n, second = k >= K1;
      const i32x4 ra = live ? (second ? A.r2 : A.r1) : none, rb = live ? (second ? B.r2 : B.r1) : none;
      const int ks = live ? (second ? k - K1 : k) : 0;
      const uint32_t p = ring0 + slot * C::STAGE + wave * 1024;
#pragma unroll
      for (int i = 0; i < C::NA; ++i) load_to_lds(ra, va[i], A.soff(ks), p + i * C::WAVES * 1024);
#pragma unroll
      for (int i = 0; i < C::NB; ++i) load_to_lds(rb, vb[i], B.soff(ks), p + C::ABYTES + i * C::WAVES * 1024);
    };
    auto products = [&](const bf16x8 (&a)[C::TM], const bf16x8 (&b)[C::TN]) {
#pragma unroll
      for (int i = 0; i < C::TM; ++i)
#pragma unroll
        for (int j = 0; j < C::TN; ++j) acc[i][j] = mfma32(a[i], b[j], acc[i][j]);
    };
#pragma unroll
    for (int s = 0; s < C::RING - 1; ++s) load(s, s);
    asm volatile("s_waitcnt vmcnt(%0)\n\ts_barrier" ::"n"(C::FLIGHT) : "memory");
    bf16x8 a0[C::TM], b0[C::TN], a1[C::TM], b1[C::TN];
    fa.get(a0, ring, 0);
    fb.get(b0, ring + C::ABYTES, 0);
    int slot = 0;
    for (int s = 0; s < n; ++s) {
      const uint8_t* cur = ring + slot * C::STAGE;
      fa.get(a1, cur, 1);
      fb.get(b1, cur + C::ABYTES, 1);
      load(s + C::RING - 1, slot == 0 ? C::RING - 1 : slot - 1);
      __builtin_amdgcn_sched_barrier(0);
      products(a0, b0);
      __builtin_amdgcn_sched_barrier(0);
      if constexpr (BK == 64) {
        fa.get(a0, cur, 2);
        fb.get(b0, cur + C::ABYTES, 2);
        __builtin_amdgcn_sched_barrier(0);
        products(a1, b1);
        __builtin_amdgcn_sched_barrier(0);
        fa.get(a1, cur, 3);
        fb.get(b1, cur + C::ABYTES, 3);
        __builtin_amdgcn_sched_barrier(0);
        products(a0, b0);
        __builtin_amdgcn_sched_barrier(0);
      }
      // stage s + 1 is in LDS, and every wave has read stage s (its slot is loaded from the next step on)
      asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" ::"n"(C::FLIGHT) : "memory");
      slot = slot == C::RING - 1 ? 0 : slot + 1;
      fa.get(a0, ring + slot * C::STAGE, 0);
      fb.get(b0, ring + slot * C::STAGE + C::ABYTES, 0);
      __builtin_amdgcn_sched_barrier(0);
      products(a1, b1);
      __builtin_amdgcn_sched_barrier(0);
    }

    // the late loads (zeros, past the last stage) are in LDS before its next user's
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");

    // acc[i][j][v] = C(m0 + wm + 32 i + acc_row(lane / 32, v), n0 + wn + 32 j + lane % 32)
    const int g = lane >> 5, col = lane & 31;
    // Stores go through a resource based at the tile: one lane offset, the
    // row and column of a register as a scalar one (64-bit addresses of 64 or
    // 128 stores would be computed before the K loop and spill).
    const int esize = OUT == 1 ? 2 : 4;
    const long ldo = OUT == 2 ? (long)C::BN : job->ldc;
    char* base;
    if constexpr (OUT == 2)
      base = reinterpret_cast<char*>(ws + (long)(w + t) * (C::BM * C::BN));
    else
      base = reinterpret_cast<char*>(job->c) + ((long)m0 * ldo + n0) * esize;
    const int rows = OUT == 2 ? C::BM : M - m0, cols = OUT == 2 ? C::BN : N - n0;
    // ends with the last row of C: rows past it are dropped by the resource, columns by the test
    const __amdgpu_buffer_rsrc_t rc =
        make_rsrc(base, (uint32_t)(((long)(min(rows, C::BM) - 1) * ldo + min(cols, C::BN)) * esize));
    const int voff = (int)(((long)(wm + 4 * g) * ldo + wn + col) * esize);
#pragma unroll
    for (int j = 0; j < C::TN; ++j) {
      if (wn + 32 * j + col < cols) {
#pragma unroll
        for (int i = 0; i < C::TM; ++i)
#pragma unroll
          for (int v = 0; v < 16; ++v) {
            const int soff = (int)(((32 * i + 8 * (v >> 2) + (v & 3)) * ldo + 32 * j) * esize);
            if constexpr (OUT == 1)
              __builtin_amdgcn_raw_buffer_store_b16((short)f32_to_bf16(acc[i][j][v]), rc, voff, soff, 0);
            else
              __builtin_amdgcn_raw_buffer_store_b32(__float_as_uint(acc[i][j][v]), rc, voff, soff, 0);
          }
      }
    }
    pos += share;
    // no wave loads the next part's stages over this one's reads
    if (pos < end) asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
  }
}

// Sum of the partials of elements (m, n .. n + 3), in workgroup order.
template <class C>
struct RangeSum {
  const float* ws;
  TileGrid tg;
  Ranges rg;
  __device__ __forceinline__ f32x4 get(int m, int n) const {
    const int t = rg.tile_at(tg.rank_of(m / C::BM, n / C::BN), tg.tiles_m * tg.tiles_n);
    const int w0 = t * rg.nk / rg.per, cnt = ((t + 1) * rg.nk - 1) / rg.per - w0 + 1;
    const float* p = ws + (long)(w0 + t) * (C::BM * C::BN) + m % C::BM * C::BN + n % C::BN;
    f32x4 s = f32x4{};
    for (int i0 = 0; i0 < cnt; i0 += 4) {  // four loads in flight
      f32x4 x[4];
#pragma unroll
      for (int e = 0; e < 4; ++e)
        x[e] = *reinterpret_cast<const f32x4*>(p + (long)min(i0 + e, cnt - 1) * (C::BM * C::BN));
#pragma unroll
      for (int e = 0; e < 4; ++e)
        if (i0 + e < cnt) {
#pragma unroll
          for (int q = 0; q < 4; ++q) s[q] += x[e][q];
        }
    }
    return s;
  }
};

template <class C, bool F32>
__global__ __launch_bounds__(256) void gemm_range_reduce_kernel(RangeSum<C> rs, void* __restrict__ c, long ldc, int M,
                                                                int N) {
  const long i = ((long)blockIdx.x * 256 + threadIdx.x) * 4;
  if (i >= (long)M * N) return;
  const int m = (int)(i / N), n = (int)(i % N);
  const f32x4 s = rs.get(m, n);
  if constexpr (F32) {
    *reinterpret_cast<f32x4*>(reinterpret_cast<float*>(c) + m * ldc + n) = s;
  } else {
    bf16x4 o;
#pragma unroll
    for (int e = 0; e < 4; ++e) o[e] = (__bf16)s[e];
    *reinterpret_cast<bf16x4*>(reinterpret_cast<bf16_t*>(c) + m * ldc + n) = o;
  }
}

// The gate epilogue of gemm_reduce_gate_kernel (gemm.hip) on range partials.
template <class C>
__global__ __launch_bounds__(256) void gemm_range_gate_kernel(RangeSum<C> rs, int M, int N, const bf16_t* __restrict__ w,
                                                              const float* __restrict__ s, bf16_t* __restrict__ c,
                                                              float* __restrict__ part) {
  __shared__ float red[256];
  const int tid = threadIdx.x;
  const long i = ((long)blockIdx.x * 256 + tid) * 4;
  float acc = 0.f;
  if (i < (long)M * N) {
    const f32x4 v = rs.get((int)(i / N), (int)(i % N));
    const float sc = *s;
    const bf16x4 wb = *reinterpret_cast<const bf16x4*>(w + i);
    bf16x4 o;
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      o[e] = (__bf16)(sc * v[e]);
      acc = fmaf(v[e], (float)wb[e], acc);
    }
    *reinterpret_cast<bf16x4*>(c + i) = o;
  }
  red[tid] = acc;
  __syncthreads();
  for (int o = 128; o > 0; o >>= 1) {
    if (tid < o) red[tid] += red[tid + o];
    __syncthreads();
  }
  if (tid == 0) part[blockIdx.x] = red[0];
}

template <class C>
static int pipe_tiles(int M, int N) {
  return (M + C::BM - 1) / C::BM * ((N + C::BN - 1) / C::BN);
}

static PipeJobs pipe_jobs(const GemmLaunch& g) {
  PipeJobs pj{};
  for (int j = 0; j < g.njobs; ++j) {
    const GemmJob& s = g.job[j];
    pj.j[j].a = PipeOp{(const bf16_t*)s.a.p1, (const bf16_t*)(s.a.p2 ? s.a.p2 : s.a.p1), s.a.ld};
    pj.j[j].b = PipeOp{(const bf16_t*)s.b.p1, (const bf16_t*)(s.b.p2 ? s.b.p2 : s.b.p1), s.b.ld};
    pj.j[j].c = s.c;
    pj.j[j].ldc = s.ldc;
  }
  return pj;
}

// Whole tiles, one per workgroup: K in whole steps, and 256 x 128 tiles for
// more than half of the CUs; below that the small tiles also fit the chip once
// (2042 x 1024 over 1024, 64 against 128 tiles: 9.2 us with the latter).
bool gemm_pipe_ok(const GemmLaunch& g) {
  return g.K % 32 == 0 && g.K1 % 32 == 0 && g.M >= 256 && g.N >= 128 && pipe_tiles<Cfg128>(g.M, g.N) * g.njobs >= 144;
}

template <class C>
static hipError_t pipe_direct(const GemmLaunch& g, const char* name, hipStream_t st) {
  const int tiles_m = (g.M + C::BM - 1) / C::BM, tiles_n = (g.N + C::BN - 1) / C::BN;
  const dim3 grid((unsigned)(tiles_m * tiles_n * g.njobs));
  const PipeJobs pj = pipe_jobs(g);
  auto run = [&](auto kernel) {
    NAYLIS_TIMED(name, st, hipLaunchKernelGGL(kernel, grid, dim3(C::NT), 0, st, pj, g.M, g.N, g.K, std::min(g.K1, g.K),
                                              tiles_m, tiles_n, Ranges{}, (float*)nullptr));
  };
  const bool ak = g.job[0].a.kcontig, bk = g.job[0].b.kcontig, f32 = g.out == kGemmOutF32;
  if (ak && bk)
    f32 ? run(gemm_pipe_kernel<C, true, true, 0>) : run(gemm_pipe_kernel<C, true, true, 1>);
  else if (ak)
    f32 ? run(gemm_pipe_kernel<C, true, false, 0>) : run(gemm_pipe_kernel<C, true, false, 1>);
  else if constexpr (!C::A_ROWS)
    return hipErrorInvalidValue;
  else if (bk)
    f32 ? run(gemm_pipe_kernel<C, false, true, 0>) : run(gemm_pipe_kernel<C, false, true, 1>);
  else
    f32 ? run(gemm_pipe_kernel<C, false, false, 0>) : run(gemm_pipe_kernel<C, false, false, 1>);
  return hipGetLastError();
}

hipError_t launch_gemm_pipe(const GemmLaunch& g, const char* name, hipStream_t st) {
  // 256 x 256 tiles do a step's work at 0.87 of the time of two 256 x 128 ones:
  // taken unless the smaller tiles save a round (2042 x 5632 over 2048, 352 tiles
  // against 176: 59 and 52 us; 4096 x 1536 over 1536, 192 against 96: 23 and 42)
  const int r128 = (pipe_tiles<Cfg128>(g.M, g.N) * g.njobs + 255) / 256;
  const int r256 = (pipe_tiles<Cfg256>(g.M, g.N) * g.njobs + 255) / 256;
  const bool k64 = g.K % 64 == 0 && g.K1 % 64 == 0;
  // 192 x 256 tiles, where they take fewer rounds than the small ones and no
  // more than the large: 2 x 2042 x 2816 over 1024 (352, 242 and 176 tiles)
  // 33.2 us with 256 x 128, 27.4 with these, 30.2 with 256 x 256; 3 x 4096 x
  // 2816 (1056, 726, 528) 77 against 90 with 256 x 256
  const int r192 = (pipe_tiles<Cfg192>(g.M, g.N) * g.njobs + 255) / 256;
  if (g.job[0].a.kcontig && k64 && r192 * 1.35 < r128 && r192 <= r256) return pipe_direct<Cfg192>(g, name, st);
  if (2 * r256 * 0.87 < r128) return pipe_direct<Cfg256>(g, name, st);
  return k64 ? pipe_direct<Cfg128>(g, name, st) : pipe_direct<Cfg128K32>(g, name, st);
}

// The smallest of the small tiles that needs at most one workgroup per CU: the
// LDS of one holds a CU, and a second round costs as much as the first (512 x
// 2816 over 1024: 176 tiles of 64 x 128 take 9.5 us, 352 of 64 x 64 14.5).
// Against gemm.hip, 2 - 3 workgroups per CU with padded tiles and one stage
// ahead: 512 x 1024 over 2816 14.7 against 16.4 us, 1021 x 1536 over 1536 11.8
// against 15.6, 2042 x 2048 over 2048 20.8 against 25.9; at K 512 level (2042 x
// 512: 5.9 against 6.3), there launch and first loads are all.
bool gemm_small_ok(const GemmLaunch& g) {
  const bool k_ok = g.K % 64 == 0 && g.K1 % 64 == 0;
  const bool rows = !g.job[0].a.kcontig && !g.job[0].b.kcontig && g.K1 == g.K;
  // with two row-contiguous operands a full chip of 128 x 128 tiles is bound by
  // LDS reads: the 64 x 64 blocks per wave of gemm.hip's tile read a third less
  // (2048 x 2048 over 2008: 27.1 against 29.3 us)
  return (k_ok || rows) && g.M >= 8 && g.N >= 8 && pipe_tiles<CfgS128>(g.M, g.N) * g.njobs <= (rows ? 255 : 256);
}

bool gemm_small_fills(int M, int N) {
  const int s32 = pipe_tiles<CfgS32>(M, N), s64 = pipe_tiles<CfgS64>(M, N), s128 = pipe_tiles<CfgS128>(M, N);
  if (s32 <= 256) return s32 >= 128;
  return s64 <= 256 || s128 <= 255;  // (gemm_small_ok: not a full chip of 128 x 128)
}

hipError_t launch_gemm_small(const GemmLaunch& g, const char* name, hipStream_t st) {
  if (pipe_tiles<CfgS32>(g.M, g.N) * g.njobs <= 256) return pipe_direct<CfgS32>(g, name, st);
  if (pipe_tiles<CfgS64>(g.M, g.N) * g.njobs <= 256) return pipe_direct<CfgS64>(g, name, st);
  return pipe_direct<CfgS128>(g, name, st);
}

// K ranges over one workgroup per CU.
constexpr int kRangeWgs = 256;

// The list's steps per tile are rounded up to what cuts it into 256 equal
// ranges, so that their starts fall on few distinct K steps.
static Ranges ranges_of(int M, int N, int K) {
  const int tiles = pipe_tiles<Cfg128>(M, N), unit = kRangeWgs / std::gcd(tiles, kRangeWgs);
  Ranges r;
  r.nk = ((K + Cfg128::BK - 1) / Cfg128::BK + unit - 1) / unit * unit;
  r.per = (int)((long)tiles * r.nk / kRangeWgs);
  r.stride = r.per / std::gcd(r.per, r.nk);
  return r;
}

// At least 1024 rows of K a workgroup (at 512 - 704 the fixed costs, 128 KB of partials
// per workgroup above all, leave it level with gemm.hip's splits or 10 - 20 %
// behind), few enough tiles that K has to be cut at all, and at most 4 % of the
// steps empty (unaligned ranges of 10016 tokens, 1024 x 1024: 47 us against 35
// with gemm.hip's splits).  Nor an odd number of tiles: the 256 ranges then start
// at 256 distinct K steps, and no two workgroups walk the same rows together
// (16384 tokens, 1152 x 1152, 45 tiles: 88 us against 71 with splits, 1032 x 1032
// 114 against 70, 1152 x 2304 164 against 123; at 128 starts, 2 mod 4 tiles, they
// are between 25 % ahead, 896 x 2432, and 3 - 8 % behind, 18 tiles).
bool gemm_ranges_ok(int M, int N, int K) {
  const int tiles = pipe_tiles<Cfg128>(M, N);
  if (K <= 0 || M < 256 || N < 128 || M % 8 || N % 8 || tiles >= 144 || tiles % 2) return false;
  const Ranges r = ranges_of(M, N, K);
  return r.per >= 16 && ((long)r.nk * Cfg128::BK - K) * 25 <= K;
}

size_t gemm_ranges_ws_bytes(int M, int N, int K) {
  return (size_t)(kRangeWgs + pipe_tiles<Cfg128>(M, N)) * Cfg128::BM * Cfg128::BN * sizeof(float);
}

hipError_t launch_gemm_ranges(const GemmLaunch& g, const char* name, hipStream_t st) {
  using C = Cfg128;
  const TileGrid tg{(g.M + C::BM - 1) / C::BM, (g.N + C::BN - 1) / C::BN};
  const Ranges rg = ranges_of(g.M, g.N, g.K);
  NAYLIS_TIMED(name, st,
               hipLaunchKernelGGL((gemm_pipe_kernel<C, false, false, 2>), dim3(kRangeWgs), dim3(C::NT), 0, st,
                                  pipe_jobs(g), g.M, g.N, g.K, g.K, tg.tiles_m, tg.tiles_n, rg, (float*)g.ws));
  const RangeSum<C> rs{(const float*)g.ws, tg, rg};
  const dim3 grid((unsigned)(((long)g.M * g.N / 4 + 255) / 256));
  if (g.gate_w != nullptr)
    NAYLIS_TIMED("gemm_reduce", st,
                 hipLaunchKernelGGL(gemm_range_gate_kernel<C>, grid, dim3(256), 0, st, rs, g.M, g.N,
                                    (const bf16_t*)g.gate_w, g.gate_s, (bf16_t*)g.job[0].c, g.gate_part));
  else if (g.out == kGemmOutF32)
    NAYLIS_TIMED("gemm_reduce", st,
                 hipLaunchKernelGGL((gemm_range_reduce_kernel<C, true>), grid, dim3(256), 0, st, rs, g.job[0].c,
                                    g.job[0].ldc, g.M, g.N));
  else
    NAYLIS_TIMED("gemm_reduce", st,
                 hipLaunchKernelGGL((gemm_range_reduce_kernel<C, false>), grid, dim3(256), 0, st, rs, g.job[0].c,
                                    g.job[0].ldc, g.M, g.N));
  return hipGetLastError();
}

}  // namespace naylis
