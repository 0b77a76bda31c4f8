// Chebyshev evolution kernels for gfx950: CSR SpMV/SpMM and the three-term
// recurrence with compensated accumulation.
//
// Row sums use TwoProduct on every real product and Neumaier's improved Kahan
// summation (Neumaier 1974) for the running sum, so the order of magnitudes
// along a row does not matter.  The batched form keeps n_rhs right-hand sides
// RHS-contiguous (element (row, j) at row*n_rhs + j): with n_rhs = 32 one
// wave64 covers two rows, every column gather reads 256 contiguous bytes, and
// the recurrence update and the Kahan accumulation are fused into the SpMM
// epilogue, so one launch per Chebyshev term touches A, T_k, T_{k-1}, the
// accumulator and its compensation exactly once.
#include "qsim_internal.hpp"
#include <utility>

namespace qsim {

// Nonzeros whose column indices, values and gathers are issued together
// before any of their products is accumulated: the gathers of a row are
// independent, so batching them overlaps their latencies (the summation
// order, and so every result bit, is unchanged).  Measured per Chebyshev
// term on the 22-qubit chain at 32 RHS: 1 -> 9.6 ms, 2 -> 6.9, 4 -> 6.2,
// 8 -> 6.9, 16 -> 8.0 (more in flight costs occupancy).
constexpr int kGather = 4;

// Neumaier step: s + c holds the running sum with the low part in c.
__device__ __forceinline__ void neu_add(float& s, float& c, float x) {
  const float t = s + x;
  if (fabsf(s) >= fabsf(x)) c += (s - t) + x;
  else c += (x - t) + s;
  s = t;
}

// Adds the complex product v * xj to (sr + cr, si + ci) with TwoProduct
// errors folded into the compensation terms.
__device__ __forceinline__ void cmac_acc(float2 v, float2 xj, float& sr, float& cr, float& si,
                                         float& ci) {
  float p, e;
  two_prod(v.x, xj.x, p, e); neu_add(sr, cr, p); cr += e;
  two_prod(-v.y, xj.y, p, e); neu_add(sr, cr, p); cr += e;
  two_prod(v.x, xj.y, p, e); neu_add(si, ci, p); ci += e;
  two_prod(v.y, xj.x, p, e); neu_add(si, ci, p); ci += e;
}

__global__ __launch_bounds__(kThreads) void k_spmv(const int32_t* __restrict__ rp,
                                                   const int32_t* __restrict__ ci,
                                                   const float2* __restrict__ val, int64_t n_rows,
                                                   const float2* __restrict__ x,
                                                   float2* __restrict__ y, float2 alpha,
                                                   float2 beta) {
  const int64_t row = (int64_t)blockIdx.x * kThreads + threadIdx.x;
  if (row >= n_rows) return;
  float sr = 0.f, cr = 0.f, si = 0.f, cc = 0.f;
  const int32_t b = rp[row], e = rp[row + 1];
  int32_t k = b;
  for (; k + kGather <= e; k += kGather) {
    int32_t c[kGather];
    float2 v[kGather], xs[kGather];
#pragma unroll
    for (int u = 0; u < kGather; ++u) { c[u] = ci[k + u]; v[u] = val[k + u]; }
#pragma unroll
    for (int u = 0; u < kGather; ++u) xs[u] = x[c[u]];
#pragma unroll
    for (int u = 0; u < kGather; ++u) cmac_acc(v[u], xs[u], sr, cr, si, cc);
  }
  for (; k < e; ++k) cmac_acc(val[k], x[ci[k]], sr, cr, si, cc);
  const float2 dot = make_float2(sr + cr, si + cc);
  const float2 r = cmulc(alpha, dot);
  float2 out = r;
  if (beta.x != 0.f || beta.y != 0.f) {
    const float2 yb = cmulc(beta, y[row]);
    out = make_float2(r.x + yb.x, r.y + yb.y);
  }
  y[row] = out;
}

__global__ __launch_bounds__(kThreads) void k_step(const float2* __restrict__ s,
                                                   const float2* __restrict__ tp,
                                                   float2* __restrict__ tn, int64_t n) {
  const int64_t i = (int64_t)blockIdx.x * kThreads + threadIdx.x;
  if (i >= n) return;
  const float2 a = s[i], b = tp[i];
  tn[i] = make_float2(2.f * a.x - b.x, 2.f * a.y - b.y);
}

__global__ __launch_bounds__(kThreads) void k_accum(float2* __restrict__ acc,
                                                    const float2* __restrict__ t, int64_t n,
                                                    float2 c) {
  const int64_t i = (int64_t)blockIdx.x * kThreads + threadIdx.x;
  if (i >= n) return;
  const float2 v = cmulc(c, t[i]);
  const float2 a = acc[i];
  acc[i] = make_float2(a.x + v.x, a.y + v.y);
}

__global__ __launch_bounds__(kThreads) void k_step_accum(const float2* __restrict__ s,
                                                         const float2* __restrict__ tp,
                                                         float2* __restrict__ tn,
                                                         float2* __restrict__ acc, int64_t n,
                                                         float2 c) {
  const int64_t i = (int64_t)blockIdx.x * kThreads + threadIdx.x;
  if (i >= n) return;
  const float2 a = s[i], b = tp[i];
  const float2 t = make_float2(2.f * a.x - b.x, 2.f * a.y - b.y);
  tn[i] = t;
  const float2 v = cmulc(c, t);
  const float2 z = acc[i];
  acc[i] = make_float2(z.x + v.x, z.y + v.y);
}

// ---------------------------------------------------------------- 32 RHS
// The batched term at 32 right-hand sides, the width of one RHS-contiguous
// row (32 x 8 B = 256 B).  One wave owns four consecutive CSR rows: lanes
// 16 q .. 16 q + 15 row r + q, each lane two RHS (one 16-byte load per
// gathered row).  Per nonzero a quarter-wave needs the column index and the
// value (the same for its 16 lanes) and one 256-byte gathered row of T_k, so
// one gather instruction fetches four rows (1 KiB).
//  * Why four rows: the gathers are bound by the number of vector memory
//    instructions in flight, not by their bytes; measured on the 22-qubit
//    chain at 32 RHS (FP64 sums), two rows per wave with 8-byte lanes take
//    4.2 ms per term and four rows with 16-byte lanes 3.7 ms, bit for bit the
//    same result.  2, 4 or 8 gathers in flight per lane measured the same
//    (1 is 5 % slower).
//  * Row data: the wave's four rows are consecutive in the CSR arrays, so it
//    stages them into its own LDS slice with coalesced full-wave loads
//    (nontemporal: the CSR is read once per term) and reads them back as
//    quarter-wave broadcasts.
//  * Row sum, ACC = kAccF64: the product of two FP32 numbers is exact in FP64
//    (24 + 24 bits < 53), so every product is converted and accumulated with
//    FP64 FMAs.  CDNA4 issues FP64 FMA at the non-packed FP32 rate, so this
//    costs 8 VALU operations per complex multiply-add against ~44 for the
//    TwoProduct + Neumaier double-float form (ACC = kAccF32c); the FP64 sum is
//    also the more accurate of the two (53-bit accumulator, exact terms).
//  * Epilogue (both forms): T_{k+1} = 2 scale (A T_k) - T_{k-1}, rounded to
//    complex64 once, and acc += c_k T_{k+1} as a Neumaier pair (acc, comp) in
//    FP32, as in the generic kernel.  T_{k-1}, acc and comp are loaded before
//    the row's gathers and streamed (nontemporal when the 32-RHS block
//    exceeds the MALL), so the cache keeps the gathered rows of T_k.
//  * Block order: order_shift s > 0 hands each XCD contiguous chunks of 2^s
//    rows, chunk x of every group of 8 chunks going to XCD x, so that a
//    gather through a low column bit stays in the XCD's own L2 while all 8
//    XCDs still walk one front through the MALL.  s = 0 is the dispatch
//    order (blocks round-robin over the XCDs).  Shifts 0, 6, 9, 12 and 19
//    measured within 4 % of each other.
constexpr int kAccF64 = 0;
constexpr int kAccF32c = 1;
constexpr int kWaves = kThreads / 64;
constexpr int kRowsPerWave = 4;
constexpr int kLanesPerRow = 64 / kRowsPerWave;            // 16
constexpr int kRhsPerLane = 32 / kLanesPerRow;             // 2
constexpr int kBlockRowsLog2 = 4;                          // 4 waves x 4 rows per workgroup
static_assert(kWaves * kRowsPerWave == 1 << kBlockRowsLog2, "rows per workgroup");
constexpr int kStageNnz = 256;      // nonzeros of a wave's four rows staged per chunk
constexpr int kSpmmOrderShift = 9;
constexpr int kGather32 = 2;        // gathers in flight per lane

typedef float f32x2_t __attribute__((ext_vector_type(2)));
template <bool NT>
__device__ __forceinline__ float2 ld2(const float2* p) {
  if constexpr (NT) {
    const f32x2_t v = __builtin_nontemporal_load(reinterpret_cast<const f32x2_t*>(p));
    return make_float2(v.x, v.y);
  } else {
    return *p;
  }
}
template <bool NT>
__device__ __forceinline__ void st2(float2* p, float2 v) {
  if constexpr (NT) {
    const f32x2_t w = {v.x, v.y};
    __builtin_nontemporal_store(w, reinterpret_cast<f32x2_t*>(p));
  } else {
    *p = v;
  }
}

// Wave-level ordering of LDS writes and reads by other lanes of the same wave.
__device__ __forceinline__ void wave_sync() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// Logical block of this workgroup under the chunked XCD order (a bijection
// on [0, gridDim.x) when gridDim.x is a multiple of 8 * chunk blocks; the
// host passes s = 0 otherwise).
__device__ __forceinline__ int64_t spmm_block(int s) {
  const int64_t b = blockIdx.x;
  if (s <= 0) return b;
  const int g = s > kBlockRowsLog2 ? s - kBlockRowsLog2 : 0;   // log2(blocks per chunk)
  const int64_t xcd = b & 7, i = b >> 3;
  const int64_t grp = i >> g, w = i & ((1ll << g) - 1);
  return ((grp * 8 + xcd) << g) + w;
}

template <int ACC>
struct RowSum;
template <>
struct RowSum<kAccF64> {
  double r = 0.0, i = 0.0;
  __device__ __forceinline__ void add(float2 v, float2 x) { add_d(v.x, v.y, x); }
  // vr, vi: an entry already rounded to complex64, held in FP64
  __device__ __forceinline__ void add_d(double vr, double vi, float2 x) {
    const double xr = x.x, xi = x.y;
    r = __builtin_fma(vr, xr, r);
    r = __builtin_fma(-vi, xi, r);
    i = __builtin_fma(vr, xi, i);
    i = __builtin_fma(vi, xr, i);
  }
  __device__ __forceinline__ void add_r(double vr, float2 x) {
    r = __builtin_fma(vr, (double)x.x, r);
    i = __builtin_fma(vr, (double)x.y, i);
  }
  // scale * sum, rounded once to FP32 after the recurrence update
  __device__ __forceinline__ float2 next(double scale, float2 tp, bool first) const {
    const double wr = r * scale, wi = i * scale;
    if (first) return make_float2((float)wr, (float)wi);
    return make_float2((float)(2.0 * wr - (double)tp.x), (float)(2.0 * wi - (double)tp.y));
  }
};
template <>
struct RowSum<kAccF32c> {
  float sr = 0.f, cr = 0.f, si = 0.f, ci = 0.f;
  __device__ __forceinline__ void add(float2 v, float2 x) { cmac_acc(v, x, sr, cr, si, ci); }
  __device__ __forceinline__ float2 next(double scale_d, float2 tp, bool first) const {
    const float scale = (float)scale_d;
    float p, q, wr, wi;
    two_prod(sr, scale, p, q); wr = p + (q + cr * scale);
    two_prod(si, scale, p, q); wi = p + (q + ci * scale);
    if (first) return make_float2(wr, wi);
    return make_float2(2.f * wr - tp.x, 2.f * wi - tp.y);
  }
};

// Split term (PASS 1 and 2).  For a matrix of N = 2^n rows whose entries
// mostly connect rows that differ either only below bit s or only at and
// above it (a Pauli Hamiltonian's X masks), the SpMM is done in two
// passes, each of whose gathers stay within 2^s (2^(n-s)) neighbouring rows
// of the order it walks, so the gathered 256-byte rows of T_k are reused
// from L2 instead of being fetched again for every row that needs them:
//   PASS 1  rows in natural order, the entries with (row ^ col) < 2^s:
//           w1 = (A_low T_k) rounded to complex64;
//   PASS 2  positions p in order, row r = rot(p) (the low n-s bits of p are
//           the high bits of r), the other entries, stored in p order:
//           w = w1 + A_high T_k (FP64), then the same recurrence epilogue.
// Entries whose mask has bits on both sides of s (at most a few per row)
// go to pass 2 and are gathered from farther away.  On a 22-qubit chain at
// 32 RHS this cuts the bytes fetched per term from 24 GB to 10 GB but gains
// only a few per cent over PASS 0 (the gathers' issue and latency, not their
// bytes, bound both forms), so callers opt in to it.
__device__ __forceinline__ int64_t split_row(int64_t p, int n, int s) {
  const int lo_bits = n - s;
  return ((p & ((int64_t(1) << lo_bits) - 1)) << s) | (p >> lo_bits);
}

// kRhsPerLane complex RHS of one lane: float2 or float4 loads and stores.
template <int EPL>
struct CVec {
  float2 c[EPL];
};
template <bool NT, int EPL>
__device__ __forceinline__ CVec<EPL> ldv(const float2* p) {
  CVec<EPL> r;
  if constexpr (EPL == 1) {
    r.c[0] = ld2<NT>(p);
  } else {
    typedef float f32x4_t __attribute__((ext_vector_type(4)));
    f32x4_t v;
    if constexpr (NT) v = __builtin_nontemporal_load(reinterpret_cast<const f32x4_t*>(p));
    else v = *reinterpret_cast<const f32x4_t*>(p);
    r.c[0] = make_float2(v.x, v.y);
    r.c[1] = make_float2(v.z, v.w);
  }
  return r;
}
template <bool NT, int EPL>
__device__ __forceinline__ void stv(float2* p, const CVec<EPL>& r) {
  if constexpr (EPL == 1) {
    st2<NT>(p, r.c[0]);
  } else {
    typedef float f32x4_t __attribute__((ext_vector_type(4)));
    const f32x4_t v = {r.c[0].x, r.c[0].y, r.c[1].x, r.c[1].y};
    if constexpr (NT) __builtin_nontemporal_store(v, reinterpret_cast<f32x4_t*>(p));
    else *reinterpret_cast<f32x4_t*>(p) = v;
  }
}

template <int ACC, bool NT, int PASS>
__global__ __launch_bounds__(kThreads) void k_cheb_spmm32(
    const int32_t* __restrict__ rp, const int32_t* __restrict__ ci, const float2* __restrict__ val,
    int64_t n_rows, double scale, const float2* __restrict__ tc, float2* __restrict__ tpn,
    float2* __restrict__ acc, float2* __restrict__ comp, float2* __restrict__ w1, float2 c,
    int first, int order_shift, int n_bits, int split) {
  constexpr int RW = kRowsPerWave, LPR = kLanesPerRow, EPL = kRhsPerLane, G = kGather32;
  __shared__ int32_t s_ci[kWaves][kStageNnz];
  __shared__ float2 s_v[kWaves][kStageNnz];
  const int wave = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
  const int lane = threadIdx.x & 63, qr = lane / LPR, jj = lane % LPR;
  const int64_t pos0 = (spmm_block(order_shift) * kWaves + wave) * RW;   // first row (position)
  if (pos0 >= n_rows) return;
  const int n_here = (int)(n_rows - pos0 < RW ? n_rows - pos0 : RW);
  const int32_t my_rp = lane <= n_here ? rp[pos0 + lane] : 0;
  const char* tcb = reinterpret_cast<const char*>(tc);
  const uint32_t lane_off = (uint32_t)jj * (8u * EPL);
  const int32_t gb = __builtin_amdgcn_readlane(my_rp, 0);        // the wave's entries [gb, ge)
  const int32_t ge = __builtin_amdgcn_readlane(my_rp, n_here);
  const bool live = qr < n_here;
  const int my_r = live ? qr : 0;   // lanes past the last row shadow the first and store nothing
  const int32_t my_b = __shfl(my_rp, my_r), my_e = live ? __shfl(my_rp, my_r + 1) : my_b;
  const int64_t pos = pos0 + my_r;
  const int64_t row = PASS == 2 ? split_row(pos, n_bits, split) : pos;
  const int64_t e_idx = row * 32 + jj * EPL;
  CVec<EPL> tp{}, a{}, k2{}, wv{};
  if constexpr (PASS != 1) {
    tp = ldv<NT, EPL>(tpn + e_idx);
    a = ldv<NT, EPL>(acc + e_idx);
    k2 = ldv<NT, EPL>(comp + e_idx);
    if constexpr (PASS == 2) wv = ldv<NT, EPL>(w1 + e_idx);
  }
  RowSum<ACC> sum[EPL];
  for (int32_t c0 = gb; c0 < ge; c0 += kStageNnz) {
    const int32_t cend = c0 + kStageNnz < ge ? c0 + kStageNnz : ge;
    wave_sync();
    for (int32_t k = c0 + lane; k < cend; k += 64) {
      s_ci[wave][k - c0] = __builtin_nontemporal_load(ci + k);
      s_v[wave][k - c0] = ld2<true>(val + k);
    }
    wave_sync();
    const int32_t lo = my_b > c0 ? my_b : c0, hi = my_e < cend ? my_e : cend;
    const int32_t* sc = s_ci[wave] - c0;
    const float2* sv = s_v[wave] - c0;
    for (int32_t k = lo; k < hi; k += G) {
      CVec<EPL> x[G];
#pragma unroll
      for (int u = 0; u < G; ++u) {
        const int32_t idx = k + u < hi ? k + u : hi - 1;
        // positions past hi gather the row's last entry again (no branch
        // between the loads) and add it with weight 0, an exact no-op
        x[u] = ldv<false, EPL>(
            reinterpret_cast<const float2*>(tcb + ((uint32_t)sc[idx] * 256u + lane_off)));
      }
#pragma unroll
      for (int u = 0; u < G; ++u) {
        const float2 v = k + u < hi ? sv[k + u] : make_float2(0.f, 0.f);
#pragma unroll
        for (int e = 0; e < EPL; ++e) sum[e].add(v, x[u].c[e]);
      }
    }
  }
  if (!live) return;
  if constexpr (PASS == 1) {
    CVec<EPL> o;
#pragma unroll
    for (int e = 0; e < EPL; ++e) o.c[e] = make_float2((float)sum[e].r, (float)sum[e].i);
    stv<NT, EPL>(w1 + e_idx, o);
    return;
  }
  CVec<EPL> tn;
#pragma unroll
  for (int e = 0; e < EPL; ++e) {
    if constexpr (PASS == 2) {
      sum[e].r += (double)wv.c[e].x;
      sum[e].i += (double)wv.c[e].y;
    }
    tn.c[e] = sum[e].next(scale, first ? make_float2(0.f, 0.f) : tp.c[e], first != 0);
    const float2 v = cmulc(c, tn.c[e]);
    neu_add(a.c[e].x, k2.c[e].x, v.x);
    neu_add(a.c[e].y, k2.c[e].y, v.y);
  }
  stv<NT, EPL>(tpn + e_idx, tn);
  stv<NT, EPL>(acc + e_idx, a);
  stv<NT, EPL>(comp + e_idx, k2);
}

// ---------------------------------------------------------------- CSR split
// Splits a CSR of N = 2^n rows at bit s: entries with (row ^ col) < 2^s go
// to the low CSR (rows in natural order), the others to the high CSR, whose
// row p is row rot(p) of the input (split_row).  Both keep each row's entry
// order.  One row (position) per thread: k_split_count sums the per-block
// counts of both outputs, k_split_scan (one workgroup) turns them into block
// offsets, k_split_fill writes row pointers, columns and values.
constexpr int kSplitThreads = 256;

__device__ __forceinline__ int64_t blk_exscan(int64_t v, int64_t* total) {
  __shared__ int64_t wsum[kSplitThreads / 64];
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
  int64_t incl = v;
  for (int d = 1; d < 64; d <<= 1) {
    const int64_t y = __shfl_up(incl, d, 64);
    if (lane >= d) incl += y;
  }
  if (lane == 63) wsum[w] = incl;
  __syncthreads();
  int64_t base = 0, all = 0;
  for (int k = 0; k < kSplitThreads / 64; ++k) {
    if (k < w) base += wsum[k];
    all += wsum[k];
  }
  __syncthreads();
  *total = all;
  return base + incl - v;
}

__device__ __forceinline__ void split_counts(const int32_t* __restrict__ rp,
                                             const int32_t* __restrict__ ci, int64_t i, int n,
                                             int s, int& nlo, int& nhi) {
  nlo = 0;
  for (int32_t k = rp[i]; k < rp[i + 1]; ++k) nlo += ((uint32_t)(ci[k] ^ (int32_t)i) >> s) == 0;
  const int64_t r = split_row(i, n, s);
  nhi = 0;
  for (int32_t k = rp[r]; k < rp[r + 1]; ++k) nhi += ((uint32_t)(ci[k] ^ (int32_t)r) >> s) != 0;
}

__global__ __launch_bounds__(kSplitThreads) void k_split_count(const int32_t* __restrict__ rp,
                                                               const int32_t* __restrict__ ci,
                                                               int64_t n_rows, int n, int s,
                                                               int64_t* __restrict__ bsum) {
  const int64_t i = (int64_t)blockIdx.x * kSplitThreads + threadIdx.x;
  int nlo = 0, nhi = 0;
  if (i < n_rows) split_counts(rp, ci, i, n, s, nlo, nhi);
  int64_t tl, th;
  blk_exscan(nlo, &tl);
  blk_exscan(nhi, &th);
  if (threadIdx.x == 0) {
    bsum[2 * blockIdx.x] = tl;
    bsum[2 * blockIdx.x + 1] = th;
  }
}

__global__ __launch_bounds__(kSplitThreads) void k_split_scan(uint64_t n_blocks,
                                                              int64_t* __restrict__ bsum,
                                                              int64_t* __restrict__ nnz2) {
  int64_t carry[2] = {0, 0};
  for (uint64_t base = 0; base < n_blocks; base += kSplitThreads) {
    const uint64_t b = base + threadIdx.x;
#pragma unroll
    for (int side = 0; side < 2; ++side) {
      const int64_t v = b < n_blocks ? bsum[2 * b + side] : 0;
      int64_t total;
      const int64_t pre = blk_exscan(v, &total);
      if (b < n_blocks) bsum[2 * b + side] = carry[side] + pre;
      carry[side] += total;
    }
  }
  if (threadIdx.x == 0) {
    nnz2[0] = carry[0];
    nnz2[1] = carry[1];
  }
}

__global__ __launch_bounds__(kSplitThreads) void k_split_fill(
    const int32_t* __restrict__ rp, const int32_t* __restrict__ ci, const float2* __restrict__ val,
    int64_t n_rows, int n, int s, const int64_t* __restrict__ boff, int32_t* __restrict__ rp_lo,
    int32_t* __restrict__ ci_lo, float2* __restrict__ val_lo, int32_t* __restrict__ rp_hi,
    int32_t* __restrict__ ci_hi, float2* __restrict__ val_hi) {
  const int64_t i = (int64_t)blockIdx.x * kSplitThreads + threadIdx.x;
  int nlo = 0, nhi = 0;
  if (i < n_rows) split_counts(rp, ci, i, n, s, nlo, nhi);
  int64_t tl, th;
  const int64_t olo = boff[2 * blockIdx.x] + blk_exscan(nlo, &tl);
  const int64_t ohi = boff[2 * blockIdx.x + 1] + blk_exscan(nhi, &th);
  if (i >= n_rows) return;
  rp_lo[i] = (int32_t)olo;
  rp_hi[i] = (int32_t)ohi;
  if (i == n_rows - 1) {
    rp_lo[n_rows] = (int32_t)(olo + nlo);
    rp_hi[n_rows] = (int32_t)(ohi + nhi);
  }
  int64_t o = olo;
  for (int32_t k = rp[i]; k < rp[i + 1]; ++k)
    if (((uint32_t)(ci[k] ^ (int32_t)i) >> s) == 0) {
      ci_lo[o] = ci[k];
      val_lo[o] = val[k];
      ++o;
    }
  const int64_t r = split_row(i, n, s);
  o = ohi;
  for (int32_t k = rp[r]; k < rp[r + 1]; ++k)
    if (((uint32_t)(ci[k] ^ (int32_t)r) >> s) != 0) {
      ci_hi[o] = ci[k];
      val_hi[o] = val[k];
      ++o;
    }
}

// Fused batched Chebyshev term for any number of right-hand sides (and for
// 32-RHS blocks beyond 4 GiB).  Thread = (row, j), j fastest; the row data
// come per lane from global memory.
template <int ACC>
__global__ __launch_bounds__(kThreads) void k_cheb_spmm(const int32_t* __restrict__ rp,
                                                        const int32_t* __restrict__ ci,
                                                        const float2* __restrict__ val,
                                                        int64_t n_rows, int n_rhs, double scale,
                                                        const float2* __restrict__ tc,
                                                        float2* __restrict__ tpn,
                                                        float2* __restrict__ acc,
                                                        float2* __restrict__ comp, float2 c,
                                                        int first) {
  const int64_t e_idx = gblock<int64_t>() * kThreads + threadIdx.x;
  const int64_t row = e_idx / n_rhs;
  const int j = (int)(e_idx - row * n_rhs);
  if (row >= n_rows) return;
  RowSum<ACC> sum;
  const int32_t b = rp[row], e = rp[row + 1];
  int32_t k = b;
  for (; k + kGather <= e; k += kGather) {
    int32_t cc[kGather];
    float2 v[kGather], xs[kGather];
#pragma unroll
    for (int u = 0; u < kGather; ++u) { cc[u] = ci[k + u]; v[u] = val[k + u]; }
#pragma unroll
    for (int u = 0; u < kGather; ++u) xs[u] = tc[(int64_t)cc[u] * n_rhs + j];
#pragma unroll
    for (int u = 0; u < kGather; ++u) sum.add(v[u], xs[u]);
  }
  for (; k < e; ++k) sum.add(val[k], tc[(int64_t)ci[k] * n_rhs + j]);
  const float2 tp = first ? make_float2(0.f, 0.f) : tpn[e_idx];
  const float2 tn = sum.next(scale, tp, first != 0);
  tpn[e_idx] = tn;
  const float2 v = cmulc(c, tn);
  float2 a = acc[e_idx], k2 = comp[e_idx];
  neu_add(a.x, k2.x, v.x);
  neu_add(a.y, k2.y, v.y);
  acc[e_idx] = a;
  comp[e_idx] = k2;
}

// Fused Chebyshev term for one right-hand side (the single-state
// chebyshev_evolve and run_hamiltonian path).  kSpmvLanes lanes share a row:
// lane l of the group takes entries b + l, b + l + kSpmvLanes, ..., so each
// load instruction reads contiguous runs of the CSR arrays instead of one
// scattered entry per lane, and the partial row sums are merged across the
// group by lane exchanges (FP64 sums add; compensated pairs merge with one
// Neumaier step).  The group's first lane runs the recurrence epilogue.
// Measured on the 22-qubit chain (33.5 entries per row): one lane per row
// (the generic kernel) 1.56 ms per term; 4, 8, 16, 32 and 64 lanes per row
// 1.26, 0.87, 0.70, 1.14 and 1.56 ms.
#ifndef QSIM_SPMV_LANES
#define QSIM_SPMV_LANES 16
#endif
constexpr int kSpmvLanes = QSIM_SPMV_LANES;

template <int ACC>
__device__ __forceinline__ void merge_lanes(RowSum<ACC>& sum) {
#pragma unroll
  for (int m = 1; m < kSpmvLanes; m <<= 1) {
    if constexpr (ACC == kAccF64) {
      sum.r += lane_xor(sum.r, m);
      sum.i += lane_xor(sum.i, m);
    } else {
      const float sr = lane_xor(sum.sr, m), cr = lane_xor(sum.cr, m);
      const float si = lane_xor(sum.si, m), ci = lane_xor(sum.ci, m);
      neu_add(sum.sr, sum.cr, sr);
      sum.cr += cr;
      neu_add(sum.si, sum.ci, si);
      sum.ci += ci;
    }
  }
}

template <int ACC, bool NT>
__global__ __launch_bounds__(kThreads) void k_cheb_spmv1(const int32_t* __restrict__ rp,
                                                         const int32_t* __restrict__ ci,
                                                         const float2* __restrict__ val,
                                                         int64_t n_rows, double scale,
                                                         const float2* __restrict__ tc,
                                                         float2* __restrict__ tpn,
                                                         float2* __restrict__ acc,
                                                         float2* __restrict__ comp, float2 c,
                                                         int first) {
  const int64_t row = (gblock<int64_t>() * kThreads + threadIdx.x) / kSpmvLanes;
  const int sub = threadIdx.x % kSpmvLanes;
  const bool live = row < n_rows;
  RowSum<ACC> sum;
  if (live) {
    const int32_t b = rp[row], e = rp[row + 1];
    int32_t k = b + sub;
    for (; k + kSpmvLanes < e; k += 2 * kSpmvLanes) {
      const int32_t c0 = __builtin_nontemporal_load(ci + k), c1 = __builtin_nontemporal_load(ci + k + kSpmvLanes);
      const float2 v0 = ld2<true>(val + k), v1 = ld2<true>(val + k + kSpmvLanes);
      const float2 x0 = tc[c0], x1 = tc[c1];
      sum.add(v0, x0);
      sum.add(v1, x1);
    }
    if (k < e) sum.add(ld2<true>(val + k), tc[__builtin_nontemporal_load(ci + k)]);
  }
  merge_lanes<ACC>(sum);   // every lane of the group, live or not, takes part
  if (!live || sub != 0) return;
  const float2 tp = first ? make_float2(0.f, 0.f) : ld2<NT>(tpn + row);
  const float2 tn = sum.next(scale, tp, first != 0);
  st2<NT>(tpn + row, tn);
  const float2 v = cmulc(c, tn);
  float2 a = ld2<NT>(acc + row), k2 = ld2<NT>(comp + row);
  neu_add(a.x, k2.x, v.x);
  neu_add(a.y, k2.y, v.y);
  st2<NT>(acc + row, a);
  st2<NT>(comp + row, k2);
}

// Matrix-free single-state term over a Pauli sum grouped by X mask (the
// tables of qsim_pauli_csr_count): row r's entries are the nonzero group
// values v_g(r) (pauli_group_value, rounded to complex64 exactly as the
// device CSR stores them) at columns r ^ xm[g], summed in group order as
// FP64 sums of exact products.  One thread per row; the group and term loops
// are uniform across the wave, so the tables come in through scalar loads.
// gconst (optional) gives, per group, the entry already rounded to complex64
// when it is the same in every row (no term has a Y|Z mask), or NaN: such a
// group costs its gather and four FMAs, nothing else.
// No index or value stream is read: per term the only HBM traffic is the
// five state vectors, and the gathers of T_k hit the caches (T_k is 32 MiB
// at 22 qubits).  Each term of an entry costs an AND, a popcount, one
// shift-or that puts the parity into the sign of 1.0, and two FP64 FMAs
// (per-term selects of +-c took 18 instructions); a 22-qubit chain term
// takes 0.15 ms (with gconst) against 0.70 ms for the CSR term.  Walking
// XCD-contiguous row ranges measured the same.
constexpr int kPauliRun = 8;   // 4: same time, 16: 3 % slower, 1: 10 % slower (22-qubit chain)
// rows per thread, kThreads apart: the scalar table loads and the loop
// control serve two rows (22-qubit chain: 1 row 0.206 ms, 2 rows 0.164 ms,
// 4 rows 0.182 ms per term, same bits)
constexpr int kPauliRows = 2;
// Entries of one group g for RR rows (uniform group, per-row values).
template <typename R, int RR>
__device__ __forceinline__ void pauli_group_rows(const R (&r)[RR], int t0, int t1,
                                                 const uint64_t* __restrict__ sm,
                                                 const double2* __restrict__ coef, double (&re)[RR],
                                                 double (&im)[RR]) {
#pragma unroll
  for (int q = 0; q < RR; ++q) re[q] = im[q] = 0.0;
  for (int t = t0; t < t1; ++t) {
    const uint64_t m = sm[t];
    const double2 c = coef[t];
#pragma unroll
    for (int q = 0; q < RR; ++q) {
      const uint32_t pc = sizeof(R) == 4 ? (uint32_t)__popc((uint32_t)r[q] & (uint32_t)m)
                                         : (uint32_t)__popcll((uint64_t)r[q] & m);
      const double sgn = __hiloint2double((int)((pc << 31) | 0x3ff00000u), 0);
      re[q] = __builtin_fma(c.x, sgn, re[q]);
      im[q] = __builtin_fma(c.y, sgn, im[q]);
    }
  }
}

template <typename R, bool NT>
__global__ __launch_bounds__(kThreads) void k_cheb_pauli1(int n_groups, const uint64_t* __restrict__ xm,
                                                          const int* __restrict__ toff,
                                                          const uint64_t* __restrict__ sm,
                                                          const double2* __restrict__ coef,
                                                          const double2* __restrict__ gconst,
                                                          int64_t n_rows, double scale,
                                                          const float2* __restrict__ tc,
                                                          float2* __restrict__ tpn,
                                                          float2* __restrict__ acc,
                                                          float2* __restrict__ comp, float2 c,
                                                          int first) {
  constexpr int RR = kPauliRows;
  const int64_t row0 = gblock<int64_t>() * (kThreads * RR) + threadIdx.x;
  if (row0 >= n_rows) return;
  const R rmask = (R)(n_rows - 1);        // n_rows = 2^n: every column stays in range
  R r[RR];
#pragma unroll
  for (int q = 0; q < RR; ++q) r[q] = (R)(row0 + q * kThreads) & rmask;   // rows past the end are not stored
  RowSum<kAccF64> sum[RR];
  // groups in runs of kPauliRun: the run's gathers are issued together (an
  // entry that turns out to be zero is gathered and not used), then the
  // values are formed and added in group order
  int g = 0;
  for (; g + kPauliRun <= n_groups; g += kPauliRun) {
    float2 x[kPauliRun][RR];
#pragma unroll
    for (int j = 0; j < kPauliRun; ++j)
#pragma unroll
      for (int q = 0; q < RR; ++q) x[j][q] = tc[(r[q] ^ (R)xm[g + j]) & rmask];
#pragma unroll
    for (int j = 0; j < kPauliRun; ++j) {
      if (gconst) {
        const double2 v = gconst[g + j];
        if (v.x == v.x) {                   // the same entry in every row (uniform branch)
          if (v.x != 0.0 || v.y != 0.0) {
#pragma unroll
            for (int q = 0; q < RR; ++q) sum[q].add_d(v.x, v.y, x[j][q]);
          }
          continue;
        }
      }
      double re[RR], im[RR];
      pauli_group_rows<R, RR>(r, toff[g + j], toff[g + j + 1], sm, coef, re, im);
#pragma unroll
      for (int q = 0; q < RR; ++q)
        if (re[q] != 0.0 || im[q] != 0.0) sum[q].add(make_float2((float)re[q], (float)im[q]), x[j][q]);
    }
  }
  for (; g < n_groups; ++g) {
    if (gconst) {
      const double2 v = gconst[g];
      if (v.x == v.x) {
        if (v.x != 0.0 || v.y != 0.0) {
#pragma unroll
          for (int q = 0; q < RR; ++q) sum[q].add_d(v.x, v.y, tc[(r[q] ^ (R)xm[g]) & rmask]);
        }
        continue;
      }
    }
    double re[RR], im[RR];
    pauli_group_rows<R, RR>(r, toff[g], toff[g + 1], sm, coef, re, im);
#pragma unroll
    for (int q = 0; q < RR; ++q)
      if (re[q] != 0.0 || im[q] != 0.0)
        sum[q].add(make_float2((float)re[q], (float)im[q]), tc[(r[q] ^ (R)xm[g]) & rmask]);
  }
#pragma unroll
  for (int q = 0; q < RR; ++q) {
    const int64_t row = row0 + q * kThreads;
    if (row >= n_rows) break;
    const float2 tp = first ? make_float2(0.f, 0.f) : ld2<NT>(tpn + row);
    const float2 tn = sum[q].next(scale, tp, first != 0);
    st2<NT>(tpn + row, tn);
    const float2 v = cmulc(c, tn);
    float2 a = ld2<NT>(acc + row), k2 = ld2<NT>(comp + row);
    neu_add(a.x, k2.x, v.x);
    neu_add(a.y, k2.y, v.y);
    st2<NT>(acc + row, a);
    st2<NT>(comp + row, k2);
  }
}

// What a matrix-free term does with T_{k+1} once its row sums are there.  The
// accumulator pair is read and written by every second term only, which adds
// c_k T_k (T_k's own rows are in LDS) and then c_{k+1} T_{k+1}: the additions
// and their order are those of one accumulation per term, and a term moves 40
// instead of 56 bytes per row on average.  The first term starts the pair from
// c_0 T_0, the last one writes acc + comp in the place of T_{k+1}.
enum : int { kChebFirst = 1, kChebInit = 2, kChebPair = 4, kChebSkip = 8, kChebLast = 16 };
struct ChebAcc {
  float2 c, c_cur;                              // c_{k+1}, c_k
  int mode;
};
template <bool NT>
__device__ __forceinline__ void cheb_store(const RowSum<kAccF64>& sum, double scale, const ChebAcc& e, float2 own,
                                           float2* __restrict__ tpn, float2* __restrict__ acc,
                                           float2* __restrict__ comp, uint64_t at) {
  const bool first = e.mode & kChebFirst;
  const float2 tp = first ? make_float2(0.f, 0.f) : ld2<NT>(tpn + at);
  const float2 tn = sum.next(scale, tp, first);
  if (!(e.mode & kChebLast)) st2<NT>(tpn + at, tn);
  if (e.mode & kChebSkip) return;
  float2 a, k2;
  if (e.mode & kChebInit) {
    a = cmulc(e.c_cur, own);
    k2 = make_float2(0.f, 0.f);
  } else {
    a = ld2<NT>(acc + at);
    k2 = ld2<NT>(comp + at);
    if (e.mode & kChebPair) {
      const float2 v = cmulc(e.c_cur, own);
      neu_add(a.x, k2.x, v.x);
      neu_add(a.y, k2.y, v.y);
    }
  }
  const float2 v = cmulc(e.c, tn);
  neu_add(a.x, k2.x, v.x);
  neu_add(a.y, k2.y, v.y);
  if (e.mode & kChebLast) {
    st2<NT>(tpn + at, make_float2(a.x + k2.x, a.y + k2.y));
  } else {
    st2<NT>(acc + at, a);
    st2<NT>(comp + at, k2);
  }
}

// Matrix-free terms over a Pauli sum with real entries.  A workgroup owns a
// tile of consecutive rows: it copies the tile's T_k into LDS, serves the
// groups whose X mask stays inside the tile from there, and loads the others
// as the contiguous partner tile (lanes permuted by the mask's low bits).
// Entries, their rounding and the FP64 sum in group order are those of
// k_cheb_pauli1, so the results have its bits; a row whose entry is zero adds
// nothing, and a group whose entry is zero in the whole wave loads nothing.
//  * Tables: one 64-byte record per group (qsim_pauli_group) holds everything
//    of a group of one or two terms, so a group costs one scalar load instead
//    of a chain of four.
//  * The entry of one or two terms is picked, not summed: the wave's part of
//    the parities on the scalar unit, the lane's part by popcounts only where a
//    mask reaches the lane bits.
struct PauliGroup {       // qsim_pauli_group
  uint64_t xm;
  uint32_t t0;
  uint16_t nt, kind;
  double same, diff, c0, c1;
  uint64_t m0, m1;
};
static_assert(sizeof(PauliGroup) == 64 && sizeof(qsim_pauli_group) == 64, "group record");
__device__ __forceinline__ bool nonzero(double v) { return (__double_as_longlong(v) << 1) != 0; }
__device__ __forceinline__ double flip_sign(double v, uint32_t bit31) {
  return __hiloint2double((int)((uint32_t)__double2hiint(v) ^ bit31), __double2loint(v));
}
__device__ __forceinline__ uint32_t par64(uint64_t m) { return (uint32_t)__builtin_popcountll(m) & 1u; }
// Entry of a one- or two-term group from the parities of its terms: +-(c0 + c1)
// where they agree, +-(c0 - c1) where they differ, the sign that of c0.
__device__ __forceinline__ double pair_entry(const PauliGroup& d, uint32_t p0, uint32_t p1) {
  return flip_sign(((p0 ^ p1) & 1u) == 0 ? d.same : d.diff, p0 << 31);
}

// Four vectors per workgroup (vector j at j * 2^n), tiles of 256 rows, lane =
// row: an entry is evaluated once for the four.  A branch merges before the
// FMAs: every kind of group yields one value per row, and one sequence of FMAs
// adds it (FMAs in each branch made the compiler copy the FP64 sums at every
// merge: 48 VALU instructions per group against 36).
// What bounds it: the T_k loads that miss L2, then the entry evaluation (VALU busy
// 49 %).  A term of 32 vectors of 20 qubits fetches 2.7 GB past L2 and writes
// 0.5, 5.8 TB/s; of 22 qubits 14.8 and 2.1, 7.0 TB/s.  Times per term of a
// Heisenberg chain against the CSR term, us: 20 qubits with 2 / 4 / 8 / 32
// vectors 273 / 278 / 385 / 838 -> 72 / 88 / 153 / 617, 22 qubits with 32 3660
// -> 2672, all with one accumulation per term; with one per two terms 565 and
// 2440 for 32.  Two and eight vectors and tiles of 512 and 1024 rows measured the same to 15 % slower.
constexpr int kPauliVecs = 4;
template <typename R, bool NT>
__global__ __launch_bounds__(kThreads) void k_cheb_pauli(int n_groups, const PauliGroup* __restrict__ tab,
                                                         const uint64_t* __restrict__ sm,
                                                         const double2* __restrict__ coef, int n_bits,
                                                         int n_rhs, int by_rhs, double scale,
                                                         const float2* __restrict__ tc,
                                                         float2* __restrict__ tpn, float2* __restrict__ acc,
                                                         float2* __restrict__ comp, ChebAcc e) {
  constexpr int C = kPauliVecs;
  constexpr uint32_t rows = kThreads;
  constexpr int b = __builtin_ctz(rows);
  __shared__ float4 X4[C * rows / 2];
  const float2* X = reinterpret_cast<const float2*>(X4);
  const uint64_t n_rows = 1ull << n_bits;
  const uint64_t n_tiles = n_rows >> b;
  const uint64_t bid = gblock<uint64_t>();
  const uint32_t ng = (uint32_t)((n_rhs + C - 1) / C);
  if (bid >= n_tiles * ng) return;              // whole workgroup: past the last tile
  uint64_t tile;
  uint32_t grp;
  if (by_rhs) {                                 // ng a multiple of 8: a group of vectors per XCD
    const uint64_t i = bid >> 3;
    grp = (uint32_t)((bid & 7u) + 8u * (i >> (n_bits - b)));
    tile = i & (n_tiles - 1);
  } else {                                      // each XCD walks its own eighth of the tiles
    grp = (uint32_t)(bid >> (n_bits - b));
    tile = bid & (n_tiles - 1);
    if (n_tiles >= 8) tile = (tile & 7u) * (n_tiles >> 3) + (tile >> 3);
  }
  uint64_t voff[C];                             // past the last vector: the last one again, not stored
#pragma unroll
  for (int j = 0; j < C; ++j) {
    const uint32_t q = grp * C + j;
    voff[j] = (uint64_t)(q < (uint32_t)n_rhs ? q : (uint32_t)n_rhs - 1) << n_bits;
  }
  const uint64_t base = tile << b;
#pragma unroll
  for (int j = 0; j < C; ++j) {
    const float4* src = reinterpret_cast<const float4*>(tc + voff[j] + base);
    for (uint32_t i = threadIdx.x; i < rows / 2; i += kThreads) X4[j * (rows / 2) + i] = src[i];
  }
  const uint32_t l = threadIdx.x;
  const R r = (R)base | (R)l;
  RowSum<kAccF64> sum[C];
  const uint32_t lane = threadIdx.x & 63u;
  const uint64_t wbase = base | (uint64_t)(__builtin_amdgcn_readfirstlane(threadIdx.x >> 6) << 6);
  // parity of the wave's part of the row under mask m
  auto wpar = [&](uint64_t m) -> uint32_t { return par64(wbase & m); };
  auto needed = [&](const PauliGroup& d) -> bool {
    if (d.kind != QSIM_PAULI_GROUP_PAIR || ((d.m0 | d.m1) & 63u)) return true;
    return nonzero(pair_entry(d, wpar(d.m0), wpar(d.m1)));
  };
  auto add_group = [&](const PauliGroup& d, const float2 (&x)[C]) {
    double v;
    if (d.kind == QSIM_PAULI_GROUP_PAIR && ((d.m0 | d.m1) & 63u)) {
      v = pair_entry(d, (uint32_t)__popc(lane & (uint32_t)d.m0) + wpar(d.m0),
                     (uint32_t)__popc(lane & (uint32_t)d.m1) + wpar(d.m1));
    } else if (d.kind == QSIM_PAULI_GROUP_TERMS) {
      v = 0.0;
#pragma unroll 4
      for (uint32_t t = d.t0; t < d.t0 + d.nt; ++t) {
        const uint64_t m = sm[t];
        v += flip_sign(coef[t].x, (wpar(m) << 31) ^ ((uint32_t)__popc(lane & (uint32_t)m) << 31));
      }
      v = (double)(float)v;
    } else {
      v = d.kind == QSIM_PAULI_GROUP_PAIR ? pair_entry(d, wpar(d.m0), wpar(d.m1)) : d.same;
    }
    asm volatile("" : "+v"(v));                 // one vector value from here on, whatever the kind
    if (v != 0.0) {
#pragma unroll
      for (int j = 0; j < C; ++j) sum[j].add_r(v, x[j]);
    }
  };
  __syncthreads();
  int g = 0;
  for (; g < n_groups && tab[g].xm < rows; ++g) {
    const PauliGroup d = tab[g];
    if (!needed(d)) continue;
    const uint32_t m = (uint32_t)d.xm;
    float2 x[C];
#pragma unroll
    for (int j = 0; j < C; ++j) x[j] = X[j * rows + (l ^ m)];
    add_group(d, x);
  }
  for (; g < n_groups; ++g) {
    const PauliGroup d = tab[g];
    if (!needed(d)) continue;
    const R m = (R)d.xm & (R)(n_rows - 1);
    float2 x[C];
#pragma unroll
    for (int j = 0; j < C; ++j) x[j] = (tc + voff[j])[r ^ m];
    add_group(d, x);
  }
#pragma unroll
  for (int j = 0; j < C; ++j)
    if (grp * C + j < (uint32_t)n_rhs)
      cheb_store<NT>(sum[j], scale, e, X[j * rows + l], tpn, acc, comp, voff[j] + r);
}

// One vector: 2^LR rows per thread, 256 apart, in tiles of 256 << LR rows.
// With one vector to serve, the chain of table loads and scalar parities of a
// group is what a term waits for, so the groups are looked at side by side:
// lane i holds group i's record and works out, once per wave and for 64 groups
// at a time, the wave's part of the parities, the entry where it is the same
// in the whole wave, and whether the group is needed at all.  The walk over the
// needed groups then takes scalars from lanes (v_readlane) and waits for T_k
// only, which it loads for U groups together.  What bounds it: on small states
// the latency of the walk (a workgroup or less per CU), from 19 qubits on the
// far loads, most of which another XCD wrote.  us per term of a Heisenberg
// chain of 12 / 16 / 19 qubits: 6.8 / 8.1 / 17.5 (k_cheb_pauli1 9.5 / 14 / 25;
// the walk with scalar table loads, as in k_cheb_pauli, 13 / 16 / 29).  A
// 19-qubit evolution 1790 -> 1270 us with the launches in one call.  Groups of
// three terms and more cost a term and row more than in k_cheb_pauli1: past 2 to
// 3.5 of them a group that kernel is the faster from 18 qubits on (the callers'
// rule).
__device__ __forceinline__ uint32_t from_lane(uint32_t v, int lane) {
  return (uint32_t)__builtin_amdgcn_readlane((int)v, lane);
}
__device__ __forceinline__ float flip_signf(float v, uint32_t bit31) {
  return __uint_as_float(__float_as_uint(v) ^ bit31);
}
template <typename R, int LR, int U, bool NT>
__global__ __launch_bounds__(kThreads) void k_cheb_pauli_one(int n_groups, const PauliGroup* __restrict__ tab,
                                                             const uint64_t* __restrict__ sm,
                                                             const double2* __restrict__ coef, int n_bits,
                                                             double scale, const float2* __restrict__ tc,
                                                             float2* __restrict__ tpn, float2* __restrict__ acc,
                                                             float2* __restrict__ comp, ChebAcc e) {
  constexpr int RR = 1 << LR, b = __builtin_ctz(kThreads) + LR;
  constexpr uint32_t rows = 1u << b;
  constexpr uint32_t qm = rows - kThreads;      // the row-of-thread bits
  __shared__ float4 X4[rows / 2];
  const float2* X = reinterpret_cast<const float2*>(X4);
  const uint64_t n_tiles = (1ull << n_bits) >> b;
  uint64_t tile = gblock<uint64_t>();
  if (tile >= n_tiles) return;                  // whole workgroup: past the last tile
  if (n_tiles >= 8) tile = (tile & 7u) * (n_tiles >> 3) + (tile >> 3);   // an eighth of the tiles per XCD
  const R base = (R)(tile << b);
  for (uint32_t i = threadIdx.x; i < rows / 2; i += kThreads) X4[i] = reinterpret_cast<const float4*>(tc + base)[i];
  const uint32_t l = threadIdx.x, lane = l & 63u;
  const R wbase = base | (R)(l & ~63u);
  auto wpar = [&](uint64_t m) -> uint32_t {
    return (uint32_t)(sizeof(R) == 4 ? __popc((uint32_t)wbase & (uint32_t)m) : __popcll((uint64_t)wbase & m)) & 1u;
  };
  auto qpar = [&](uint32_t m, int q) -> uint32_t { return (uint32_t)__popc(m & (uint32_t)(q * kThreads)); };
  RowSum<kAccF64> sum[RR];
  bool loaded = false;
  for (int g0 = 0; g0 < n_groups; g0 += 64) {
    // lane i: group g0 + i
    const bool valid = (int)lane < n_groups - g0;
    const PauliGroup d = tab[valid ? g0 + (int)lane : n_groups - 1];
    const uint32_t reach = (uint32_t)(d.m0 | d.m1);
    const uint32_t p0 = wpar(d.m0), p1 = wpar(d.m1);
    const bool pair = d.kind == QSIM_PAULI_GROUP_PAIR, terms = d.kind == QSIM_PAULI_GROUP_TERMS;
    const float same = (float)d.same, diff = (float)d.diff;      // FP32 values
    const float vu = pair ? flip_signf(p0 == p1 ? same : diff, p0 << 31) : same;
    const bool uni = !terms && !(pair && (reach & (63u | qm)));
    const uint64_t is_uni = __ballot(uni), is_terms = __ballot(terms), is_q = __ballot(pair && (reach & qm));
    const uint64_t odd0 = __ballot(p0 != 0), odd1 = __ballot(p1 != 0);
    uint64_t todo = __ballot(valid && !(uni && vu == 0.f));
    const uint32_t xlo = (uint32_t)d.xm, xhi = (uint32_t)(d.xm >> 32), m0 = (uint32_t)d.m0, m1 = (uint32_t)d.m1;
    const uint32_t same_b = __float_as_uint(same), diff_b = __float_as_uint(diff), vu_b = __float_as_uint(vu);
    if (!loaded) __syncthreads();
    loaded = true;
    while (todo) {
      int gi[U];
      float2 x[U][RR];
#pragma unroll
      for (int u = 0; u < U; ++u) {
        gi[u] = todo ? __builtin_ctzll(todo) : -1;
        todo &= todo - 1;
        if (gi[u] < 0) continue;
        R xm = (R)from_lane(xlo, gi[u]);
        if constexpr (sizeof(R) == 8) xm |= (R)from_lane(xhi, gi[u]) << 32;
        if (xm < rows) {
#pragma unroll
          for (int q = 0; q < RR; ++q) x[u][q] = X[(l + q * kThreads) ^ (uint32_t)xm];
        } else {
#pragma unroll
          for (int q = 0; q < RR; ++q) x[u][q] = tc[(base | (R)(l + q * kThreads)) ^ xm];
        }
      }
#pragma unroll
      for (int u = 0; u < U; ++u) {
        if (gi[u] < 0) continue;
        const int g = gi[u];
        float v[RR];
        if (is_uni >> g & 1) {
          const float w = __uint_as_float(from_lane(vu_b, g));
#pragma unroll
          for (int q = 0; q < RR; ++q) v[q] = w;
        } else {
          if (is_terms >> g & 1) {
            const uint32_t t0 = from_lane(d.t0, g), nt = from_lane(d.nt, g);
            double w[RR];
#pragma unroll
            for (int q = 0; q < RR; ++q) w[q] = 0.0;
            for (uint32_t c0 = 0; c0 < nt; c0 += 64) {
              const uint32_t left = nt - c0 < 64u ? nt - c0 : 64u;
              const uint32_t t = t0 + c0 + (lane < left ? lane : left - 1);
              const uint64_t m = sm[t];
              const double cs = flip_sign(coef[t].x, wpar(m) << 31);
              const uint32_t mlo = (uint32_t)m, chi = (uint32_t)__double2hiint(cs), clo = (uint32_t)__double2loint(cs);
#pragma unroll 4
              for (uint32_t j = 0; j < left; ++j) {
                const uint32_t mj = from_lane(mlo, j);
                const uint32_t s = from_lane(chi, j) ^ ((uint32_t)__popc(lane & mj) << 31);
                const uint32_t lo = from_lane(clo, j);
#pragma unroll
                for (int q = 0; q < RR; ++q) w[q] += __hiloint2double((int)(s ^ (qpar(mj, q) << 31)), (int)lo);
              }
            }
#pragma unroll
            for (int q = 0; q < RR; ++q) v[q] = (float)w[q];
          } else {
            const uint32_t a0 = from_lane(m0, g), a1 = from_lane(m1, g);
            const float vs = __uint_as_float(from_lane(same_b, g)), vd = __uint_as_float(from_lane(diff_b, g));
            const uint32_t q0 = (uint32_t)__popc(lane & a0) + (uint32_t)(odd0 >> g & 1);
            const uint32_t q1 = (uint32_t)__popc(lane & a1) + (uint32_t)(odd1 >> g & 1);
            if (LR && (is_q >> g & 1)) {
#pragma unroll
              for (int q = 0; q < RR; ++q) {
                const uint32_t r0 = q0 + qpar(a0, q), r1 = q1 + qpar(a1, q);
                v[q] = flip_signf(((r0 ^ r1) & 1u) ? vd : vs, r0 << 31);
              }
            } else {
              const float w = flip_signf(((q0 ^ q1) & 1u) ? vd : vs, q0 << 31);
#pragma unroll
              for (int q = 0; q < RR; ++q) v[q] = w;
            }
          }
#pragma unroll
          for (int q = 0; q < RR; ++q)            // a row whose entry is zero takes nothing from T_k
            if (v[q] == 0.f) x[u][q] = make_float2(0.f, 0.f);
        }
#pragma unroll
        for (int q = 0; q < RR; ++q) {
          asm volatile("" : "+v"(v[q]));          // one vector value from here on, whatever the kind
          sum[q].add_r((double)v[q], x[u][q]);
        }
      }
    }
  }
  if (!loaded) __syncthreads();
#pragma unroll
  for (int q = 0; q < RR; ++q)
    cheb_store<NT>(sum[q], scale, e, X[l + q * kThreads], tpn, acc, comp, (uint64_t)base + l + q * kThreads);
}

struct PauliTerm {        // a matrix-free Hamiltonian with real entries, and the vectors
  int n_groups;
  const PauliGroup* groups;
  const uint64_t* sm;
  const double2* coef;
  int n, n_rhs;
  double scale;
};

template <typename R, int LR, int U>
static void launch_pauli_one(hipStream_t s, const PauliTerm& h, const float2* tc, float2* tpn, float2* acc,
                             float2* comp, const ChebAcc& e) {
  auto* kern = nt_for_bytes(32ull << h.n) ? k_cheb_pauli_one<R, LR, U, true> : k_cheb_pauli_one<R, LR, U, false>;
  hipLaunchKernelGGL(kern, grid1d((1ull << h.n) / (kThreads << LR)), dim3(kThreads), 0, s, h.n_groups, h.groups,
                     h.sm, h.coef, h.n, h.scale, tc, tpn, acc, comp, e);
}

template <typename R>
static void launch_pauli(hipStream_t s, const PauliTerm& h, const float2* tc, float2* tpn, float2* acc, float2* comp,
                         const ChebAcc& e) {
  if (h.n_rhs == 1) {
    // us per evolution of a Heisenberg chain (t = 1, 43 to 70 terms) at 1 / 2 / 4
    // rows per thread: 12 qubits 420 / 478 / 564, 16 qubits 580 / 670 / 796,
    // 18 qubits 921 / 929 / 1015, 19 qubits 1313 / 1234 / 1270, 20 qubits 2204 /
    // 1916 / 1906, 21 qubits 4054 / 3292 / 3183, 22 qubits 7900 / 6143 / 5732
    // (8 rows: 6258 there); more rows share the work on a group but leave fewer
    // waves.  Four groups' loads together, two where four rows already are.
    if (h.n <= 18) launch_pauli_one<R, 0, 4>(s, h, tc, tpn, acc, comp, e);
    else if (h.n <= 20) launch_pauli_one<R, 1, 4>(s, h, tc, tpn, acc, comp, e);
    else launch_pauli_one<R, 2, 2>(s, h, tc, tpn, acc, comp, e);
    return;
  }
  const uint64_t ng = ceil_div((uint64_t)h.n_rhs, kPauliVecs);
  const uint64_t blocks = ng * ((1ull << h.n) / kThreads);
  // T_k, T_{k-1} and the accumulator pair stream together: nontemporal once
  // the four exceed the MALL (20 qubits, 32 right-hand sides: 622 against
  // 659 us; 8, which fit: 171 against 155 us)
  const bool nt = nt_for_bytes((32ull * h.n_rhs) << h.n);
  // a group of vectors per XCD while its T_k (32 B a row) is a few L2s large:
  // 16 qubits, 32 right-hand sides 38 against 44 us, 20 qubits 609 against
  // 622; 22 qubits 2890 against 2733 us
  const int by_rhs = ng % 8 == 0 && h.n <= 20;
  auto* kern = nt ? k_cheb_pauli<R, true> : k_cheb_pauli<R, false>;
  hipLaunchKernelGGL(kern, grid1d(blocks), dim3(kThreads), 0, s, h.n_groups, h.groups, h.sm, h.coef, h.n, h.n_rhs,
                     by_rhs, h.scale, tc, tpn, acc, comp, e);
}

static int check_pauli(const PauliTerm& h, const void* t_cur, const void* t_prev_next, const void* acc,
                       const void* comp) {
  if (h.n < QSIM_PAULI_BATCH_MIN_QUBITS || h.n > QSIM_MAX_QUBITS)
    return fail(QSIM_ERANGE, "n_qubits=%d outside %d..%d", h.n, QSIM_PAULI_BATCH_MIN_QUBITS, QSIM_MAX_QUBITS);
  if (h.n_groups < 0 || h.n_rhs < 1 || h.n_rhs > (1 << 20))
    return fail(QSIM_EINVAL, "bad sizes (n_groups=%d, n_rhs=%d)", h.n_groups, h.n_rhs);
  if ((h.n_groups > 0 && (!h.groups || !h.sm || !h.coef)) || !t_cur || !t_prev_next || !acc || !comp)
    return fail(QSIM_EINVAL, "NULL pointer argument");
  return QSIM_OK;
}

__global__ __launch_bounds__(kThreads) void k_cheb_init(float2* __restrict__ acc,
                                                        float2* __restrict__ comp,
                                                        const float2* __restrict__ t, int64_t n,
                                                        float2 c) {
  const int64_t i = (int64_t)blockIdx.x * kThreads + threadIdx.x;
  if (i >= n) return;
  acc[i] = cmulc(c, t[i]);
  comp[i] = make_float2(0.f, 0.f);
}

__global__ __launch_bounds__(kThreads) void k_cheb_finish(float2* __restrict__ out,
                                                          const float2* __restrict__ acc,
                                                          const float2* __restrict__ comp,
                                                          int64_t n) {
  const int64_t i = (int64_t)blockIdx.x * kThreads + threadIdx.x;
  if (i >= n) return;
  const float2 a = acc[i], k = comp[i];
  out[i] = make_float2(a.x + k.x, a.y + k.y);
}

// Order shift for a grid of `blocks` 32-RHS workgroups (2^kBlockRowsLog2
// rows each): the requested shift when the chunks tile the grid exactly,
// else 0.
static int spmm_order(int64_t blocks, int shift) {
  const int64_t chunk = shift > kBlockRowsLog2 ? int64_t(1) << (shift - kBlockRowsLog2) : 1;
  return blocks % (8 * chunk) == 0 ? shift : 0;
}

static int log2_exact(int64_t v) {
  if (v <= 0 || (v & (v - 1))) return -1;
  int n = 0;
  while ((int64_t(1) << n) < v) ++n;
  return n;
}

static inline float2 f2(double re, double im) { return make_float2((float)re, (float)im); }

}  // namespace qsim

using namespace qsim;

extern "C" {

int qsim_spmv_csr(void* stream, const void* row_ptr, const void* col_idx, const void* values,
                  int64_t n_rows, const void* x, void* y, double alpha_re, double alpha_im,
                  double beta_re, double beta_im) {
  if (n_rows < 0) return fail(QSIM_EINVAL, "n_rows < 0");
  if (n_rows == 0) return QSIM_OK;
  if (!row_ptr || !col_idx || !values || !x || !y) return fail(QSIM_EINVAL, "NULL pointer argument");
  hipLaunchKernelGGL(k_spmv, dim3(ceil_div(n_rows, kThreads)), dim3(kThreads), 0, as_stream(stream),
                     (const int32_t*)row_ptr, (const int32_t*)col_idx, (const float2*)values, n_rows,
                     (const float2*)x, (float2*)y, f2(alpha_re, alpha_im), f2(beta_re, beta_im));
  return launch_status("spmv_csr");
}

int qsim_chebyshev_step(void* stream, const void* s, const void* t_prev, void* t_next, int64_t n) {
  if (n < 0) return fail(QSIM_EINVAL, "n < 0");
  if (n == 0) return QSIM_OK;
  if (!s || !t_prev || !t_next) return fail(QSIM_EINVAL, "NULL pointer argument");
  hipLaunchKernelGGL(k_step, dim3(ceil_div(n, kThreads)), dim3(kThreads), 0, as_stream(stream),
                     (const float2*)s, (const float2*)t_prev, (float2*)t_next, n);
  return launch_status("chebyshev_step");
}

int qsim_chebyshev_accum(void* stream, void* accum, const void* t, int64_t n, double c_re,
                         double c_im) {
  if (n < 0) return fail(QSIM_EINVAL, "n < 0");
  if (n == 0) return QSIM_OK;
  if (!accum || !t) return fail(QSIM_EINVAL, "NULL pointer argument");
  hipLaunchKernelGGL(k_accum, dim3(ceil_div(n, kThreads)), dim3(kThreads), 0, as_stream(stream),
                     (float2*)accum, (const float2*)t, n, f2(c_re, c_im));
  return launch_status("chebyshev_accum");
}

int qsim_chebyshev_step_accum(void* stream, const void* s, const void* t_prev, void* t_next,
                              void* accum, int64_t n, double c_re, double c_im) {
  if (n < 0) return fail(QSIM_EINVAL, "n < 0");
  if (n == 0) return QSIM_OK;
  if (!s || !t_prev || !t_next || !accum) return fail(QSIM_EINVAL, "NULL pointer argument");
  hipLaunchKernelGGL(k_step_accum, dim3(ceil_div(n, kThreads)), dim3(kThreads), 0,
                     as_stream(stream), (const float2*)s, (const float2*)t_prev, (float2*)t_next,
                     (float2*)accum, n, f2(c_re, c_im));
  return launch_status("chebyshev_step_accum");
}

int qsim_cheb_spmm_step(void* stream, const void* row_ptr, const void* col_idx, const void* values,
                        int64_t n_rows, int n_rhs, double scale, const void* t_cur,
                        void* t_prev_next, void* acc, void* comp, double c_re, double c_im,
                        int first, int accumulate) {
  if (n_rows < 0 || n_rhs < 1) return fail(QSIM_EINVAL, "bad sizes (n_rows=%lld, n_rhs=%d)",
                                           (long long)n_rows, n_rhs);
  if (accumulate != QSIM_CHEB_ACC_FP64 && accumulate != QSIM_CHEB_ACC_FP32C)
    return fail(QSIM_EINVAL, "unknown accumulate mode %d", accumulate);
  if (n_rows == 0) return QSIM_OK;
  if (!row_ptr || !col_idx || !values || !t_cur || !t_prev_next || !acc || !comp)
    return fail(QSIM_EINVAL, "NULL pointer argument");
  hipStream_t s = as_stream(stream);
  const float2 cf = f2(c_re, c_im);
  const bool f64 = accumulate == QSIM_CHEB_ACC_FP64;
  // the 32-RHS kernel addresses T_k with 32-bit byte offsets (<= 2^24 rows)
  if (n_rhs == 32 && n_rows <= (int64_t(1) << 24)) {
    const int64_t blocks = (int64_t)ceil_div((uint64_t)n_rows, kWaves * kRowsPerWave);
    const int order = spmm_order(blocks, kSpmmOrderShift);
    const bool nt = nt_for_bytes((uint64_t)n_rows * 256u);
    auto* kern = f64 ? (nt ? k_cheb_spmm32<kAccF64, true, 0> : k_cheb_spmm32<kAccF64, false, 0>)
                     : (nt ? k_cheb_spmm32<kAccF32c, true, 0> : k_cheb_spmm32<kAccF32c, false, 0>);
    hipLaunchKernelGGL(kern, dim3((unsigned)blocks), dim3(kThreads), 0, s, (const int32_t*)row_ptr,
                       (const int32_t*)col_idx, (const float2*)values, n_rows, scale,
                       (const float2*)t_cur, (float2*)t_prev_next, (float2*)acc, (float2*)comp,
                       (float2*)nullptr, cf, first, order, 0, 0);
    return launch_status("cheb_spmm_step");
  }
  if (n_rhs == 1) {
    const int64_t threads = n_rows * kSpmvLanes;
    const bool nt = nt_for_bytes((uint64_t)n_rows * 8u);
    auto* kern = f64 ? (nt ? k_cheb_spmv1<kAccF64, true> : k_cheb_spmv1<kAccF64, false>)
                     : (nt ? k_cheb_spmv1<kAccF32c, true> : k_cheb_spmv1<kAccF32c, false>);
    hipLaunchKernelGGL(kern, grid1d(ceil_div(threads, kThreads)), dim3(kThreads), 0, s,
                       (const int32_t*)row_ptr, (const int32_t*)col_idx, (const float2*)values, n_rows,
                       scale, (const float2*)t_cur, (float2*)t_prev_next, (float2*)acc, (float2*)comp,
                       cf, first);
    return launch_status("cheb_spmm_step");
  }
  const int64_t total = n_rows * (int64_t)n_rhs;
  auto* kern = f64 ? k_cheb_spmm<kAccF64> : k_cheb_spmm<kAccF32c>;
  hipLaunchKernelGGL(kern, grid1d(ceil_div(total, kThreads)), dim3(kThreads), 0, s,
                     (const int32_t*)row_ptr, (const int32_t*)col_idx, (const float2*)values,
                     n_rows, n_rhs, scale, (const float2*)t_cur, (float2*)t_prev_next, (float2*)acc,
                     (float2*)comp, cf, first);
  return launch_status("cheb_spmm_step");
}

int qsim_cheb_pauli_step(void* stream, int n_qubits, int n_groups, const void* xm, const void* toff,
                         const void* sm, const void* coef, const void* gconst, double scale, const void* t_cur,
                         void* t_prev_next, void* acc, void* comp, double c_re, double c_im,
                         int first) {
  if (n_qubits < 1 || n_qubits > QSIM_MAX_QUBITS)
    return fail(QSIM_ERANGE, "n_qubits=%d outside 1..%d", n_qubits, QSIM_MAX_QUBITS);
  if (n_groups < 0) return fail(QSIM_EINVAL, "n_groups < 0");
  if ((n_groups > 0 && (!xm || !toff || !sm || !coef)) || !t_cur || !t_prev_next || !acc || !comp)
    return fail(QSIM_EINVAL, "NULL pointer argument");
  const int64_t n_rows = int64_t(1) << n_qubits;
  const bool nt = nt_for_bytes((uint64_t)n_rows * 8u);
  auto* kern = n_qubits > 32 ? (nt ? k_cheb_pauli1<uint64_t, true> : k_cheb_pauli1<uint64_t, false>)
                             : (nt ? k_cheb_pauli1<uint32_t, true> : k_cheb_pauli1<uint32_t, false>);
  hipLaunchKernelGGL(kern, grid1d(ceil_div((uint64_t)n_rows, kThreads * kPauliRows)), dim3(kThreads), 0,
                     as_stream(stream), n_groups, (const uint64_t*)xm, (const int*)toff,
                     (const uint64_t*)sm, (const double2*)coef, (const double2*)gconst, n_rows, scale,
                     (const float2*)t_cur,
                     (float2*)t_prev_next, (float2*)acc, (float2*)comp, f2(c_re, c_im), first);
  return launch_status("cheb_pauli_step");
}

int qsim_cheb_pauli_batch_step(void* stream, int n_qubits, int n_groups, const void* groups, const void* sm,
                               const void* coef, int n_rhs, double scale, const void* t_cur, void* t_prev_next,
                               void* acc, void* comp, double c_re, double c_im, int first) {
  const PauliTerm h = {n_groups, (const PauliGroup*)groups, (const uint64_t*)sm, (const double2*)coef, n_qubits,
                       n_rhs, scale};
  if (int rc = check_pauli(h, t_cur, t_prev_next, acc, comp)) return rc;
  if (((uintptr_t)t_cur & 15u) != 0) return fail(QSIM_EINVAL, "t_cur must be 16-byte aligned");
  const ChebAcc e = {f2(c_re, c_im), make_float2(0.f, 0.f), first ? kChebFirst : 0};
  (n_qubits > 32 ? launch_pauli<uint64_t> : launch_pauli<uint32_t>)(as_stream(stream), h, (const float2*)t_cur,
                                                                    (float2*)t_prev_next, (float2*)acc,
                                                                    (float2*)comp, e);
  return launch_status("cheb_pauli_batch_step");
}

int qsim_cheb_pauli_evolve(void* stream, int n_qubits, int n_groups, const void* groups, const void* sm,
                           const void* coef, int n_rhs, double scale, void* t0, void* t1, void* acc, void* comp,
                           const double* coeffs, int n_terms) {
  const PauliTerm h = {n_groups, (const PauliGroup*)groups, (const uint64_t*)sm, (const double2*)coef, n_qubits,
                       n_rhs, scale};
  if (int rc = check_pauli(h, t0, t1, acc, comp)) return rc;
  if (!coeffs) return fail(QSIM_EINVAL, "NULL pointer argument");
  if (n_terms < 1) return fail(QSIM_EINVAL, "n_terms < 1");
  if ((((uintptr_t)t0 | (uintptr_t)t1) & 15u) != 0) return fail(QSIM_EINVAL, "t0 and t1 must be 16-byte aligned");
  auto* launch = n_qubits > 32 ? launch_pauli<uint64_t> : launch_pauli<uint32_t>;
  float2 *cur = (float2*)t0, *prv = (float2*)t1;
  for (int k = 1; k <= n_terms; ++k) {
    ChebAcc e = {f2(coeffs[2 * k], coeffs[2 * k + 1]), f2(coeffs[2 * k - 2], coeffs[2 * k - 1]), 0};
    if (k == 1) e.mode = kChebFirst | kChebInit;
    else if (k % 2) e.mode = kChebPair;
    else if (k < n_terms) e.mode = kChebSkip;
    if (k == n_terms) e.mode |= kChebLast;
    launch(as_stream(stream), h, cur, prv, (float2*)acc, (float2*)comp, e);
    if (int rc = launch_status("cheb_pauli_evolve")) return rc;
    std::swap(cur, prv);
  }
  return QSIM_OK;
}

int qsim_cheb_init_acc(void* stream, void* acc, void* comp, const void* t, int64_t n, double c_re,
                       double c_im) {
  if (n < 0) return fail(QSIM_EINVAL, "n < 0");
  if (n == 0) return QSIM_OK;
  if (!acc || !comp || !t) return fail(QSIM_EINVAL, "NULL pointer argument");
  hipLaunchKernelGGL(k_cheb_init, dim3(ceil_div(n, kThreads)), dim3(kThreads), 0, as_stream(stream),
                     (float2*)acc, (float2*)comp, (const float2*)t, n, f2(c_re, c_im));
  return launch_status("cheb_init_acc");
}

int qsim_cheb_finish(void* stream, void* out, const void* acc, const void* comp, int64_t n) {
  if (n < 0) return fail(QSIM_EINVAL, "n < 0");
  if (n == 0) return QSIM_OK;
  if (!out || !acc || !comp) return fail(QSIM_EINVAL, "NULL pointer argument");
  hipLaunchKernelGGL(k_cheb_finish, dim3(ceil_div(n, kThreads)), dim3(kThreads), 0,
                     as_stream(stream), (float2*)out, (const float2*)acc, (const float2*)comp, n);
  return launch_status("cheb_finish");
}

int64_t qsim_csr_split_workspace_bytes(int64_t n_rows) {
  if (n_rows < 1) return -1;
  const int64_t blocks = (int64_t)ceil_div((uint64_t)n_rows, kSplitThreads);
  return (2 * blocks + 2) * (int64_t)sizeof(int64_t);
}

static int check_split(int64_t n_rows, int split_bit, int& n) {
  n = log2_exact(n_rows);
  if (n < 2 || n_rows > (int64_t(1) << 30))
    return fail(QSIM_EINVAL, "the CSR split needs 2^n rows, 4 <= rows <= 2^30 (got %lld)", (long long)n_rows);
  if (split_bit < 1 || split_bit >= n)
    return fail(QSIM_EINVAL, "split_bit %d outside 1..%d", split_bit, n - 1);
  return QSIM_OK;
}

int qsim_csr_split_count(void* stream, const void* row_ptr, const void* col_idx, int64_t n_rows,
                         int split_bit, void* workspace, int64_t* nnz_lo, int64_t* nnz_hi) {
  int n = 0;
  if (int rc = check_split(n_rows, split_bit, n)) return rc;
  if (!row_ptr || !col_idx || !workspace || !nnz_lo || !nnz_hi) return fail(QSIM_EINVAL, "NULL pointer argument");
  hipStream_t s = as_stream(stream);
  const uint64_t blocks = ceil_div((uint64_t)n_rows, kSplitThreads);
  int64_t* bsum = (int64_t*)workspace;
  int64_t* tot = bsum + 2 * blocks;
  hipLaunchKernelGGL(k_split_count, dim3((unsigned)blocks), dim3(kSplitThreads), 0, s,
                     (const int32_t*)row_ptr, (const int32_t*)col_idx, n_rows, n, split_bit, bsum);
  if (int rc = launch_status("csr_split: count")) return rc;
  hipLaunchKernelGGL(k_split_scan, dim3(1), dim3(kSplitThreads), 0, s, blocks, bsum, tot);
  if (int rc = launch_status("csr_split: scan")) return rc;
  int64_t h[2] = {0, 0};
  hipError_t e = hipMemcpyAsync(h, tot, sizeof h, hipMemcpyDeviceToHost, s);
  if (e == hipSuccess) e = hipStreamSynchronize(s);
  if (e != hipSuccess) return fail(QSIM_EHIP, "csr_split: %s", hipGetErrorString(e));
  if (h[0] > INT32_MAX || h[1] > INT32_MAX) return fail(QSIM_ERANGE, "split CSR beyond int32 nonzeros");
  *nnz_lo = h[0];
  *nnz_hi = h[1];
  return QSIM_OK;
}

int qsim_csr_split_fill(void* stream, const void* row_ptr, const void* col_idx, const void* values,
                        int64_t n_rows, int split_bit, const void* workspace, void* rp_lo,
                        void* ci_lo, void* val_lo, void* rp_hi, void* ci_hi, void* val_hi) {
  int n = 0;
  if (int rc = check_split(n_rows, split_bit, n)) return rc;
  if (!row_ptr || !col_idx || !values || !workspace || !rp_lo || !ci_lo || !val_lo || !rp_hi ||
      !ci_hi || !val_hi)
    return fail(QSIM_EINVAL, "NULL pointer argument");
  const uint64_t blocks = ceil_div((uint64_t)n_rows, kSplitThreads);
  hipLaunchKernelGGL(k_split_fill, dim3((unsigned)blocks), dim3(kSplitThreads), 0, as_stream(stream),
                     (const int32_t*)row_ptr, (const int32_t*)col_idx, (const float2*)values, n_rows, n,
                     split_bit, (const int64_t*)workspace, (int32_t*)rp_lo, (int32_t*)ci_lo,
                     (float2*)val_lo, (int32_t*)rp_hi, (int32_t*)ci_hi, (float2*)val_hi);
  return launch_status("csr_split: fill");
}

int qsim_cheb_spmm_step_split(void* stream, const void* rp_lo, const void* ci_lo, const void* val_lo,
                              const void* rp_hi, const void* ci_hi, const void* val_hi, int64_t n_rows,
                              int split_bit, int n_rhs, double scale, const void* t_cur,
                              void* t_prev_next, void* acc, void* comp, void* w1, double c_re,
                              double c_im, int first) {
  int n = 0;
  if (int rc = check_split(n_rows, split_bit, n)) return rc;
  if (n_rhs != 32) return fail(QSIM_EINVAL, "the split term runs 32 right-hand sides (got %d)", n_rhs);
  if (n_rows > (int64_t(1) << 24)) return fail(QSIM_ERANGE, "the split term handles at most 2^24 rows");
  if (!rp_lo || !ci_lo || !val_lo || !rp_hi || !ci_hi || !val_hi || !t_cur || !t_prev_next || !acc ||
      !comp || !w1)
    return fail(QSIM_EINVAL, "NULL pointer argument");
  hipStream_t s = as_stream(stream);
  const float2 cf = f2(c_re, c_im);
  const int64_t blocks = (int64_t)ceil_div((uint64_t)n_rows, kWaves * kRowsPerWave);
  // each XCD walks one contiguous eighth of the rows (positions) in both passes
  const int order = spmm_order(blocks, n >= 3 ? n - 3 : 0);
  const bool nt = nt_for_bytes((uint64_t)n_rows * 256u);
  auto* k1 = nt ? k_cheb_spmm32<kAccF64, true, 1> : k_cheb_spmm32<kAccF64, false, 1>;
  auto* k2 = nt ? k_cheb_spmm32<kAccF64, true, 2> : k_cheb_spmm32<kAccF64, false, 2>;
  hipLaunchKernelGGL(k1, dim3((unsigned)blocks), dim3(kThreads), 0, s, (const int32_t*)rp_lo,
                     (const int32_t*)ci_lo, (const float2*)val_lo, n_rows, scale, (const float2*)t_cur,
                     (float2*)t_prev_next, (float2*)acc, (float2*)comp, (float2*)w1, cf, first, order,
                     n, split_bit);
  if (int rc = launch_status("cheb_spmm_step_split: low pass")) return rc;
  hipLaunchKernelGGL(k2, dim3((unsigned)blocks), dim3(kThreads), 0, s, (const int32_t*)rp_hi,
                     (const int32_t*)ci_hi, (const float2*)val_hi, n_rows, scale, (const float2*)t_cur,
                     (float2*)t_prev_next, (float2*)acc, (float2*)comp, (float2*)w1, cf, first, order,
                     n, split_bit);
  return launch_status("cheb_spmm_step_split: high pass");
}

}  // extern "C"
