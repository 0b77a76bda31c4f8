// Pauli-string expectation values, Pauli-string application and the
// stochastic noise channels (one Kraus branch per call) for gfx950.
//
// A Pauli string is given by two masks: x (qubits carrying X or Y) and z
// (qubits carrying Z or Y).  With y = popcount(x & z) (the number of Y's),
//   P = i^y X^x Z^z,   (P psi)_i = i^y (-1)^popcount((i ^ x) & z) psi_{i ^ x}.
// Its expectation pairs every index i0 whose highest x bit is clear with its
// partner j = i0 ^ x.  With zc = conj(psi_i0) psi_j and s = (-1)^popcount(i0 & z):
//   <psi|P|psi> = sum_{i0} s * ( (-1)^(y/2)     * 2 Re zc   if y is even,
//                                (-1)^((y-1)/2) * 2 Im zc   if y is odd ),
// and for x = 0 it is sum_i s(i) |psi_i|^2.  Products of FP32 amplitudes are
// exact in FP64; every sum is FP64 in a fixed order (per lane, then a wave
// butterfly, then the waves of a workgroup, then the workgroups in index
// order), so results are deterministic.  The reference reduces in FP32 with
// atomicAdd and handles a Z string or one X/Y qubit only
// (bwk/csrc/expectation_sm120.cu:45-163).
//
// Memory layout follows the gate kernels: a wave owns a window of 64
// float4 slots (128 amplitudes, 1 KiB).  When x < 128 the partner of every
// amplitude is in the same window (a cross-lane swap by x >> 1, plus a swap
// inside the float4 when x & 1); when x >= 128 the wave owns the window pair
// (w, w ^ (x >> 7)) with bit h - 7 of w clear, h the highest bit of x.  Each
// amplitude is read once, by whole-line 1 KiB loads.
#include <algorithm>
#include <vector>

#include "qsim_internal.hpp"

namespace qsim {

constexpr int kExpMaxTerms = 8;   // terms sharing one x mask per state pass

struct ExpTerms {
  uint64_t z[kExpMaxTerms];
  double fac[kExpMaxTerms];       // +-1 (x = 0) or +-2 (x != 0)
  int out[kExpMaxTerms];          // output slot, -1 = discard (padding)
  int im;                         // every term of the pass takes Im(zc) (else Re(zc))
};

__device__ __forceinline__ double wsum64(double v) {
#pragma unroll
  for (int m = 32; m >= 1; m >>= 1) v += lane_xor(v, m);
  return v;
}

// Pass 1.  Units are windows (KIND 0: x == 0; KIND 1: 0 < x < 128) or window
// pairs (KIND 2: x >= 128); workgroup b reduces units [b*chunk, (b+1)*chunk),
// wave k of it takes units k, k+4, ...  part[b*NT + j] = the workgroup's sum
// for term j.
//
// Amplitude i = 128 w + 2 lane + c (window w, lane, c = 0/1 in the float4),
// so the sign (-1)^popcount(i & z) factors into a lane constant (bits 0..6,
// folded with the term's factor and, for KIND 1, with the "highest x bit
// clear" selection into k_c) and a window sign that is the same for the
// whole wave (computed on the scalar unit).  Per slot and term that leaves
// t = v_0 k_0 + v_1 k_1 and acc += ws * t, with v_c = |a_c|^2 (KIND 0) or
// Re / Im of conj(a_c) * partner_c.
template <int NT, int KIND, bool NTL>
__global__ __launch_bounds__(kThreads) void k_expect(const float4* __restrict__ st, uint64_t n4,
                                                     uint64_t n_units, uint64_t chunk, uint64_t x,
                                                     int hw, ExpTerms a, double* __restrict__ part) {
  __shared__ double sh[NT][4];
  const int lane = threadIdx.x & 63;
  const int wid = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const uint64_t beg = (uint64_t)blockIdx.x * chunk;
  const uint64_t end = beg + chunk < n_units ? beg + chunk : n_units;
  const int xl = (int)((x >> 1) & 63), csw = (int)(x & 1);
  const int h = x ? 63 - __clzll(x) : 0;
  const uint64_t xw = x >> 7;
  double acc[NT], k0[NT], k1[NT];
#pragma unroll
  for (int j = 0; j < NT; ++j) {
    acc[j] = 0.0;
    const uint32_t zl = (uint32_t)(a.z[j] & 127);
    const uint32_t i0 = 2 * lane, i1 = 2 * lane + 1;
    const bool t0 = KIND != 1 || !((i0 >> h) & 1), t1 = KIND != 1 || !((i1 >> h) & 1);
    k0[j] = t0 ? ((__popc(i0 & zl) & 1) ? -a.fac[j] : a.fac[j]) : 0.0;
    k1[j] = t1 ? ((__popc(i1 & zl) & 1) ? -a.fac[j] : a.fac[j]) : 0.0;
  }
  constexpr int U = KIND == 2 ? 2 : 4;   // units in flight per wave
  const float4 zero = make_float4(0.f, 0.f, 0.f, 0.f);
  for (uint64_t u0 = beg + wid; u0 < end; u0 += 4 * U) {
    float4 v[U], p[U];
    uint64_t wk[U];
#pragma unroll
    for (int k = 0; k < U; ++k) {
      const uint64_t u = u0 + 4 * k;
      wk[k] = KIND == 2 ? ins0(u, hw) : u;
      const uint64_t sl = wk[k] * 64 + lane;
      const bool ok = u < end && sl < n4;
      v[k] = ok ? ld4<NTL>(st + sl) : zero;
      if (KIND == 2) p[k] = ok ? ld4<NTL>(st + ((wk[k] ^ xw) * 64 + lane)) : zero;
    }
#pragma unroll
    for (int k = 0; k < U; ++k) {
      if (KIND == 1) p[k] = shfl_xor4(v[k], xl);
      if (KIND == 2) p[k] = shfl_xor4(p[k], xl);
      if (u0 + 4 * k >= end) continue;
      double v0, v1;
      if (KIND == 0) {
        v0 = (double)v[k].x * v[k].x + (double)v[k].y * v[k].y;
        v1 = (double)v[k].z * v[k].z + (double)v[k].w * v[k].w;
      } else {
        const float2 a0 = lo2(v[k]), a1 = hi2(v[k]);
        const float2 b0 = csw ? hi2(p[k]) : lo2(p[k]), b1 = csw ? lo2(p[k]) : hi2(p[k]);
        if (a.im) {
          v0 = (double)a0.x * b0.y - (double)a0.y * b0.x;
          v1 = (double)a1.x * b1.y - (double)a1.y * b1.x;
        } else {
          v0 = (double)a0.x * b0.x + (double)a0.y * b0.y;
          v1 = (double)a1.x * b1.x + (double)a1.y * b1.y;
        }
      }
      const uint64_t wb = wk[k] * 128;
#pragma unroll
      for (int j = 0; j < NT; ++j) {
        const double ws = (__popcll(wb & a.z[j]) & 1) ? -1.0 : 1.0;
        // k and ws are 0, +-1 or +-2, so the products are exact and the
        // fused forms round exactly as the separate ones would
        const double t = __builtin_fma(v1, k1[j], v0 * k0[j]);
        acc[j] = __builtin_fma(ws, t, acc[j]);
      }
    }
  }
#pragma unroll
  for (int j = 0; j < NT; ++j) {
    const double r = wsum64(acc[j]);
    if (lane == 0) sh[j][wid] = r;
  }
  __syncthreads();
  if (threadIdx.x < NT) {
    const int j = threadIdx.x;
    part[(uint64_t)blockIdx.x * NT + j] = (sh[j][0] + sh[j][1]) + (sh[j][2] + sh[j][3]);
  }
}

// Pass 2: one workgroup sums each of the NT columns of part[nb][NT] in index
// order and writes term j to out[a.out[j]] (padding terms are dropped).
template <int NT>
__global__ __launch_bounds__(kThreads) void k_expect_final(const double* __restrict__ part, int nb,
                                                           ExpTerms a, double* __restrict__ out) {
  __shared__ double sh[NT][4];
  const int lane = threadIdx.x & 63, wid = threadIdx.x >> 6;
  double acc[NT];
#pragma unroll
  for (int j = 0; j < NT; ++j) acc[j] = 0.0;
  for (int b = threadIdx.x; b < nb; b += kThreads) {
#pragma unroll
    for (int j = 0; j < NT; ++j) acc[j] += part[(int64_t)b * NT + j];
  }
#pragma unroll
  for (int j = 0; j < NT; ++j) {
    const double r = wsum64(acc[j]);
    if (lane == 0) sh[j][wid] = r;
  }
  __syncthreads();
  if (threadIdx.x < NT) {
    const int j = threadIdx.x;
    if (a.out[j] >= 0) out[a.out[j]] = (sh[j][0] + sh[j][1]) + (sh[j][2] + sh[j][3]);
  }
}

template <int NT, int KIND>
static void launch_expect(hipStream_t s, const void* state, int n, uint64_t x, const ExpTerms& a,
                          double* part, double* out) {
  const uint64_t n4 = (1ull << n) / 2;
  const uint64_t windows = ceil_div(n4, 64);
  const uint64_t n_units = KIND == 2 ? windows / 2 : windows;
  const int hw = KIND == 2 ? (63 - __builtin_clzll(x)) - 7 : 0;
  const uint64_t want = ceil_div(n_units, 16);   // 4 waves x 4 units per workgroup
  const int blocks = (int)(want < (uint64_t)kRedBlocks ? (want ? want : 1) : kRedBlocks);
  const uint64_t chunk = ceil_div(n_units, blocks);
  // NTL: nontemporal loads above the MALL size
  if (nt_for_qubits(n))
    hipLaunchKernelGGL((k_expect<NT, KIND, true>), dim3(blocks), dim3(kThreads), 0, s,
                       (const float4*)state, n4, n_units, chunk, x, hw, a, part);
  else
    hipLaunchKernelGGL((k_expect<NT, KIND, false>), dim3(blocks), dim3(kThreads), 0, s,
                       (const float4*)state, n4, n_units, chunk, x, hw, a, part);
  hipLaunchKernelGGL((k_expect_final<NT>), dim3(1), dim3(kThreads), 0, s, part, blocks, a, out);
}

template <int NT>
static void launch_expect_kind(hipStream_t s, const void* state, int n, uint64_t x,
                               const ExpTerms& a, double* part, double* out) {
  if (x == 0) launch_expect<NT, 0>(s, state, n, x, a, part, out);
  else if (x < 128) launch_expect<NT, 1>(s, state, n, x, a, part, out);
  else launch_expect<NT, 2>(s, state, n, x, a, part, out);
}

// Tiled pass: many term groups per read of the state.  A workgroup copies a
// tile of 2^M amplitudes (M qubits, among them the lowest 4, so that loads are
// whole 128-byte lines) into LDS and evaluates there every group whose x mask
// lies inside the tile's qubits.  x and the part of z inside the tile arrive
// as tile-local masks; the rest of z gives one sign per tile.
//
// A unit of work is a group (up to 8 terms of one x mask and one Y parity)
// and one of 2^seg equal parts of its index pairs.  A wave takes them 64 slots
// (two amplitudes each) at a time: with i0 = the slots whose highest x bit is
// clear, a slot index splits into a lane part and a wave part, so both LDS
// addresses are a lane constant plus a wave constant, and the sign of a term
// is a lane constant (applied once, to the unit's sum) times a wave sign,
// taken from a bit mask over the unit's steps that one ballot computes.  Every
// unit belongs to one wave, which adds its reduced sum to the unit's LDS slot
// tile after tile; slots are added in order at the end, so sums are
// deterministic as before.
//
// What bounds it: vector issue (busy 59 % of the time before groups shared
// units, 29 % of it conversions to FP64), then the tile loads, which do not
// overlap it.  The 4 n - 3 terms of a Heisenberg chain, plain passes (two
// launches and a read of the state per group) -> tiled passes -> units of two
// groups: 20 / 22 / 24 / 26 qubits 302 / - / 1208 / - -> 43 / 83 / 254 / 975 ->
// 38.5 / 72 / 212 / 804 us; 12 and 16 qubits 151 and 245 -> 27 and 38.  Measured
// and not taken, at 28 qubits and 4000 us: the next tile loaded into registers
// during the evaluation 4290 us, tiles of 2^12 at 256 threads 4556, 1024 threads
// 4675 (two parts a group; 512 threads there 4713).
struct ExpGroup {
  uint16_t x;                     // tile-local x mask
  uint8_t h, im;                  // its highest bit; Im(zc) instead of Re(zc)
  uint16_t t0, nt;                // terms [t0, t0 + nt), nt <= kExpMaxTerms
  uint16_t zl[4];                 // tile-local z masks of the first four
  uint16_t x2;                    // not 0: two groups, the second with this x mask (exp_unit2)
  uint8_t lo, hi;                 // their pivot bits, lo < hi
};
struct ExpTerm {
  uint64_t z;                     // z mask outside the tile
  uint16_t zl;                    // tile-local z mask
  int16_t fac;                    // +-1 (x = 0) or +-2
  int32_t out;
};
constexpr int kPassGroups = 64, kPassTerms = 144, kPassBlocks = 512, kPassThreads = 512;
constexpr int kPassWaves = kPassThreads / 64, kExpTileMax = 13, kExpTileMin = 10;
// A pass of two groups already beats two plain passes: 24 qubits 30 against
// 49 us, 28 qubits 340 against 635; a single group stays on the plain pass.
constexpr int kPassMinGroups = 2;
constexpr size_t kPassWindow = 2048;   // groups looked at per pass: planning stays linear in their number
// Smallest state whose groups share units: energies of chains of 12 / 14 / 18
// qubits 27.3 / 39.4 / 39.6 us apart against 29.4 / 40.5 / 40.8 joined, 20 / 22 /
// 24 / 26 qubits 43 / 83 / 254 / 975 against 38.5 / 72 / 212 / 804.
constexpr int kJoinMinQubits = 20;
struct ExpPass {
  uint32_t tq[4];                 // tile qubits, ascending, one byte each; the first four are 0..3
  int n_groups, n_terms, seg;
  ExpGroup g[kPassGroups];
  ExpTerm t[kPassTerms];
};
static_assert(sizeof(ExpPass) <= 3712, "kernel arguments");
__host__ __device__ inline int exp_tq(const ExpPass& a, int j) { return (int)((a.tq[j >> 2] >> (8 * (j & 3))) & 255u); }

// Sums of a unit kept per term: the lanes are added over the lane bits whose
// exchange is a DPP or permlane move (0, 1, 3, 5); bits 2 and 4, whose exchange
// goes through the LDS unit, stay apart until the end.
constexpr int kSlotLanes = 4;

// Kinds of a group: x = 0; x = 1 (pairs inside a slot); x > 1 even; x > 1 odd.
enum { kDiag, kInSlot, kPair, kPairSwap };

// Adds a unit's lane sums of term j, with its lane and tile signs, to its slot.
__device__ __forceinline__ void exp_unit_sum(const ExpPass& a, const ExpGroup& g, int j, double acc, uint32_t il,
                                             uint64_t base, uint32_t lane, double* slot) {
  const ExpTerm t = a.t[g.t0 + j];
  const int minus = (__popc(il & (uint32_t)(t.zl >> 1)) + __popcll(base & t.z)) & 1;
  double r = acc * (double)(minus ? -t.fac : t.fac);
  r += lane_xor(r, 1);
  r += lane_xor(r, 2);
  r += lane_xor(r, 8);
  r += lane_xor(r, 32);
  if ((lane & 0x2b) == 0) slot[(j << a.seg) * kSlotLanes + (lane >> 4) * 2 + (lane >> 2 & 1)] += r;
}

// A unit's sums for its NT terms: steps of 64 slots from slot step p0 on.
template <int NT, bool IM, int KIND>
__device__ __forceinline__ void exp_unit(const char* Xb, const ExpPass& a, const ExpGroup g, uint32_t p0,
                                         uint32_t steps, uint64_t base, uint32_t lane, double* slot) {
  constexpr int U = 4;
  constexpr bool pair = KIND >= kPair;
  const int hs = (int)g.h - 1;
  const uint32_t xs = g.x >> 1, lm = pair && hs < 6 ? 127u : 63u;
  auto clear_h = [&](uint32_t p) -> uint32_t { return pair ? ins0(p, hs) : p; };
  const uint32_t il = clear_h(lane);
  const uint32_t la = il * 16, lb = (il ^ (xs & lm)) * 16, xw = xs & ~lm;
  double acc[NT], c1[NT];
  uint64_t neg[NT];                       // bit k: the wave sign of step k is -1
#pragma unroll
  for (int j = 0; j < NT; ++j) {
    const uint32_t z = j < 4 ? g.zl[j] : a.t[g.t0 + (j < g.nt ? j : 0)].zl;
    acc[j] = 0.0;
    c1[j] = (z & 1) ? -1.0 : 1.0;
    neg[j] = __ballot(__popc(clear_h((p0 + lane) * 64) & (z >> 1)) & 1);
  }
  for (uint32_t k0 = 0; k0 < steps; k0 += U) {
#pragma unroll
    for (int q = 0; q < U; ++q) {
      const uint32_t iw = clear_h((p0 + k0 + q) * 64);
      const float4 u = *reinterpret_cast<const float4*>(Xb + (la + iw * 16));
      double v0, v1 = 0.0;
      auto prod = [](float2 x, float2 y) -> double {
        return IM ? (double)x.x * y.y - (double)x.y * y.x : (double)x.x * y.x + (double)x.y * y.y;
      };
      if (KIND == kDiag) {
        v0 = prod(lo2(u), lo2(u));
        v1 = prod(hi2(u), hi2(u));
      } else if (KIND == kInSlot) {
        v0 = prod(lo2(u), hi2(u));
      } else {
        const float4 w = *reinterpret_cast<const float4*>(Xb + (lb + (iw ^ xw) * 16));
        v0 = prod(lo2(u), KIND == kPairSwap ? hi2(w) : lo2(w));
        v1 = prod(hi2(u), KIND == kPairSwap ? lo2(w) : hi2(w));
      }
#pragma unroll
      for (int j = 0; j < NT; ++j) {
        const uint32_t m = (uint32_t)(neg[j] >> k0);
        const double t = KIND == kInSlot ? v0 : __builtin_fma(c1[j], v1, v0);
        acc[j] = __builtin_fma(__hiloint2double((m >> q & 1u) ? (int)0xbff00000 : 0x3ff00000, 0), t, acc[j]);
      }
    }
  }
#pragma unroll
  for (int j = 0; j < NT; ++j) {
    if (j >= g.nt) continue;
    exp_unit_sum(a, g, j, acc[j], il, base, lane, slot);
  }
}

// A unit of two groups (even x masks, real parts, NA and NB terms): the four
// slots i, i ^ x, i ^ x2 and i ^ x ^ x2 hold two pairs of either group, so
// four slots are converted to FP64 for four pairs, where two units convert four
// for two.  i runs over the slots with both pivot bits clear; the sign of the
// second pair of a group is that of the first times the other mask's.
template <int NA, int NB>
__device__ __forceinline__ void exp_unit2(const char* Xb, const ExpPass& a, const ExpGroup g, uint32_t p0,
                                          uint32_t steps, uint64_t base, uint32_t lane, double* slot) {
  constexpr int U = 2, NT = NA + NB;
  auto clear = [&](uint32_t p) -> uint32_t { return ins0(ins0(p, (int)g.lo - 1), (int)g.hi - 1); };
  const uint32_t il = clear(lane), la = il * 16;
  const uint32_t xa = (g.x >> 1) * 16u, xb = (g.x2 >> 1) * 16u;
  double acc[NT], c1[NT], c2[NT];
  uint64_t neg[NT];                       // bit k: the wave sign of step k is -1
#pragma unroll
  for (int j = 0; j < NT; ++j) {
    const uint32_t z = g.zl[j];
    acc[j] = 0.0;
    c1[j] = (z & 1) ? -1.0 : 1.0;
    c2[j] = (__popc(z & (j < NA ? g.x2 : g.x)) & 1) ? -1.0 : 1.0;
    neg[j] = __ballot(__popc(clear((p0 + lane) * 64) & (z >> 1)) & 1);
  }
  auto dot = [](const double (&x)[4], const double (&y)[4], int e) -> double {
    return x[2 * e] * y[2 * e] + x[2 * e + 1] * y[2 * e + 1];
  };
  for (uint32_t k0 = 0; k0 < steps; k0 += U) {
#pragma unroll
    for (int q = 0; q < U; ++q) {
      const uint32_t iw = clear((p0 + k0 + q) * 64) * 16;
      auto slot_at = [&](uint32_t x, double (&d)[4]) {
        const float4 v = *reinterpret_cast<const float4*>(Xb + (la ^ (iw ^ x)));
        d[0] = v.x; d[1] = v.y; d[2] = v.z; d[3] = v.w;
      };
      double v0[4], va[4], vb[4], vc[4];
      slot_at(0, v0);
      slot_at(xa, va);
      slot_at(xb, vb);
      slot_at(xa ^ xb, vc);
      double p[2][2], r[2][2];              // first and second pair of either group, per amplitude of a slot
#pragma unroll
      for (int e = 0; e < 2; ++e) {
        p[0][e] = dot(v0, va, e);
        r[0][e] = dot(vb, vc, e);
        p[1][e] = dot(v0, vb, e);
        r[1][e] = dot(va, vc, e);
      }
#pragma unroll
      for (int j = 0; j < NT; ++j) {
        const int b = j < NA ? 0 : 1;
        const uint32_t m = (uint32_t)(neg[j] >> k0);
        const double t = __builtin_fma(c1[j], __builtin_fma(c2[j], r[b][1], p[b][1]),
                                       __builtin_fma(c2[j], r[b][0], p[b][0]));
        acc[j] = __builtin_fma(__hiloint2double((m >> q & 1u) ? (int)0xbff00000 : 0x3ff00000, 0), t, acc[j]);
      }
    }
  }
#pragma unroll
  for (int j = 0; j < NT; ++j) exp_unit_sum(a, g, j, acc[j], il, base, lane, slot);
}

template <int M, bool NTL>
__global__ __launch_bounds__(kPassThreads) void k_expect_tile(ExpPass args, const float4* __restrict__ st,
                                                              uint64_t n_tiles, double* __restrict__ part) {
  // read in place by scalar loads: indexed through `args` itself, the compiler
  // copied all of it to scratch (93 terms, 24 qubits: 783 against 272 us)
  const ExpPass& a = *(const ExpPass*)__builtin_amdgcn_kernarg_segment_ptr();
  extern __shared__ float4 X4[];
  const char* Xb = reinterpret_cast<const char*>(X4);
  double* slots = reinterpret_cast<double*>(X4 + (1 << (M - 1)));
  constexpr int TB = __builtin_ctz(kPassThreads);
  constexpr int SLOTS = (1 << (M - 1)) / kPassThreads;
  const uint32_t tid = threadIdx.x, lane = tid & 63;
  const uint32_t wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int per_term = kSlotLanes << a.seg;
  const uint32_t units = (uint32_t)a.n_groups << a.seg;
  auto group = [&](uint32_t u) -> ExpGroup { return a.g[(u < units ? u : units - 1) >> a.seg]; };
  for (int i = tid; i < a.n_terms * per_term; i += kPassThreads) slots[i] = 0.0;
  uint64_t toff = 0;
#pragma unroll
  for (int j = 0; j < TB; ++j) toff |= (uint64_t)((tid >> j) & 1) << (exp_tq(a, j + 1) - 1);
  for (uint64_t tile = blockIdx.x; tile < n_tiles; tile += gridDim.x) {
    uint64_t base = tile;
#pragma unroll
    for (int j = 0; j < M; ++j) base = ins0(base, exp_tq(a, j));
    float4 v[SLOTS];
#pragma unroll
    for (int k = 0; k < SLOTS; ++k) {
      uint64_t off = base >> 1;
#pragma unroll
      for (int j = TB; j < M - 1; ++j) off |= (uint64_t)((k >> (j - TB)) & 1) << (exp_tq(a, j + 1) - 1);
      v[k] = ld4<NTL>(st + (off + toff));
    }
    __syncthreads();              // the tile before has been read
#pragma unroll
    for (int k = 0; k < SLOTS; ++k) X4[k * kPassThreads + tid] = v[k];
    __syncthreads();
    ExpGroup next = group(wave);
    for (uint32_t u = wave; u < units; u += kPassWaves) {
      const ExpGroup g = next;
      next = group(u + kPassWaves);
      const uint32_t part_no = u & ((1u << a.seg) - 1u);
      const uint32_t steps = (1u << (g.x2 ? M - 9 : g.x > 1 ? M - 8 : M - 7)) >> a.seg;
      double* slot = slots + (((uint32_t)g.t0 << a.seg) + part_no) * kSlotLanes;
#define QSIM_UNIT(NT, IM, KIND) exp_unit<NT, IM, KIND>(Xb, a, g, part_no * steps, steps, base, lane, slot)
#define QSIM_UNIT_NT(IM, KIND)                 \
  do {                                         \
    if (g.nt == 1) QSIM_UNIT(1, IM, KIND);     \
    else if (g.nt == 2) QSIM_UNIT(2, IM, KIND); \
    else QSIM_UNIT(8, IM, KIND);               \
  } while (0)
      if (g.x2) {
        const uint32_t s0 = part_no * steps;
        if (g.nt == 2) exp_unit2<1, 1>(Xb, a, g, s0, steps, base, lane, slot);
        else if (g.nt == 3) exp_unit2<1, 2>(Xb, a, g, s0, steps, base, lane, slot);
        else exp_unit2<2, 2>(Xb, a, g, s0, steps, base, lane, slot);
      } else if (g.x == 0) {
        if (g.nt <= 4) QSIM_UNIT(4, false, kDiag);
        else QSIM_UNIT(8, false, kDiag);
      } else if (g.x == 1) {
        if (g.im) QSIM_UNIT(8, true, kInSlot);
        else QSIM_UNIT(8, false, kInSlot);
      } else if (g.im) {
        if (g.x & 1) QSIM_UNIT_NT(true, kPairSwap);
        else QSIM_UNIT_NT(true, kPair);
      } else {
        if (g.x & 1) QSIM_UNIT_NT(false, kPairSwap);
        else QSIM_UNIT_NT(false, kPair);
      }
#undef QSIM_UNIT_NT
#undef QSIM_UNIT
    }
  }
  __syncthreads();
  for (int t = tid; t < a.n_terms; t += kPassThreads) {
    double r = 0.0;
    for (int i = 0; i < per_term; ++i) r += slots[t * per_term + i];
    part[(uint64_t)t * gridDim.x + blockIdx.x] = r;
  }
}

// One wave per term adds its nb partials in index order per lane, then the lanes.
__global__ __launch_bounds__(64) void k_expect_tile_final(const double* __restrict__ part, int nb, ExpPass a,
                                                          double* __restrict__ out) {
  double r = 0.0;
  for (int b = threadIdx.x; b < nb; b += 64) r += part[(uint64_t)blockIdx.x * nb + b];
  r = wsum64(r);
  if (threadIdx.x == 0) out[a.t[blockIdx.x].out] = r;
}

template <int M>
static void launch_expect_tile(hipStream_t s, const void* state, int n, const ExpPass& a, double* part, double* out) {
  const uint64_t tiles = 1ull << (n - M);
  const int blocks = (int)std::min<uint64_t>(tiles, kPassBlocks);
  const size_t lds = (sizeof(float2) << M) + ((size_t)a.n_terms * kSlotLanes * sizeof(double) << a.seg);
  auto* kern = nt_for_qubits(n) ? k_expect_tile<M, true> : k_expect_tile<M, false>;
  hipLaunchKernelGGL(kern, dim3(blocks), dim3(kPassThreads), lds, s, a, (const float4*)state, tiles, part);
  hipLaunchKernelGGL(k_expect_tile_final, dim3(a.n_terms), dim3(64), 0, s, part, blocks, a, out);
}

// Workspace (doubles): a plain pass's partials [kRedBlocks][kExpMaxTerms] or a
// tiled pass's [kPassTerms][kPassBlocks].
constexpr int64_t kExpWsDoubles =
    std::max((int64_t)kRedBlocks * kExpMaxTerms, (int64_t)kPassTerms * kPassBlocks);

// One group: terms order[beg, beg + cnt) with one x mask and Y parity.
struct TermGroup {
  uint64_t x;
  int im, beg, cnt;
  bool done;
};

static int pair_factor(uint64_t x, uint64_t z) {
  return x == 0 ? 1 : ((__builtin_popcountll(x & z) >> 1) & 1) ? -2 : 2;
}
// The bits of v at the positions set in m, packed (v within m).
static uint32_t pack_bits(uint64_t v, uint64_t m) {
  uint32_t r = 0;
  for (int j = 0; m; ++j, m &= m - 1)
    if (v & m & (0 - m)) r |= 1u << j;
  return r;
}

static int expectation_impl(hipStream_t s, const void* state, int n, int64_t n_terms,
                            const uint64_t* xm, const uint64_t* zm, double* ws, double* out) {
  if (int rc = check_n(n)) return rc;
  if (n_terms < 0) return fail(QSIM_EINVAL, "n_terms < 0");
  if (n_terms == 0) return QSIM_OK;
  if (!state || !xm || !zm || !ws || !out) return fail(QSIM_EINVAL, "NULL pointer argument");
  const uint64_t lim = 1ull << n;
  for (int64_t k = 0; k < n_terms; ++k)
    if (xm[k] >= lim || zm[k] >= lim)
      return fail(QSIM_EINVAL, "Pauli term %lld: mask has a qubit >= n_qubits (%d)", (long long)k, n);
  // terms sharing an x mask and the parity of their Y count (Re or Im of
  // the pair products) share the pair products: visit them grouped, in input
  // order within a group
  std::vector<int64_t> order(n_terms);
  for (int64_t k = 0; k < n_terms; ++k) order[k] = k;
  auto key = [xm, zm](int64_t k) {
    return std::make_pair(xm[k], __builtin_popcountll(xm[k] & zm[k]) & 1);
  };
  std::stable_sort(order.begin(), order.end(),
                   [&key](int64_t a, int64_t b) { return key(a) < key(b); });
  std::vector<TermGroup> groups;
  for (int64_t g = 0; g < n_terms;) {
    const auto k0 = key(order[g]);
    int cnt = 1;
    while (g + cnt < n_terms && cnt < kExpMaxTerms && key(order[g + cnt]) == k0) ++cnt;
    groups.push_back({k0.first, k0.second, (int)g, cnt, false});
    g += cnt;
  }
  // Tiled passes: the first group not done opens a tile, and every later one
  // whose x mask still fits joins.
  const int m = n < kExpTileMin ? 0 : n < kExpTileMax ? n : kExpTileMax;
  for (size_t first = 0; m && first < groups.size(); ++first) {
    if (groups[first].done || __builtin_popcountll(groups[first].x | 15) > m) continue;
    uint64_t tile = 15;
    std::vector<size_t> in;
    int terms = 0;
    const size_t last = std::min(groups.size(), first + kPassWindow);
    for (size_t i = first; i < last && in.size() < (size_t)kPassGroups; ++i) {
      const TermGroup& g = groups[i];
      if (g.done || __builtin_popcountll(tile | g.x) > m || terms + g.cnt > kPassTerms) continue;
      tile |= g.x;
      terms += g.cnt;
      in.push_back(i);
    }
    if (in.size() < (size_t)kPassMinGroups) continue;
    for (int q = 0; __builtin_popcountll(tile) < m; ++q) tile |= 1ull << q;
    ExpPass a = {};
    uint64_t rest = tile;
    for (int j = 0; j < m; ++j, rest &= rest - 1) a.tq[j >> 2] |= (uint32_t)__builtin_ctzll(rest) << (8 * (j & 3));
    a.n_terms = terms;
    int t = 0;
    auto add_terms = [&](ExpGroup& e, TermGroup& g) {
      for (int j = 0; j < g.cnt; ++j, ++t, ++e.nt) {
        const int64_t k = order[g.beg + j];
        a.t[t] = {zm[k] & ~tile, (uint16_t)pack_bits(zm[k] & tile, tile), (int16_t)pair_factor(g.x, zm[k]), (int32_t)k};
        if (e.nt < 4) e.zl[e.nt] = a.t[t].zl;
      }
      g.done = true;
    };
    // groups of one or two terms that share a unit, in pairs as they come, where
    // there are tiles enough to keep the chip busy
    auto joins = [&](const TermGroup& g) {
      return n >= kJoinMinQubits && g.x && !(g.x & 1) && !g.im && g.cnt <= 2;
    };
    for (size_t i = 0; i < in.size(); ++i) {
      TermGroup* g = &groups[in[i]];
      if (g->done) continue;
      TermGroup* other = nullptr;
      for (size_t k = i + 1; k < in.size() && joins(*g) && !other; ++k)
        if (!groups[in[k]].done && joins(groups[in[k]])) other = &groups[in[k]];
      if (other && other->cnt < g->cnt) std::swap(g, other);
      ExpGroup& e = a.g[a.n_groups++];
      const uint32_t x = pack_bits(g->x, tile);
      e.x = (uint16_t)x;
      e.h = (uint8_t)(x ? 31 - __builtin_clz(x) : 0);
      e.im = (uint8_t)g->im;
      e.t0 = (uint16_t)t;
      add_terms(e, *g);
      if (other) {
        const uint32_t x2 = pack_bits(other->x, tile), y = x2 >> e.h & 1 ? x2 ^ x : x2;
        const int h2 = 31 - __builtin_clz(y);
        e.x2 = (uint16_t)x2;
        e.lo = (uint8_t)std::min<int>(e.h, h2);
        e.hi = (uint8_t)std::max<int>(e.h, h2);
        add_terms(e, *other);
      }
    }
    // the fewest parts that give each wave a unit (28 qubits, 93 terms: 3.99 ms
    // with one part, 4.59 with two, 4.90 with four; 2 groups: 355 us with two
    // parts, 340 with four), and at least 4 steps a unit of one group
    a.seg = std::min(a.n_groups >= kPassWaves ? 0 : a.n_groups >= kPassWaves / 2 ? 1 : 2, m - 10);
    switch (m) {
      case 10: launch_expect_tile<10>(s, state, n, a, ws, out); break;
      case 11: launch_expect_tile<11>(s, state, n, a, ws, out); break;
      case 12: launch_expect_tile<12>(s, state, n, a, ws, out); break;
      default: launch_expect_tile<13>(s, state, n, a, ws, out); break;
    }
    if (int rc = launch_status("expectation")) return rc;
  }
  for (const TermGroup& g : groups) {
    if (g.done) continue;
    const uint64_t x = g.x;
    const int cnt = g.cnt;
    ExpTerms a = {};
    a.im = g.im;
    for (int j = 0; j < cnt; ++j) {
      const int64_t k = order[g.beg + j];
      a.z[j] = zm[k];
      a.out[j] = (int)k;
      a.fac[j] = pair_factor(x, zm[k]);
    }
    for (int j = cnt; j < kExpMaxTerms; ++j) { a.out[j] = -1; a.fac[j] = 0.0; }
    if (cnt == 1) launch_expect_kind<1>(s, state, n, x, a, ws, out);
    else if (cnt == 2) launch_expect_kind<2>(s, state, n, x, a, ws, out);
    else if (cnt <= 4) launch_expect_kind<4>(s, state, n, x, a, ws, out);
    else launch_expect_kind<8>(s, state, n, x, a, ws, out);
    if (int rc = launch_status("expectation")) return rc;
  }
  return QSIM_OK;
}

// ------------------------------------------------------------ apply P
// psi <- P psi, exact: every output amplitude is an input amplitude with its
// components swapped and/or negated.  KIND as for k_expect; one wave per
// window (KIND 0, 1) or window pair (KIND 2).  KIND 3 is x = 0 with no z bit
// below 7: the sign is one per window, (-1)^popcount(w & (z >> 7)), so only
// the half of the windows whose sign is -1 is visited (unit u inserts the
// highest bit hw of z >> 7 into u, set so that the parity is odd).
__device__ __forceinline__ float2 quarter_turn(float2 a, int k) {
  switch (k & 3) {
    case 0: return a;
    case 1: return make_float2(-a.y, a.x);     // * i
    case 2: return make_float2(-a.x, -a.y);    // * -1
    default: return make_float2(a.y, -a.x);    // * -i
  }
}

// New slot s from partner float4 p: amplitude i = 2s + c takes
// i^y (-1)^popcount((i ^ x) & z) psi_{i ^ x}.
__device__ __forceinline__ float4 pauli_slot(float4 p, uint64_t s, uint64_t x, uint64_t z, int y,
                                             int csw) {
  float2 r[2];
#pragma unroll
  for (int c = 0; c < 2; ++c) {
    const uint64_t i = 2 * s + c;
    const float2 b = (c ^ csw) ? hi2(p) : lo2(p);
    r[c] = quarter_turn(b, y + 2 * (int)(__popcll((i ^ x) & z) & 1));
  }
  return cat4(r[0], r[1]);
}

template <int KIND, bool NT>
__global__ __launch_bounds__(kThreads) void k_pauli_apply(float4* __restrict__ st, uint64_t n4,
                                                          uint64_t n_units, uint64_t x, uint64_t z,
                                                          int y, int hw) {
  const uint64_t u = xcd_block<uint64_t>() * 4 + (threadIdx.x >> 6);
  if (u >= n_units) return;
  const int lane = threadIdx.x & 63;
  if (KIND == 3) {
    const uint64_t w0 = ins0(u, hw);
    const uint64_t w = (__popcll(w0 & (z >> 7)) & 1) ? w0 : (w0 | (1ull << hw));
    const uint64_t s = w * 64 + lane;
    const float4 v = ld4<NT>(st + s);
    st4<NT>(st + s, make_float4(-v.x, -v.y, -v.z, -v.w));
    return;
  }
  const int xl = (int)((x >> 1) & 63), csw = (int)(x & 1);
  if (KIND == 2) {
    const uint64_t w0 = ins0(u, hw), w1 = w0 ^ (x >> 7);
    const uint64_t s0 = w0 * 64 + lane, s1 = w1 * 64 + lane;
    const float4 v0 = ld4<NT>(st + s0), v1 = ld4<NT>(st + s1);
    const float4 p0 = shfl_xor4(v1, xl), p1 = shfl_xor4(v0, xl);
    st4<NT>(st + s0, pauli_slot(p0, s0, x, z, y, csw));
    st4<NT>(st + s1, pauli_slot(p1, s1, x, z, y, csw));
    return;
  }
  const uint64_t s = u * 64 + lane;
  const bool ok = s < n4;
  const float4 v = ok ? ld4<NT>(st + s) : make_float4(0.f, 0.f, 0.f, 0.f);
  const float4 p = KIND == 1 ? shfl_xor4(v, xl) : v;
  if (ok) st4<NT>(st + s, pauli_slot(p, s, x, z, y, csw));
}

template <bool NT>
static void launch_pauli(hipStream_t s, void* state, uint64_t n4, uint64_t windows, uint64_t x,
                         uint64_t z, int y) {
  if (x == 0 && (z & 127) == 0) {
    const int hw = (63 - __builtin_clzll(z >> 7));
    hipLaunchKernelGGL((k_pauli_apply<3, NT>), grid1d(ceil_div(windows / 2, 4)), dim3(kThreads), 0, s,
                       (float4*)state, n4, windows / 2, x, z, y, hw);
  } else if (x == 0) {
    hipLaunchKernelGGL((k_pauli_apply<0, NT>), grid1d(ceil_div(windows, 4)), dim3(kThreads), 0, s,
                       (float4*)state, n4, windows, x, z, y, 0);
  } else if (x < 128) {
    hipLaunchKernelGGL((k_pauli_apply<1, NT>), grid1d(ceil_div(windows, 4)), dim3(kThreads), 0, s,
                       (float4*)state, n4, windows, x, z, y, 0);
  } else {
    const int hw = (63 - __builtin_clzll(x)) - 7;
    hipLaunchKernelGGL((k_pauli_apply<2, NT>), grid1d(ceil_div(windows / 2, 4)), dim3(kThreads), 0, s,
                       (float4*)state, n4, windows / 2, x, z, y, hw);
  }
}

static int pauli_apply_impl(hipStream_t s, void* state, int n, uint64_t x, uint64_t z) {
  if (int rc = check_n(n)) return rc;
  if (!state) return fail(QSIM_EINVAL, "state is NULL");
  const uint64_t lim = 1ull << n;
  if (x >= lim || z >= lim) return fail(QSIM_EINVAL, "Pauli mask has a qubit >= n_qubits (%d)", n);
  if (x == 0 && z == 0) return QSIM_OK;
  const uint64_t n4 = (1ull << n) / 2;
  const uint64_t windows = ceil_div(n4, 64);
  const int y = __builtin_popcountll(x & z) & 3;
  if (nt_for_qubits(n)) launch_pauli<true>(s, state, n4, windows, x, z, y);
  else launch_pauli<false>(s, state, n4, windows, x, z, y);
  return launch_status("apply_pauli_string");
}

// ------------------------------------------------------------ damping channels
// One Kraus branch of amplitude damping (kind 0: E0 = diag(1, sqrt(1-g)),
// E1 = [[0, sqrt(g)], [0, 0]]) or dephasing (kind 1: E0 as before,
// E1 = diag(0, sqrt(g))) on qubit t.  From res = (total, S0) of the FP64
// reduction, S1 = total - S0 is the weight with bit t = 1; branch 1 has
// probability g * S1 / total.  The chosen branch is written as a 2x2 matrix
// that also renormalises the state to unit norm (E0: 1/sqrt(S0 + (1-g) S1);
// E1: 1/sqrt(g S1) times sqrt(g)), all in FP64, and applied by the dense
// 2x2 gate kernel.
__global__ void k_channel_branch(const double* __restrict__ res, int kind, double g, double u,
                                 float2* __restrict__ mat, int* __restrict__ branch) {
  if (threadIdx.x != 0 || blockIdx.x != 0) return;
  const double tot = res[0], s0 = res[1];
  const double s1 = tot - s0 > 0.0 ? tot - s0 : 0.0;
  const double p1 = tot > 0.0 ? g * s1 / tot : 0.0;
  const int b = u < p1 ? 1 : 0;
  float2 m[4];
  for (int k = 0; k < 4; ++k) m[k] = make_float2(0.f, 0.f);
  if (b == 0) {
    const double nrm = s0 + (1.0 - g) * s1;
    const double r = nrm > 0.0 ? 1.0 / sqrt(nrm) : 0.0;
    m[0] = make_float2((float)r, 0.f);
    m[3] = make_float2((float)(r * sqrt(1.0 - g)), 0.f);
  } else {
    const double r = s1 > 0.0 ? 1.0 / sqrt(s1) : 0.0;
    m[kind == 0 ? 1 : 3] = make_float2((float)r, 0.f);
  }
  for (int k = 0; k < 4; ++k) mat[k] = m[k];
  *branch = b;
}

static int damping_impl(void* stream, void* state, int n, int t, double g, double u, void* workspace,
                        int* branch, int kind, const char* what) {
  if (int rc = check_n(n)) return rc;
  if (int rc = check_q(t, n, "target_qubit")) return rc;
  if (!state || !workspace || !branch) return fail(QSIM_EINVAL, "NULL pointer argument");
  if (!(g >= 0.0 && g <= 1.0)) return fail(QSIM_EINVAL, "%s: probability %g outside [0, 1]", what, g);
  hipStream_t s = as_stream(stream);
  double* ws = (double*)workspace;
  if (int rc = reduce_impl(s, state, n, 1, t, ws)) return rc;
  // the pass-1 partials are consumed by pass 2, so their space holds the
  // branch matrix; the branch index goes next to the results
  float2* mat = (float2*)ws;
  int* dev_branch = (int*)(ws + 2 * kRedBlocks + 4);
  hipLaunchKernelGGL(k_channel_branch, dim3(1), dim3(64), 0, s, ws + 2 * kRedBlocks, kind, g, u,
                     mat, dev_branch);
  if (int rc = launch_status(what)) return rc;
  M2 unused = {};
  if (int rc = gate1q_impl(stream, state, 1, n, mat, unused, t)) return rc;
  int host = -1;
  if (hipMemcpyAsync(&host, dev_branch, sizeof(int), hipMemcpyDeviceToHost, s) != hipSuccess)
    return fail(QSIM_EHIP, "%s: copy failed", what);
  if (hipStreamSynchronize(s) != hipSuccess) return fail(QSIM_EHIP, "%s: sync failed", what);
  *branch = host;
  return QSIM_OK;
}

}  // namespace qsim

using namespace qsim;

extern "C" {

int64_t qsim_expectation_workspace_bytes(int n_qubits) {
  (void)n_qubits;
  return kExpWsDoubles * (int64_t)sizeof(double);
}

int qsim_expectation_paulis(void* stream, const void* state, int n_qubits, int64_t n_terms,
                            const uint64_t* x_masks, const uint64_t* z_masks, void* workspace,
                            void* out_dev) {
  clear_error();
  return expectation_impl(as_stream(stream), state, n_qubits, n_terms, x_masks, z_masks,
                          (double*)workspace, (double*)out_dev);
}

int qsim_expectation_z(void* stream, const void* state, int n_qubits, uint64_t z_mask,
                       void* workspace, void* out_dev) {
  clear_error();
  const uint64_t x = 0;
  return expectation_impl(as_stream(stream), state, n_qubits, 1, &x, &z_mask, (double*)workspace,
                          (double*)out_dev);
}

int qsim_expectation_pauli(void* stream, const void* state, int n_qubits, uint64_t z_mask,
                           int xy_qubit, int op, void* workspace, void* out_dev) {
  clear_error();
  if (op < 0 || op > 2) return fail(QSIM_EINVAL, "op must be 0=I/Z, 1=X, 2=Y (got %d)", op);
  if (op == 0) return qsim_expectation_z(stream, state, n_qubits, z_mask, workspace, out_dev);
  if (int rc = check_n(n_qubits)) return rc;
  if (int rc = check_q(xy_qubit, n_qubits, "xy_qubit")) return rc;
  // the Z string acts on the other qubits: a z bit on xy_qubit is ignored
  const uint64_t bit = 1ull << xy_qubit;
  const uint64_t x = bit, z = (z_mask & ~bit) | (op == 2 ? bit : 0);
  return expectation_impl(as_stream(stream), state, n_qubits, 1, &x, &z, (double*)workspace,
                          (double*)out_dev);
}

int qsim_apply_pauli_string(void* stream, void* state, int n_qubits, uint64_t x_mask,
                            uint64_t z_mask) {
  clear_error();
  return pauli_apply_impl(as_stream(stream), state, n_qubits, x_mask, z_mask);
}

int qsim_apply_depolarizing(void* stream, void* state, int n_qubits, int target, double p,
                            double random_val, int* branch) {
  clear_error();
  if (int rc = check_n(n_qubits)) return rc;
  if (int rc = check_q(target, n_qubits, "target_qubit")) return rc;
  if (!state || !branch) return fail(QSIM_EINVAL, "NULL pointer argument");
  if (!(p >= 0.0 && p <= 1.0)) return fail(QSIM_EINVAL, "depolarizing: p = %g outside [0, 1]", p);
  // identity on [0, 1-p); then X, Y, Z on three intervals of width p/3
  int b = 0;
  if (!(random_val < 1.0 - p)) {
    const double r = random_val - (1.0 - p), third = p / 3.0;
    b = r < third ? 1 : (r < 2.0 * third ? 2 : 3);
  }
  *branch = b;
  if (b == 0) return QSIM_OK;
  const uint64_t bit = 1ull << target;
  const uint64_t x = b == 3 ? 0 : bit, z = b == 1 ? 0 : bit;
  return pauli_apply_impl(as_stream(stream), state, n_qubits, x, z);
}

int qsim_apply_amplitude_damping(void* stream, void* state, int n_qubits, int target, double gamma,
                                 double random_val, void* workspace, int* branch) {
  clear_error();
  return damping_impl(stream, state, n_qubits, target, gamma, random_val, workspace, branch, 0,
                      "amplitude_damping");
}

int qsim_apply_dephasing(void* stream, void* state, int n_qubits, int target, double lam,
                         double random_val, void* workspace, int* branch) {
  clear_error();
  return damping_impl(stream, state, n_qubits, target, lam, random_val, workspace, branch, 1,
                      "dephasing");
}

}  // extern "C"
