// Block passes for gfx950: many dense 4-qubit blocks per trip through HBM.
//
// A pass is a set of m state qubits (the tile, 10..13 of them) and a list of
// 4-qubit blocks on tile qubits.  One workgroup copies one tile of 2^m
// amplitudes into LDS, applies every block of the list to it on the matrix
// cores, and writes the tile back: the state crosses memory once per pass
// instead of once per block.
//
// A block is the real 32 x 32 matrix [[Re, -Im], [Im, Re]] of its 16 x 16
// complex matrix, with rows and columns interleaved (index 2 r + part), acting
// on the 32 real components of each group of 16 amplitudes.  One wave takes a
// set of 32 groups: D (32 x 32) = A (32 x 32) B (32 x 32).  Lane (h = l / 32,
// c = l % 32) holds amplitudes 4 q + 2 h + e (q < 4, e < 2) of group c, both
// as B operand and as D result (register 4 q + 2 e + part), so a set is read
// and written as whole amplitudes at the same eight LDS addresses.
//
// Arithmetic: FP32 amplitudes as sums of three bf16 (hi + mid + lo, each
// rounded to nearest, 3 x 8 bits), exact for magnitudes from 2^-100 to 2^127:
// below, the last bits of lo fall under the smallest bf16, and the top 2^-8 of
// FP32's range rounds hi up to infinity.  Coefficients are three bf16 within
// 2^-26 of their FP64 value (closer than FP32), multiplied on
// v_mfma_f32_32x32x16_bf16 with FP32 accumulation.  Products of two bf16 are
// exact.  The hi*hi sums have an accumulator of their own, where they are all
// but exact; the five smaller products (lo with hi, mid with mid, mid with hi;
// the three left out are below 2^-26 of a term) are summed from the smallest up
// in a second one, and one FP32 addition joins the two.  Error of the norm
// against FP64: 1.9e-7 after 24 random blocks on 13 qubits, 5.0e-7 on the FP32
// matrix instructions; SU(4) volume 28 qubits 5.4e-7 against 1.2e-6.
// Accumulating everything in one chain doubles the error of structured blocks
// (27-qubit QFT 5.7e-7 against 3.5e-7).  A permutation block moves amplitudes of
// that range bit for bit (hi + (mid + lo) has no rounding).  The FP32
// instructions run at 1/16 of the bf16 rate and, measured here, not beside VALU
// work: 277 us per block at 28 qubits (218 at their peak) against 190 us.
//
// LDS addresses are linear over GF(2): amplitude j of the tile sits at
// sw(j) = j with bits 5..9 and 10..13 folded onto bits 0..4.  The planner
// picks the five group bits that run over the 32 lanes so that each residue
// (bit mod 5) occurs once where it can, which spreads the lanes over all
// banks whatever the block's qubits are.  The block record holds the swizzled
// index of each single bit, so an address is an XOR of record entries.
//
// What bounds it: issue, of vector instructions before products, with waits that
// the waves at hand do not all cover.  At 28 qubits and 3.5 blocks a pass the
// counters give a set 144 vector instructions, 12 of them products; 88 split its
// amplitudes, 16 join the accumulators.  Of all SIMD cycles 34 % run a product
// and 47 % a vector instruction (at 4 cycles each), half of the products'
// cycles beside a vector instruction, so 36 % issue neither; a wave spends 29 %
// of its time at a wait or barrier and 47 % ready but not picked.  The tile's
// bytes cross memory once each way (2.15 GB) and hide in part: 1.08 ms a pass
// with 3.5 blocks, 0.68 for the bytes alone.
// Fewer vector instructions did help: LDS addresses without the array's base,
// slots stored as two amplitudes instead of four selects, scalar bases in
// global addresses (163 -> 148 a set) took the depth-24 SU(4) circuit at 24
// qubits from 1752 to 1707 us, depth 28 at 28 qubits from 40.3 to 39.7 ms.
// Measured and not taken: residues by v_dot2c_f32_bf16 (32 instructions fewer
// at twice the cycles, no gain), the next tile loaded into registers beside the
// blocks by workgroups that stay (42.4 ms), consecutive blocks on the same wave
// bits without the barrier between them (40.5 ms), the next set's amplitudes
// loaded beside the products (208 us a block against 190).
// Two workgroups of 8 waves per CU (13-qubit tiles) are the best of 4, 8 and 16
// waves for states that fill the chip; a 12-qubit tile takes 8 waves for the
// sake of states of at most 21 qubits, which leave a CU one or two tiles (20
// qubits: 175 us against 192 with 4 waves).  92 launches of 5-qubit blocks took
// 76.7 ms for the depth-28 circuit, 32 passes of 143 blocks take 39.7.
#include "qsim_internal.hpp"
#include <string.h>
#include <algorithm>

namespace qsim {

static_assert(sizeof(qsim_pass_rec) == 48, "batch pass record");

typedef float f32x16 __attribute__((ext_vector_type(16)));
typedef float f32x2v __attribute__((ext_vector_type(2)));
typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));

struct PassGeom {
  uint32_t w[4];         // tile qubits, ascending, one byte each; the first is 0
  __host__ __device__ int tq(int j) const { return (int)((w[j >> 2] >> (8 * (j & 3))) & 255u); }
};

constexpr uint32_t pass_sw(uint32_t j) { return j ^ ((j >> 5) & 31u) ^ ((j >> 10) & 31u); }

constexpr int kFrags = 6;     // bf16 fragments of a block: parts hi, mid, lo x halves of the K range

__device__ __forceinline__ bf16x8 as_frag(float4 v) { return __builtin_bit_cast(bf16x8, v); }
__device__ __forceinline__ uint32_t pk_bf16(float a, float b) {
  const f32x2v v = {a, b};
  return __builtin_bit_cast(uint32_t, __builtin_convertvector(v, bf16x2));
}
// x = hi + mid + lo (exactly in the range above), each a pair of bf16 rounded to nearest.
__device__ __forceinline__ void split3(float2 x, uint32_t& hi, uint32_t& mid, uint32_t& lo) {
  hi = pk_bf16(x.x, x.y);
  const float rx = x.x - __uint_as_float(hi << 16), ry = x.y - __uint_as_float(hi & 0xffff0000u);
  mid = pk_bf16(rx, ry);
  lo = pk_bf16(rx - __uint_as_float(mid << 16), ry - __uint_as_float(mid & 0xffff0000u));
}
// The B fragments of a set: amplitudes 4 t .. 4 t + 3 of a lane are half t of
// its K range.
__device__ __forceinline__ void split_set(const float2 x[8], bf16x8 b[kFrags]) {
#pragma unroll
  for (int t = 0; t < 2; ++t) {
    uint32_t w[3][4];
#pragma unroll
    for (int p = 0; p < 4; ++p) split3(x[4 * t + p], w[0][p], w[1][p], w[2][p]);
#pragma unroll
    for (int k = 0; k < 3; ++k) {
      const uint4 v = make_uint4(w[k][0], w[k][1], w[k][2], w[k][3]);
      b[2 * k + t] = __builtin_bit_cast(bf16x8, v);
    }
  }
}
template <int KA, int KB>
__device__ __forceinline__ f32x16 mul_parts(const bf16x8 a[kFrags], const bf16x8 b[kFrags], f32x16 acc) {
  acc = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a[2 * KA], b[2 * KB], acc, 0, 0, 0);
  return __builtin_amdgcn_mfma_f32_32x32x16_bf16(a[2 * KA + 1], b[2 * KB + 1], acc, 0, 0, 0);
}

// An amplitude at a byte offset of LDS.  The tile is the only thing there and
// starts at 0, so an offset is an address: through the array's symbol the
// compiler adds that 0 at every access, after the XORs.
typedef __attribute__((address_space(3))) f32x2v lds_amp;
__device__ __forceinline__ float2 lds_get(uint32_t at) {
  const f32x2v v = *(const lds_amp*)at;
  return make_float2(v.x, v.y);
}
__device__ __forceinline__ void lds_put(uint32_t at, float x, float y) {
  const f32x2v v = {x, y};
  *(lds_amp*)at = v;
}

// One tile of one pass, by a workgroup of W waves.  OFF holds the byte offset
// of a thread's place in a tile: 32 bits up to 29 qubits, so that an address is
// a scalar base and one register.
template <int M, int W, bool NT, typename OFF>
__device__ __forceinline__ void pass_tile(float4* __restrict__ st, uint64_t tile, const PassGeom& g,
                                          const uint4* __restrict__ blocks, const float4* __restrict__ frags,
                                          int n_blocks) {
  constexpr int T = 64 * W;
  constexpr int SLOTS = (1 << (M - 1)) / T;           // float4 slots per thread
  constexpr int TB = __builtin_ctz(T);                // slot bits that run over the threads
  constexpr int SETS = 1 << (M - 9);
  constexpr int SPW = SETS >= W ? SETS / W : 1;       // sets per wave
  const int tid = threadIdx.x;
  const int lane = tid & 63, h = lane >> 5;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  uint64_t base = tile;
#pragma unroll
  for (int j = 0; j < M; ++j) base = ins0(base, g.tq(j));
  OFF toff = 0;
#pragma unroll
  for (int j = 0; j < TB; ++j) toff |= (OFF)((tid >> j) & 1) << (g.tq(j + 1) + 3);
  const uint32_t tsw = pass_sw(2u * tid) * 8u;
  auto place = [&](int k) -> float4* {                // slot k of the thread; the first tile qubit is 0
    uint64_t at = base;
#pragma unroll
    for (int j = TB; j < M - 1; ++j) at |= (uint64_t)((k >> (j - TB)) & 1) << g.tq(j + 1);
    return reinterpret_cast<float4*>(reinterpret_cast<char*>(st) + at * 8u + toff);
  };
  {
    float4 v[SLOTS];
#pragma unroll
    for (int k = 0; k < SLOTS; ++k) v[k] = ld4<NT>(place(k));
#pragma unroll
    for (int k = 0; k < SLOTS; ++k) {
      // the slot's two amplitudes are neighbours in LDS, in either order
      const uint32_t p = tsw ^ pass_sw(2u * k * T) * 8u;
      lds_put(p, v[k].x, v[k].y);
      lds_put(p ^ 8u, v[k].z, v[k].w);
    }
  }
  bf16x8 a[kFrags];
  auto load_frags = [&](int b) {
    // a base in the middle: every fragment within an instruction's offset of it
    const float4* fb = frags + (size_t)b * (64 * kFrags) + 64 * (kFrags / 2);
#pragma unroll
    for (int q = 0; q < kFrags; ++q) a[q] = as_frag((fb + 64 * (q - kFrags / 2))[lane]);
  };
  load_frags(0);
  uint4 d0 = blocks[0], d1 = blocks[1];
  __syncthreads();
  for (int b = 0; b < n_blocks; ++b) {
    // record: row[4], lane[5], set[5] (16-bit swizzled single-bit indices)
    const uint32_t r0 = (d0.x & 0xffffu) * 8u, r1 = (d0.x >> 16) * 8u, r2 = (d0.y & 0xffffu) * 8u,
                   r3 = (d0.y >> 16) * 8u;
    uint32_t lb = h ? r1 : 0u;            // row bit 1 is the lane half
    lb ^= (lane & 1) ? (d0.z & 0xffffu) * 8u : 0u;
    lb ^= (lane & 2) ? (d0.z >> 16) * 8u : 0u;
    lb ^= (lane & 4) ? (d0.w & 0xffffu) * 8u : 0u;
    lb ^= (lane & 8) ? (d0.w >> 16) * 8u : 0u;
    lb ^= (lane & 16) ? (d1.x & 0xffffu) * 8u : 0u;
    const uint32_t sb[4] = {(d1.x >> 16) * 8u, (d1.y & 0xffffu) * 8u, (d1.y >> 16) * 8u, (d1.z & 0xffffu) * 8u};
    uint32_t ro[8];                       // amplitude 4 q + e of a lane at index 2 q + e
#pragma unroll
    for (int s = 0; s < 8; ++s) ro[s] = ((s & 1) ? r0 : 0u) ^ ((s & 2) ? r2 : 0u) ^ ((s & 4) ? r3 : 0u);
    const int nb = b + 1 < n_blocks ? b + 1 : b;
    const uint4 e0 = blocks[2 * nb], e1 = blocks[2 * nb + 1];
    if (SETS >= W || wave < SETS) {
      uint32_t sbase[SPW];
#pragma unroll
      for (int i = 0; i < SPW; ++i) {
        const int set = wave + W * i;
        sbase[i] = lb;
#pragma unroll
        for (int j = 0; j < M - 9; ++j) sbase[i] ^= ((set >> j) & 1) ? sb[j] : 0u;
      }
#pragma unroll
      for (int i = 0; i < SPW; ++i) {
        float2 x[8];
#pragma unroll
        for (int s = 0; s < 8; ++s) x[s] = lds_get(sbase[i] ^ ro[s]);
        bf16x8 bp[kFrags];
        split_set(x, bp);
        f32x16 big = {0.f}, small = {0.f};
        big = mul_parts<0, 0>(a, bp, big);
        small = mul_parts<0, 2>(a, bp, small);
        small = mul_parts<2, 0>(a, bp, small);
        small = mul_parts<1, 1>(a, bp, small);
        small = mul_parts<0, 1>(a, bp, small);
        small = mul_parts<1, 0>(a, bp, small);
        if (i + 1 == SPW) {
          // the next block's fragments travel while the results are written
          load_frags(nb);
        }
#pragma unroll
        for (int s = 0; s < 8; ++s)
          lds_put(sbase[i] ^ ro[s], big[2 * s] + small[2 * s], big[2 * s + 1] + small[2 * s + 1]);
      }
    }
    __syncthreads();
    d0 = e0;
    d1 = e1;
  }
#pragma unroll
  for (int k = 0; k < SLOTS; ++k) {
    const uint32_t p = tsw ^ pass_sw(2u * k * T) * 8u;
    const float2 u = lds_get(p), w = lds_get(p ^ 8u);
    st4<NT>(place(k), make_float4(u.x, u.y, w.x, w.y));
  }
}

template <int M, int W, bool NT, typename OFF>
__global__ __launch_bounds__(64 * W, 4) void k_pass(float4* __restrict__ st, uint64_t n_tiles, PassGeom g,
                                                    const uint4* __restrict__ blocks,
                                                    const float4* __restrict__ frags, int n_blocks) {
  const uint64_t tile = gblock<uint64_t>();
  if (tile >= n_tiles) return;                        // whole workgroup: past the last tile
  pass_tile<M, W, NT, OFF>(st, tile, g, blocks, frags, n_blocks);
}

// One pass of each of n_recs states in one launch: workgroup b takes the tile
// b - tile_begin of the record it falls to, found by one load per lane and a
// ballot (records ascend; more than 64 take further rounds).  pass_tile does
// not depend on W or on the tile's place in the grid, so a state's bits are
// those of its passes run alone.  What bounds it is the latency of a pass, a
// tile or less per CU: a step of 6 states of 15 to 17 qubits takes 13 us, and
// replaces three to four launches of 5-qubit block steps of 7.5 us, 5 us apart.
constexpr int kBatchWaves = 8;
__global__ __launch_bounds__(64 * kBatchWaves, 4) void k_pass_batch(const qsim_pass_rec* __restrict__ recs, int n_recs,
                                                                    const uint4* __restrict__ blocks,
                                                                    const float4* __restrict__ frags) {
  const uint64_t b = blockIdx.x;
  const int lane = threadIdx.x & 63;
  int at = -1;                                        // records before it begin at or below b
  for (int r0 = 0; r0 < n_recs; r0 += 64) {
    const int r = r0 + lane;
    const int c = __popcll(__ballot(r < n_recs && recs[r < n_recs ? r : 0].tile_begin <= b));
    at += c;
    if (c < 64) break;
  }
  const qsim_pass_rec& rec = recs[__builtin_amdgcn_readfirstlane(at)];
  PassGeom g;
#pragma unroll
  for (int j = 0; j < 4; ++j) g.w[j] = reinterpret_cast<const uint32_t*>(rec.tile_qubits)[j];
  float4* st = reinterpret_cast<float4*>(rec.state);
  const uint4* bl = blocks + 2 * (size_t)rec.first_block;
  const float4* fr = frags + (size_t)rec.first_block * (64 * kFrags);
  const uint64_t tile = b - rec.tile_begin;
  switch (rec.tile_bits) {
    case 10: pass_tile<10, kBatchWaves, false, uint64_t>(st, tile, g, bl, fr, rec.n_blocks); break;
    case 11: pass_tile<11, kBatchWaves, false, uint64_t>(st, tile, g, bl, fr, rec.n_blocks); break;
    case 12: pass_tile<12, kBatchWaves, false, uint64_t>(st, tile, g, bl, fr, rec.n_blocks); break;
    default: pass_tile<13, kBatchWaves, false, uint64_t>(st, tile, g, bl, fr, rec.n_blocks); break;
  }
}

template <int M, int W>
static void launch_pass(hipStream_t s, void* state, int n, const PassGeom& g, const qsim_pass_block* blocks,
                        const void* frags, int n_blocks) {
  const uint64_t tiles = 1ull << (n - M);
  const size_t lds = sizeof(float2) << M;
  auto* kern = n > 29             ? k_pass<M, W, true, uint64_t>
               : nt_for_qubits(n) ? k_pass<M, W, true, uint32_t>
                                  : k_pass<M, W, false, uint32_t>;
  hipLaunchKernelGGL(kern, grid1d(tiles), dim3(64 * W), lds, s, (float4*)state, tiles, g, (const uint4*)blocks,
                     (const float4*)frags, n_blocks);
}

// Host check of one record: the swizzled indices of m distinct tile bits.
static bool block_ok(const qsim_pass_block& b, int m) {
  uint32_t seen = 0;
  for (int j = 0; j < m; ++j) {
    const uint32_t v = b.bit[j];
    if (v == 0 || v >> m) return false;
    const int p = 31 - __builtin_clz(v);
    if (v != pass_sw(1u << p) || (seen >> p & 1)) return false;
    seen |= 1u << p;
  }
  return true;
}

}  // namespace qsim

using namespace qsim;

extern "C" {

int qsim_apply_passes(void* stream, void* state, int n_qubits, const qsim_pass* passes, int n_passes,
                      const qsim_pass_block* blocks_host, const void* blocks_dev, const void* frags_dev,
                      int n_blocks) {
  clear_error();
  if (int rc = check_n(n_qubits)) return rc;
  if (n_passes < 0 || n_blocks < 0) return fail(QSIM_EINVAL, "negative count");
  if (n_passes == 0) return QSIM_OK;
  if (!state || !passes || !blocks_host || !blocks_dev || !frags_dev)
    return fail(QSIM_EINVAL, "NULL pointer argument");
  for (int i = 0; i < n_passes; ++i) {
    const qsim_pass& p = passes[i];
    const int m = __builtin_popcountll(p.tile_mask);
    if (p.tile_mask >> n_qubits) return fail(QSIM_EINVAL, "pass %d: tile qubits above n_qubits", i);
    if (!(p.tile_mask & 1)) return fail(QSIM_EINVAL, "pass %d: the tile must hold qubit 0", i);
    if (m < QSIM_PASS_MIN_TILE || m > QSIM_PASS_MAX_TILE)
      return fail(QSIM_ERANGE, "pass %d: tile of %d qubits outside %d..%d", i, m, QSIM_PASS_MIN_TILE,
                  QSIM_PASS_MAX_TILE);
    if (p.first_block < 0 || p.n_blocks < 1 || p.n_blocks > n_blocks - p.first_block)
      return fail(QSIM_EINVAL, "pass %d: blocks [%d, +%d) beyond the %d passed", i, p.first_block, p.n_blocks,
                  n_blocks);
    for (int b = 0; b < p.n_blocks; ++b)
      if (!block_ok(blocks_host[p.first_block + b], m))
        return fail(QSIM_EINVAL, "pass %d: block record %d is not a record of a %d-qubit tile", i,
                    p.first_block + b, m);
  }
  hipStream_t s = as_stream(stream);
  for (int i = 0; i < n_passes; ++i) {
    const qsim_pass& p = passes[i];
    PassGeom g;
    memset(&g, 0, sizeof g);
    int m = 0;
    for (int q = 0; q < n_qubits; ++q)
      if (p.tile_mask >> q & 1) {
        g.w[m >> 2] |= (uint32_t)q << (8 * (m & 3));
        ++m;
      }
    const qsim_pass_block* bd = (const qsim_pass_block*)blocks_dev + p.first_block;
    const uint16_t* fd = (const uint16_t*)frags_dev + (size_t)p.first_block * QSIM_PASS_BLOCK_BF16;
    switch (m) {
      case 10: launch_pass<10, 4>(s, state, n_qubits, g, bd, fd, p.n_blocks); break;
      case 11: launch_pass<11, 4>(s, state, n_qubits, g, bd, fd, p.n_blocks); break;
      case 12: launch_pass<12, 8>(s, state, n_qubits, g, bd, fd, p.n_blocks); break;
      default: launch_pass<13, 8>(s, state, n_qubits, g, bd, fd, p.n_blocks); break;
    }
    if (int rc = launch_status("apply_passes")) return rc;
  }
  return QSIM_OK;
}

int qsim_apply_pass_batch(void* stream, const qsim_pass_rec* recs_host, const void* recs_dev, int64_t n_recs,
                          const qsim_pass_block* blocks_host, const void* blocks_dev, const void* frags_dev,
                          int64_t n_blocks) {
  clear_error();
  if (n_recs < 0 || n_blocks < 0) return fail(QSIM_EINVAL, "negative count");
  if (n_recs == 0) return QSIM_OK;
  if (n_recs > (1 << 20)) return fail(QSIM_ERANGE, "%lld records in one batch", (long long)n_recs);
  if (!recs_host || !recs_dev || !blocks_host || !blocks_dev || !frags_dev)
    return fail(QSIM_EINVAL, "NULL pointer argument");
  uint64_t tiles = 0;
  int max_m = 0;
  for (int64_t i = 0; i < n_recs; ++i) {
    const qsim_pass_rec& r = recs_host[i];
    const int m = r.tile_bits;
    if (!r.state || (r.state & 15u)) return fail(QSIM_EINVAL, "record %lld: state NULL or not 16-byte aligned", (long long)i);
    if (int rc = check_n(r.n_qubits)) return rc;
    if (m < QSIM_PASS_MIN_TILE || m > QSIM_PASS_MAX_TILE || m > r.n_qubits)
      return fail(QSIM_ERANGE, "record %lld: tile of %d qubits", (long long)i, m);
    if (r.tile_qubits[0] != 0) return fail(QSIM_EINVAL, "record %lld: the tile must hold qubit 0", (long long)i);
    for (int j = 1; j < m; ++j)
      if (r.tile_qubits[j] <= r.tile_qubits[j - 1] || r.tile_qubits[j] >= r.n_qubits)
        return fail(QSIM_EINVAL, "record %lld: tile qubits not ascending below n_qubits", (long long)i);
    if (r.tile_begin != tiles) return fail(QSIM_EINVAL, "record %lld: tile_begin is not the prefix sum", (long long)i);
    if (r.first_block < 0 || r.n_blocks < 1 || r.n_blocks > n_blocks - r.first_block)
      return fail(QSIM_EINVAL, "record %lld: blocks [%d, +%d) beyond the %lld passed", (long long)i, r.first_block,
                  r.n_blocks, (long long)n_blocks);
    for (int b = 0; b < r.n_blocks; ++b)
      if (!block_ok(blocks_host[r.first_block + b], m))
        return fail(QSIM_EINVAL, "record %lld: block record %d is not a record of a %d-qubit tile", (long long)i,
                    r.first_block + b, m);
    tiles += 1ull << (r.n_qubits - m);
    max_m = std::max(max_m, m);
  }
  if (tiles > 0x7fffffffull) return fail(QSIM_ERANGE, "batch too large (%llu tiles)", (unsigned long long)tiles);
  hipLaunchKernelGGL(k_pass_batch, dim3((unsigned)tiles), dim3(64 * kBatchWaves), sizeof(float2) << max_m,
                     as_stream(stream), (const qsim_pass_rec*)recs_dev, (int)n_recs, (const uint4*)blocks_dev,
                     (const float4*)frags_dev);
  return launch_status("apply_pass_batch");
}

}  // extern "C"
