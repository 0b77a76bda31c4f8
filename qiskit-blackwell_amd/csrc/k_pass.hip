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
// set of 32 groups: D (32 x 32) = A (32 x 32) B (32 x 32) in 16
// v_mfma_f32_32x32x2_f32 with FP32 accumulation.
//   A[i][2 s + h]: lane (h = l / 32, i = l % 32), packed by the planner in
//     fragment order [s / 4][l][s % 4], so a wave reads it as four
//     contiguous 1 KiB loads.
//   B[2 s + h][c]: part h (0 = re, 1 = im) of amplitude s of group c: one
//     ds_read_b32 per slice s, 64 lanes on 64 banks.
//   D[i][c]: register q * 4 + 2 e + part of lane (h, c) is part `part` of
//     amplitude 4 q + 2 h + e, so results leave as whole amplitudes
//     (ds_write_b64).
//
// LDS addresses are linear over GF(2): amplitude j of the tile sits at
// sw(j) = j with bits 5..9 and 10..13 folded onto bits 0..4.  The planner
// picks the five group bits that run over the 32 lanes so that each residue
// (bit mod 5) occurs once where it can, which spreads the lanes over all
// banks whatever the block's qubits are.  The block record holds the swizzled
// index of each single bit, so an address is an XOR of record entries.
//
// What bounds it: 128 flop per amplitude and block at the FP32 MFMA rate
// (256 for a 5-qubit block, while a 4-qubit block absorbs about 3/4 of the ops
// of a 5-qubit one) once a pass has three or more blocks; the trip through
// memory below that.  At 28 qubits a block takes 277 us on top of the others
// (218 at the matrix peak; tiles of 11, 12 or 13 qubits and 4, 8 or 16 waves
// all measure 267-299) and a pass of one block 0.9 ms (0.68 for its bytes).
// The depth-28 SU(4) circuit: 92 launches of 5-qubit blocks 76.7 ms, 32 passes
// of 147 blocks 52.4 ms; depth 24 at 24 qubits 3.85 -> 2.44 ms.
#include "qsim_internal.hpp"
#include <string.h>
#include <algorithm>

namespace qsim {

typedef float f32x16 __attribute__((ext_vector_type(16)));

struct PassGeom {
  uint8_t tq[16];        // tile qubits, ascending; tq[0] = 0
};

constexpr uint32_t pass_sw(uint32_t j) { return j ^ ((j >> 5) & 31u) ^ ((j >> 10) & 31u); }

template <int M, int W, bool NT>
__global__ __launch_bounds__(64 * W) void k_pass(float4* __restrict__ st, uint64_t n_tiles, PassGeom g,
                                                 const uint4* __restrict__ blocks,
                                                 const float4* __restrict__ mats, int n_blocks) {
  constexpr int T = 64 * W;
  constexpr int SLOTS = (1 << (M - 1)) / T;           // float4 slots per thread
  constexpr int TB = __builtin_ctz(T);                // slot bits that run over the threads
  constexpr int SETS = 1 << (M - 9);
  constexpr int SPW = SETS >= W ? SETS / W : 1;       // sets per wave
  extern __shared__ float4 X4[];
  char* Xb = reinterpret_cast<char*>(X4);
  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  uint64_t base = gblock<uint64_t>();
  if (base >= n_tiles) return;                        // whole workgroup: past the last tile
#pragma unroll
  for (int j = 0; j < M; ++j) base = ins0(base, g.tq[j]);
  base >>= 1;                                         // in slots; tq[0] = 0
  uint64_t toff = 0;
#pragma unroll
  for (int j = 0; j < TB; ++j) toff |= (uint64_t)((tid >> j) & 1) << (g.tq[j + 1] - 1);
  const uint32_t tsw = pass_sw(2u * tid);
  uint64_t koff[SLOTS];
#pragma unroll
  for (int k = 0; k < SLOTS; ++k) {
    koff[k] = base;
#pragma unroll
    for (int j = TB; j < M - 1; ++j) koff[k] |= (uint64_t)((k >> (j - TB)) & 1) << (g.tq[j + 1] - 1);
  }
  {
    float4 v[SLOTS];
#pragma unroll
    for (int k = 0; k < SLOTS; ++k) v[k] = ld4<NT>(st + (koff[k] + toff));
#pragma unroll
    for (int k = 0; k < SLOTS; ++k) {
      // an odd swizzled index swaps the two amplitudes of a slot
      const uint32_t p = tsw ^ pass_sw(2u * k * T);
      const bool odd = p & 1;
      X4[p >> 1] = make_float4(odd ? v[k].z : v[k].x, odd ? v[k].w : v[k].y, odd ? v[k].x : v[k].z,
                               odd ? v[k].y : v[k].w);
    }
  }
  const int h = lane >> 5;
  float4 a[4];
#pragma unroll
  for (int q = 0; q < 4; ++q) a[q] = mats[q * 64 + lane];
  uint4 d0 = blocks[0], d1 = blocks[1];
  __syncthreads();
  for (int b = 0; b < n_blocks; ++b) {
    // record: row[4], lane[5], set[5] (16-bit swizzled single-bit indices)
    const uint32_t r0 = (d0.x & 0xffffu) * 8u, r1 = (d0.x >> 16) * 8u, r2 = (d0.y & 0xffffu) * 8u,
                   r3 = (d0.y >> 16) * 8u;
    uint32_t lb = 4u * h;
    lb ^= (lane & 1) ? (d0.z & 0xffffu) * 8u : 0u;
    lb ^= (lane & 2) ? (d0.z >> 16) * 8u : 0u;
    lb ^= (lane & 4) ? (d0.w & 0xffffu) * 8u : 0u;
    lb ^= (lane & 8) ? (d0.w >> 16) * 8u : 0u;
    lb ^= (lane & 16) ? (d1.x & 0xffffu) * 8u : 0u;
    const uint32_t sb[5] = {(d1.x >> 16) * 8u, (d1.y & 0xffffu) * 8u, (d1.y >> 16) * 8u, (d1.z & 0xffffu) * 8u,
                            (d1.z >> 16) * 8u};
    uint32_t ro[16];
#pragma unroll
    for (int s = 0; s < 16; ++s)
      ro[s] = ((s & 1) ? r0 : 0u) ^ ((s & 2) ? r1 : 0u) ^ ((s & 4) ? r2 : 0u) ^ ((s & 8) ? r3 : 0u);
    // the next block's fragments and record arrive while this one runs
    const int nb = b + 1 < n_blocks ? b + 1 : b;
    float4 an[4];
#pragma unroll
    for (int q = 0; q < 4; ++q) an[q] = mats[(size_t)nb * 256 + q * 64 + lane];
    const uint4 e0 = blocks[2 * nb], e1 = blocks[2 * nb + 1];
    const float* af = reinterpret_cast<const float*>(a);
    if (SETS >= W || wave < SETS) {
      float x[SPW][16];
      uint32_t sbase[SPW];
#pragma unroll
      for (int i = 0; i < SPW; ++i) {
        const int set = wave + W * i;
        uint32_t so = 0;
#pragma unroll
        for (int j = 0; j < M - 9; ++j) so ^= ((set >> j) & 1) ? sb[j] : 0u;
        sbase[i] = lb ^ so;
#pragma unroll
        for (int s = 0; s < 16; ++s) x[i][s] = *reinterpret_cast<const float*>(Xb + (sbase[i] ^ ro[s]));
      }
#pragma unroll
      for (int i = 0; i < SPW; ++i) {
        f32x16 acc = {0.f};
#pragma unroll
        for (int s = 0; s < 16; ++s) acc = __builtin_amdgcn_mfma_f32_32x32x2f32(af[s], x[i][s], acc, 0, 0, 0);
        // rows 4 q + 2 h + e: row bit 1 is the lane half
        const uint32_t wb = sbase[i] ^ (h ? (r1 ^ 4u) : 0u);
#pragma unroll
        for (int q = 0; q < 4; ++q)
#pragma unroll
          for (int e = 0; e < 2; ++e)
            *reinterpret_cast<float2*>(Xb + (wb ^ ro[4 * q + e])) =
                make_float2(acc[4 * q + 2 * e], acc[4 * q + 2 * e + 1]);
      }
    }
    __syncthreads();
#pragma unroll
    for (int q = 0; q < 4; ++q) a[q] = an[q];
    d0 = e0;
    d1 = e1;
  }
#pragma unroll
  for (int k = 0; k < SLOTS; ++k) {
    const uint32_t p = tsw ^ pass_sw(2u * k * T);
    const bool odd = p & 1;
    const float4 v = X4[p >> 1];
    st4<NT>(st + (koff[k] + toff), make_float4(odd ? v.z : v.x, odd ? v.w : v.y, odd ? v.x : v.z, odd ? v.y : v.w));
  }
}

template <int M, int W>
static void launch_pass(hipStream_t s, void* state, int n, const PassGeom& g, const qsim_pass_block* blocks,
                        const float* mats, int n_blocks) {
  const uint64_t tiles = 1ull << (n - M);
  const size_t lds = sizeof(float2) << M;
  if (nt_for_qubits(n))
    hipLaunchKernelGGL((k_pass<M, W, true>), grid1d(tiles), dim3(64 * W), lds, s, (float4*)state, tiles, g,
                       (const uint4*)blocks, (const float4*)mats, n_blocks);
  else
    hipLaunchKernelGGL((k_pass<M, W, false>), grid1d(tiles), dim3(64 * W), lds, s, (float4*)state, tiles, g,
                       (const uint4*)blocks, (const float4*)mats, n_blocks);
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
                      const qsim_pass_block* blocks_host, const void* blocks_dev, const void* mats_dev,
                      int n_blocks) {
  clear_error();
  if (int rc = check_n(n_qubits)) return rc;
  if (n_passes < 0 || n_blocks < 0) return fail(QSIM_EINVAL, "negative count");
  if (n_passes == 0) return QSIM_OK;
  if (!state || !passes || !blocks_host || !blocks_dev || !mats_dev)
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
      if (p.tile_mask >> q & 1) g.tq[m++] = (uint8_t)q;
    const qsim_pass_block* bd = (const qsim_pass_block*)blocks_dev + p.first_block;
    const float* md = (const float*)mats_dev + (size_t)p.first_block * QSIM_PASS_BLOCK_FLOATS;
    switch (m) {
      case 10: launch_pass<10, 4>(s, state, n_qubits, g, bd, md, p.n_blocks); break;
      case 11: launch_pass<11, 4>(s, state, n_qubits, g, bd, md, p.n_blocks); break;
      case 12: launch_pass<12, 8>(s, state, n_qubits, g, bd, md, p.n_blocks); break;
      default: launch_pass<13, 8>(s, state, n_qubits, g, bd, md, p.n_blocks); break;
    }
    if (int rc = launch_status("apply_passes")) return rc;
  }
  return QSIM_OK;
}

}  // extern "C"
