// Host-side runtime of libqsim_gfx950.so: the dense-block planner.  Pure
// C++ (no HIP headers, no kernels), compiled by the host compiler, so it
// also builds under the host sanitizers (tests/test_planner_sanitizers.py).
//
// Planner.  Ops arrive in circuit order, each with up to 8 qubits and a
// dense FP64 matrix on them (row bit j <-> qubit j of the op).  A block is
// a set S of at most k qubits together with the ops it absorbs: scanning the
// remaining ops in order, an op joins when its qubits lie in S and none of
// them was touched by an earlier op left out of the block (so every op still
// follows its predecessors).  A seed is any remaining op that no earlier
// remaining op touches; up to kSeeds of them are tried and the block that
// absorbs the most ops per unit of kernel time (block_score) is kept (ties go
// to the earliest).
//  * effort 0: S grows greedily from the seed's qubits, an op joining while
//    the union stays <= k; a depth-28 random SU(4) circuit on 28 qubits
//    takes 100 blocks (120 with the first op as the only seed).
//  * effort 1: in addition, every S made of the seed's qubits and up to
//    k - |seed| of the qubits that the next kSearchWindow ops connect to the
//    seed is scored.  The depth-30 SU(4) circuit on 30 qubits then took 108
//    blocks instead of 119 (28 qubits, depth 28: 92 instead of 100) when
//    scored by count, for about 5 ms of host time.  A 40-op window gave 110 and 93 blocks in twice the
//    time, a 20-op window 112 and 96.
// The block matrix is the FP64 product of the members in circuit order, each
// applied to the rows of the running 2^k x 2^k matrix.  Blocks are padded with
// the lowest unused qubits from kPadFrom up (then below it) to exactly
// min(k, n) qubits.  An op wider than k
// becomes a passthrough entry for the caller to run on its own kernel.
#include "qsim_gfx950.h"
#include "host_error.hpp"
#include <stdint.h>
#include <algorithm>
#include <string.h>
#include <new>
#include <vector>

namespace qsim {

constexpr int kSeeds = 32;
constexpr int kSearchWindow = 30;     // ops after the seed whose qubits may join S (effort 1)
constexpr int kSearchQubits = 16;     // at most this many candidate qubits per seed
// First padding qubit.  A padded qubit only selects the block kernel: a low one
// can put qubit 0 or a third qubit of 0..4 into the block, whose kernels are
// slower, and a lowest block qubit of 12 streams well.  The 30-qubit SU(4)
// step ran 363-364 ms against 369 ms with padding from qubit 0 (108 blocks
// either way; 368 ms from 16, 20 or 24).
constexpr int kPadFrom = 12;
// Blocks are compared by ops absorbed per unit of kernel time, in thousandths
// of a block with no qubit in 0..3: qubit 0 in the block 1.10, three or more
// block qubits in 0..4 (the LDS-staged kernel) 1.31, the ratios of their mean
// launch times in the 30-qubit SU(4) trace.  Scored by count alone, that
// circuit took 108 blocks (20 with qubit 0, 3 LDS-staged) and 367 ms per
// fused step; scored per cost, 107 blocks (15 and 2) and 361 ms.  The ratios
// hold for states above the 256 MiB MALL (n > 25); smaller states and the
// other widths (one kernel for every qubit set) are scored by count.
constexpr long long kCostQ0 = 1100, kCostLow3 = 1310;

static inline long long block_score(int n_ops, uint64_t S, bool weigh) {
  long long c = 1000;
  if (weigh) c = (S & 1ull) ? kCostQ0 : (__builtin_popcountll(S & 31ull) >= 3 ? kCostLow3 : 1000);
  return (long long)n_ops * 1000000 / c;
}

// Ops of rem (in order) that the qubit set S absorbs: an op joins when its
// qubits lie in S and no earlier op left out touched any of them.  With
// `out` null only the count is returned, and the scan stops once every
// qubit of S is blocked.
static int absorb_set(const std::vector<int>& rem, const std::vector<uint64_t>& mask, uint64_t S,
                      std::vector<int>* out) {
  uint64_t blocked = 0;
  int cnt = 0;
  for (int i : rem) {
    const uint64_t m = mask[i];
    if ((m & blocked) == 0 && (m & ~S) == 0) {
      ++cnt;
      if (out) out->push_back(i);
    } else {
      blocked |= m;
      if (!out && (blocked & S) == S) break;
    }
  }
  return cnt;
}

// Block matrix kept as separate real and imaginary D x D arrays so that the
// row updates below run as contiguous loops over the columns.
//
// rows of (re, im) (row bit b <-> block bit b) <- u (on block bits pos[0..kq))
// times those rows; u is row-major complex (re, im interleaved).
// One- and two-qubit ops (the common case) go through local row buffers, so
// the column loops vectorise without alias checks (with an AVX2 clone where
// the host has it); the operation order is that of the general form below
// (each product rounded, then summed over t from 0.0), so both give the same
// bits.
template <int KQ>
__attribute__((target_clones("avx2", "default")))
static void apply_rows_small(double* re, double* im, int D, const double* u, const int* pos) {
  constexpr int d = 1 << KQ;
  constexpr int kMaxD = 1 << QSIM_MAX_BLOCK_QUBITS;
  double ur[d][d], ui[d][d];
  for (int s = 0; s < d; ++s)
    for (int t = 0; t < d; ++t) {
      ur[s][t] = u[2 * (s * d + t)];
      ui[s][t] = u[2 * (s * d + t) + 1];
    }
  uint32_t pm = 0;
  for (int j = 0; j < KQ; ++j) pm |= 1u << pos[j];
  double xr[d][kMaxD], xi[d][kMaxD], yr[d][kMaxD], yi[d][kMaxD];
  for (int base = 0; base < D; ++base) {
    if (base & pm) continue;
    double* pr[d];
    double* pi[d];
    for (int s = 0; s < d; ++s) {
      int r = base;
      for (int j = 0; j < KQ; ++j)
        if (s >> j & 1) r |= 1 << pos[j];
      pr[s] = re + (size_t)r * D;
      pi[s] = im + (size_t)r * D;
      memcpy(xr[s], pr[s], sizeof(double) * D);
      memcpy(xi[s], pi[s], sizeof(double) * D);
    }
    for (int s = 0; s < d; ++s)
      for (int c = 0; c < D; ++c) {
        double ar = 0.0, ai = 0.0;
        for (int t = 0; t < d; ++t) {
          ar += ur[s][t] * xr[t][c] - ui[s][t] * xi[t][c];
          ai += ur[s][t] * xi[t][c] + ui[s][t] * xr[t][c];
        }
        yr[s][c] = ar;
        yi[s][c] = ai;
      }
    for (int s = 0; s < d; ++s) {
      memcpy(pr[s], yr[s], sizeof(double) * D);
      memcpy(pi[s], yi[s], sizeof(double) * D);
    }
  }
}

static void apply_rows(double* re, double* im, int D, const double* u, const int* pos, int kq,
                       double* tre, double* tim) {
  if (kq == 1) return apply_rows_small<1>(re, im, D, u, pos);
  if (kq == 2) return apply_rows_small<2>(re, im, D, u, pos);
  const int d = 1 << kq;
  uint32_t pm = 0;
  for (int j = 0; j < kq; ++j) pm |= 1u << pos[j];
  int idx[256];
  for (int base = 0; base < D; ++base) {
    if (base & pm) continue;
    for (int s = 0; s < d; ++s) {
      int r = base;
      for (int j = 0; j < kq; ++j)
        if (s >> j & 1) r |= 1 << pos[j];
      idx[s] = r;
    }
    for (int t = 0; t < d; ++t) {
      memcpy(tre + (size_t)t * D, re + (size_t)idx[t] * D, sizeof(double) * D);
      memcpy(tim + (size_t)t * D, im + (size_t)idx[t] * D, sizeof(double) * D);
    }
    for (int s = 0; s < d; ++s) {
      double* ore = re + (size_t)idx[s] * D;
      double* oim = im + (size_t)idx[s] * D;
      const double* us = u + 2 * (size_t)s * d;
      for (int c = 0; c < D; ++c) ore[c] = oim[c] = 0.0;
      for (int t = 0; t < d; ++t) {
        const double ur = us[2 * t], ui = us[2 * t + 1];
        const double* xr = tre + (size_t)t * D;
        const double* xi = tim + (size_t)t * D;
        for (int c = 0; c < D; ++c) {
          ore[c] += ur * xr[c] - ui * xi[c];
          oim[c] += ur * xi[c] + ui * xr[c];
        }
      }
    }
  }
}

// ------------------------------------------------------------------ passes
// Pass planner.  A pass is a tile (a set T of at most tile_bits qubits that
// holds the low_bits lowest ones) and the ops it absorbs, by the rule of
// absorb_set.  From each start (the low qubits alone, and with the qubits of
// each op that no earlier remaining op touches) T grows by the op on its
// frontier that adds the most absorbed ops per added qubit; the T that
// absorbs the most ops is kept and filled up with the lowest unused qubits.
// Ops wider than a block are never absorbed.
constexpr int kPassK = 4;             // qubits per block
constexpr int kPassD = 1 << kPassK;

struct PassPlan {
  int n, m;
  uint64_t low;
  std::vector<uint64_t> mask;       // per op; wide ops carry kWide as well
  std::vector<int> rem;
};
constexpr uint64_t kWide = 1ull << 63;   // in no tile, so the op is never absorbed

static uint64_t grow_tile(const PassPlan& p, uint64_t S, int* absorbed) {
  const uint64_t all = (1ull << p.n) - 1;
  int base = absorb_set(p.rem, p.mask, S, nullptr);
  while (__builtin_popcountll(S) < p.m) {
    uint64_t blocked = 0, best = 0;
    int best_gain = -1, best_add = 1;
    for (int i : p.rem) {
      const uint64_t mk = p.mask[i];
      if ((mk & blocked) == 0 && (mk & ~S) == 0) continue;      // absorbed already
      if ((mk & blocked) == 0 && !(mk & kWide)) {
        const uint64_t un = S | mk;
        const int add = __builtin_popcountll(mk & ~S);
        if (__builtin_popcountll(un) <= p.m) {
          const int gain = absorb_set(p.rem, p.mask, un, nullptr) - base;
          if (best_gain < 0 || (long long)gain * best_add > (long long)best_gain * add) {
            best_gain = gain;
            best_add = add;
            best = un;
          }
        }
      }
      blocked |= mk;
      if ((blocked & all) == all) break;
    }
    if (best_gain < 0) break;
    S = best;
    base += best_gain;
  }
  *absorbed = base;
  return S;
}

// Swizzled LDS index of tile bit p: bits 5..9 and 10..13 fold onto bits 0..4.
static uint16_t pass_index(int p) {
  const uint32_t j = 1u << p;
  return (uint16_t)(j ^ ((j >> 5) & 31u) ^ ((j >> 10) & 31u));
}

// Record of a block on tile bits row[0..4): the lane bits take one bit of each
// residue mod 5 (the LDS bank bits they fold onto) where one is free, then the
// rest in ascending order.
static void pass_record(qsim_pass_block* rec, int m, const int* row) {
  memset(rec, 0, sizeof *rec);
  uint32_t used = 0;
  int at = 0;
  for (int j = 0; j < kPassK; ++j) {
    used |= 1u << row[j];
    rec->bit[at++] = pass_index(row[j]);
  }
  int lane[5];
  for (int j = 0; j < 5; ++j) {
    lane[j] = -1;
    for (int p = j; p < m && lane[j] < 0; p += 5)
      if (!(used >> p & 1)) {
        lane[j] = p;
        used |= 1u << p;
      }
  }
  for (int j = 0; j < 5; ++j) {
    for (int p = 0; p < m && lane[j] < 0; ++p)
      if (!(used >> p & 1)) {
        lane[j] = p;
        used |= 1u << p;
      }
    rec->bit[at++] = pass_index(lane[j]);
  }
  for (int p = 0; p < m; ++p)
    if (!(used >> p & 1)) rec->bit[at++] = pass_index(p);
}

// x rounded to the nearest bf16 (ties to even); coefficients are finite.
static uint16_t bf16_bits(float x) {
  uint32_t u;
  memcpy(&u, &x, 4);
  return (uint16_t)((u + 0x7fffu + ((u >> 16) & 1u)) >> 16);
}
static float bf16_value(uint16_t b) {
  const uint32_t u = (uint32_t)b << 16;
  float x;
  memcpy(&x, &u, 4);
  return x;
}

// A fragments of the 16 x 16 complex matrix u: row i = 2 r + part of its real
// 32 x 32 form, split into hi + mid + lo, each the bf16 nearest to what the
// parts before it leave (so the sum is within 2^-26 of the FP64 coefficient,
// closer than its FP32 rounding).  Part k, half t of the K range: out[k][t][lane = 32 h + i][j], j the component (amplitude
// 4 q + 2 h + e, part c) with j = 4 (q - 2 t) + 2 e + c.
static void pass_fragments(uint16_t* out, const double* u) {
  for (int t = 0; t < 2; ++t)
    for (int h = 0; h < 2; ++h)
      for (int i = 0; i < 2 * kPassD; ++i)
        for (int j = 0; j < 8; ++j) {
          const int amp = 4 * (2 * t + (j >> 2)) + 2 * h + ((j >> 1) & 1), c = j & 1;
          const double* e = u + 2 * ((i >> 1) * kPassD + amp);
          const int part = i & 1;
          double v = part == c ? e[0] : (part ? e[1] : -e[1]);
          for (int k = 0; k < 3; ++k) {
            const uint16_t b = bf16_bits((float)v);
            out[((2 * k + t) * 64 + 32 * h + i) * 8 + j] = b;
            v -= (double)bf16_value(b);
          }
        }
}

}  // namespace qsim

using namespace qsim;

extern "C" {

int qsim_plan_blocks_search(int n_qubits, int k, int effort, int n_ops, const int32_t* op_nq,
                            const int32_t* op_qubits, const double* op_mats, int32_t* out_ref,
                            int32_t* block_qubits, double* block_mats, int* n_out) {
  if (effort < 0 || effort > 1) return fail(QSIM_EINVAL, "effort %d outside 0..1", effort);
  if (n_qubits < 1 || n_qubits > QSIM_MAX_QUBITS) return fail(QSIM_ERANGE, "n_qubits=%d", n_qubits);
  if (k < 1 || k > QSIM_MAX_BLOCK_QUBITS) return fail(QSIM_ERANGE, "block size k=%d outside 1..%d", k,
                                                      QSIM_MAX_BLOCK_QUBITS);
  if (n_ops < 0) return fail(QSIM_EINVAL, "n_ops < 0");
  if (!n_out || (n_ops > 0 && (!op_nq || !op_qubits || !op_mats || !out_ref || !block_qubits ||
                               !block_mats)))
    return fail(QSIM_EINVAL, "NULL pointer argument");
  const int kk = k < n_qubits ? k : n_qubits;
  const int D = 1 << kk;
  const bool weigh = kk == 5 && n_qubits > 25;
  std::vector<uint64_t> mask(n_ops);
  std::vector<size_t> moff(n_ops);
  size_t off = 0;
  for (int i = 0; i < n_ops; ++i) {
    const int nq = op_nq[i];
    if (nq < 1 || nq > 8) return fail(QSIM_EINVAL, "op %d has %d qubits (1..8)", i, nq);
    uint64_t m = 0;
    for (int j = 0; j < nq; ++j) {
      const int q = op_qubits[i * 8 + j];
      if (q < 0 || q >= n_qubits) return fail(QSIM_EINVAL, "op %d: qubit %d out of range", i, q);
      if (m >> q & 1) return fail(QSIM_EINVAL, "op %d: repeated qubit %d", i, q);
      m |= 1ull << q;
    }
    mask[i] = m;
    moff[i] = off;
    off += (size_t)1 << (2 * nq);
  }
  std::vector<int> rem(n_ops), keep, best;
  for (int i = 0; i < n_ops; ++i) rem[i] = i;
  std::vector<int> chosen;
  int n_entries = 0, n_blocks = 0;
  std::vector<double> mre((size_t)D * D), mim((size_t)D * D), tre((size_t)256 * D),
      tim((size_t)256 * D);
  uint64_t best_bq = 0;
  while (!rem.empty()) {
    // try up to kSeeds eligible seeds; keep the block that absorbs the most ops
    best.clear();
    best_bq = 0;
    uint64_t before = 0;   // qubits of the remaining ops ahead of the candidate seed
    int tried = 0;
    for (size_t sc = 0; sc < rem.size() && tried < kSeeds; before |= mask[rem[sc]], ++sc) {
      const uint64_t ms = mask[rem[sc]];
      if (ms & before) continue;                          // not movable to the front
      if (__builtin_popcountll(ms) > kk) continue;        // wider than a block
      ++tried;
      uint64_t bq = ms, blocked = 0;
      chosen.clear();
      for (size_t t = 0; t < rem.size(); ++t) {
        const int i = rem[t];
        const uint64_t m = mask[i];
        if (t == sc) {
          chosen.push_back(i);
          continue;
        }
        if (m & blocked) {
          blocked |= m;
          continue;
        }
        const uint64_t un = bq | m;
        if (__builtin_popcountll(un) <= kk) {
          bq = un;
          chosen.push_back(i);
        } else {
          blocked |= m;
        }
        // a full block whose qubits are all blocked can take nothing more
        if (t > sc && __builtin_popcountll(bq) == kk && (blocked & bq) == bq) break;
      }
      if (best.empty() || block_score((int)chosen.size(), bq, weigh) > block_score((int)best.size(), best_bq, weigh)) {
        best = chosen;
        best_bq = bq;
      }
      if (effort >= 1) {
        // qubits the next ops connect to the seed, then every S of the
        // seed's qubits and up to kk - |seed| of them
        uint64_t conn = ms;
        const size_t wend = std::min(rem.size(), sc + (size_t)kSearchWindow);
        for (size_t t = sc; t < wend; ++t)
          if (mask[rem[t]] & conn) conn |= mask[rem[t]];
        int extra[kSearchQubits], ne = 0;
        for (int q = 0; q < n_qubits && ne < kSearchQubits; ++q)
          if ((conn >> q & 1) && !(ms >> q & 1)) extra[ne++] = q;
        const int room = kk - __builtin_popcountll(ms);
        // subsets of extra with 1..room members (Gosper's next-combination)
        long long best_sc = block_score((int)best.size(), best_bq, weigh);
        uint64_t best_s = 0;
        for (int r = 1; r <= room && r <= ne; ++r) {
          for (uint32_t sub = (1u << r) - 1; sub < (1u << ne);) {
            uint64_t S = ms;
            for (int e = 0; e < ne; ++e)
              if (sub >> e & 1) S |= 1ull << extra[e];
            const long long sc = block_score(absorb_set(rem, mask, S, nullptr), S, weigh);
            if (sc > best_sc) {
              best_sc = sc;
              best_s = S;
            }
            const uint32_t c = sub & (0u - sub), nx = sub + c;
            sub = (((nx ^ sub) >> 2) / c) | nx;
          }
        }
        if (best_s) {
          best.clear();
          absorb_set(rem, mask, best_s, &best);
          uint64_t u = 0;
          for (int i : best) u |= mask[i];
          best_bq = u;
        }
      }
    }
    if (best.empty()) {  // every candidate is wider than k: the first op passes through
      out_ref[n_entries++] = -1 - rem[0];
      rem.erase(rem.begin());
      continue;
    }
    chosen = best;
    uint64_t bq = best_bq;
    keep.clear();
    {
      size_t c = 0;
      for (int i : rem) {
        if (c < chosen.size() && chosen[c] == i) ++c;
        else keep.push_back(i);
      }
    }
    rem.swap(keep);
    int bqs[8], nb = 0;
    for (int q = 0; q < n_qubits && nb < 8; ++q)
      if (bq >> q & 1) bqs[nb++] = q;
    // padding qubits: the lowest unused from kPadFrom up, then below it
    for (int pass = 0; pass < 2; ++pass)
      for (int q = pass ? 0 : std::min(kPadFrom, n_qubits); q < n_qubits && nb < kk; ++q)
        if (!(bq >> q & 1)) { bqs[nb++] = q; bq |= 1ull << q; }
    // ascending order
    for (int a = 0; a < nb; ++a)
      for (int b = a + 1; b < nb; ++b)
        if (bqs[b] < bqs[a]) { int t = bqs[a]; bqs[a] = bqs[b]; bqs[b] = t; }
    std::fill(mre.begin(), mre.end(), 0.0);
    std::fill(mim.begin(), mim.end(), 0.0);
    for (int r = 0; r < D; ++r) mre[(size_t)r * D + r] = 1.0;
    for (int i : chosen) {
      const int nq = op_nq[i];
      int pos[8];
      for (int j = 0; j < nq; ++j) {
        const int q = op_qubits[i * 8 + j];
        for (int b = 0; b < nb; ++b)
          if (bqs[b] == q) pos[j] = b;
      }
      apply_rows(mre.data(), mim.data(), D, op_mats + 2 * moff[i], pos, nq, tre.data(), tim.data());
    }
    for (int b = 0; b < 8; ++b) block_qubits[n_blocks * 8 + b] = b < nb ? bqs[b] : -1;
    double* dst = block_mats + (size_t)n_blocks * D * D * 2;
    for (size_t e = 0; e < (size_t)D * D; ++e) {
      dst[2 * e] = mre[e];
      dst[2 * e + 1] = mim[e];
    }
    out_ref[n_entries++] = n_blocks++;
  }
  *n_out = n_entries;
  return QSIM_OK;
}

int qsim_plan_blocks(int n_qubits, int k, int n_ops, const int32_t* op_nq, const int32_t* op_qubits,
                     const double* op_mats, int32_t* out_ref, int32_t* block_qubits,
                     double* block_mats, int* n_out) {
  return qsim_plan_blocks_search(n_qubits, k, 0, n_ops, op_nq, op_qubits, op_mats, out_ref,
                                 block_qubits, block_mats, n_out);
}

int qsim_count_blocks(int n_qubits, int k, int n_ops, const uint64_t* op_masks, int* n_blocks) {
  if (n_qubits < 1 || n_qubits > QSIM_MAX_QUBITS) return fail(QSIM_ERANGE, "n_qubits=%d", n_qubits);
  if (k < 1 || k > QSIM_MAX_BLOCK_QUBITS) return fail(QSIM_ERANGE, "block size k=%d outside 1..%d", k,
                                                      QSIM_MAX_BLOCK_QUBITS);
  if (n_ops < 0) return fail(QSIM_EINVAL, "n_ops < 0");
  if (!n_blocks || (n_ops > 0 && !op_masks)) return fail(QSIM_EINVAL, "NULL pointer argument");
  const uint64_t all = (1ull << n_qubits) - 1;
  for (int i = 0; i < n_ops; ++i)
    if (op_masks[i] == 0 || (op_masks[i] & ~all)) return fail(QSIM_EINVAL, "op %d: qubit set outside the state", i);
  try {
    std::vector<uint64_t> rem(op_masks, op_masks + n_ops);
    size_t head = 0;                     // ops before it are done
    int blocks = 0;
    while (head < rem.size()) {
      // ops left out are moved up behind the ones not looked at
      uint64_t set = 0, blocked = 0;
      size_t t = head, left = 0;
      for (; t < rem.size() && (blocked & all) != all; ++t) {
        const uint64_t m = rem[t];
        if (!(m & blocked) && __builtin_popcountll(set | m) <= k) {
          set |= m;
        } else {
          blocked |= m;
          rem[head + left++] = m;
        }
      }
      std::copy_backward(rem.begin() + head, rem.begin() + head + left, rem.begin() + t);
      head = t - left;
      if (set) ++blocks;
      else ++head;                       // wider than a block, and so is all beside it: passes through
    }
    *n_blocks = blocks;
    return QSIM_OK;
  } catch (const std::bad_alloc&) {
    return fail(QSIM_ENOMEM, "block count: out of host memory");
  }
}

int qsim_plan_passes(int n_qubits, int tile_bits, int low_bits, int n_ops, const int32_t* op_nq,
                     const int32_t* op_qubits, const double* op_mats, int32_t* out_ref,
                     qsim_pass* passes, qsim_pass_block* blocks, uint16_t* frags, int* n_out,
                     int* n_blocks) {
  if (n_qubits < QSIM_PASS_MIN_TILE || n_qubits > QSIM_MAX_QUBITS)
    return fail(QSIM_ERANGE, "n_qubits=%d outside %d..%d", n_qubits, QSIM_PASS_MIN_TILE, QSIM_MAX_QUBITS);
  if (tile_bits < QSIM_PASS_MIN_TILE || tile_bits > QSIM_PASS_MAX_TILE)
    return fail(QSIM_ERANGE, "tile of %d qubits outside %d..%d", tile_bits, QSIM_PASS_MIN_TILE, QSIM_PASS_MAX_TILE);
  const int m = std::min(tile_bits, n_qubits);
  if (low_bits < 1 || low_bits > m - kPassK)
    return fail(QSIM_EINVAL, "low_bits %d outside 1..%d", low_bits, m - kPassK);
  if (n_ops < 0) return fail(QSIM_EINVAL, "n_ops < 0");
  if (!n_out || !n_blocks || (n_ops > 0 && (!op_nq || !op_qubits || !op_mats || !out_ref || !passes || !blocks ||
                                            !frags)))
    return fail(QSIM_EINVAL, "NULL pointer argument");
  try {
    PassPlan p;
    p.n = n_qubits;
    p.m = m;
    p.low = (1ull << low_bits) - 1;
    p.mask.resize(n_ops);
    std::vector<size_t> moff(n_ops);
    size_t off = 0;
    for (int i = 0; i < n_ops; ++i) {
      const int nq = op_nq[i];
      if (nq < 1 || nq > 8) return fail(QSIM_EINVAL, "op %d has %d qubits (1..8)", i, nq);
      uint64_t mk = 0;
      for (int j = 0; j < nq; ++j) {
        const int q = op_qubits[i * 8 + j];
        if (q < 0 || q >= n_qubits) return fail(QSIM_EINVAL, "op %d: qubit %d out of range", i, q);
        if (mk >> q & 1) return fail(QSIM_EINVAL, "op %d: repeated qubit %d", i, q);
        mk |= 1ull << q;
      }
      p.mask[i] = mk | (nq > kPassK ? kWide : 0);
      moff[i] = off;
      off += (size_t)1 << (2 * nq);
    }
    p.rem.resize(n_ops);
    for (int i = 0; i < n_ops; ++i) p.rem[i] = i;
    const uint64_t all = (1ull << n_qubits) - 1;
    std::vector<int> chosen, keep, sub_nq, sub_q, ref, bq;
    std::vector<double> sub_m, bm;
    std::vector<uint64_t> starts;
    int np = 0, nb = 0, ne = 0;
    while (!p.rem.empty()) {
      // candidate tiles
      uint64_t best_S = 0;
      int best_cnt = 0;
      starts.assign(1, p.low);
      uint64_t blocked = 0;
      for (int i : p.rem) {
        const uint64_t mk = p.mask[i];
        if (!(mk & blocked) && !(mk & kWide)) {
          const uint64_t un = p.low | mk;
          if (std::find(starts.begin(), starts.end(), un) == starts.end()) starts.push_back(un);
        }
        blocked |= mk;
        if ((blocked & all) == all) break;
      }
      for (uint64_t s0 : starts) {
        int cnt = 0;
        const uint64_t S = m == n_qubits ? all : grow_tile(p, s0, &cnt);
        if (m == n_qubits) cnt = absorb_set(p.rem, p.mask, S, nullptr);
        if (cnt > best_cnt) {
          best_cnt = cnt;
          best_S = S;
        }
        if (m == n_qubits) break;
      }
      if (best_cnt == 0) {               // the first op is wider than a block
        out_ref[ne++] = -1 - p.rem[0];
        p.rem.erase(p.rem.begin());
        continue;
      }
      for (int q = 0; q < n_qubits && __builtin_popcountll(best_S) < m; ++q) best_S |= 1ull << q;
      chosen.clear();
      absorb_set(p.rem, p.mask, best_S, &chosen);
      keep.clear();
      {
        size_t c = 0;
        for (int i : p.rem) {
          if (c < chosen.size() && chosen[c] == i) ++c;
          else keep.push_back(i);
        }
      }
      p.rem.swap(keep);
      // the pass's ops on tile-local qubits, packed into blocks
      const int ns = (int)chosen.size();
      sub_nq.resize(ns);
      sub_q.assign((size_t)ns * 8, -1);
      sub_m.clear();
      for (int c = 0; c < ns; ++c) {
        const int i = chosen[c], nq = op_nq[i];
        sub_nq[c] = nq;
        for (int j = 0; j < nq; ++j)
          sub_q[c * 8 + j] = __builtin_popcountll(best_S & ((1ull << op_qubits[i * 8 + j]) - 1));
        const double* u = op_mats + 2 * moff[i];
        sub_m.insert(sub_m.end(), u, u + ((size_t)2 << (2 * nq)));
      }
      ref.resize(ns);
      bq.resize((size_t)ns * 8);
      bm.resize((size_t)ns * kPassD * kPassD * 2);
      int n_ent = 0;
      if (int rc = qsim_plan_blocks_search(m, kPassK, 1, ns, sub_nq.data(), sub_q.data(), sub_m.data(), ref.data(),
                                           bq.data(), bm.data(), &n_ent))
        return rc;
      passes[np].tile_mask = best_S;
      passes[np].first_block = nb;
      passes[np].n_blocks = n_ent;        // every entry is a block: no op here is wider than one
      for (int b = 0; b < n_ent; ++b, ++nb) {
        pass_record(blocks + nb, m, &bq[(size_t)b * 8]);
        pass_fragments(frags + (size_t)nb * QSIM_PASS_BLOCK_BF16, &bm[(size_t)b * kPassD * kPassD * 2]);
      }
      out_ref[ne++] = np++;
    }
    *n_out = ne;
    *n_blocks = nb;
    return QSIM_OK;
  } catch (const std::bad_alloc&) {
    return fail(QSIM_ENOMEM, "pass planner: out of host memory");
  }
}

}  // extern "C"
