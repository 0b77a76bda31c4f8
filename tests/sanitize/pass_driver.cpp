// Host driver for qsim_plan_passes and qsim_count_blocks (csrc/host_plan.cpp)
// built with the host sanitizers by tests/test_pass_planner_sanitizers.py.
// Random op lists of 1..8 qubits go into buffers of exactly the promised
// capacity; each plan, replayed in FP64 from its block records and matrix
// fragments, equals the ops applied one by one, and malformed arguments are
// rejected.  Exit status 0 on success.
#include <complex>
#include <cstdarg>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <random>
#include <vector>

#include "qsim_gfx950.h"

namespace qsim {
static char g_msg[256];
int fail(int code, const char* fmt, ...) {
  va_list ap;
  va_start(ap, fmt);
  vsnprintf(g_msg, sizeof g_msg, fmt, ap);
  va_end(ap);
  return code;
}
void clear_error() { g_msg[0] = 0; }
}  // namespace qsim

using cd = std::complex<double>;

// psi <- u on qubits q (row bit j <-> q[j]), u row-major.
static void apply(std::vector<cd>& psi, const std::vector<cd>& u, const std::vector<int>& q) {
  const size_t d = (size_t)1 << q.size();
  uint64_t m = 0;
  for (int x : q) m |= 1ull << x;
  std::vector<cd> in(d);
  std::vector<uint64_t> idx(d);
  for (uint64_t b = 0; b < psi.size(); ++b) {
    if (b & m) continue;
    for (size_t s = 0; s < d; ++s) {
      uint64_t i = b;
      for (size_t j = 0; j < q.size(); ++j)
        if (s >> j & 1) i |= 1ull << q[j];
      idx[s] = i;
      in[s] = psi[i];
    }
    for (size_t r = 0; r < d; ++r) {
      cd acc = 0;
      for (size_t c = 0; c < d; ++c) acc += u[r * d + c] * in[c];
      psi[idx[r]] = acc;
    }
  }
}

static double bf16(uint16_t b) {
  const uint32_t u = (uint32_t)b << 16;
  float x;
  memcpy(&x, &u, 4);
  return x;
}

// The 16 x 16 matrix of a block's fragments [3 parts][2 halves][64 lanes][8].
static std::vector<cd> matrix(const uint16_t* f) {
  std::vector<cd> u(256);
  for (int t = 0; t < 2; ++t)
    for (int lane = 0; lane < 64; ++lane)
      for (int j = 0; j < 8; ++j) {
        double v = 0;
        for (int k = 0; k < 3; ++k) v += bf16(f[((2 * k + t) * 64 + lane) * 8 + j]);
        const int row = lane & 31, amp = 4 * (2 * t + (j >> 2)) + 2 * (lane >> 5) + ((j >> 1) & 1);
        if (row & 1) continue;                            // the real row gives Re and -Im
        cd& e = u[(row >> 1) * 16 + amp];
        if (j & 1) e.imag(-v);
        else e.real(v);
      }
  return u;
}

#define CHECK(c, ...)              \
  do {                             \
    if (!(c)) {                    \
      std::printf(__VA_ARGS__);    \
      std::printf("\n");           \
      return 1;                    \
    }                              \
  } while (0)

int main() {
  std::mt19937_64 rng(2718);
  std::normal_distribution<double> nd;
  int n_passes = 0, passthrough = 0;
  for (int trial = 0; trial < 80; ++trial) {
    const int n = 10 + (int)(rng() % 4), tile = 10 + (int)(rng() % 4), m = (int)(rng() % 30);
    const int tm = tile < n ? tile : n, low = 1 + (int)(rng() % (tm - 4));
    std::vector<int32_t> nq(m), qs(8 * (size_t)m, -1);
    std::vector<double> mats;
    std::vector<std::vector<cd>> us(m);
    std::vector<std::vector<int>> oq(m);
    std::vector<uint64_t> masks(m);
    for (int i = 0; i < m; ++i) {
      const int w = rng() % 6 ? 1 + (int)(rng() % 4) : 5 + (int)(rng() % (trial % 8 ? 1 : 4));
      std::vector<int> perm(n);
      for (int a = 0; a < n; ++a) perm[a] = a;
      for (int a = 0; a < w; ++a) std::swap(perm[a], perm[a + rng() % (n - a)]);
      nq[i] = w;
      masks[i] = 0;
      for (int a = 0; a < w; ++a) {
        qs[8 * i + a] = perm[a];
        masks[i] |= 1ull << perm[a];
      }
      oq[i].assign(perm.begin(), perm.begin() + w);
      for (int e = 0; e < (1 << (2 * w)); ++e) {
        const cd v = cd(nd(rng), nd(rng)) / std::sqrt(2.0 * (1 << w));      // norm of about 1
        us[i].push_back(v);
        mats.push_back(v.real());
        mats.push_back(v.imag());
      }
    }
    std::vector<int32_t> ref(m);
    std::vector<qsim_pass> passes(m);
    std::vector<qsim_pass_block> blocks(m);
    std::vector<uint16_t> frags((size_t)m * QSIM_PASS_BLOCK_BF16);
    int n_out = -1, nb = -1;
    const int rc = qsim_plan_passes(n, tile, low, m, nq.data(), qs.data(), mats.data(), ref.data(), passes.data(),
                                    blocks.data(), frags.data(), &n_out, &nb);
    CHECK(rc == QSIM_OK && n_out >= 0 && n_out <= m && nb >= 0 && nb <= m, "trial %d: rc=%d n_out=%d nb=%d (%s)",
          trial, rc, n_out, nb, qsim::g_msg);
    std::vector<cd> a(1ull << n), b;
    for (auto& x : a) x = cd(nd(rng), nd(rng));
    b = a;
    for (int i = 0; i < m; ++i) apply(a, us[i], oq[i]);
    int next_pass = 0, next_block = 0;
    for (int e = 0; e < n_out; ++e) {
      if (ref[e] < 0) {
        const int i = -1 - ref[e];
        CHECK(i < m && nq[i] > 4, "trial %d: bad passthrough %d", trial, i);
        apply(b, us[i], oq[i]);
        ++passthrough;
        continue;
      }
      CHECK(ref[e] == next_pass, "trial %d: pass %d out of order", trial, ref[e]);
      const qsim_pass& p = passes[next_pass++];
      CHECK(__builtin_popcountll(p.tile_mask) == tm && !(p.tile_mask >> n) &&
                (p.tile_mask & ((1ull << low) - 1)) == (1ull << low) - 1 && p.first_block == next_block && p.n_blocks > 0,
            "trial %d: pass %d is malformed", trial, ref[e]);
      std::vector<int> tq;
      for (int q = 0; q < n; ++q)
        if (p.tile_mask >> q & 1) tq.push_back(q);
      for (int k = 0; k < p.n_blocks; ++k, ++next_block) {
        std::vector<int> q;
        for (int j = 0; j < 4; ++j) q.push_back(tq[31 - __builtin_clz((unsigned)blocks[next_block].bit[j])]);
        apply(b, matrix(&frags[(size_t)next_block * QSIM_PASS_BLOCK_BF16]), q);
      }
      ++n_passes;
    }
    CHECK(next_block == nb, "trial %d: %d blocks of %d in passes", trial, next_block, nb);
    double err = 0, scale = 0;
    for (size_t i = 0; i < a.size(); ++i) {
      err += std::norm(a[i] - b[i]);
      scale += std::norm(a[i]);
    }
    // coefficients within 2^-26 of about 1, 32 to a row, at most 30 blocks of norm about 1..2
    CHECK(err <= 1e-9 * (scale + 1e-9), "trial %d: plan differs by %.3e of %.3e", trial, err, scale);
    int cnt = -1, most = 0;
    for (int i = 0; i < m; ++i) most += nq[i] <= 5;
    CHECK(qsim_count_blocks(n, 5, m, masks.data(), &cnt) == QSIM_OK && cnt >= (most > 0) && cnt <= most,
          "trial %d: %d blocks of %d ops", trial, cnt, most);
  }
  // malformed arguments
  const int32_t nq1[1] = {2};
  const int32_t q1[8] = {0, 9, -1, -1, -1, -1, -1, -1}, q2[8] = {4, 4, -1, -1, -1, -1, -1, -1},
                q3[8] = {4, 12, -1, -1, -1, -1, -1, -1};
  std::vector<double> u1(32, 0.25);
  int32_t out[1];
  qsim_pass ps[1];
  qsim_pass_block bl[1];
  std::vector<uint16_t> fr(QSIM_PASS_BLOCK_BF16);
  int no = 0, nb = 0;
  auto plan = [&](int n, int tile, int low, const int32_t* q, int* cnt) {
    return qsim_plan_passes(n, tile, low, 1, nq1, q, u1.data(), out, ps, bl, fr.data(), cnt, &nb);
  };
  CHECK(plan(12, 10, 4, q1, &no) == QSIM_OK && no == 1 && nb == 1, "a plan of one op was refused");
  CHECK(plan(9, 10, 4, q1, &no) && plan(35, 10, 4, q1, &no) && plan(12, 9, 4, q1, &no) && plan(12, 14, 4, q1, &no) &&
            plan(12, 10, 0, q1, &no) && plan(12, 10, 7, q1, &no) && plan(12, 10, 4, q2, &no) &&
            plan(12, 10, 4, q3, &no) && plan(12, 10, 4, q1, nullptr),
        "malformed plan arguments accepted");
  const uint64_t zero = 0, high = 1ull << 12, one = 3;
  CHECK(qsim_count_blocks(12, 5, 1, &zero, &no) && qsim_count_blocks(12, 5, 1, &high, &no) &&
            qsim_count_blocks(12, 0, 1, &one, &no) && qsim_count_blocks(0, 5, 1, &one, &no) &&
            qsim_count_blocks(12, 5, -1, &one, &no) && qsim_count_blocks(12, 5, 1, nullptr, &no) &&
            qsim_count_blocks(12, 5, 1, &one, nullptr),
        "malformed count arguments accepted");
  std::printf("pass planner ok: 80 random plans of %d passes replayed (%d passthrough entries)\n", n_passes, passthrough);
  return 0;
}
