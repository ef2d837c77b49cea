// Host check of the flexible chains (csrc/flex_chain.cpp): for every length
// that gets one, replays the engine's addressing (csrc/flex_engine.hpp) and
// compares it with the Stockham definition.
//   * the shapes multiply to n and cover every butterfly within the points and
//     threads allowed;
//   * b / L by the reciprocal is exact;
//   * each stage reads element b + m N/R where the previous one wrote it;
//   * no two elements share an LDS slot, and all lie below lper;
//   * thread / divisor by the reciprocal is exact over a block.
// Prints the number of chains checked; exits 1 at the first fault.
#include <cstdio>
#include <cstdlib>
#include <vector>

#include "../../perf-libs-fft_amd/csrc/flex_chain.hpp"

using namespace plf;

static uint32_t umulhi(uint32_t a, uint32_t b) { return (uint32_t)(((uint64_t)a * b) >> 32); }

#define CHECK(c)                                                    \
  do {                                                              \
    if (!(c)) {                                                     \
      std::printf("n=%ld: %s (line %d)\n", (long)n, #c, __LINE__);  \
      std::exit(1);                                                 \
    }                                                               \
  } while (0)

static void check(int64_t n, int pts, int block, int csize, const FlexDesc &d) {
  const int threads = flex_threads(d);
  CHECK(d.n == n && d.ns >= 1 && d.ns <= kFlexStages);
  CHECK(d.tpt >= 1 && d.tpb >= 1 && threads <= block);
  CHECK(flex_lds(d, csize) <= 160 * 1024);
  const int div = d.lanes ? d.tpb : d.tpt;
  for (int t = 0; t < threads; ++t) CHECK((div == 1 ? t : (int)umulhi(t, d.magic)) == t / div);
  int64_t L = 1;
  for (int s = 0; s < d.ns; ++s) {
    const FlexStage &st = d.st[s];
    CHECK(st.shape >= 0 && st.shape < kFlexShapeCount);
    const int R = kFlexShapes[st.shape].r, K = kFlexShapes[st.shape].k;
    CHECK(st.L == L && st.nb == n / R && n % (L * R) == 0);
    CHECK((int64_t)K * d.tpt >= st.nb && K * R <= (pts > R ? pts : R));
    if (d.ns == 1) CHECK(K == 1 && st.nb == 1);
    for (int64_t b = 0; L > 1 && b < st.nb; ++b) CHECK((int64_t)umulhi(b, st.magic) == b / L);
    if (s + 1 < d.ns) {
      // where this stage writes logical element q L R + j + m L
      std::vector<int64_t> at(n, -1);
      std::vector<char> used(d.lper, 0);
      for (int64_t b = 0; b < st.nb; ++b)
        for (int m = 0; m < R; ++m) {
          const int64_t q = b / L, j = b % L, p = q * st.wr_gp + j + m * L;
          CHECK(p >= 0 && p < d.lper && !used[p]);
          used[p] = 1;
          at[q * L * R + j + m * L] = p;
        }
      const FlexStage &nx = d.st[s + 1];
      const int R2 = kFlexShapes[nx.shape].r;
      const int64_t L2 = L * R;
      for (int64_t b = 0; b < n / R2; ++b)
        for (int m = 0; m < R2; ++m)
          CHECK((b / L2) * nx.rd_gp + b % L2 + (int64_t)m * nx.rd_step == at[b + m * (n / R2)]);
    } else {
      CHECK(st.nb == L && n <= d.lper);  // the last stage's stride is its N / R
    }
    L *= R;
  }
  CHECK(L == n);
}

int main() {
  long count = 0;
  const int cfg[][4] = {// pts, block, csize, lanes
                        {20, 512, 8, 0}, {20, 1024, 8, 0}, {16, 256, 16, 0},
                        {16, 512, 16, 0}, {20, 1024, 8, 16}, {16, 512, 16, 8}};
  for (const auto &c : cfg)
    for (int64_t n = 2; n < (1 << 15); ++n) {
      int64_t r = n;
      for (int p : {2, 3, 5, 7, 11, 13})
        while (r % p == 0) r /= p;
      FlexDesc d;
      const bool ok = flex_choose(n, c[0], c[1], c[2], 160 * 1024, c[3], &d);
      if (r != 1) CHECK(!ok);
      if (!ok) continue;
      check(n, c[0], c[1], c[2], d);
      ++count;
    }
  std::printf("%ld chains\n", count);
  return 0;
}
