// flex_chain.cpp -- choice of a flexible chain (flex_engine.hpp).
#include "flex_chain.hpp"

#include <algorithm>
#include <cstring>
#include <set>

namespace plf {

namespace {

// Radices of the engine with their VALU work per point (butterfly, twiddles,
// addresses) plus one exchange; the sum over a chain ranks it.
struct RadixCost {
  int r;
  double c;
};
const RadixCost kRadix[] = {{16, 40}, {15, 43}, {13, 45}, {12, 38}, {11, 42}, {10, 39}, {9, 42},
                            {8, 36},  {7, 39},  {6, 36},  {5, 37},  {4, 33},  {3, 35},  {2, 32}};
// per thread and stage: barriers, stage description, loop control; and where
// no other blocks hide the barriers and the LDS accesses
constexpr double kStageOverhead = 150, kStageWait = 670;

// the compiled shape of radix r with at least kb butterflies, or -1
int shape_for(int r, int64_t kb, int pts) {
  int best = -1;
  for (int i = 0; i < kFlexShapeCount; ++i)
    if (kFlexShapes[i].r == r && kFlexShapes[i].k >= kb && r * kFlexShapes[i].k <= std::max(pts, r) &&
        (best < 0 || kFlexShapes[i].k < kFlexShapes[best].k))
      best = i;
  return best;
}

double radix_cost(int r) {
  for (const auto &k : kRadix)
    if (k.r == r) return k.c;
  return 1e9;
}

void multisets(int64_t n, size_t from, std::vector<int> &cur, std::vector<std::vector<int>> &out) {
  if (n == 1) {
    out.push_back(cur);
    return;
  }
  if (cur.size() == kFlexStages) return;
  for (size_t i = from; i < sizeof(kRadix) / sizeof(kRadix[0]); ++i) {
    const int r = kRadix[i].r;
    if (n % r) continue;
    cur.push_back(r);
    multisets(n / r, i, cur, out);
    cur.pop_back();
  }
}

// Passes that a wave's access at addr(lane) takes beyond the least, over the
// bank slots of one element each.
template <class F>
int conflicts(int slots, F &&addr) {
  int worst = 0;
  for (int h = 0; h < 64; h += slots) {
    int cnt[32] = {0};
    int64_t at[32][32];  // the distinct addresses of each slot
    for (int l = h; l < h + slots; ++l) {
      const int64_t a = addr(l);
      const int s = (int)(a % slots);
      if (std::find(at[s], at[s] + cnt[s], a) != at[s] + cnt[s]) continue;  // broadcast
      at[s][cnt[s]++] = a;
      worst = std::max(worst, cnt[s]);
    }
  }
  return worst - 1;
}

}  // namespace

bool flex_choose(int64_t n, int pts, int block, int csize, int64_t lds_max, int lanes,
                 FlexDesc *out, const FlexWait *wait) {
  if (n < 2 || n >= (1 << 15)) return false;
  const bool idle = wait && wait->members > 0;
  std::vector<std::vector<int>> sets;
  std::vector<int> cur;
  multisets(n, 0, cur, sets);
  double best = 0;
  std::vector<int> chain;
  int best_tpt = 0, best_tpb = 0;
  for (const auto &c : sets) {
    std::set<int> cand;
    for (int r : c)
      for (const auto &sh : kFlexShapes)
        if (sh.r == r) cand.insert((int)((n / r + sh.k - 1) / sh.k));
    if (wait && wait->spare) cand.insert({2, 4, 8, 16});  // threads beyond the butterflies
    for (int tpt : cand) {
      if (tpt > block || tpt < 1) continue;
      double work = 0;
      int first = 0;  // points of the first stage a thread
      bool ok = true;
      for (int r : c) {
        const int64_t nb = n / r;
        const int sh = shape_for(r, (nb + tpt - 1) / tpt, pts);
        if (sh < 0) {
          ok = false;
          break;
        }
        work += (double)kFlexShapes[sh].k * r * radix_cost(r) + (idle ? kStageWait : kStageOverhead);
        if (r == c.front()) first = kFlexShapes[sh].k * r;
      }
      if (!ok) continue;
      if (wait)
        work += wait->real * (2.0 * n / tpt) * (idle ? 1.0 : 1.0 + 8.0 / tpt) + wait->first * first;
      // members per block: the fullest waves among blocks of up to 512
      // threads (or one member), LDS permitting (half of a CU's, so that two
      // blocks share it, where a block holds several members); a waiting
      // batch takes one wave's members until the chip is full
      const int64_t mem = (n + n / 8 + 34) * csize;
      if ((n + 2) * csize > lds_max) continue;
      const int most = lanes ? lanes : 512;
      int tmax = std::min(most, std::max(1, std::min(block, lanes ? block : 512) / tpt));
      tmax = (int)std::min<int64_t>(tmax, std::max<int64_t>(1, std::min<int64_t>(lds_max, lds_max / 2) / mem));
      const int least = lanes ? tmax : idle ? std::min(tmax, std::max(1, 64 / tpt)) : 1;
      for (int tpb = least; tpb <= tmax; ++tpb) {
        const int threads = (tpt * tpb + 63) / 64 * 64;
        if (threads > block) break;
        double cost = work * threads / ((double)tpb * n);
        if (idle) {
          const int64_t all = (wait->members + tpb - 1) / tpb * threads;
          cost = work * std::max(1.0, (double)all / wait->resident);
        }
        if (!lanes && !idle && threads < 192)
          cost *= 1.0 + 0.1 * (192 - threads) / 64;  // few waves a block
        if (threads > 256) cost *= 1.03;                                       // wider barriers
        if (lanes) cost *= 1.0 + 0.5 * (lanes - tpb) / lanes;                  // shorter runs
        if (!best_tpt || cost < best) {
          best = cost;
          best_tpt = tpt;
          best_tpb = tpb;
          chain = c;
        }
      }
    }
  }
  if (!best_tpt) return false;

  FlexDesc d;
  std::memset(&d, 0, sizeof(d));
  d.n = (int)n;
  d.ns = (int)chain.size();
  d.tpt = best_tpt;
  d.tpb = best_tpb;
  d.lanes = lanes ? 1 : 0;
  const int div = lanes ? best_tpb : best_tpt;
  d.magic = div > 1 ? (uint32_t)(((uint64_t(1) << 32) + div - 1) / div) : 0;
  int64_t L = 1, off = 0;
  for (int s = 0; s < d.ns; ++s) {
    FlexStage &st = d.st[s];
    st.L = (int)L;
    st.nb = (int)(n / chain[s]);
    st.shape = shape_for(chain[s], (st.nb + best_tpt - 1) / best_tpt, pts);
    st.twoff = (int)off;
    st.magic = L > 1 ? (uint32_t)(((uint64_t(1) << 32) + L - 1) / L) : 0;
    if (s > 0) off += L * (chain[s] - 1);
    L *= chain[s];
  }
  // exchange layouts: groups of G = L R elements, GP apart
  const int slots = csize == 8 ? 32 : 16;
  int64_t lper = n;
  for (int s = 0; s + 1 < d.ns; ++s) {
    const int64_t Ls = d.st[s].L, G = Ls * chain[s];
    int64_t bp = 0, bc = 0;
    for (int64_t p = 0; p <= std::max<int64_t>(1, std::min<int64_t>(G / 8, 33)); ++p) {
      const int64_t GP = G + p, lp = n / G * GP;
      if (p > 0 && (lp + 1) * csize * best_tpb > lds_max) break;
      auto where = [&](int l, int64_t group) {
        const int64_t g = lanes ? l % best_tpb : l / best_tpt;
        const int64_t b = lanes ? l / best_tpb : l % best_tpt;
        return g * (lp | 1) + (b / group) * GP + b % group;
      };
      const int64_t c = 64 * (conflicts(slots, [&](int l) { return where(l, Ls); }) +
                              conflicts(slots, [&](int l) { return where(l, G); })) + p;
      if (p == 0 || c < bc) {
        bc = c;
        bp = p;
      }
      if (c < 64) break;  // none: a larger pad cannot rank better
    }
    const int64_t GP = G + bp;
    d.st[s].wr_gp = (int)GP;
    d.st[s + 1].rd_gp = (int)GP;
    d.st[s + 1].rd_step = (int)(d.st[s + 1].nb / G * GP);
    lper = std::max(lper, n / G * GP);
  }
  d.lper = (int)(lper | 1);  // members on different banks
  *out = d;
  return true;
}

std::vector<int> flex_radices(const FlexDesc &d) {
  std::vector<int> c;
  for (int s = 0; s < d.ns; ++s) c.push_back(kFlexShapes[d.st[s].shape].r);
  return c;
}

}  // namespace plf
