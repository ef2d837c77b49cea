// flex_plan.cpp -- plan nodes on the flexible-chain kernels
// (kernels_flex.hpp): complex transforms, and real transforms of even length.
#include <algorithm>
#include <cstdint>
#include <sstream>

#include "flex_chain.hpp"
#include "flex_registry.hpp"
#include "plan.hpp"

namespace plf {

const std::vector<FlexEntry> &flex_registry() {
  static const std::vector<FlexEntry> reg = [] {
    std::vector<FlexEntry> r;
    register_flex_f32(r);
    register_flex_f64(r);
    register_flex_real_f32(r);
    register_flex_real_f64(r);
    register_flex_h(r);
    return r;
  }();
  return reg;
}

static const char *flex_kind_name(int k) {
  static const char *names[] = {"c2c", "r2c", "c2r", "dct2", "dct3"};
  return names[k];
}

// The entry and chain for engine length m: the smallest block size that
// holds a member. 20 points a thread in FP32 (92 registers), 16 in FP64.
static const FlexEntry *flex_find(int kind, int64_t m, int prec, bool bwd, int lanes,
                                  FlexDesc *d, const FlexWait *wait = nullptr) {
  const int pts = prec_compute_bytes(prec) == 8 ? 16 : 20;
  const FlexEntry *big = nullptr;
  for (const auto &e : flex_registry()) {
    if (e.kind != kind || e.prec != prec || e.bwd != bwd) continue;
    if (!lanes && flex_choose(m, pts, e.block, 2 * prec_compute_bytes(prec), 160 * 1024, 0, d, wait))
      return &e;
    big = &e;
  }
  if (lanes && big &&
      flex_choose(m, pts, big->block, 2 * prec_compute_bytes(prec), 160 * 1024, lanes, d)) {
    for (const auto &e : flex_registry())
      if (e.kind == kind && e.prec == prec && e.bwd == bwd && flex_threads(*d) <= e.block)
        return &e;
  }
  return nullptr;
}

// Real transforms move a member's reals or bins through LDS outside the chain.
// The chain of least work per member leaves that to few threads (2 for a
// DCT-II of 60), which a full chip hides and a small batch waits for: DCT-II
// of 60 FP32, 256 members, 9.6 us, 6.6 on the runtime chain's 16 threads, and
// 5.0 with 16 threads here; of 3000, 64 members, 13.8, 10.8 and 9.4. So a batch
// of at most half the threads that the chip runs well at once takes the chain
// of least predicted time (units of flex_chain.cpp's work, fitted to 4300
// measured pairs of chains; the DCT-III also computes a bin in its first
// loads). Above that line it is the slower one (DCT-II of 300 FP64, 2048
// members: 13.7 against 10.2 us with 75 threads against 15), and members of
// more than 2048 pairs have a hundred threads or more already (R2C of 12000:
// 10.8 against 10.1 us). C2R moves its reals in the chain's own stages.
//
// On a full chip the loads and stores of a DCT-II of 8 to 256 pairs count too,
// per real and more the fewer lanes share a line (of 32, 2^19 members, FP32
// 154 -> 57 us on 4 threads instead of one, FP64 314 -> 99; of 64, 2^18 members,
// 144 -> 62). Shorter members lose (of 8, 2^21 members, 72 -> 81), longer ones
// have ten threads and more, and in between, with more than half of the
// resident threads but not all, least work per member is best (FP64 of 20,
// 52428 members: 11.3 against 13.4).
static bool flex_wait(int kind, int64_t m, int prec, int64_t howmany, const FlexDesc &d,
                      FlexWait *w) {
  if (m > 2048 || (kind != FK_R2C && kind != FK_DCT2 && kind != FK_DCT3)) return false;
  const int64_t resident = (int64_t)cu_count() * (prec_compute_bytes(prec) == 8 ? 256 : 512);
  const int64_t threads = (howmany + d.tpb - 1) / d.tpb * flex_threads(d);
  if (threads > resident / 2) {
    *w = FlexWait{0, 0, prec_compute_bytes(prec) == 8 ? 8.0 : 20.0, 0, false};
    return kind == FK_DCT2 && m >= 8 && m <= 256 && threads >= resident;
  }
  // (R2C: its first loads come from memory; repeated by spare threads they cost time)
  *w = FlexWait{howmany, resident, kind == FK_DCT2 ? 130.0 : 55.0, kind == FK_DCT3 ? 300.0 : 0.0,
                kind != FK_R2C};
  return true;
}

class FlexNode : public Node {
 public:
  // p with its distances zeroed for one member; m: engine length
  FlexNode(const FlexEntry *e, const FlexDesc &d, const Problem &p, int64_t m)
      : e_(e), d_(d), p_(p), m_(m) {}
  hipError_t init() {
    hipError_t err = upload_table(tw_, stockham_twiddles(flex_radices(d_)), p_.prec);
    if (err == hipSuccess) err = desc_.upload(&d_, sizeof(d_));
    if (err == hipSuccess && e_->kind != FK_C2C)
      err = upload_table(aux0_, root_table(2 * m_, m_ + 1), p_.prec);
    // w_k = exp(-i pi k / 2n) = W_{4n}^k, n = 2m
    if (err == hipSuccess && (e_->kind == FK_DCT2 || e_->kind == FK_DCT3))
      err = upload_table(aux1_, root_table(8 * m_, m_ + 1), p_.prec);
    return err;
  }
  hipError_t enqueue(const void *in, void *out, void *, hipStream_t s) const override {
    if (p_.howmany <= 0) return hipSuccess;
    FlexArgs f{};
    KArgs &a = f.a;
    a.in = in;
    a.out = out;
    a.tw = tw_.p;
    a.aux0 = aux0_.p;
    a.aux1 = aux1_.p;
    a.count = p_.howmany;
    a.istride = p_.istride;
    a.idist = p_.idist;
    a.ostride = p_.ostride;
    a.odist = p_.odist;
    a.n = m_;
    f.d = static_cast<const FlexDesc *>(desc_.p);
    if (e_->kind == FK_R2C || e_->kind == FK_C2R) {
      // real side as complex pairs: unit stride, even distance, aligned base
      const bool r2c = e_->kind == FK_R2C;
      const size_t pair = 2 * (size_t)prec_real_bytes(p_.prec);
      const int64_t rs = r2c ? p_.istride : p_.ostride, rd = r2c ? p_.idist : p_.odist;
      if (rs == 1 && rd % 2 == 0 && (uintptr_t)(r2c ? in : out) % pair == 0) a.flags |= 1;
    }
    if (e_->kind == FK_C2C) {
      // neighbouring tiles of columns share lines unless the rows are whole
      // 4 KiB (as TileColumnsNode)
      const int64_t pitch = p_.istride * 2 * prec_real_bytes(p_.prec);
      if (d_.lanes && pitch % 4096) a.flags |= 1;
    }
    if (p_.adjoint) a.flags |= 2;
    const int csize = 2 * prec_compute_bytes(p_.prec);
    return e_->launch(f, (p_.howmany + d_.tpb - 1) / d_.tpb, flex_threads(d_),
                      flex_lds(d_, csize), s);
  }
  std::string describe() const override {
    std::ostringstream o;
    o << "(flex_" << flex_kind_name(e_->kind) << "_" << prec_name(p_.prec)
      << (e_->bwd ? "_bwd" : "_fwd") << "_n" << p_.n << "_r";
    const std::vector<int> c = flex_radices(d_);
    for (size_t i = 0; i < c.size(); ++i) o << (i ? "x" : "") << c[i];
    o << "_t" << d_.tpt << "_b" << d_.tpb << (d_.lanes ? "_lanes" : "") << " n=" << p_.n
      << " batch=" << p_.howmany << " is=" << p_.istride << " id=" << p_.idist
      << " os=" << p_.ostride << " od=" << p_.odist << ")";
    return o.str();
  }

 private:
  const FlexEntry *e_;
  FlexDesc d_;
  Problem p_;
  int64_t m_;
  DevMem tw_, desc_, aux0_, aux1_;
};

// Node for a length without a compiled chain, or null (a prime factor above
// 13, no room, or spans past the kernels' 32-bit offsets) with *why untouched
// unless the device fails.
std::unique_ptr<Node> build_flex_node(const Problem &pp, std::string *why) {
  Problem p = pp;
  if (p.howmany <= 1) p.idist = p.odist = 0;
  int kind = FK_C2C;
  bool bwd = p.dir > 0;
  int64_t m = p.n;
  if (p.kind != K_C2C) {
    if (p.n % 2) return nullptr;
    m = p.n / 2;
    bwd = false;
    if (p.kind == K_R2C) kind = FK_R2C;
    else if (p.kind == K_C2R) kind = FK_C2R;
    else if (p.r2r_kind == 1 || p.r2r_kind == 5) kind = FK_DCT2, bwd = p.r2r_kind == 5;
    else if (p.r2r_kind == 2 || p.r2r_kind == 6) kind = FK_DCT3, bwd = p.r2r_kind == 6;
    else return nullptr;
  }
  // columns: lanes along the members that share a line. Fewer than eight members
  // fill half a line at most (us without and with, FP32: 360 points 5.6 and 6.5
  // for 4 members, 6.0 and 6.5 for 8; 100 points 5.6 and 4.4 for 8; 1500 11.4 and
  // 8.1). Long members that leave a block two or three of them wait for it until
  // there are some 64 (3000 points FP32 17.0 and 17.6 for 32, 19.1 and 17.3 for
  // 64, 43.6 and 27.9 for 512, 307 and 191 for 4096; 2000 points FP64 7.8 and 9.4
  // for 8, 12.5 and 9.9 for 64, 70 and 48 for 1024); with one there is nothing to
  // share.
  const int lanes = kind == FK_C2C && p.howmany >= 8 && p.idist < p.istride && p.odist < p.ostride
                        ? 128 / (2 * prec_compute_bytes(p.prec))
                        : 0;
  FlexDesc d;
  const FlexEntry *e = flex_find(kind, m, p.prec, bwd, lanes, &d);
  if (lanes && e && (d.tpb < 2 || (d.tpb < 4 && p.howmany < 64))) e = nullptr;
  if (lanes && !e) e = flex_find(kind, m, p.prec, bwd, 0, &d);
  if (!e) return nullptr;
  FlexWait w;
  if (flex_wait(kind, m, p.prec, p.howmany, d, &w)) {
    FlexDesc other;
    if (const FlexEntry *o = flex_find(kind, m, p.prec, bwd, 0, &other, &w)) e = o, d = other;
  }
  const int64_t rb = prec_real_bytes(p.prec);
  const int64_t ie = kind == FK_C2C || kind == FK_C2R ? 2 * rb : rb;
  auto span = [&](int64_t dist, int64_t stride) {
    const int64_t big = int64_t(1) << 40;
    if (dist > big || stride > big / (p.n + 1)) return big;
    return d.tpb * dist + (p.n + 1) * stride;
  };
  const int64_t limit = int64_t(1) << 32;
  if (span(p.idist, p.istride) >= limit / ie) return nullptr;
  if (kind == FK_C2C && span(p.odist, p.ostride) >= limit / ie) return nullptr;
  auto node = std::make_unique<FlexNode>(e, d, p, m);
  const hipError_t err = node->init();
  if (err != hipSuccess) {
    *why = std::string("device upload failed: ") + hipGetErrorString(err);
    return nullptr;
  }
  return node;
}

}  // namespace plf
