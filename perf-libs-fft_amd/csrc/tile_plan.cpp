// tile_plan.cpp -- plan nodes on the tile kernels (kernels_tile.hpp): columns
// of a matrix, and the four-step with a blocked workspace.
#include <algorithm>
#include <cmath>
#include <cstdint>
#include <sstream>

#include "plan.hpp"
#include "tile_registry.hpp"

namespace plf {

std::string TileEntry::name() const {
  static const char *kinds[] = {"tile_c2c", "tile_col", "tile_row"};
  std::ostringstream o;
  o << kinds[kind] << "_" << prec_name(prec) << (bwd ? "_bwd" : "_fwd") << "_n" << n << "_r";
  for (size_t i = 0; i < chain.size(); ++i) o << (i ? "x" : "") << chain[i];
  o << "_w" << w;
  return o.str();
}

const std::vector<TileEntry> &tile_registry() {
  static const std::vector<TileEntry> reg = [] {
    std::vector<TileEntry> r;
    register_tiles_f32(r);
    register_tiles_f64(r);
    register_tiles_h(r);
    return r;
  }();
  return reg;
}

int cu_count() {
  int dev = 0, c = 0;
  if (hipGetDevice(&dev) != hipSuccess ||
      hipDeviceGetAttribute(&c, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess)
    return 256;
  return c > 0 ? c : 256;
}

static const TileEntry *find_tile(int kind, int64_t n, int prec, bool bwd, int wb = 0) {
  for (const auto &e : tile_registry())
    if (e.kind == kind && e.n == n && e.prec == prec && e.bwd == bwd && (!wb || e.wb == wb))
      return &e;
  return nullptr;
}

// ---------------------------------------------------------------------------
// columns
// ---------------------------------------------------------------------------
class TileColumnsNode : public Node {
 public:
  TileColumnsNode(const TileEntry *e, const Problem &p) : e_(e), p_(p) {}
  hipError_t init() { return upload_table(tw_, stockham_twiddles(e_->chain), p_.prec); }
  hipError_t enqueue(const void *in, void *out, void *, hipStream_t s) const override {
    KArgs a{};
    a.in = in;
    a.out = out;
    a.tw = tw_.p;
    a.count = p_.howmany;
    a.istride = p_.istride;
    a.idist = p_.idist;
    a.ostride = p_.ostride;
    a.odist = p_.odist;
    a.n = p_.n;
    // Block order: with a row pitch of whole 4 KiB every tile starts on a
    // line boundary and neighbouring tiles on all XCDs keep the DRAM pages of
    // a row open (65536 columns of 256: 59 against 63 us); any other pitch
    // puts neighbours, which share lines, on one XCD (16001 columns of 1024:
    // 77 against 97 us).
    const int64_t pitch = p_.istride * 2 * prec_real_bytes(p_.prec);
    a.flags = pitch % 4096 ? 1 : 0;
    return e_->launch(a, (p_.howmany + e_->w - 1) / e_->w, e_->lds, s);
  }
  std::string describe() const override {
    std::ostringstream o;
    o << "(" << e_->name() << " n=" << p_.n << " batch=" << p_.howmany << " is=" << p_.istride
      << " id=" << p_.idist << " os=" << p_.ostride << " od=" << p_.odist << ")";
    return o.str();
  }

 private:
  const TileEntry *e_;
  Problem p_;
  DevMem tw_;
};

// Members closer together than their elements on both sides: lanes along the
// members (a line holds up to 16 of them) instead of along the elements (a
// line each). Few tiles wait for the block's chain, and the general kernel's
// smaller blocks may be faster: below a quarter of the chip's CUs in tiles for 64
// and 512 points, an eighth in FP64 and for 2048, else a 32nd. In us, general
// kernel and tiles, on 8 / 16 / 32 tiles: FP32 128 points 6.1 4.4 / 6.2 4.4 / 6.3
// 4.4, 256 6.2 5.3 / 6.3 5.4 / 6.4 5.5, 512 7.0 8.1 / 7.1 8.3 / 7.5 8.3, 1024
// 10.6 8.6 / 11.1 8.9 / 11.5 9.2, 2048 13.6 18.1 / 15.5 18.5 / 22.6 19.1; FP64
// 256 5.0 4.6 / 5.1 4.7 / 5.1 4.8, 512 5.6 7.6 / 5.7 7.8 / 6.6 7.9, 1024 7.8 7.9 /
// 8.1 8.4 / 9.3 9.0; f16 64 4.2 4.9 / 4.2 5.0 / 4.2 5.0, 512 7.4 9.7 / 8.0 9.8 /
// 9.7 9.7, 1024 13.1 10.3 / 14.6 11.6 / 18.6 13.7; 64 points FP32 and FP64 alike.
std::unique_ptr<Node> build_columns_node(const Problem &p, std::string *why) {
  if (p.howmany < 2 || p.idist >= p.istride || p.odist >= p.ostride) return nullptr;
  const TileEntry *e = find_tile(TK_C2C, p.n, p.prec, p.dir > 0);
  if (!e) return nullptr;
  const int share = p.n == 64 || p.n == 512 ? 4 : p.n == 2048 || p.prec == P_F64 ? 8 : 32;
  if ((p.howmany + e->w - 1) / e->w < cu_count() / share) return nullptr;
  auto node = std::make_unique<TileColumnsNode>(e, p);
  const hipError_t err = node->init();
  if (err != hipSuccess) {
    *why = std::string("device upload failed: ") + hipGetErrorString(err);
    return nullptr;
  }
  return node;
}

// ---------------------------------------------------------------------------
// four-step
// ---------------------------------------------------------------------------
class TileFourStepNode : public Node {
 public:
  TileFourStepNode(const TileEntry *col, const TileEntry *row, const Problem &p, int64_t chunk)
      : col_(col), row_(row), p_(p), chunk_(chunk), n1_(col->n), n2_(row->n) {}

  hipError_t init() {
    hipError_t err = upload_table(tw1_, stockham_twiddles(col_->chain), p_.prec);
    if (err == hipSuccess) err = upload_table(tw2_, stockham_twiddles(row_->chain), p_.prec);
    if (err != hipSuccess) return err;
    // T1[c][b] = W_N^{c b} (b < NB) and T2[c][m] = W_N^{c NB m} (m < RL), each
    // rounded once
    const int64_t n = n1_ * n2_, RL = col_->chain.back(), NB = n1_ / RL;
    const SplitRoots root(n);
    std::vector<double> t1(2 * n2_ * NB), t2(2 * n2_ * RL);
    for (int64_t c = 0; c < n2_; ++c) {
      for (int64_t b = 0; b < NB; ++b) root(c * b, &t1[2 * (c * NB + b)]);
      for (int64_t m = 0; m < RL; ++m) root((c * NB * m) % n, &t2[2 * (c * RL + m)]);
    }
    err = upload_table(t1_, t1, p_.prec);
    if (err == hipSuccess) err = upload_table(t2_, t2, p_.prec);
    return err;
  }
  size_t per_bytes() const { return (size_t)(n1_ * n2_) * 2 * prec_compute_bytes(p_.prec); }
  size_t workspace_bytes() const override { return (size_t)chunk_ * per_bytes(); }
  size_t min_workspace_bytes() const override { return per_bytes(); }
  hipError_t enqueue(const void *in, void *out, void *work, hipStream_t s) const override {
    return run(in, out, work, chunk_, s);
  }
  hipError_t enqueue_capped(const void *in, void *out, void *work, size_t cap,
                            hipStream_t s) const override {
    const int64_t fit = (int64_t)(cap / per_bytes());
    if (fit < 1) return hipErrorInvalidValue;
    return run(in, out, work, std::min(chunk_, fit), s);
  }
  // column pass then row pass over `chunk` members at a time
  hipError_t run(const void *in, void *out, void *work, int64_t chunk, hipStream_t s) const {
    const int64_t n = n1_ * n2_;
    const int64_t id = p_.howmany > 1 ? p_.idist : 0, od = p_.howmany > 1 ? p_.odist : 0;
    const int64_t ie = 2 * (int64_t)prec_real_bytes(p_.prec);
    // a side is accessed in whole lines (and then past the caches, since
    // nothing touches a line twice) when members and tiles fill whole lines
    auto lines = [&](const void *p, int64_t stride, int64_t dist, int w) {
      return stride == 1 && (uintptr_t)p % 128 == 0 && (dist * ie) % 128 == 0 &&
             (w * ie) % 128 == 0;
    };
    for (int64_t b0 = 0; b0 < p_.howmany; b0 += chunk) {
      const int64_t cb = std::min(chunk, p_.howmany - b0);
      KArgs a{};
      a.in = static_cast<const char *>(in) + b0 * id * ie;
      a.out = work;
      a.tw = tw1_.p;
      a.aux0 = t1_.p;
      a.aux1 = t2_.p;
      a.istride = p_.istride;
      a.idist = id;
      a.n1 = n1_;
      a.n2 = n2_;
      a.bigdist = n;
      const KLaunch cl = lines(a.in, p_.istride, id, col_->w) ? col_->launch_nt : col_->launch;
      hipError_t err = cl(a, cb * (n2_ / col_->w), col_->lds, s);
      if (err != hipSuccess) return err;
      KArgs b{};
      b.in = work;
      b.out = static_cast<char *>(out) + b0 * od * ie;
      b.tw = tw2_.p;
      b.ostride = p_.ostride;
      b.odist = od;
      b.n1 = n1_;
      b.n2 = n2_;
      b.bigdist = n;
      const KLaunch rl = lines(b.out, p_.ostride, od, row_->w) ? row_->launch_nt : row_->launch;
      err = rl(b, cb * (n1_ / row_->w), row_->lds, s);
      if (err != hipSuccess) return err;
    }
    return hipSuccess;
  }
  std::string describe() const override {
    std::ostringstream o;
    o << "(fourstep n=" << n1_ * n2_ << " = " << n1_ << "x" << n2_ << " chunk=" << chunk_
      << " batch=" << p_.howmany << " " << col_->name() << " " << row_->name() << ")";
    return o.str();
  }

 private:
  const TileEntry *col_, *row_;
  Problem p_;
  int64_t chunk_, n1_, n2_;
  DevMem tw1_, tw2_, t1_, t2_;
};

// The balanced split n1 <= n2 <= 2 n1 with tile kernels for both sides
// (powers of two up to 2^22); the others keep the passes of kernels.hpp. So do
// FP32 and FP64 batches whose passes have fewer blocks than the chip has CUs:
// those wait for single blocks, and the narrower tiles with fewer points per
// thread of kernels.hpp answer sooner (2^18 FP32: 19 against 26 us for 4
// members, 24 against 27 for 8 (128 blocks), 68 against 52 for 32; 2^18 FP64:
// 21 against 23 us for 4, 34 against 33 for 8 (256 blocks)). The 16-bit types
// have only runtime chains there and always take the tiles (f16, passes against
// tiles: 65536 17.3 and 12.4 us for one member, 22.1 and 14.5 for 16, 59.6 and
// 25.9 for 64; 2^18 24.6 and 22.0, 32 and 26 for 8, 216 and 91 for 64; 2^20 36.8
// and 23.7, 642 and 401 for 64).
std::unique_ptr<Node> build_tile_fourstep_node(const Problem &p, std::string *why) {
  for (const auto &row : tile_registry()) {
    if (row.kind != TK_ROW || row.prec != p.prec || row.bwd != (p.dir > 0)) continue;
    if (p.n % row.n) continue;
    const int64_t n1 = p.n / row.n;
    if (n1 != row.n && 2 * n1 != row.n) continue;
    const TileEntry *col = find_tile(TK_COL, n1, p.prec, p.dir > 0, row.wb);
    if (!col) continue;
    const int64_t blocks = p.howmany * std::min(row.n / col->w, col->n / row.w);
    if (prec_real_bytes(p.prec) >= 4 && blocks < cu_count()) continue;
    auto node = std::make_unique<TileFourStepNode>(col, &row, p,
                                                   fourstep_chunk(p.n, p.prec, p.howmany));
    const hipError_t err = node->init();
    if (err != hipSuccess) {
      *why = std::string("device upload failed: ") + hipGetErrorString(err);
      return nullptr;
    }
    return node;
  }
  return nullptr;
}

}  // namespace plf
