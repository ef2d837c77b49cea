// kernels_flex.hpp -- batched transforms of any length with prime factors up
// to 13 on the flexible-chain engine.
#pragma once

#include "flex_engine.hpp"
#include "flex_registry.hpp"
#include "kernels.hpp"

namespace plf {

// Member g < tpb of the block and thread t < tpt of it. Threads past tpt * tpb
// work along on the block's last member and store nothing.
struct FlexThread {
  int g, t;
  bool live;
};
__device__ __forceinline__ FlexThread flex_thread(const FlexDesc &d) {
  const int tid = threadIdx.x;
  const int div = d.lanes ? d.tpb : d.tpt;
  const int q = div == 1 ? tid : (int)__umulhi((uint32_t)tid, d.magic), r = tid - q * div;
  const int g = d.lanes ? r : q, t = d.lanes ? q : r;
  const bool live = g < d.tpb && t < d.tpt;
  return {g < d.tpb ? g : d.tpb - 1, t < d.tpt ? t : d.tpt - 1, live};
}

// batched C2C: in[b*idist + e*istride] -> out[b*odist + k*ostride]. Block
// bases in scalar registers, 32-bit offsets per lane: tpb members and one
// member's span stay below 4 GiB (flex_plan.cpp checks). Plain accesses: a
// member's rows are rarely whole lines, and non-temporal stores of partial
// lines reach HBM as such.
template <typename S, bool BWD, int BLOCK>
__global__ void __launch_bounds__(BLOCK) k_flex_c2c(FlexArgs f) {
  using ST = StorageT<S>;
  using E = typename ST::E;
  using C = typename ST::C;
  const KArgs &a = f.a;
  const FlexThread th = flex_thread(*f.d);
  // flags bit0: consecutive blocks on one XCD (they share lines)
  const int64_t blk = (a.flags & 1) ? xcd_block(blockIdx.x, gridDim.x) : (int64_t)blockIdx.x;
  const int64_t tr0 = blk * f.d->tpb;
  const bool valid = tr0 + th.g < a.count;
  const uint32_t g = valid ? th.g : 0;
  const E *in = static_cast<const E *>(a.in) + tr0 * a.idist;
  E *out = static_cast<E *>(a.out) + tr0 * a.odist;
  const uint32_t is = (uint32_t)a.istride, os = (uint32_t)a.ostride;
  const uint32_t gi = g * (uint32_t)a.idist, go = g * (uint32_t)a.odist;
  FlexEngine<C, false>::run(
      *f.d, dyn_lds<C>() + th.g * f.d->lper, static_cast<const cpx<C> *>(a.tw), th.t, th.live,
      valid,
      [&](int b, int o) {
        const cpx<C> v = ST::ld(at_u32(in + (int64_t)o * is, gi + b * is));
        return BWD ? cswap(v) : v;
      },
      [&](int b, int o, cpx<C> v) {
        const_cast<E &>(at_u32(out + (int64_t)o * os, go + b * os)) =
            ST::st(BWD ? cswap(v) : v);
      });
}

// One member of a real transform of even length n = 2m (kernels_real.hpp
// states the transforms): a.n = m, flags, aux0, aux1 as there. Real-side
// strides count reals, complex-side strides complex values.
template <typename S, bool UNUSED, int BLOCK>
__global__ void __launch_bounds__(BLOCK) k_flex_r2c(FlexArgs f) {
  using ST = StorageT<S>;
  using E = typename ST::E;
  using Rs = typename ST::Rs;
  using C = typename ST::C;
  const KArgs &a = f.a;
  const FlexThread th = flex_thread(*f.d);
  const int64_t tr0 = (int64_t)blockIdx.x * f.d->tpb;
  const bool valid = tr0 + th.g < a.count;
  const uint32_t g = valid ? th.g : 0;
  const int m = (int)a.n, tpt = f.d->tpt;
  const Rs *x = static_cast<const Rs *>(a.in) + tr0 * a.idist;
  const uint32_t is = (uint32_t)a.istride, gi = g * (uint32_t)a.idist;
  cpx<C> *lds = dyn_lds<C>() + th.g * f.d->lper;
  const cpx<C> *tw = static_cast<const cpx<C> *>(a.tw);
  auto drop = [](int, int, cpx<C>) {};
  if (a.flags & 1) {  // reals in pairs
    FlexEngine<C, true>::run(
        *f.d, lds, tw, th.t, th.live, valid,
        [&](int b, int o) {
          return ST::ld(at_u32(reinterpret_cast<const E *>(x) + o, gi / 2 + b));
        },
        drop);
  } else {
    FlexEngine<C, true>::run(
        *f.d, lds, tw, th.t, th.live, valid,
        [&](int b, int o) {
          const Rs *p = x + (int64_t)(2 * o) * is;
          const uint32_t e = gi + 2 * b * is;
          return cpx<C>{ST::ldr(at_u32(p, e)), ST::ldr(at_u32(p + is, e))};
        },
        drop);
  }
  if (!valid || !th.live) return;
  const cpx<C> *W = static_cast<const cpx<C> *>(a.aux0);
  E *out = static_cast<E *>(a.out) + (tr0 + th.g) * a.odist;
  const int64_t os = a.ostride;
  const C h = (a.flags & 2) ? C(1) : C(0.5);
  for (int k = th.t; 2 * k <= m; k += tpt) {
    if (k == 0) {
      const cpx<C> z0 = lds[0];
      out[0] = ST::st({z0.x + z0.y, C(0)});
      out[(int64_t)m * os] = ST::st({z0.x - z0.y, C(0)});
      continue;
    }
    const cpx<C> A = lds[k], B = lds[m - k];
    const cpx<C> xe = {h * (A.x + B.x), h * (A.y - B.y)};
    const cpx<C> xo = {h * (A.y + B.y), h * (B.x - A.x)};  // -i (A - conj B) h
    const cpx<C> wx = cmul(W[k], xo);
    out[(int64_t)k * os] = ST::st(cadd(xe, wx));
    if (2 * k != m) out[(int64_t)(m - k) * os] = ST::st({xe.x - wx.x, wx.y - xe.y});
  }
}

template <typename S, bool UNUSED, int BLOCK>
__global__ void __launch_bounds__(BLOCK) k_flex_c2r(FlexArgs f) {
  using ST = StorageT<S>;
  using E = typename ST::E;
  using Rs = typename ST::Rs;
  using C = typename ST::C;
  const KArgs &a = f.a;
  const FlexThread th = flex_thread(*f.d);
  const int64_t tr0 = (int64_t)blockIdx.x * f.d->tpb;
  const bool valid = tr0 + th.g < a.count;
  const uint32_t g = valid ? th.g : 0;
  const int m = (int)a.n;
  const E *X = static_cast<const E *>(a.in) + tr0 * a.idist;
  const uint32_t is = (uint32_t)a.istride, gi = g * (uint32_t)a.idist;
  Rs *y = static_cast<Rs *>(a.out) + (tr0 + g) * a.odist;
  const int64_t os = a.ostride;
  const bool pair = a.flags & 1;
  const C hw = (a.flags & 2) ? C(0.5) : C(1);
  const cpx<C> *W = static_cast<const cpx<C> *>(a.aux0);
  FlexEngine<C, false>::run(
      *f.d, dyn_lds<C>() + th.g * f.d->lper, static_cast<const cpx<C> *>(a.tw), th.t, th.live,
      valid,
      in_bursts<4>([&](int b, int o) {
        const int e = b + o;
        cpx<C> A = ST::ld(at_u32(X + (int64_t)o * is, gi + b * is));
        cpx<C> B = ST::ld(at_u32(X, gi + (m - e) * is));
        // X[0] and X[m] count as real, whatever their imaginary parts hold
        A = {e == 0 ? A.x : hw * A.x, e == 0 ? C(0) : hw * A.y};
        B = {e == 0 ? B.x : hw * B.x, e == 0 ? C(0) : hw * B.y};
        const cpx<C> s = {A.x + B.x, A.y - B.y};        // A + conj B
        const cpx<C> d = {A.x - B.x, A.y + B.y};        // A - conj B
        const cpx<C> wd = cconj_mul(d, at_u32(W + o, b));  // W^{-e} (A - conj B)
        return cswap(cpx<C>{s.x - wd.y, s.y + wd.x});   // s + i wd, swapped
      }),
      [&](int b, int o, cpx<C> v) {
        v = cswap(v);
        const int e = b + o;
        if (pair) {
          reinterpret_cast<E *>(y)[e] = ST::st(v);
        } else {
          y[(int64_t)(2 * e) * os] = ST::str(v.x);
          y[(int64_t)(2 * e + 1) * os] = ST::str(v.y);
        }
      });
}

// DCT-II / DST-II (two = true) and DCT-III / DST-III of even n through LDS,
// as k_dct2_even and k_dct3_even.
template <typename S, bool DST, int BLOCK>
__global__ void __launch_bounds__(BLOCK) k_flex_dct2(FlexArgs f) {
  using ST = StorageT<S>;
  using Rs = typename ST::Rs;
  using C = typename ST::C;
  const KArgs &a = f.a;
  const FlexThread th = flex_thread(*f.d);
  const int64_t tr = (int64_t)blockIdx.x * f.d->tpb + th.g;
  const bool valid = tr < a.count;
  const int m = (int)a.n, n = 2 * m, tpt = f.d->tpt, t = th.t;
  const Rs *x = static_cast<const Rs *>(a.in) + (valid ? tr * a.idist : 0);
  const int64_t is = a.istride, os = a.ostride;
  cpx<C> *lds = dyn_lds<C>() + th.g * f.d->lper;
  C *lr = reinterpret_cast<C *>(lds);
  if (th.live) {
#pragma unroll 8
    for (int o = t; o < n; o += tpt) {
      const C v = ST::ldr(x[(int64_t)o * is]);
      lr[(o & 1) ? n - (o + 1) / 2 : o / 2] = (DST && (o & 1)) ? -v : v;
    }
  }
  __syncthreads();
  FlexEngine<C, true, true>::run(
      *f.d, lds, static_cast<const cpx<C> *>(a.tw), t, th.live, valid,
      [&](int b, int o) { return lds[b + o]; }, [](int, int, cpx<C>) {});
  if (!valid || !th.live) return;
  Rs *y = static_cast<Rs *>(a.out) + tr * a.odist;
  const cpx<C> *W = static_cast<const cpx<C> *>(a.aux0);
  const cpx<C> *w = static_cast<const cpx<C> *>(a.aux1);
  const C h = C(0.5), two = C(2);
  const C s0 = (a.flags & 2) ? C(0.5) : C(1);
  auto put = [&](int o, C v) { y[(int64_t)(DST ? n - 1 - o : o) * os] = ST::str(v); };
  auto emit = [&](int k, cpx<C> V) {  // y_k and y_{n-k} from V_k
    const cpx<C> r = cmul(w[k], V);
    put(k, two * r.x);
    put(n - k, -two * r.y);
  };
  for (int k = t; 2 * k <= m; k += tpt) {
    if (k == 0) {
      const cpx<C> z0 = lds[0];
      put(0, s0 * two * (z0.x + z0.y));
      put(m, two * (z0.x - z0.y) * w[m].x);
      continue;
    }
    const cpx<C> A = lds[k], B = lds[m - k];
    const cpx<C> xe = {h * (A.x + B.x), h * (A.y - B.y)};
    const cpx<C> xo = {h * (A.y + B.y), h * (B.x - A.x)};
    const cpx<C> wx = cmul(W[k], xo);
    emit(k, cadd(xe, wx));
    if (2 * k != m) emit(m - k, {xe.x - wx.x, wx.y - xe.y});
  }
}

template <typename S, bool DST, int BLOCK>
__global__ void __launch_bounds__(BLOCK) k_flex_dct3(FlexArgs f) {
  using ST = StorageT<S>;
  using Rs = typename ST::Rs;
  using C = typename ST::C;
  const KArgs &a = f.a;
  const FlexThread th = flex_thread(*f.d);
  const int64_t tr = (int64_t)blockIdx.x * f.d->tpb + th.g;
  const bool valid = tr < a.count;
  const int m = (int)a.n, n = 2 * m, tpt = f.d->tpt, t = th.t;
  const Rs *x = static_cast<const Rs *>(a.in) + (valid ? tr * a.idist : 0);
  const int64_t is = a.istride, os = a.ostride;
  cpx<C> *lds = dyn_lds<C>() + th.g * f.d->lper;
  C *lu = reinterpret_cast<C *>(lds);
  const cpx<C> *W = static_cast<const cpx<C> *>(a.aux0);
  const cpx<C> *w = static_cast<const cpx<C> *>(a.aux1);
  const C s0 = (a.flags & 2) ? C(2) : C(1);
  if (th.live) {
#pragma unroll 8
    for (int o = t; o < n; o += tpt) {
      const C v = ST::ldr(x[(int64_t)o * is]);
      const int k = DST ? n - 1 - o : o;
      lu[k] = k == 0 ? s0 * v : v;
    }
  }
  __syncthreads();
  FlexEngine<C, true, true>::run(
      *f.d, lds, static_cast<const cpx<C> *>(a.tw), t, th.live, valid,
      in_bursts<2>([&](int b, int o) {
        const int e = b + o;
        // X_e and X_{m-e}: (u_k - i u_{n-k}) conj(w_k), u_n = 0
        const C un = lu[e == 0 ? 0 : n - e];
        const cpx<C> A = cconj_mul(cpx<C>{lu[e], e == 0 ? C(0) : -un}, at_u32(w + o, b));
        const cpx<C> B = cconj_mul(cpx<C>{lu[m - e], -lu[m + e]}, at_u32(w, m - e));
        const cpx<C> sm = {A.x + B.x, A.y - B.y}, d = {A.x - B.x, A.y + B.y};
        const cpx<C> wd = cconj_mul(d, at_u32(W + o, b));
        return cswap(cpx<C>{sm.x - wd.y, sm.y + wd.x});
      }),
      [](int, int, cpx<C>) {});
  if (!valid || !th.live) return;
  // swap(lds[e]) = v_{2e} + i v_{2e+1}; y[o] = v_i, i = o/2 (o even) or
  // n - (o+1)/2 (o odd, negated for DST)
  Rs *y = static_cast<Rs *>(a.out) + tr * a.odist;
#pragma unroll 4
  for (int o = t; o < n; o += tpt) {
    const int i = (o & 1) ? n - (o + 1) / 2 : o / 2;
    const C v = lu[2 * (i >> 1) + 1 - (i & 1)];
    y[(int64_t)o * os] = ST::str((DST && (o & 1)) ? -v : v);
  }
}

}  // namespace plf
