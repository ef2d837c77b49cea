// kernels_conv.hpp -- prime lengths: fused Bluestein (chirp-z) and Rader
// kernels, one block per member with everything resident in LDS.
//
// Bluestein (src/planner/strategies/bluestein.hpp:66-146): with the chirp
// c_k = exp(-i pi (k^2 mod 2n) / n) (phase reduced in integers on the host),
//   X = c .* IDFT_M( DFT_M(x .* c, zero-padded to M) .* B ),
//   B = DFT_M(b) / M,  b_k = b_{M-k} = conj(c_k) for 0 <= k < n, else 0.
// Rader (src/planner/strategies/rader.hpp:36-124), n prime, m = n - 1,
// generator g, perm[k] = g^k mod n:
//   a_k = x[perm[k]],  A = DFT_m(a),  X[0] = x0 + A[0],
//   conv = IDFT_m(A .* B),  B = DFT_m(b) / m,  b_{(m-k) mod m} = W_n^{perm[k]},
//   X[perm[(m - e) mod m]] = x0 + conv[e].
// Both run the forward engine twice in one kernel: the inverse DFT is
// swap(DFT(swap(.))). A backward transform swaps at the first load and the
// final store, like the other kernels.
#pragma once

#include "kernels.hpp"
#include "tile_engine.hpp"

namespace plf {

// aux0: B (M entries), aux1: chirp c (n entries); a.n = M, a.n1 = n.
// Gathered launch (aux2 = BlueMember records, one per transform; a mixed
// batch's members and rows of equal M): length, offsets, output stride and
// table offsets per record, unit input stride.
template <typename S, bool BWD, int TPB, class Eng>
__global__ void __launch_bounds__(Eng::TPT *TPB) k_bluestein(KArgs a) {
  using ST = StorageT<S>;
  using E = typename ST::E;
  using C = typename Eng::C;
  constexpr int TPT = Eng::TPT;
  const int g = threadIdx.x / TPT;
  const int t = threadIdx.x % TPT;
  const int64_t tr = (int64_t)blockIdx.x * TPB + g;
  const bool valid = tr < a.count;
  const int M = (int)a.n;
  const BlueMember *mt = static_cast<const BlueMember *>(a.aux2);
  const BlueMember *rec = mt ? mt + (valid ? tr : 0) : nullptr;
  const int n = mt ? (int)rec->n : (int)a.n1;
  const E *in = static_cast<const E *>(a.in) + (mt ? rec->in_off : valid ? tr * a.idist : 0);
  E *out = static_cast<E *>(a.out) + (mt ? rec->out_off : valid ? tr * a.odist : 0);
  cpx<C> *lds = dyn_lds<C>() + g * Eng::lds_per(M);
  const cpx<C> *tw = static_cast<const cpx<C> *>(a.tw);
  const cpx<C> *B = static_cast<const cpx<C> *>(a.aux0) + (mt ? rec->B_off : 0);
  const cpx<C> *chirp = static_cast<const cpx<C> *>(a.aux1) + (mt ? rec->chirp_off : 0);
  const int64_t is = mt ? 1 : a.istride, os = mt ? rec->ostride : a.ostride;
  // zero padding: skipped where it is all padding (o >= n, the same for
  // every thread), otherwise selected after a load of element 0
  auto load = [&](int b, int o) {
    if (o >= n) return cpx<C>{C(0), C(0)};
    const int e = b + o < n ? b + o : 0;
    cpx<C> v = ST::ld(in[(int64_t)e * is]);
    if (BWD) v = cswap(v);
    v = cmul(v, chirp[e]);
    return cpx<C>{b + o < n ? v.x : C(0), b + o < n ? v.y : C(0)};
  };
  auto store = [&](int e, cpx<C> v) {
    if (e < n) {
      cpx<C> r = cmul(cswap(v), chirp[e]);
      out[(int64_t)e * os] = ST::st(BWD ? cswap(r) : r);
    }
  };
  Eng::template run<true>(a.desc, lds, tw, t, valid, load, [&](int, cpx<C>) {});
  for (int e = t; e < M; e += TPT) {
    const int p = lds_pad<Eng::PAD>(e);
    lds[p] = cswap(cmul(lds[p], B[e]));
  }
  __syncthreads();
  Eng::template run<false, true>(
      a.desc, lds, tw, t, valid, [&](int) { return cpx<C>{C(0), C(0)}; }, store);
}

// k_bluestein of a compile-time padded length on the two-transform tile engine
// (ConvTile): TPB members of TPT threads. Bound by LDS latency and the two
// transforms' arithmetic. FP64 members of 1399 (M = 4096, 5996 of them) 187
// -> 144 us against the engine that passes the first transform's result
// through LDS, FP32 members of 59 (M = 128, 280000) 140 -> 114 us.
template <typename S, bool BWD, int TPB, int TPT, class Ch>
__global__ void __launch_bounds__(TPT *TPB) k_bluestein_tile(KArgs a) {
  using ST = StorageT<S>;
  using E = typename ST::E;
  using C = typename ST::C;
  using T = ConvTile<C, TPB, TPT, Ch>;
  constexpr int R0 = Ch::radix(0), NB0 = Ch::N / R0;
  const int tid = threadIdx.x;
  const int t = tid % TPT;
  const int64_t tr = (int64_t)blockIdx.x * TPB + tid / TPT;
  const bool valid = tr < a.count;
  const BlueMember *mt = static_cast<const BlueMember *>(a.aux2);
  const BlueMember *rec = mt ? mt + (valid ? tr : 0) : nullptr;
  const int n = mt ? (int)rec->n : (int)a.n1;
  const E *in = static_cast<const E *>(a.in) + (mt ? rec->in_off : valid ? tr * a.idist : 0);
  E *out = static_cast<E *>(a.out) + (mt ? rec->out_off : valid ? tr * a.odist : 0);
  const cpx<C> *B = static_cast<const cpx<C> *>(a.aux0) + (mt ? rec->B_off : 0) + t;
  const cpx<C> *chirp = static_cast<const cpx<C> *>(a.aux1) + (mt ? rec->chirp_off : 0);
  const int64_t is = mt ? 1 : a.istride, os = mt ? rec->ostride : a.ostride;
  T::run(
      reinterpret_cast<C *>(dyn_lds<C>()), static_cast<const cpx<C> *>(a.tw), tid,
      [&](int b, int m) {
        // n <= M / 2 + 1, as M >= 2n - 2: the upper half is padding; below it
        // padding is selected after a load of element 0
        if (2 * m * NB0 > Ch::N) return cpx<C>{C(0), C(0)};
        const int o = b + m * NB0, e = o < n ? o : 0;
        cpx<C> v = ST::ld(in[(int64_t)e * is]);
        v = cmul(BWD ? cswap(v) : v, chirp[e]);
        return cpx<C>{o < n ? v.x : C(0), o < n ? v.y : C(0)};
      },
      [&](cpx<C> (&v)[T::KB][T::R]) {
#pragma unroll
        for (int k = 0; k < T::KB; ++k)
#pragma unroll
          for (int m = 0; m < T::R; ++m) v[k][m] = cswap(cmul(v[k][m], B[k * TPT + m * T::NB]));
      },
      [&](int b, const cpx<C> (&v)[R0]) {
        if (!valid) return;
#pragma unroll
        for (int m = 0; m < R0; ++m) {
          if (2 * m * NB0 > Ch::N) continue;
          const int e = b + m * NB0;
          if (e < n) {
            const cpx<C> r = cmul(cswap(v[m]), chirp[e]);
            out[(int64_t)e * os] = ST::st(BWD ? cswap(r) : r);
          }
        }
      });
}

// aux0: B (m entries), aux1: perm (int32, m entries); a.n = m, a.n1 = n.
template <typename S, bool BWD, int TPB, class Eng>
__global__ void __launch_bounds__(Eng::TPT *TPB) k_rader(KArgs a) {
  using ST = StorageT<S>;
  using E = typename ST::E;
  using C = typename Eng::C;
  constexpr int TPT = Eng::TPT;
  const int g = threadIdx.x / TPT;
  const int t = threadIdx.x % TPT;
  const int64_t tr = (int64_t)blockIdx.x * TPB + g;
  const bool valid = tr < a.count;
  const int m = (int)a.n;
  const E *in = static_cast<const E *>(a.in) + (valid ? tr * a.idist : 0);
  E *out = static_cast<E *>(a.out) + (valid ? tr * a.odist : 0);
  cpx<C> *lds = dyn_lds<C>() + g * Eng::lds_per(m);
  const cpx<C> *tw = static_cast<const cpx<C> *>(a.tw);
  const cpx<C> *B = static_cast<const cpx<C> *>(a.aux0);
  const int *perm = static_cast<const int *>(a.aux1);
  const int64_t is = a.istride, os = a.ostride;
  cpx<C> x0 = {C(0), C(0)};
  if (valid) {
    x0 = ST::ld(in[0]);
    if (BWD) x0 = cswap(x0);
  }
  auto load = [&](int e) {
    cpx<C> v = ST::ld(in[(int64_t)perm[e] * is]);
    return BWD ? cswap(v) : v;
  };
  auto store = [&](int e, cpx<C> v) {
    const int k = perm[e == 0 ? 0 : m - e];
    const cpx<C> r = cadd(x0, cswap(v));
    out[(int64_t)k * os] = ST::st(BWD ? cswap(r) : r);
  };
  auto first = [&](cpx<C> A) {  // X_0 = x_0 + A_0
    if (valid) {
      const cpx<C> y0 = cadd(x0, A);
      out[0] = ST::st(BWD ? cswap(y0) : y0);
    }
  };
  Eng::template run<true>(a.desc, lds, tw, t, valid, load, [&](int, cpx<C>) {});
  for (int e = t; e < m; e += TPT) {
    const int p = lds_pad<Eng::PAD>(e);
    const cpx<C> A = lds[p];
    if (e == 0) first(A);
    lds[p] = cswap(cmul(A, B[e]));
  }
  __syncthreads();
  Eng::template run<false, true>(
      a.desc, lds, tw, t, valid, [&](int) { return cpx<C>{C(0), C(0)}; }, store);
}

}  // namespace plf
