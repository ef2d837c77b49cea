// kernels_cz.hpp -- chirp-z (Bluestein whose DFT_M is a four-step) and
// Rader (prime n, N = n - 1 a four-step length) in three HBM passes on the
// compile-time column / row engines.
//
// With M = n1 * n2 >= 2n - 2, c_j the chirp and B = DFT_M(b) / M
// (bluestein.hpp:66-98), y = conj-chirp o IDFT_M(B o DFT_M(c o x)) is the
// DFT of x. The passes over a member's workspace (M complex, row-major
// n1 x n2):
//   1. column c2: a_j = x_j c_j (j = c2 + n2 e < n, else 0), DFT_n1 over e,
//      times W_M^{c2 k1}, into row k1, column c2;
//   2. row k1: DFT_n2 gives A[k1 + n1 k2]; times B (stored row-major by k1),
//      swapped; the inverse transform's four-step, taken with the sides
//      exchanged, starts with a DFT_n2 over the same row, so it runs on the
//      same registers, is twiddled by W_M^{k1 m2} and written back in place;
//   3. column m2: DFT_n1 over k1 gives bin m = m2 + n2 m1; swapped back,
//      times c_m, stored for m < n.
// The backward transform is swap o forward o swap on the input and output.
//
// KArgs of all three: tw = the engine's Stockham twiddles, aux0 = W_M split
// table (lo: 2^shift entries, then hi), n = engine length, n1, n2 = the
// sides, bigdist = the transform length n, count = columns (members * n2) or
// rows (members * n1). Pass 1: in = input (storage type, istride, idist),
// out = workspace, aux1 = chirp. Pass 2: out = workspace, aux0 = its own
// twiddles (k_cz_row_mid), aux1 = B. Pass 3:
// in = workspace, out = output (ostride, odist), aux1 = chirp.
// Gathered launch (aux2 = CzMember records, one per member of the launch;
// the members of a mixed-length batch that share M): each member's length,
// unit-stride offsets, workspace and table offsets come from its record.
#pragma once

#include "kernels.hpp"
#include "tile_engine.hpp"

namespace plf {

template <typename C>
__device__ __forceinline__ cpx<C> cz_twiddle(const cpx<C> *__restrict__ split, int shift,
                                             int64_t e) {
  const cpx<C> *hi = split + (int64_t(1) << shift);
  return cmul(hi[e >> shift], split[e & ((int64_t(1) << shift) - 1)]);
}

template <typename S, bool BWD, int TPB, class Eng>
__global__ void __launch_bounds__(Eng::TPT *TPB) k_cz_col_in(KArgs a) {
  using ST = StorageT<S>;
  using E = typename ST::E;
  using C = typename Eng::C;
  const int g = threadIdx.x % TPB;
  const int t = threadIdx.x / TPB;
  const int64_t col = xcd_block(blockIdx.x, gridDim.x) * TPB + g;
  const bool valid = col < a.count;
  const int64_t n1 = a.n1, n2 = a.n2;
  const int64_t bi = valid ? col / n2 : 0, c2 = valid ? col % n2 : 0;
  const CzMember *mt = static_cast<const CzMember *>(a.aux2);
  const int64_t nn = mt ? mt[bi].n : a.bigdist;
  const E *in = static_cast<const E *>(a.in) + (mt ? mt[bi].in_off : bi * a.idist);
  cpx<C> *ws = static_cast<cpx<C> *>(a.out) + (mt ? mt[bi].ws_off : bi * n1 * n2) + c2;
  const cpx<C> *split = static_cast<const cpx<C> *>(a.aux0);
  const cpx<C> *chirp = static_cast<const cpx<C> *>(a.aux1) + (mt ? mt[bi].chirp_off : 0);
  const int64_t is = mt ? 1 : a.istride;
  const int shift = a.shift;
  cpx<C> *lds = dyn_lds<C>() + g * Eng::lds_per(a.n);
  Eng::template run<false>(
      a.desc, lds, static_cast<const cpx<C> *>(a.tw), t, valid,
      [&](int b, int o) {
        // zero padding: skipped where it is all padding (the same for every
        // thread), otherwise selected after a load of element 0
        if (n2 * o >= nn) return cpx<C>{C(0), C(0)};
        const int64_t j0 = c2 + n2 * (b + o), j = j0 < nn ? j0 : 0;
        cpx<C> v = ST::ld(in[j * is]);
        v = cmul(BWD ? cswap(v) : v, chirp[j]);
        return cpx<C>{j0 < nn ? v.x : C(0), j0 < nn ? v.y : C(0)};
      },
      [&](int k1, cpx<C> v) { ws[(int64_t)k1 * n2] = cmul(v, cz_twiddle(split, shift, c2 * k1)); });
}

// Row pass, on the two-transform tile engine (ConvTile): W rows of TPT threads
// (n1 % W == 0). aux0: T1[k1][b] = W_M^{k1 b} (b < N / R, R the chain's first
// radix), then T2[k1][m] = W_M^{k1 m N / R}: the twiddle of output b + m N / R
// is the product of an entry per thread and one that the row's threads share.
// Storage types and directions do not matter to it. Rows of 256 of 512 members
// of 65536 (268 MB each way): 206 -> 141 us against two transforms through LDS.
template <typename C, int W, int TPT, class Ch>
__global__ void __launch_bounds__(TPT *W) k_cz_row_mid(KArgs a) {
  using T = ConvTile<C, W, TPT, Ch>;
  constexpr int N = Ch::N, R0 = Ch::radix(0), NB0 = N / R0;
  const int tid = threadIdx.x;
  const int t = tid % TPT;
  const uint32_t n1 = (uint32_t)a.n1, tpm = n1 / W;  // tiles per member
  const uint32_t bx = (uint32_t)xcd_block(blockIdx.x, gridDim.x);
  const uint32_t bi = bx / tpm, k1 = (bx % tpm) * W + tid / TPT;
  const CzMember *mt = static_cast<const CzMember *>(a.aux2);
  cpx<C> *row = static_cast<cpx<C> *>(a.out) + (mt ? mt[bi].ws_off : (int64_t)bi * n1 * N) +
                (int64_t)k1 * N;
  const cpx<C> *B = static_cast<const cpx<C> *>(a.aux1) + (mt ? mt[bi].B_off : 0) +
                    (int64_t)k1 * N + t;
  const cpx<C> *t1 = static_cast<const cpx<C> *>(a.aux0) + (int64_t)k1 * NB0;
  const cpx<C> *t2 = static_cast<const cpx<C> *>(a.aux0) + (int64_t)n1 * NB0 + (int64_t)k1 * R0;
  // Rader (aux3 set): bin 0 of the forward transform, A_0 = sum of the
  // permuted inputs, goes to the member's slot for X_0 = x_0 + A_0
  cpx<C> *slot = static_cast<cpx<C> *>(a.aux3);
  T::run(
      reinterpret_cast<C *>(dyn_lds<C>()), static_cast<const cpx<C> *>(a.tw), tid,
      [&](int b, int m) { return row[b + m * NB0]; },
      [&](cpx<C> (&v)[T::KB][T::R]) {
        if (slot && k1 == 0 && t == 0) slot[2 * bi + 1] = v[0][0];
#pragma unroll
        for (int k = 0; k < T::KB; ++k)
#pragma unroll
          for (int m = 0; m < T::R; ++m) v[k][m] = cswap(cmul(v[k][m], B[k * TPT + m * T::NB]));
      },
      [&](int b, const cpx<C> (&v)[R0]) {
        const cpx<C> wb = t1[b];
#pragma unroll
        for (int m = 0; m < R0; ++m)
          row[b + m * NB0] = cmul(v[m], m == 0 ? wb : cmul(wb, t2[m]));
      });
}

template <typename S, bool BWD, int TPB, class Eng>
__global__ void __launch_bounds__(Eng::TPT *TPB) k_cz_col_out(KArgs a) {
  using ST = StorageT<S>;
  using E = typename ST::E;
  using C = typename Eng::C;
  const int g = threadIdx.x % TPB;
  const int t = threadIdx.x / TPB;
  const int64_t col = xcd_block(blockIdx.x, gridDim.x) * TPB + g;
  const bool valid = col < a.count;
  const int64_t n1 = a.n1, n2 = a.n2;
  const int64_t bi = valid ? col / n2 : 0, c2 = valid ? col % n2 : 0;
  const CzMember *mt = static_cast<const CzMember *>(a.aux2);
  const int64_t nn = mt ? mt[bi].n : a.bigdist;
  const cpx<C> *ws = static_cast<const cpx<C> *>(a.in) + (mt ? mt[bi].ws_off : bi * n1 * n2) + c2;
  E *out = static_cast<E *>(a.out) + (mt ? mt[bi].out_off : bi * a.odist);
  const cpx<C> *chirp = static_cast<const cpx<C> *>(a.aux1) + (mt ? mt[bi].chirp_off : 0);
  const int64_t os = mt ? 1 : a.ostride;
  cpx<C> *lds = dyn_lds<C>() + g * Eng::lds_per(a.n);
  Eng::template run<false>(
      a.desc, lds, static_cast<const cpx<C> *>(a.tw), t, valid,
      [&](int e) { return ws[(int64_t)e * n2]; },
      [&](int m1, cpx<C> v) {
        const int64_t m = c2 + n2 * m1;
        if (m < nn) {
          const cpx<C> y = cmul(cswap(v), chirp[m]);
          out[m * os] = ST::st(BWD ? cswap(y) : y);
        }
      });
}

// Rader in three passes for a prime n with N = n - 1 = n1 * n2 (the
// reference's rader.hpp:51-90, with its convolution on the four-step
// passes above). g generates the nonzero residues mod n, perm[p] = g^p mod n,
// a_p = x[perm[p]] and b_p = W_n^{perm[(N - p) mod N]}; with B = DFT_N(b) / N,
// X[perm[(N - q) mod N]] = x_0 + (a (*) b)_q and X_0 = x_0 + sum_p a_p.
// The row pass is k_cz_row_mid with aux3 set (it keeps A_0 = sum_p a_p).
// KArgs as for the chirp-z passes, except: aux1 = perm (int32, N entries)
// in the column passes, aux3 = two slots per member of the launch (x_0,
// A_0; compute precision) and bigdist unused (no padding).
template <typename S, bool BWD, int TPB, class Eng>
__global__ void __launch_bounds__(Eng::TPT *TPB) k_rd_col_in(KArgs a) {
  using ST = StorageT<S>;
  using E = typename ST::E;
  using C = typename Eng::C;
  const int g = threadIdx.x % TPB;
  const int t = threadIdx.x / TPB;
  const int64_t col = xcd_block(blockIdx.x, gridDim.x) * TPB + g;
  const bool valid = col < a.count;
  const int64_t n1 = a.n1, n2 = a.n2;
  const int64_t bi = valid ? col / n2 : 0, c2 = valid ? col % n2 : 0;
  const E *in = static_cast<const E *>(a.in) + bi * a.idist;
  cpx<C> *ws = static_cast<cpx<C> *>(a.out) + bi * n1 * n2 + c2;
  const cpx<C> *split = static_cast<const cpx<C> *>(a.aux0);
  const int *perm = static_cast<const int *>(a.aux1) + c2;
  const int64_t is = a.istride;
  const int shift = a.shift;
  if (valid && c2 == 0 && t == 0) {
    const cpx<C> x0 = ST::ld(in[0]);
    static_cast<cpx<C> *>(a.aux3)[2 * bi] = BWD ? cswap(x0) : x0;
  }
  cpx<C> *lds = dyn_lds<C>() + g * Eng::lds_per(a.n);
  Eng::template run<false>(
      a.desc, lds, static_cast<const cpx<C> *>(a.tw), t, valid,
      [&](int e) {
        const cpx<C> v = ST::ld(in[(int64_t)perm[n2 * e] * is]);
        return BWD ? cswap(v) : v;
      },
      [&](int k1, cpx<C> v) { ws[(int64_t)k1 * n2] = cmul(v, cz_twiddle(split, shift, c2 * k1)); });
}

template <typename S, bool BWD, int TPB, class Eng>
__global__ void __launch_bounds__(Eng::TPT *TPB) k_rd_col_out(KArgs a) {
  using ST = StorageT<S>;
  using E = typename ST::E;
  using C = typename Eng::C;
  const int g = threadIdx.x % TPB;
  const int t = threadIdx.x / TPB;
  const int64_t col = xcd_block(blockIdx.x, gridDim.x) * TPB + g;
  const bool valid = col < a.count;
  const int64_t n1 = a.n1, n2 = a.n2, N = n1 * n2;
  const int64_t bi = valid ? col / n2 : 0, c2 = valid ? col % n2 : 0;
  const cpx<C> *ws = static_cast<const cpx<C> *>(a.in) + bi * N + c2;
  E *out = static_cast<E *>(a.out) + bi * a.odist;
  const int *perm = static_cast<const int *>(a.aux1);
  const cpx<C> *slot = static_cast<const cpx<C> *>(a.aux3) + 2 * bi;
  const cpx<C> x0 = slot[0];
  const int64_t os = a.ostride;
  cpx<C> *lds = dyn_lds<C>() + g * Eng::lds_per(a.n);
  Eng::template run<false>(
      a.desc, lds, static_cast<const cpx<C> *>(a.tw), t, valid,
      [&](int e) { return ws[(int64_t)e * n2]; },
      [&](int m1, cpx<C> v) {
        const int64_t q = c2 + n2 * m1;
        const cpx<C> r = cadd(x0, cswap(v));
        out[(int64_t)perm[q == 0 ? 0 : N - q] * os] = ST::st(BWD ? cswap(r) : r);
        if (q == 0) {
          const cpx<C> y0 = cadd(x0, slot[1]);
          out[0] = ST::st(BWD ? cswap(y0) : y0);
        }
      });
}

}  // namespace plf
