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
// KArgs of all three: tw = the engine's Stockham twiddles, n = engine length,
// n1, n2 = the sides, bigdist = the transform length n, count = columns (members * n2) or
// rows (members * n1). Pass 1: in = input (storage type, istride, idist),
// out = workspace, aux0 = its twiddles (CzTile::put), aux1 = chirp. Pass 2: out = workspace, aux0 = its own
// twiddles (k_cz_row_mid), aux1 = B. Pass 3:
// in = workspace, out = output (ostride, odist), aux1 = chirp.
// Gathered launch (aux2 = CzMember records, one per member of the launch;
// the members of a mixed-length batch that share M): each member's length,
// unit-stride offsets, workspace and table offsets come from its record.
#pragma once

#include "kernels.hpp"
#include "tile_engine.hpp"

namespace plf {

// A block's tile of a column pass: W neighbouring columns c of one member
// (n2 % W == 0), lanes along the columns, on the split exchange. The chirp-z
// passes are bound by memory, Rader's by their 8-byte gathers and scatters
// (a line each). 512 members of 65537: in 270 -> 236 us, out 267 -> 255 us
// against the full exchange with a split twiddle table; 800 members of 20011,
// all three passes, 472 -> 420 us.
template <typename C, int W, int TPT, class Ch>
struct CzTile {
  using T = TileEngine<C, W, TPT, Ch, true, true>;
  static constexpr int R0 = Ch::radix(0), NB0 = Ch::N / R0;
  static constexpr int RL = Ch::radix(Ch::count - 1), NBL = Ch::N / RL;
  uint32_t n2, bi, c;
  int t;
  __device__ __forceinline__ explicit CzTile(const KArgs &a) {
    n2 = (uint32_t)a.n2;
    const uint32_t tpm = n2 / W, bx = (uint32_t)xcd_block(blockIdx.x, gridDim.x);
    bi = bx / tpm;
    c = (bx % tpm) * W + threadIdx.x % W;
    t = threadIdx.x / W;
  }
  // outputs b + m NBL of the column, twiddled by W_M^{c k1}, to the workspace;
  // T1[b][c] and T2[m][c] are read along the columns (the split table of the
  // other exponents took two gathers an element)
  __device__ __forceinline__ void put(const KArgs &a, cpx<C> *ws, int b,
                                      const cpx<C> (&v)[RL]) const {
    const cpx<C> *t1 = static_cast<const cpx<C> *>(a.aux0);
    const cpx<C> *t2 = t1 + (uint32_t)NBL * n2;
    const cpx<C> wb = at_u32(t1, (uint32_t)b * n2 + c);
    cpx<C> y[RL];
#pragma unroll
    for (int m = 0; m < RL; ++m)
      y[m] = cmul(v[m], m == 0 ? wb : cmul(wb, at_u32(t2, (uint32_t)m * n2 + c)));
#pragma unroll
    for (int m = 0; m < RL; ++m) ws[(uint32_t)(b + m * NBL) * n2 + c] = y[m];
  }
};

template <typename S, bool BWD, int W, int TPT, class Ch>
__global__ void __launch_bounds__(W *TPT) k_cz_col_in(KArgs a) {
  using ST = StorageT<S>;
  using E = typename ST::E;
  using C = typename ST::C;
  using Z = CzTile<C, W, TPT, Ch>;
  const Z z(a);
  const CzMember *mt = static_cast<const CzMember *>(a.aux2);
  const uint32_t nn = (uint32_t)(mt ? mt[z.bi].n : a.bigdist);
  const E *in = static_cast<const E *>(a.in) + (mt ? mt[z.bi].in_off : z.bi * a.idist);
  cpx<C> *ws = static_cast<cpx<C> *>(a.out) +
               (mt ? mt[z.bi].ws_off : (int64_t)z.bi * Ch::N * z.n2);
  const cpx<C> *chirp = static_cast<const cpx<C> *>(a.aux1) + (mt ? mt[z.bi].chirp_off : 0);
  const int64_t is = mt ? 1 : a.istride;
  Z::T::run(
      reinterpret_cast<C *>(dyn_lds<C>()), static_cast<const cpx<C> *>(a.tw), threadIdx.x,
      [&](int b, int m) {
        // n <= M / 2 + 1, as M >= 2n - 2: the upper half is padding; below it
        // padding is selected after a load of element 0
        if (2 * m * Z::NB0 > Ch::N) return cpx<C>{C(0), C(0)};
        const uint32_t j0 = z.c + z.n2 * (uint32_t)(b + m * Z::NB0), j = j0 < nn ? j0 : 0;
        cpx<C> v = ST::ld(in[j * is]);
        v = cmul(BWD ? cswap(v) : v, chirp[j]);
        return cpx<C>{j0 < nn ? v.x : C(0), j0 < nn ? v.y : C(0)};
      },
      [&](int b, const cpx<C> (&v)[Z::RL]) { z.put(a, ws, b, v); });
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

template <typename S, bool BWD, int W, int TPT, class Ch>
__global__ void __launch_bounds__(W *TPT) k_cz_col_out(KArgs a) {
  using ST = StorageT<S>;
  using E = typename ST::E;
  using C = typename ST::C;
  using Z = CzTile<C, W, TPT, Ch>;
  const Z z(a);
  const CzMember *mt = static_cast<const CzMember *>(a.aux2);
  const uint32_t nn = (uint32_t)(mt ? mt[z.bi].n : a.bigdist);
  const cpx<C> *ws = static_cast<const cpx<C> *>(a.in) +
                     (mt ? mt[z.bi].ws_off : (int64_t)z.bi * Ch::N * z.n2);
  E *out = static_cast<E *>(a.out) + (mt ? mt[z.bi].out_off : z.bi * a.odist);
  const cpx<C> *chirp = static_cast<const cpx<C> *>(a.aux1) + (mt ? mt[z.bi].chirp_off : 0);
  const int64_t os = mt ? 1 : a.ostride;
  Z::T::run(
      reinterpret_cast<C *>(dyn_lds<C>()), static_cast<const cpx<C> *>(a.tw), threadIdx.x,
      [&](int b, int m) { return ws[(uint32_t)(b + m * Z::NB0) * z.n2 + z.c]; },
      [&](int b, const cpx<C> (&v)[Z::RL]) {
#pragma unroll
        for (int m = 0; m < Z::RL; ++m) {
          if (2 * m * Z::NBL > Ch::N) continue;  // n <= M / 2 + 1
          const uint32_t j = z.c + z.n2 * (uint32_t)(b + m * Z::NBL);
          if (j < nn) {
            const cpx<C> y = cmul(cswap(v[m]), chirp[j]);
            out[j * os] = ST::st(BWD ? cswap(y) : y);
          }
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
template <typename S, bool BWD, int W, int TPT, class Ch>
__global__ void __launch_bounds__(W *TPT) k_rd_col_in(KArgs a) {
  using ST = StorageT<S>;
  using E = typename ST::E;
  using C = typename ST::C;
  using Z = CzTile<C, W, TPT, Ch>;
  const Z z(a);
  const E *in = static_cast<const E *>(a.in) + z.bi * a.idist;
  cpx<C> *ws = static_cast<cpx<C> *>(a.out) + (int64_t)z.bi * Ch::N * z.n2;
  const int *perm = static_cast<const int *>(a.aux1);
  const int64_t is = a.istride;
  if (z.c == 0 && z.t == 0) {
    const cpx<C> x0 = ST::ld(in[0]);
    static_cast<cpx<C> *>(a.aux3)[2 * z.bi] = BWD ? cswap(x0) : x0;
  }
  Z::T::run(
      reinterpret_cast<C *>(dyn_lds<C>()), static_cast<const cpx<C> *>(a.tw), threadIdx.x,
      [&](int b, int m) {
        const cpx<C> v = ST::ld(in[perm[z.n2 * (uint32_t)(b + m * Z::NB0) + z.c] * is]);
        return BWD ? cswap(v) : v;
      },
      [&](int b, const cpx<C> (&v)[Z::RL]) { z.put(a, ws, b, v); });
}

template <typename S, bool BWD, int W, int TPT, class Ch>
__global__ void __launch_bounds__(W *TPT) k_rd_col_out(KArgs a) {
  using ST = StorageT<S>;
  using E = typename ST::E;
  using C = typename ST::C;
  using Z = CzTile<C, W, TPT, Ch>;
  const Z z(a);
  const uint32_t N = Ch::N * z.n2;
  const cpx<C> *ws = static_cast<const cpx<C> *>(a.in) + (int64_t)z.bi * N;
  E *out = static_cast<E *>(a.out) + z.bi * a.odist;
  const int *perm = static_cast<const int *>(a.aux1);
  const cpx<C> *slot = static_cast<const cpx<C> *>(a.aux3) + 2 * z.bi;
  const cpx<C> x0 = slot[0];
  const int64_t os = a.ostride;
  Z::T::run(
      reinterpret_cast<C *>(dyn_lds<C>()), static_cast<const cpx<C> *>(a.tw), threadIdx.x,
      [&](int b, int m) { return ws[(uint32_t)(b + m * Z::NB0) * z.n2 + z.c]; },
      [&](int b, const cpx<C> (&v)[Z::RL]) {
        int64_t at[Z::RL];
#pragma unroll
        for (int m = 0; m < Z::RL; ++m) {
          const uint32_t q = z.c + z.n2 * (uint32_t)(b + m * Z::NBL);
          at[m] = perm[q == 0 ? 0 : N - q] * os;
        }
#pragma unroll
        for (int m = 0; m < Z::RL; ++m) {
          const cpx<C> r = cadd(x0, cswap(v[m]));
          out[at[m]] = ST::st(BWD ? cswap(r) : r);
        }
        if (z.c == 0 && b == 0) {
          const cpx<C> y0 = cadd(x0, slot[1]);
          out[0] = ST::st(BWD ? cswap(y0) : y0);
        }
      });
}

}  // namespace plf
