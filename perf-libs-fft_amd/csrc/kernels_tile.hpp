// kernels_tile.hpp -- complex transforms on the tile engine (tile_engine.hpp).
//
//   k_tile_c2c  columns of a matrix: members at distance 1, elements at a
//               stride (both sides)
//   k_tile_col  four-step pass A and
//   k_tile_row  four-step pass B for N = n1 * n2 with compile-time sides
//
// Four-step: X[k1 + n1 k2] = sum_c W_n2^{c k2} W_N^{c k1} sum_e x[c + n2 e] W_n1^{e k1}.
// The workspace holds the twiddled columns in blocks of WB rows,
//   ws[(k1 / WB)][c][k1 % WB],
// so that pass A, whose last stage runs on map B, writes WB consecutive k1
// (whole 128-byte lines), pass B's tile of WB rows is one contiguous piece of
// n2 * WB elements, and its outputs are WB consecutive bins: neither pass
// transposes through LDS, and both fit the split exchange.
#pragma once

#include "kernels.hpp"
#include "tile_engine.hpp"

namespace plf {

// KArgs::flags of k_tile_c2c
constexpr int kTileXcd = 1;  // columns: consecutive tiles on one XCD

// ---------------------------------------------------------------------------
// columns: KArgs in, out, tw, count, istride, idist, ostride, odist. Bound by
// the lines it opens: a tile touches N lines a whole row apart, and where the
// rows do not start on line boundaries a line is shared with the next tile
// (kTileXcd puts both in one L2; plain accesses, so that it merges the halves:
// 16001 columns of 1024 in 77 us against 97 us in dispatch order and 157 us
// with non-temporal stores). 16384 columns of 1024 (134 MB each way): 64 us,
// 173 us on k_c2c, whose lanes run along a column (64 lines an instruction).
// ---------------------------------------------------------------------------
template <typename S, bool BWD, int W, int TPT, int WAVES, class Ch>
__global__ void __launch_bounds__(W *TPT) __attribute__((amdgpu_waves_per_eu(WAVES)))
k_tile_c2c(KArgs a) {
  using ST = StorageT<S>;
  using E = typename ST::E;
  using C = typename ST::C;
  using T = TileEngine<C, W, TPT, Ch, true, true>;
  const int tid = threadIdx.x;
  const int64_t bx = (a.flags & kTileXcd) ? xcd_block(blockIdx.x, gridDim.x) : (int64_t)blockIdx.x;
  const int64_t tr = bx * W + T::col_in(tid);
  const bool valid = tr < a.count;
  const E *in = static_cast<const E *>(a.in) + (valid ? tr * a.idist : 0);
  E *out = static_cast<E *>(a.out) + (valid ? tr * a.odist : 0);
  const int64_t is = a.istride, os = a.ostride;
  constexpr int NB0 = Ch::N / Ch::radix(0), RL = Ch::radix(Ch::count - 1), NBL = Ch::N / RL;
  T::run(
      reinterpret_cast<C *>(dyn_lds<C>()), static_cast<const cpx<C> *>(a.tw), tid,
      [&](int b, int m) {
        if (!valid) return cpx<C>{C(0), C(0)};
        const cpx<C> v = ST::ld(in[(int64_t)b * is + (int64_t)(m * NB0) * is]);
        return BWD ? cswap(v) : v;
      },
      [&](int b, const cpx<C> (&v)[RL]) {
        if (!valid) return;
        E *o = out + (int64_t)b * os;
#pragma unroll
        for (int m = 0; m < RL; ++m)
          o[(int64_t)(m * NBL) * os] = ST::st(BWD ? cswap(v[m]) : v[m]);
      });
}

// ---------------------------------------------------------------------------
// four-step pass A: one block per W columns (n2 % W == 0, n1 % WB == 0).
// aux0: T1[c][b] = W_N^{c b}, b < NB; aux1: T2[c][m] = W_N^{c NB m}, m < RL
// (RL the last radix, NB = n1 / RL): the twiddle of k1 = b + m NB is the
// product of one table entry per thread and RL entries per column.
// KArgs: in, out (workspace), tw, istride, idist, n2, bigdist.
// ---------------------------------------------------------------------------
// NT: the input is read in whole lines, once each, so past the caches; also
// the workspace, always.
template <typename S, bool BWD, int W, int TPT, int WB, int WAVES, bool NT, class Ch>
__global__ void __launch_bounds__(W *TPT) __attribute__((amdgpu_waves_per_eu(WAVES)))
k_tile_col(KArgs a) {
  using ST = StorageT<S>;
  using E = typename ST::E;
  using C = typename ST::C;
  using T = TileEngine<C, W, TPT, Ch, true, false>;
  constexpr int NB0 = Ch::N / Ch::radix(0), RL = Ch::radix(Ch::count - 1), NBL = Ch::N / RL;
  static_assert(NBL % WB == 0 || WB % NBL == 0, "k1 = b + m NB splits at WB");
  const int tid = threadIdx.x;
  const uint32_t n2 = (uint32_t)a.n2, tpm = n2 / W;  // tiles per member
  const uint32_t bi = blockIdx.x / tpm, c0 = (blockIdx.x % tpm) * W;
  const int64_t is = a.istride, step = (int64_t)n2 * is;
  const E *in = static_cast<const E *>(a.in) + (int64_t)bi * a.idist +
                (int64_t)(c0 + T::col_in(tid)) * is;
  const uint32_t c = c0 + T::col_out(tid);
  cpx<C> *ws = static_cast<cpx<C> *>(a.out) + (int64_t)bi * a.bigdist + c * WB;
  const cpx<C> *t1 = static_cast<const cpx<C> *>(a.aux0) + c * NBL;
  const cpx<C> *t2 = static_cast<const cpx<C> *>(a.aux1) + c * RL;
  T::run(
      reinterpret_cast<C *>(dyn_lds<C>()), static_cast<const cpx<C> *>(a.tw), tid,
      [&](int b, int m) {
        const E *p = in + ((int64_t)b * step + (m * NB0) * step);
        const cpx<C> v = NT ? ST::ldnt(p) : ST::ld(*p);
        return BWD ? cswap(v) : v;
      },
      [&](int b, const cpx<C> (&v)[RL]) {
        const cpx<C> wb = t1[b];
#pragma unroll
        for (int m = 0; m < RL; ++m) {
          const cpx<C> y = cmul(v[m], m == 0 ? wb : cmul(wb, t2[m]));
          const uint32_t hi = NBL % WB == 0 ? b / WB + m * (NBL / WB) : m / (WB / NBL);
          const uint32_t lo = NBL % WB == 0 ? b % WB : b + (m % (WB / NBL)) * NBL;
          StorageT<C>::stnt(ws + (hi * (n2 * WB) + lo), y);
        }
      });
}

// ---------------------------------------------------------------------------
// four-step pass B: one block per WB rows; the tile is the contiguous piece
// [k1 / WB] of the workspace. KArgs: in (workspace), out, tw, ostride, odist,
// n1, bigdist. NT: the output is written in whole lines.
// ---------------------------------------------------------------------------
template <typename S, bool BWD, int WB, int TPT, int WAVES, bool NT, class Ch>
__global__ void __launch_bounds__(WB *TPT) __attribute__((amdgpu_waves_per_eu(WAVES)))
k_tile_row(KArgs a) {
  using ST = StorageT<S>;
  using E = typename ST::E;
  using C = typename ST::C;
  using T = TileEngine<C, WB, TPT, Ch, true, true>;
  constexpr int NB0 = Ch::N / Ch::radix(0), RL = Ch::radix(Ch::count - 1), NBL = Ch::N / RL;
  const int tid = threadIdx.x;
  const uint32_t n1 = (uint32_t)a.n1, tpm = n1 / WB;
  const uint32_t bi = blockIdx.x / tpm, q = blockIdx.x % tpm;
  const int g = T::col_in(tid);
  const cpx<C> *ws = static_cast<const cpx<C> *>(a.in) + (int64_t)bi * a.bigdist +
                     (int64_t)q * (Ch::N * WB) + g;
  const int64_t os = a.ostride, step = (int64_t)n1 * os;
  E *out = static_cast<E *>(a.out) + (int64_t)bi * a.odist + (int64_t)(q * WB + g) * os;
  T::run(
      reinterpret_cast<C *>(dyn_lds<C>()), static_cast<const cpx<C> *>(a.tw), tid,
      [&](int b, int m) { return StorageT<C>::ldnt(ws + (b + m * NB0) * WB); },
      [&](int b, const cpx<C> (&v)[RL]) {
        E *o = out + b * step;
#pragma unroll
        for (int m = 0; m < RL; ++m) {
          const cpx<C> y = BWD ? cswap(v[m]) : v[m];
          if constexpr (NT) ST::stnt(o + (m * NBL) * step, y);
          else o[(m * NBL) * step] = ST::st(y);
        }
      });
}

}  // namespace plf
