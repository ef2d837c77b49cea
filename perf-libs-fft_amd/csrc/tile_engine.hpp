// tile_engine.hpp -- W transforms of one length per block, through the split
// (real, then imaginary) LDS exchange.
//
// The engine of the strided kernels (kernels_tile.hpp): a block of W * TPT
// threads runs W member columns of length N. Every stage but the last deals
// its butterflies with map AIN, the last one with map AOUT; the exchange in
// between crosses the whole block's LDS, so changing the map there costs
// nothing:
//   A (true)   column = thread % W, butterfly thread / W: neighbouring lanes
//              hold neighbouring columns (members at distance 1)
//   B (false)  butterfly = thread % TPT, column thread / TPT: neighbouring
//              lanes hold neighbouring elements of one column
// An access of a strided side then covers W consecutive elements (a 128-byte
// line) and an access of a contiguous side min(TPT, 64) of them.
//
// LDS holds one scalar per element, column g at g * LPER. An element has one
// pad slot every 16 and LPER is 1/2 + 1/(2W) of the banks modulo all of them, so that
// the 64/W butterflies x W columns of a wave (map A) and the 64 consecutive
// elements (map B) both spread over the banks, at the first stage's stride
// of 16 as at the later ones' stride of 1.
#pragma once

#include "engine.hpp"

namespace plf {

template <typename C, int W, int TPT, class Ch, bool AIN, bool AOUT>
struct TileEngine {
  static constexpr int N = Ch::N;
  static constexpr int NS = Ch::count;
  static constexpr int BANKS = 256 / (int)sizeof(C);
  static constexpr int LPER = [] {
    const int want = (BANKS / 2 + (BANKS / 2 / W > 0 ? BANKS / 2 / W : 1)) % BANKS;
    int l = N + N / 16 + 1;
    while (l % BANKS != want) ++l;
    return l;
  }();
  static constexpr size_t LDS_BYTES = (size_t)W * LPER * sizeof(C);
  static_assert(NS >= 2, "one exchange at least");

  // Map B alone, members within one wave: the exchange stays in the wave, whose
  // LDS accesses are executed in order, so no barrier is needed.
  static constexpr bool WAVE = !AIN && !AOUT && 64 % TPT == 0;
  static __device__ __forceinline__ void sync() {
    if constexpr (WAVE) {
      __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
      __builtin_amdgcn_wave_barrier();
      __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
    } else {
      __syncthreads();
    }
  }

  template <int SI>
  struct St {
    static constexpr int R = Ch::radix(SI);
    static constexpr int L = Ch::L(SI);
    static constexpr int NB = N / R;
    static constexpr int KB = NB / TPT;
    static constexpr bool A = SI == NS - 1 ? AOUT : AIN;
    static_assert(NB % TPT == 0, "whole butterflies per thread");
  };
  static __device__ __forceinline__ int col(bool a, int tid) { return a ? tid % W : tid / TPT; }
  static __device__ __forceinline__ int thr(bool a, int tid) { return a ? tid / W : tid % TPT; }
  // this thread's column at the loads and at the stores
  static __device__ __forceinline__ int col_in(int tid) { return col(AIN, tid); }
  static __device__ __forceinline__ int col_out(int tid) { return col(AOUT, tid); }

  template <int SI>
  static __device__ __forceinline__ void compute(cpx<C> (&v)[St<SI>::KB][St<SI>::R],
                                                 const cpx<C> *__restrict__ tw, int tid) {
    using T = St<SI>;
    const int t = thr(T::A, tid);
#pragma unroll
    for (int k = 0; k < T::KB; ++k) {
      if constexpr (SI > 0) {
        const int j = (t + k * TPT) % T::L;
#pragma unroll
        for (int m = 1; m < T::R; ++m)
          v[k][m] = cmul(v[k][m], tw[Ch::tw_offset(SI) + (m - 1) * T::L + j]);
      }
      Dft<T::R, C>::run(v[k]);
    }
  }

  template <int SI, int COMP>
  static __device__ __forceinline__ void put(C *lds, const cpx<C> (&v)[St<SI>::KB][St<SI>::R],
                                             int tid) {
    using T = St<SI>;
    const int t = thr(T::A, tid);
    C *c = lds + col(T::A, tid) * LPER;
#pragma unroll
    for (int k = 0; k < T::KB; ++k) {
      const int b = t + k * TPT;
      const int base = (b / T::L) * T::L * T::R + b % T::L;
#pragma unroll
      for (int m = 0; m < T::R; ++m)
        c[lds_pad_step<4, T::L>(base, m)] = COMP ? v[k][m].y : v[k][m].x;
    }
  }

  template <int SI, int COMP>
  static __device__ __forceinline__ void get(const C *lds, cpx<C> (&v)[St<SI>::KB][St<SI>::R],
                                             int tid) {
    using T = St<SI>;
    const int t = thr(T::A, tid);
    const C *c = lds + col(T::A, tid) * LPER;
#pragma unroll
    for (int k = 0; k < T::KB; ++k)
#pragma unroll
      for (int m = 0; m < T::R; ++m) {
        const C x = c[lds_pad_step<4, T::NB>(t + k * TPT, m)];
        if (COMP) v[k][m].y = x;
        else v[k][m].x = x;
      }
  }

  template <int SI, class Store>
  static __device__ __forceinline__ void from(cpx<C> (&v)[St<SI>::KB][St<SI>::R], C *lds,
                                              const cpx<C> *__restrict__ tw, int tid,
                                              Store &store) {
    using T = St<SI>;
    compute<SI>(v, tw, tid);
    if constexpr (SI == NS - 1 && std::is_invocable_v<Store &, decltype(v)>) {
      store(v);
    } else if constexpr (SI == NS - 1) {
      const int t = thr(T::A, tid);
#pragma unroll
      for (int k = 0; k < T::KB; ++k) store(t + k * TPT, v[k]);
    } else {
      cpx<C> w[St<SI + 1>::KB][St<SI + 1>::R];
      put<SI, 0>(lds, v, tid);
      sync();
      get<SI + 1, 0>(lds, w, tid);
      sync();
      put<SI, 1>(lds, v, tid);
      sync();
      get<SI + 1, 1>(lds, w, tid);
      if constexpr (SI + 1 < NS - 1) sync();  // the next exchange rewrites LDS
      from<SI + 1>(w, lds, tw, tid, store);
    }
  }

  // load(b, m): element b + m * (N / R0) of this thread's input column.
  // store(b, v): v[m] = element b + m * (N / RL) of its output column, or
  // store(v): all of them, v[k][m] for b = thr(AOUT, tid) + k * TPT.
  template <class Load, class Store>
  static __device__ __forceinline__ void run(C *lds, const cpx<C> *__restrict__ tw, int tid,
                                             Load &&load, Store &&store) {
    using T = St<0>;
    cpx<C> v[T::KB][T::R];
    const int t = thr(T::A, tid);
#pragma unroll
    for (int k = 0; k < T::KB; ++k)
#pragma unroll
      for (int m = 0; m < T::R; ++m) v[k][m] = load(t + k * TPT, m);
    from<0>(v, lds, tw, tid, store);
  }
};

// The chain in reverse order.
template <class Ch, class = std::make_integer_sequence<int, Ch::count>>
struct ReversedChain;
template <class Ch, int... I>
struct ReversedChain<Ch, std::integer_sequence<int, I...>> {
  using type = Chain<Ch::radix(Ch::count - 1 - I)...>;
};

// Two transforms of one length with a product in between (the convolutions of
// kernels_conv.hpp and kernels_cz.hpp), W members of TPT threads. The last
// stage of the first leaves a thread elements b + m * (N / RL), which are the
// inputs of a first stage of radix RL: the second transform runs the chain in
// reverse and takes them from registers. Against a transform through LDS in
// natural order, a pass over LDS and the second transform's stage 0 this saves
// one of 2 NS - 1 exchanges, and the split exchange half of the LDS.
template <typename C, int W, int TPT, class Ch>
struct ConvTile {
  using First = TileEngine<C, W, TPT, Ch, false, false>;
  using Second = TileEngine<C, W, TPT, typename ReversedChain<Ch>::type, false, false>;
  static constexpr int N = Ch::N;
  static constexpr int R = Ch::radix(Ch::count - 1);  // the radix on both sides of the product
  static constexpr int NB = N / R, KB = NB / TPT;
  static constexpr size_t LDS_BYTES =
      First::LDS_BYTES > Second::LDS_BYTES ? First::LDS_BYTES : Second::LDS_BYTES;

  // tw: the chain's twiddles, then those of the reversed chain. load(b, m) as
  // TileEngine::run; mid(v): v[k][m] = element t + k TPT + m NB of the first
  // transform, replaced by the second's input; store(b, v) as TileEngine::run.
  template <class Load, class Mid, class Store>
  static __device__ __forceinline__ void run(C *lds, const cpx<C> *__restrict__ tw, int tid,
                                             Load &&load, Mid &&mid, Store &&store) {
    First::run(lds, tw, tid, load, [&](cpx<C> (&v)[KB][R]) {
      mid(v);
      First::sync();  // the first's last reads are done
      Second::template from<0>(v, lds, tw + Ch::tw_size(), tid, store);
    });
  }
};

}  // namespace plf
