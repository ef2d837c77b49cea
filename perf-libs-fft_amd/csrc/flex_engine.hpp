// flex_engine.hpp -- the runtime-chain Stockham engine with a runtime number
// of threads per member.
//
// Serves the lengths without a compile-time chain. A member of length n runs
// on any number tpt of threads (50 for 1000 = 10.10.10), tpb members a block,
// so that few lanes idle where n is no multiple of a power of two. A stage's
// radix, butterflies per thread and place in the chain (first, middle, last)
// are compile-time (kFlexShapes; one straight-line body each, no predicated
// loads); what depends on n is laid out by the host (flex_chain.cpp):
//   * the division by L, the product of the earlier radices, is a multiply
//     by a reciprocal (exact below 2^16);
//   * an exchange stores its groups of L R elements GP = L R + pad apart, the
//     pad chosen for the banks. As L R divides the next stage's N / R', its
//     inputs are group b / (L R) + m (N / R') / (L R), element b mod (L R):
//     both sides address base + m * (uniform step), with no per-element
//     padding arithmetic.
// Lanes past the last butterfly repeat it and skip the store.
#pragma once

#include "engine.hpp"
#include "flex_args.hpp"

namespace plf {

enum FlexPlace : int { FP_FIRST = 0, FP_MID = 1, FP_LAST = 2, FP_ONLY = 3 };

// TO_LDS: the result stays in LDS in natural order, unpadded (after a
// barrier). LDS_IN: the load callback reads the member's LDS (the caller has
// put a barrier before), so the first stage waits for all of them to be read.
template <typename C, bool TO_LDS, bool LDS_IN = false>
struct FlexEngine {
  // live: the thread belongs to a member of the block; valid: that member is
  // one of the batch.
  template <int R, int K, int PLACE, class Load, class Store>
  static __device__ __forceinline__ void stage(const FlexStage &s, cpx<C> *lds,
                                               const cpx<C> *__restrict__ tw, int t, int tpt,
                                               bool live, bool valid, Load &load, Store &store) {
    constexpr bool FIRST = PLACE == FP_FIRST || PLACE == FP_ONLY;
    constexpr bool LAST = PLACE == FP_LAST || PLACE == FP_ONLY;
    // opaque copy: keeps the address arithmetic of the other bodies from
    // being hoisted out of the stage loop and held in registers
    asm volatile("" : "+v"(t));
    const int NB = s.nb, L = s.L;
    cpx<C> v[K][R];
    int q[K], j[K];
#pragma unroll
    for (int k = 0; k < K; ++k) {
      int b = t + k * tpt;
      b = b < NB ? b : NB - 1;
      if constexpr (FIRST) {
        q[k] = b;
        j[k] = 0;
#pragma unroll
        for (int m = 0; m < R; ++m) {
          v[k][m] = load(b, m * NB);
          burst_after<Load>(v[k], m);
        }
      } else {
        q[k] = (int)__umulhi((uint32_t)b, s.magic);
        j[k] = b - q[k] * L;
        const cpx<C> *src = lds + (q[k] * s.rd_gp + j[k]);
#pragma unroll
        for (int m = 0; m < R; ++m) v[k][m] = src[m * s.rd_step];
      }
    }
#pragma unroll
    for (int k = 0; k < K; ++k) {
      if constexpr (!FIRST) {
        const cpx<C> *w = tw + s.twoff;
#pragma unroll
        for (int m = 1; m < R; ++m)
          v[k][m] = cmul(v[k][m], at_u32(w + (m - 1) * L, (uint32_t)j[k]));
      }
      Dft<R, C>::run(v[k]);
    }
    if constexpr ((!FIRST || LDS_IN) && (!LAST || TO_LDS)) __syncthreads();  // all reads done
#pragma unroll
    for (int k = 0; k < K; ++k) {
      const int b = t + k * tpt;
      const bool act = live && b < NB;
      if constexpr (LAST && !TO_LDS) {
        if (act && valid) {
#pragma unroll
          for (int m = 0; m < R; ++m) store(b, m * NB, v[k][m]);
        }
      } else {
        if (act) {
          // last: natural order, unpadded (L = NB, one group)
          cpx<C> *dst = lds + (LAST ? b : q[k] * s.wr_gp + j[k]);
#pragma unroll
          for (int m = 0; m < R; ++m) dst[m * L] = v[k][m];
        }
      }
    }
    if constexpr (!LAST || TO_LDS) __syncthreads();
  }

  template <int PLACE, int I, class Load, class Store>
  static __device__ __forceinline__ void dispatch(const FlexStage &s, cpx<C> *lds,
                                                  const cpx<C> *__restrict__ tw, int t, int tpt,
                                                  bool live, bool valid, Load &load,
                                                  Store &store) {
    // a binary tree of uniform branches over the shapes
    constexpr int LO = I >> 8, HI = I & 255;
    if constexpr (HI - LO == 1) {
      // a member of one butterfly has one a thread
      if constexpr (PLACE != FP_ONLY || kFlexShapes[LO].k == 1)
        stage<kFlexShapes[LO].r, kFlexShapes[LO].k, PLACE>(s, lds, tw, t, tpt, live, valid, load,
                                                         store);
    } else {
      constexpr int MID = (LO + HI) / 2;
      if (s.shape < MID)
        dispatch<PLACE, (LO << 8) | MID>(s, lds, tw, t, tpt, live, valid, load, store);
      else
        dispatch<PLACE, (MID << 8) | HI>(s, lds, tw, t, tpt, live, valid, load, store);
    }
  }

  // load(b, o): element b + o of the member (o uniform); store(b, o, value).
  template <class Load, class Store>
  static __device__ __forceinline__ void run(const FlexDesc &d, cpx<C> *lds,
                                             const cpx<C> *__restrict__ tw, int t, bool live,
                                             bool valid, Load &&load, Store &&store) {
    const int ns = d.ns;
    if (ns == 1) {
      dispatch<FP_ONLY, kFlexShapeCount>(d.st[0], lds, tw, t, d.tpt, live, valid, load, store);
      return;
    }
    dispatch<FP_FIRST, kFlexShapeCount>(d.st[0], lds, tw, t, d.tpt, live, valid, load, store);
    for (int i = 1; i < ns - 1; ++i)
      dispatch<FP_MID, kFlexShapeCount>(d.st[i], lds, tw, t, d.tpt, live, valid, load, store);
    dispatch<FP_LAST, kFlexShapeCount>(d.st[ns - 1], lds, tw, t, d.tpt, live, valid, load, store);
  }
};

}  // namespace plf
