// flex_chain.hpp -- choice of a flexible chain (flex_engine.hpp).
#pragma once

#include <stddef.h>
#include <stdint.h>

#include <vector>

#include "flex_args.hpp"

namespace plf {

// A block's time beyond its chain, in the units of a chain's work
// (flex_chain.cpp): per real of a member that a thread moves between memory and
// LDS, and per point of the first stage, where the loads compute. spare: reals
// are moved by more threads than there are butterflies.
// members > 0: a batch of so many, for which `resident` threads run at once.
// members = 0: a full chip; a real costs more the fewer threads move a member's
// (each opens a line of its own).
struct FlexWait {
  int64_t members, resident;
  double real, first;
  bool spare;
};

// The chain, thread count and LDS layout for members of length n (2 <= n <
// 2^15) at up to `pts` points per thread and `block` threads per block, with
// elements of `csize` bytes: least predicted cost, LDS up to `lds_max` bytes.
// False if n has a prime factor above 13 or does not fit.
// lanes > 0: that many neighbouring members per row of threads (members
// closer together than their elements), or fewer if they do not fit.
// wait: with the work outside the chain; for members > 0 the least predicted
// time of a batch that leaves the chip partly idle, instead of the least work
// per member.
bool flex_choose(int64_t n, int pts, int block, int csize, int64_t lds_max, int lanes,
                 FlexDesc *out, const FlexWait *wait = nullptr);
std::vector<int> flex_radices(const FlexDesc &d);
inline int flex_threads(const FlexDesc &d) { return (d.tpt * d.tpb + 63) / 64 * 64; }
inline size_t flex_lds(const FlexDesc &d, int csize) { return (size_t)d.tpb * d.lper * csize; }

}  // namespace plf
