// flex_args.hpp -- host and device description of a flexible chain
// (flex_engine.hpp).
#pragma once

#include <stdint.h>

namespace plf {

constexpr int kFlexStages = 8;

// The stage shapes the engine compiles: radix and butterflies per thread.
struct FlexShape {
  int r, k;
};
constexpr FlexShape kFlexShapes[] = {
    {2, 1}, {2, 2}, {2, 4}, {2, 7}, {3, 1},  {3, 2},  {3, 3},  {3, 4},  {3, 5},  {4, 1},  {4, 2},
    {4, 3}, {4, 4}, {5, 1}, {5, 2}, {5, 3},  {6, 1},  {6, 2},  {7, 1},  {7, 2},  {8, 1},  {8, 2},
    {9, 1}, {9, 2}, {10, 1}, {10, 2}, {11, 1}, {12, 1}, {13, 1}, {15, 1}, {16, 1}};
constexpr int kFlexShapeCount = sizeof(kFlexShapes) / sizeof(kFlexShapes[0]);

struct FlexStage {
  int shape;             // index into kFlexShapes
  int L, nb;             // product of the earlier radices, n / radix
  int twoff;             // twiddles of this stage (complex entries)
  uint32_t magic;        // ceil(2^32 / L): b / L = umulhi(b, magic), b < 2^16
  int rd_gp, rd_step;    // inputs from LDS: group distance, distance of consecutive inputs
  int wr_gp;             // outputs to LDS: distance of the groups of L * radix
};

struct FlexDesc {
  int n, ns, tpt, tpb;
  int lanes;           // 1: neighbouring threads in neighbouring members, else in one member
  uint32_t magic;      // thread / (lanes ? tpb : tpt) = umulhi(thread, magic), divisor > 1
  int lper;            // LDS complex slots per member
  FlexStage st[kFlexStages];
};

}  // namespace plf
