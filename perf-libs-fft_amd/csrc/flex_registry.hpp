// flex_registry.hpp -- host-side table of the flexible-chain kernels
// (kernels_flex.hpp).
#pragma once

#include <hip/hip_runtime.h>

#include <vector>

#include "flex_args.hpp"
#include "kernel_args.hpp"

namespace plf {

struct FlexArgs {
  KArgs a;
  const FlexDesc *d;  // device memory
};

enum FlexKind : int { FK_C2C = 0, FK_R2C = 1, FK_C2R = 2, FK_DCT2 = 3, FK_DCT3 = 4 };

using FlexLaunch = hipError_t (*)(const FlexArgs &, int64_t grid, int threads, size_t lds,
                                  hipStream_t);

struct FlexEntry {
  int kind, prec;
  bool bwd;   // C2C direction; DCT kinds: the DST
  int block;  // most threads per block
  FlexLaunch launch;
};

// Entries of one kind, precision and direction in ascending block order.
const std::vector<FlexEntry> &flex_registry();
void register_flex_f32(std::vector<FlexEntry> &r);
void register_flex_f64(std::vector<FlexEntry> &r);
void register_flex_real_f32(std::vector<FlexEntry> &r);
void register_flex_real_f64(std::vector<FlexEntry> &r);
void register_flex_h(std::vector<FlexEntry> &r);

}  // namespace plf
