// flex_launch.hpp -- launch wrapper and registration of the flexible-chain
// kernels (device side).
#pragma once

#include "kernels_flex.hpp"
#include "registry.hpp"

namespace plf {

template <void (*K)(FlexArgs)>
hipError_t launch_flex(const FlexArgs &f, int64_t grid, int threads, size_t lds, hipStream_t s) {
  if (lds > 65536) {
    static const hipError_t attr =
        hipFuncSetAttribute(reinterpret_cast<const void *>(K),
                            hipFuncAttributeMaxDynamicSharedMemorySize, 160 * 1024);
    if (attr != hipSuccess) return attr;
  }
  hipLaunchKernelGGL(K, dim3((unsigned)grid), dim3(threads), lds, s, f);
  return hipGetLastError();
}

// Up to BLOCK threads a block; entries of one kind in ascending order.
template <typename S, int BLOCK>
void add_flex_c2c(std::vector<FlexEntry> &r, int prec) {
  r.push_back({FK_C2C, prec, false, BLOCK, &launch_flex<&k_flex_c2c<S, false, BLOCK>>});
  r.push_back({FK_C2C, prec, true, BLOCK, &launch_flex<&k_flex_c2c<S, true, BLOCK>>});
}
template <typename S, int BLOCK>
void add_flex_real(std::vector<FlexEntry> &r, int prec) {
  r.push_back({FK_R2C, prec, false, BLOCK, &launch_flex<&k_flex_r2c<S, false, BLOCK>>});
  r.push_back({FK_C2R, prec, false, BLOCK, &launch_flex<&k_flex_c2r<S, false, BLOCK>>});
  r.push_back({FK_DCT2, prec, false, BLOCK, &launch_flex<&k_flex_dct2<S, false, BLOCK>>});
  r.push_back({FK_DCT2, prec, true, BLOCK, &launch_flex<&k_flex_dct2<S, true, BLOCK>>});
  r.push_back({FK_DCT3, prec, false, BLOCK, &launch_flex<&k_flex_dct3<S, false, BLOCK>>});
  r.push_back({FK_DCT3, prec, true, BLOCK, &launch_flex<&k_flex_dct3<S, true, BLOCK>>});
}

}  // namespace plf
