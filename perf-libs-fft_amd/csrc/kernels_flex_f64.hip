// kernels_flex_f64.hip -- FP64 complex transforms of lengths without a compiled chain.
#include "flex_launch.hpp"

namespace plf {

// 256 threads: the widest stages take 172 registers, two waves per SIMD.
void register_flex_f64(std::vector<FlexEntry> &r) {
  add_flex_c2c<double, 256>(r, P_F64);
  add_flex_c2c<double, 512>(r, P_F64);
}

}  // namespace plf
