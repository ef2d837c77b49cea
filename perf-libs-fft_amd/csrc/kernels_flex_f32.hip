// kernels_flex_f32.hip -- FP32 complex transforms of lengths without a compiled chain.
#include "flex_launch.hpp"

namespace plf {

void register_flex_f32(std::vector<FlexEntry> &r) {
  add_flex_c2c<float, 512>(r, P_F32);
  add_flex_c2c<float, 1024>(r, P_F32);
}

}  // namespace plf
