// kernels_flex_real_f32.hip -- FP32 real transforms of even lengths without a compiled chain.
#include "flex_launch.hpp"

namespace plf {

void register_flex_real_f32(std::vector<FlexEntry> &r) {
  add_flex_real<float, 512>(r, P_F32);
  add_flex_real<float, 1024>(r, P_F32);
}

}  // namespace plf
