// kernels_flex_real_f64.hip -- FP64 real transforms of even lengths without a compiled chain.
#include "flex_launch.hpp"

namespace plf {

void register_flex_real_f64(std::vector<FlexEntry> &r) {
  add_flex_real<double, 256>(r, P_F64);
  add_flex_real<double, 512>(r, P_F64);
}

}  // namespace plf
