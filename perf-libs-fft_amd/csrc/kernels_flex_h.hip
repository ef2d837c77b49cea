// kernels_flex_h.hip -- f16 / bf16 storage: complex transforms of lengths without a compiled chain.
#include "flex_launch.hpp"

namespace plf {

void register_flex_h(std::vector<FlexEntry> &r) {
  add_flex_c2c<half_pair, 512>(r, P_F16);
  add_flex_c2c<half_pair, 1024>(r, P_F16);
  add_flex_c2c<bf16_pair, 512>(r, P_BF16);
  add_flex_c2c<bf16_pair, 1024>(r, P_BF16);
}

}  // namespace plf
