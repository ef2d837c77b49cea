// kernels_f64_cz.hip -- FP64 three-pass chirp-z and Rader kernels (the
// column and row engines of the four-step passes, sides 64..512).
#include "kernels_cz.hpp"
#include "launch.hpp"

namespace plf {

void register_kernels_f64_cz(std::vector<KEntry> &r) {
  using S = double;
  constexpr int P = P_F64;
  PLF_CZ_COLS(S, P,    8,  16, 8, 8);
  PLF_CZ_COLS(S, P,    8,  16, 16, 8);
  PLF_CZ_COLS(S, P,   16,  16, 16, 16);
  PLF_CZ_COLS(S, P,   32,   8, 16, 2, 16);
  PLF_CZ_MID(S, P,    8,  32, 8, 8);
  PLF_CZ_MID(S, P,    8,  32, 16, 8);
  PLF_CZ_MID(S, P,   16,  16, 16, 16);
  PLF_CZ_MID(S, P,   64,   4, 8, 8, 8);
  // row sides with a factor 3, for M = 3 * 2^k
  PLF_CZ_MID(S, P,    4,  64, 8, 12);
  PLF_CZ_MID(S, P,    8,  32, 8, 3, 8);
  PLF_CZ_MID(S, P,   16,  16, 8, 6, 8);
}

}  // namespace plf
