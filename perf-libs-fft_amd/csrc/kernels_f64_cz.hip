// kernels_f64_cz.hip -- FP64 three-pass chirp-z and Rader kernels
// (kernels_cz.hpp), sides 64..512.
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
  // row sides with a factor 3, for M = 3 * 2^k: 12 points a thread. A thread's
  // two transforms are the time of a batch of few members (10007: 16.4 us for
  // one and 99 for 256, against 22.1 and 107 with 24 points, 230 registers).
  // 384 on 8 rows a block: 20011 19.1 us for one member and 380 for 419, 22.2
  // and 397 with 24 points, 18.1 and 384 on 4 rows, which take 60 against 57
  // for 64 members.
  PLF_CZ_MID(S, P,    8,  16, 12, 2, 4);
  PLF_CZ_MID(S, P,   16,   8, 4, 12, 4);
  PLF_CZ_MID(S, P,   32,   8, 4, 4, 4, 6);
}

}  // namespace plf
