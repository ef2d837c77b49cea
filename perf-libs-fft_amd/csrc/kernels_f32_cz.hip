// kernels_f32_cz.hip -- three-pass chirp-z and Rader kernels with FP32 arithmetic
// (kernels_cz.hpp; f32, f16 and bf16 storage), sides 64..1024.
#include "kernels_cz.hpp"
#include "launch.hpp"

namespace plf {

// sides 64..1024 with FP32 arithmetic for storage S
template <typename S, int P>
void register_cz_f32_compute(std::vector<KEntry> &r) {
  PLF_CZ_COLS(S, P,    8,  32, 8, 8);
  PLF_CZ_COLS(S, P,    8,  32, 16, 8);
  PLF_CZ_COLS(S, P,   16,  16, 16, 16);
  PLF_CZ_COLS(S, P,   32,  16, 16, 2, 16);
  PLF_CZ_COLS(S, P,   64,  16, 16, 4, 16);
  PLF_CZ_MID(S, P,    8,  32, 8, 8);
  PLF_CZ_MID(S, P,    8,  32, 16, 8);
  PLF_CZ_MID(S, P,   16,  16, 16, 16);
  PLF_CZ_MID(S, P,   32,   8, 16, 2, 16);
  PLF_CZ_MID(S, P,   64,   4, 16, 4, 16);
  // row sides with a factor 3, for M = 3 * 2^k (192 on 12 points a thread: 10007
  // 15.7 us for one member and 187 for 838, 20.6 and 194 on 24)
  PLF_CZ_MID(S, P,    4,  64, 8, 12);
  PLF_CZ_MID(S, P,   16,   8, 4, 12, 4);
  PLF_CZ_MID(S, P,   16,  16, 8, 6, 8);
  PLF_CZ_MID(S, P,   32,   8, 8, 12, 8);
}

void register_kernels_f32_cz(std::vector<KEntry> &r) {
  register_cz_f32_compute<float, P_F32>(r);
  register_cz_f32_compute<half_pair, P_F16>(r);
  register_cz_f32_compute<bf16_pair, P_BF16>(r);
}

}  // namespace plf
