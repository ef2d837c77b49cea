// kernels_conv_bf16.hip -- bf16 Bluestein / Rader kernel configurations.
#include "kernels_conv.hpp"
#include "launch.hpp"

namespace plf {

void register_kernels_conv_bf16(std::vector<KEntry> &r) {
    using S = bf16_pair;
    constexpr int P = P_BF16;
    // powers of two on the tile engine, before the smooth lengths of the runtime
    // chain (the FP32 kernels: 1.1 to 1.3x against the compiled full-exchange
    // engine, which is itself ahead of the runtime chain)
    PLF_BLUE_TILE(S, P,    8,  32, 8, 8);
    PLF_BLUE_TILE(S, P,    8,  32, 16, 8);
    PLF_BLUE_TILE(S, P,   16,  16, 16, 16);
    PLF_BLUE_TILE(S, P,   32,   8, 16, 2, 16);
    PLF_BLUE_TILE(S, P,   64,   4, 16, 4, 16);
    PLF_BLUE_TILE(S, P,  128,   2, 16, 8, 16);
    PLF_BLUE_TILE(S, P,  256,   1, 16, 16, 16);
    PLF_BLUE_TILE(S, P,  512,   1, 16, 2, 16, 16);
    PLF_BLUE_TILE(S, P, 1024,   1, 16, 4, 16, 16);
    PLF_DYNAMIC(k_bluestein, KK_BLUE, S, P,  64,   4, 16);
    PLF_DYNAMIC(k_bluestein, KK_BLUE, S, P, 256,   1, 16);
    PLF_DYNAMIC(k_bluestein, KK_BLUE, S, P, 1024,  1, 16);
    PLF_DYNAMIC(k_rader, KK_RADER, S, P,   64,   4, 16);
    PLF_DYNAMIC(k_rader, KK_RADER, S, P,  256,   1, 16);
    PLF_DYNAMIC(k_rader, KK_RADER, S, P, 1024,   1, 16);
}

}  // namespace plf
