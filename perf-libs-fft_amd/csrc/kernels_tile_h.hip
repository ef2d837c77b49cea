// kernels_tile_h.hip -- f16 / bf16 storage, FP32 arithmetic: tile kernels
// for columns and four-step passes.
#include "tile_launch.hpp"

namespace plf {

// Us per pass of 512 MiB of FP32 workspace.
template <typename S, int P>
static void register_half(std::vector<TileEntry> &r) {
  add_tile_c2c<S, 64, 4, 8, 16, 4>(r, P);
  add_tile_c2c<S, 32, 8, 8, 16, 8>(r, P);
  add_tile_c2c<S, 32, 16, 8, 16, 16>(r, P);
  add_tile_c2c<S, 32, 32, 8, 16, 16, 2>(r, P);
  add_tile_c2c<S, 16, 64, 8, 16, 16, 4>(r, P);
  add_tile_col<S, 32, 16, 32, 5, 16, 16>(r, P);
  add_tile_col<S, 32, 32, 32, 7, 16, 2, 16>(r, P);  // 202 us; 16x32 319
  add_tile_col<S, 32, 32, 16, 7, 16, 2, 16>(r, P);
  add_tile_col<S, 16, 64, 16, 8, 16, 4, 16>(r, P);  // 244; 32x32 356
  add_tile_row<S, 32, 16, 8, 16, 16>(r, P);
  add_tile_row<S, 32, 32, 8, 16, 2, 16>(r, P);
  add_tile_row<S, 16, 64, 8, 16, 4, 16>(r, P);
}

void register_tiles_h(std::vector<TileEntry> &r) {
  register_half<half_pair, P_F16>(r);
  register_half<bf16_pair, P_BF16>(r);
}

}  // namespace plf
