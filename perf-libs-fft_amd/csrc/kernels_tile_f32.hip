// kernels_tile_f32.hip -- FP32 tile kernels: columns and four-step passes.
#include "tile_launch.hpp"

namespace plf {

// Chains, widths and register caps are the fastest of the sweeps over 512 MiB
// each way (us per pass; W columns, WB rows per block of the workspace).
void register_tiles_f32(std::vector<TileEntry> &r) {
  using S = float;
  constexpr int P = P_F32;
  //               W  TPT WB waves  chain
  add_tile_c2c<S, 64, 4, 8, 16, 4>(r, P);
  add_tile_c2c<S, 32, 8, 8, 16, 8>(r, P);
  add_tile_c2c<S, 32, 16, 8, 16, 16>(r, P);
  add_tile_c2c<S, 32, 16, 4, 16, 32>(r, P);
  add_tile_c2c<S, 16, 32, 4, 32, 32>(r, P);  // 64 us; 16x16x4 on 64 threads 74
  add_tile_c2c<S, 16, 64, 4, 32, 8, 8>(r, P);
  // pass A (k_col: 279 at 256, 325 at 1024)
  add_tile_col<S, 32, 16, 32, 5, 16, 16>(r, P);  // 203; 64 registers spill: 239
  add_tile_col<S, 32, 16, 32, 4, 16, 32>(r, P);  // 212; 16x16x2: 227
  add_tile_col<S, 32, 16, 16, 4, 16, 32>(r, P);
  add_tile_col<S, 16, 32, 16, 4, 32, 32>(r, P);  // 227; 16x16x4 on 64 threads 238
  add_tile_col<S, 16, 64, 16, 4, 32, 8, 8>(r, P);  // 295; 8 columns a tile 335
  // pass B (k_row: 203 at 256, 262 at 1024)
  add_tile_row<S, 32, 16, 8, 16, 16>(r, P);     // 179
  add_tile_row<S, 32, 32, 8, 16, 2, 16>(r, P);  // 187; 8x8x8 190
  add_tile_row<S, 16, 64, 8, 16, 4, 16>(r, P);  // 199; 32x32 212
  add_tile_row<S, 16, 64, 4, 16, 16, 8>(r, P);  // 244; 8 rows a tile 251
}

}  // namespace plf
