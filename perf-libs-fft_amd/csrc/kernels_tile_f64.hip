// kernels_tile_f64.hip -- FP64 tile kernels: columns and four-step passes.
#include "tile_launch.hpp"

namespace plf {

// As kernels_tile_f32.hip (us per pass of 512 MiB each way).
void register_tiles_f64(std::vector<TileEntry> &r) {
  using S = double;
  constexpr int P = P_F64;
  add_tile_c2c<S, 32, 8, 8, 8, 8>(r, P);
  add_tile_c2c<S, 32, 8, 4, 16, 8>(r, P);
  add_tile_c2c<S, 16, 16, 4, 16, 16>(r, P);
  add_tile_c2c<S, 16, 32, 4, 16, 16, 2>(r, P);
  add_tile_c2c<S, 8, 64, 4, 16, 16, 4>(r, P);
  // pass A (k_col: 297 at 1024)
  add_tile_col<S, 32, 8, 16, 4, 16, 8>(r, P);
  // (a last radix of 16 keeps the table T1, N / RL entries, small)
  add_tile_col<S, 16, 16, 16, 4, 16, 16>(r, P);     // 189; 8x8x4 191
  add_tile_col<S, 16, 32, 16, 4, 16, 2, 16>(r, P);  // 207
  add_tile_col<S, 8, 32, 8, 4, 16, 2, 16>(r, P);    // 204
  add_tile_col<S, 8, 64, 8, 4, 16, 4, 16>(r, P);    // 215
  add_tile_col<S, 8, 128, 8, 4, 16, 8, 16>(r, P);   // 232; 16x16x8 242
  // pass B (k_row: 263 at 1024)
  add_tile_row<S, 16, 16, 4, 16, 16>(r, P);     // 183
  add_tile_row<S, 16, 32, 4, 16, 16, 2>(r, P);  // 178
  add_tile_row<S, 8, 64, 4, 16, 16, 4>(r, P);   // 188
  add_tile_row<S, 8, 128, 4, 16, 16, 8>(r, P);  // 230
}

}  // namespace plf
