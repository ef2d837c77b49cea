// tile_launch.hpp -- registration of the tile kernels (device side).
#pragma once

#include "kernels_tile.hpp"
#include "launch.hpp"
#include "tile_registry.hpp"

namespace plf {

inline void add_tile(std::vector<TileEntry> &r, int kind, int prec, int n, int w, int wb,
                     std::initializer_list<int> chain, size_t lds, KLaunch fwd, KLaunch bwd,
                     KLaunch fwd_nt = nullptr, KLaunch bwd_nt = nullptr) {
  r.push_back(TileEntry{kind, prec, false, n, w, wb, chain, lds, fwd, fwd_nt});
  r.push_back(TileEntry{kind, prec, true, n, w, wb, chain, lds, bwd, bwd_nt});
}

template <typename S, int W, int TPT, int WAVES, int... Rs>
void add_tile_c2c(std::vector<TileEntry> &r, int prec) {
  using Ch = Chain<Rs...>;
  using T = TileEngine<typename StorageT<S>::C, W, TPT, Ch, true, true>;
  add_tile(r, TK_C2C, prec, Ch::N, W, 0, {Rs...}, T::LDS_BYTES,
           &launch_k<&k_tile_c2c<S, false, W, TPT, WAVES, Ch>, W * TPT>,
           &launch_k<&k_tile_c2c<S, true, W, TPT, WAVES, Ch>, W * TPT>);
}

template <typename S, int W, int TPT, int WB, int WAVES, int... Rs>
void add_tile_col(std::vector<TileEntry> &r, int prec) {
  using Ch = Chain<Rs...>;
  using T = TileEngine<typename StorageT<S>::C, W, TPT, Ch, true, false>;
  add_tile(r, TK_COL, prec, Ch::N, W, WB, {Rs...}, T::LDS_BYTES,
           &launch_k<&k_tile_col<S, false, W, TPT, WB, WAVES, false, Ch>, W * TPT>,
           &launch_k<&k_tile_col<S, true, W, TPT, WB, WAVES, false, Ch>, W * TPT>,
           &launch_k<&k_tile_col<S, false, W, TPT, WB, WAVES, true, Ch>, W * TPT>,
           &launch_k<&k_tile_col<S, true, W, TPT, WB, WAVES, true, Ch>, W * TPT>);
}

template <typename S, int WB, int TPT, int WAVES, int... Rs>
void add_tile_row(std::vector<TileEntry> &r, int prec) {
  using Ch = Chain<Rs...>;
  using T = TileEngine<typename StorageT<S>::C, WB, TPT, Ch, true, true>;
  add_tile(r, TK_ROW, prec, Ch::N, WB, WB, {Rs...}, T::LDS_BYTES,
           &launch_k<&k_tile_row<S, false, WB, TPT, WAVES, false, Ch>, WB * TPT>,
           &launch_k<&k_tile_row<S, true, WB, TPT, WAVES, false, Ch>, WB * TPT>,
           &launch_k<&k_tile_row<S, false, WB, TPT, WAVES, true, Ch>, WB * TPT>,
           &launch_k<&k_tile_row<S, true, WB, TPT, WAVES, true, Ch>, WB * TPT>);
}

}  // namespace plf
