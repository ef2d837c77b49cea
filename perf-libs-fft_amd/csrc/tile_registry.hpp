// tile_registry.hpp -- host-side table of the compiled tile kernels
// (kernels_tile.hpp).
#pragma once

#include <string>
#include <vector>

#include "registry.hpp"

namespace plf {

enum TileKind : int { TK_C2C = 0, TK_COL = 1, TK_ROW = 2 };

struct TileEntry {
  int kind, prec;
  bool bwd;
  int n;       // engine length
  int w;       // columns (TK_ROW: rows) per block
  int wb;      // TK_COL / TK_ROW: rows per block of the workspace layout
  std::vector<int> chain;
  size_t lds;  // bytes per block
  KLaunch launch;
  KLaunch launch_nt;  // TK_COL / TK_ROW: outer side in whole lines, past the caches
  std::string name() const;
};

const std::vector<TileEntry> &tile_registry();
void register_tiles_f32(std::vector<TileEntry> &r);
void register_tiles_f64(std::vector<TileEntry> &r);
void register_tiles_h(std::vector<TileEntry> &r);

}  // namespace plf
