// Which tile shape each cloth on the tiled grid kernel is launched with (host code).
#pragma once

#include <cstdint>
#include <vector>

#include "kernels.hpp"

namespace fpsim {

inline uint64_t tile_count(uint64_t rows, uint64_t cols, int shape) {
  const uint64_t tr = (uint64_t)fp::kTileRows[shape], tc = (uint64_t)fp::kTileCols[shape];
  return ((rows + tr - 1) / tr) * ((cols + tc - 1) / tc);
}

// Most 8x8 tiles that the exact kernel takes in place of the default shapes: three to a CU.  Up to
// there a step is one tile's chain of dependent work and the twelve-wave form is the faster (5.1 us
// against 8.7 up to 128 x 128 vertices, 256 tiles; 7.8 against 8.8 at 192 x 192, 576 tiles); at 224 x
// 224, 784 tiles, both take 9.0, and beyond it the larger tiles' fewer operations win (256 x 256: 9.1
// against 9.7).  The surrogate's big step runs over the same tiles, a lane per vertex; there too the 8x8
// tiles' shorter face phase is the faster up to the line (4.6 to 5.4 us from 16 x 16 to 192 x 192 vertices,
// 15x15 tiles 5.0 to 6.2).
constexpr uint64_t kSmallTiles = 768;
// Tiles resident at once: six workgroups of the fast kernel (seven of the exact one's lane-per-vertex form)
// on each of 256 CUs.
constexpr uint64_t kResidentTiles = 1536;

struct ClothTiles {
  uint32_t rows, cols;
  int shape;    // the default for its size, or what the caller asked for
  bool chosen;  // asked for by the caller: launched as it is
};

// The shape a cloth is launched with on its own: the fast kernel has one quad per thread, 15x15 and 7x31
// tiles; 16x16 becomes 15x15.
inline int own_shape(int shape, bool fast) { return fast && shape == fp::TILE_16x16 ? (int)fp::TILE_15x15 : shape; }

// The launch shape of every cloth.  A chosen shape stays; the others take 8x8 where the simulation is
// small and exact, and otherwise share one shape while all the tiles together are resident at once: meshes
// of different shapes cost a launch per shape and step, a launch is then one tile's latency and a second one
// as long again, so they take the shape that most tiles have.
inline std::vector<int> launch_shapes(const std::vector<ClothTiles>& cloths, bool fast) {
  uint64_t n_small = 0, per_shape[fp::N_TILE_SHAPES] = {};
  for (const auto& c : cloths) {
    n_small += tile_count(c.rows, c.cols, fp::TILE_8x8);
    per_shape[own_shape(c.shape, fast)] += tile_count(c.rows, c.cols, own_shape(c.shape, fast));
  }
  const bool small = !fast && n_small <= kSmallTiles;
  int common = 0;
  for (int sh = 1; sh < fp::N_TILE_SHAPES; ++sh)
    if (per_shape[sh] > per_shape[common]) common = sh;
  uint64_t n_common = 0;
  for (const auto& c : cloths) n_common += tile_count(c.rows, c.cols, c.chosen ? own_shape(c.shape, fast) : common);
  const bool one_shape = n_common <= kResidentTiles;
  std::vector<int> out;
  for (const auto& c : cloths)
    out.push_back(c.chosen ? own_shape(c.shape, fast)
                  : small  ? (int)fp::TILE_8x8
                           : one_shape ? common : own_shape(c.shape, fast));
  return out;
}

}  // namespace fpsim
