// The host's choice of launch shapes (feriphys_amd/csrc/tile_rule.hpp) behind a C entry point.
#include "../../feriphys_amd/csrc/tile_rule.hpp"

extern "C" void rule(uint32_t n, const uint32_t* rows, const uint32_t* cols, const int32_t* shape,
                     const int32_t* chosen, int32_t fast, int32_t* out) {
  std::vector<fpsim::ClothTiles> c;
  for (uint32_t i = 0; i < n; ++i) c.push_back(fpsim::ClothTiles{rows[i], cols[i], shape[i], chosen[i] != 0});
  const std::vector<int> s = fpsim::launch_shapes(c, fast != 0);
  for (uint32_t i = 0; i < n; ++i) out[i] = s[i];
}
