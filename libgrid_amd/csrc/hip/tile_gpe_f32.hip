#include "tile_pass.hpp"

int lg::tile::launch_gpe_f32(const hgrid_tile *p) { return launch_potential<float2, TGPE>(p); }
