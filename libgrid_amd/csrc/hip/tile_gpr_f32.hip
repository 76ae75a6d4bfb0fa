#include "tile_pass.hpp"

int lg::tile::launch_gpr_f32(const hgrid_tile *p) { return launch_potential<float2, TGPR>(p); }
