#include "tile_pass.hpp"

int lg::tile::launch_mrg_f32(const hgrid_tile *p) { return launch_potential<float2, TMRG>(p); }
