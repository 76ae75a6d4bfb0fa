#include "tile_pass.hpp"

int lg::tile::launch_kinetic_f32(const hgrid_tile *p) { return launch_kinetic<float2>(p); }
