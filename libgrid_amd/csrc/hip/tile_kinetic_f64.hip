#include "tile_pass.hpp"

int lg::tile::launch_kinetic_f64(const hgrid_tile *p) { return launch_kinetic<double2>(p); }
