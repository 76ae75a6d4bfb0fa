#include "tile_pass.hpp"

int lg::tile::launch_mrg_f64(const hgrid_tile *p) { return launch_potential<double2, TMRG>(p); }
