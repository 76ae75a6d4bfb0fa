#include "row_pass.hpp"

int lg::row::launch_f32(const hgrid_pass *p) { return launch_len<float2>(p); }
