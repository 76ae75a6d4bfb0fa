#include "row_pass.hpp"

int lg::row::launch_f32s_f64(const hgrid_pass *p) { return launch_len<double2, float2>(p); }
