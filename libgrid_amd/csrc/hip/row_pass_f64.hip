#include "row_pass.hpp"

int lg::row::launch_f64(const hgrid_pass *p) { return launch_len<double2>(p); }
