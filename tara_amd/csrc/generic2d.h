// derive2csh / derive2css on grids the fused passes do not take (generic2d.hip).
#pragma once
#include "csh2d.h"

namespace tara {

// Whether the fused csh2d passes take an nx x ny grid.
bool csh_fast_grid(int nx, int ny);
// out = the right-hand side of the nh x ny host spectrum in, or (step) one RK4
// step of size dt from it.  Synchronous, on the null stream.
int gen_csh_host(int nx, int ny, const CshPhys& ph, const double* in, double* out, bool step, double dt);

}  // namespace tara
