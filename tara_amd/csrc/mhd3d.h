// Host interface of the 3D compressible isothermal MHD pipeline.
#pragma once
#include <vector>

#include "common.h"
#include "csh2d.h"  // EventTimer

namespace tara {

enum MhdMode { MHD_RHS = 0, MHD_AB2 = 1 };

// Plan + scratch of one (nx, ny, nz) grid.  Device spectra use the reference's
// kx-fastest layout with the row length padded to ld = Nh rounded up to 8,
// element (i, j, k) at (k*Ny + j)*ld + i; padding columns are kept at zero (those of
// b, in which host copies pack their rows, where a live tile reaches past Nh).
struct MhdPlan {
    int nx = 0, ny = 0, nz = 0, nh = 0, ld = 0;
    double lx = 0, ly = 0, lz = 0, mu = 0, eta = 0, cs = 0;
    size_t fsz = 0;            // elements per field (ld * ny * nz)
    DevBuf a;                  // 7 fields: inverse-transformed state (rho, rho u, B)
    DevBuf az;                 // stepping only (mhd_plan_stepping): 7 fields, the state's inverse z transform
    DevBuf b;                  // 12 fields: u (3), momentum fluxes (6), induction fluxes (3)
    DevBuf kx, ky, kz, imin;
    // The modes that the dealiasing leaves alive: no other mode ever changes.
    int ktiles = 0;            // tiles of 8 kx columns that hold one
    int nlive = 0;             // tiles (ky row j, kx tile x; id j*(ld/8) + x) that hold one, listed in live
    DevBuf live;               // int[nlive]
    DevBuf yskip;              // int2[ktiles]: rows [x, y) of a kx tile hold none
    DevBuf bad;                // int: set when an AB2 step's new state holds a non-finite value
    const double2* tw_y = nullptr;
    const double2* tw_z = nullptr;
    const double2* tw_z4 = nullptr;  // radix cap 4 (z forward pass at 4 elements per thread)
    const double2* tw_x = nullptr;  // length nx, radix cap 4 (x pass)
};

int mhd_plan_init(MhdPlan& p, int nx, int ny, int nz, double lx, double ly, double lz, double mu, double eta,
                  double cs);
// Allocates what mhd_advance needs beyond a right-hand side.
int mhd_plan_stepping(MhdPlan& p);
// nsteps AB2 steps of st with history hist (f_{n-1} in, f_n out; zero outside
// the live modes).  A step writes the new momentum (st[1..3]) to mom[0..2] and
// exchanges the pointers; both sets hold the same values outside the live modes.
// Timing classes as mhd_rhs_stage.
int mhd_advance(const MhdPlan& p, double2* st[7], double2* mom[3], double2* const hist[7], int nsteps, double dt,
                hipStream_t s, EventTimer* tm);
// One right-hand side on the 7 live state fields st[0..6] = rho, rho ux, rho uy,
// rho uz, Bx, By, Bz (device, padded layout), written to out[0..6], which the
// caller has zeroed once: only tiles that hold a live mode are written.  Timing
// classes: 0 inverse z and y, 1 x, 2 forward y, 3 forward z and assembly.
int mhd_rhs_stage(const MhdPlan& p, double2* const st[7], double2* const out[7], hipStream_t s, EventTimer* tm);

}  // namespace tara
