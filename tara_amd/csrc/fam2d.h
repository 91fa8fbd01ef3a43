// Host interface of the 2D compressible families: isothermal hydro
// (derive2coh) and compressible MHD (derive2com).
#pragma once
#include "common.h"
#include "csh2d.h"  // EventTimer

namespace tara {

enum F2Mode { F2_RHS = 0, F2_AB2 = 1 };

// Plan + scratch of one (nx, ny) grid.  Device spectra are kx-fastest with the
// row padded to ld = Nh rounded up to 8: element (i, j) at j*ld + i; padding
// columns are kept at zero.  kx, ky follow the reference's expression
// 2 pi (i-1)/Lx with the caller's pi and box (src/derive2coh.f95:59-60).
struct F2Plan {
    int nx = 0, ny = 0, nh = 0, ld = 0;
    size_t fsz = 0;            // elements per field (ld * ny)
    double pi = 0, lx = 0, ly = 0;
    DevBuf a;                  // inverse-y-transformed fields
    DevBuf b;                  // products after the x pass
    DevBuf c, d, k;            // com only: first-round x output, d uy/dy before x, u / forcing spectra
    DevBuf sines;              // com only: the forcing's sin(kf x), sin(kf y) (per call)
    DevBuf kx, ky, imin;       // imin[j]: modes with i >= imin[j] are dealiased away
    DevBuf bad;                // one int: set when an AB2 update stores a NaN or Inf
    const double2* tw_y = nullptr;
    const double2* tw_x = nullptr;  // length nx, radix cap 4
};

struct CohPhys {
    double mux = 0, muy = 0, cs = 0;
};
struct ComPhys {
    double mu = 0, eta = 0, cs = 0, kf = 0, amp = 0;
};

// family: 0 = coh (3 fields), 1 = com (6 fields)
int f2_plan_init(F2Plan& p, int family, int nx, int ny, double pi, double lx, double ly);
// One RHS of st (device, padded) into out.
int coh_rhs(const F2Plan& p, const CohPhys& ph, double2* const st[3], double2* const out[3], hipStream_t s);
int com_rhs(const F2Plan& p, const ComPhys& ph, double2* const st[6], double2* const out[6], hipStream_t s);
// nsteps AB2 steps of st with history hist (f_{n-1} in, f_n out).  A step writes
// the fields that others of its workgroups still read to a second set and
// exchanges the pointers: coh state and history (st2, hist2), com momentum (st[1],
// st[2]; mom).  Timing classes: 0 the call's inverse y pass, 1 x (com: with the
// passes between), 2 forward y.
int coh_advance(const F2Plan& p, const CohPhys& ph, double2* st[3], double2* hist[3], double2* st2[3], double2* hist2[3],
                int nsteps, double dt, hipStream_t s, EventTimer* tm);
int com_advance(const F2Plan& p, const ComPhys& ph, double2* st[6], double2* mom[2], double2* const hist[6], int nsteps,
                double dt, hipStream_t s, EventTimer* tm);
// Pointwise updates over n complex elements: AB2, Euler, and the degenerate
// "RK4" / predictor-corrector forms of the coh steppers.
enum F2Point { F2P_AB2 = 0, F2P_EULER = 1, F2P_RK4_DEGEN = 2, F2P_PC_DEGEN = 3 };
int f2_pointwise(int kind, const double2* w, double2* wn, const double2* fo, const double2* fn, double dt, size_t n,
                 hipStream_t st);

}  // namespace tara
