// Device pieces shared by the 2D incompressible passes (csh2d.hip: the passes of
// large grids and batches; csh2d_small.hip: those of grids too small to fill
// the chip): layouts, wavenumbers, the paired c2r and the stage update.
#pragma once
#include "common.h"
#include "csh2d.h"
#include "passes.h"
#include "rfft.h"

namespace tara {

// The register-resident transform of the y passes (csh_yem elements per thread).
template <int NY>
using RY = RF<NY, csh_yem(NY)>;

// Columns per workgroup of the y passes: at least 256 threads.
template <int N>
struct YShape {
    static constexpr int T = RY<N>::T;
    static constexpr int CB = T >= 256 ? 1 : 256 / T;
    static constexpr int NT = CB * T;
};
// Offset of element (kx = i, ky = j) in an 8-row-blocked intermediate.
__device__ __forceinline__ size_t blk8(int i, int j, int nh)
{
    return ((size_t)(j >> 3) * nh + i) * 8 + (j & 7);
}

// Offset of element (i, j) in the intermediates G0..G3: groups of 2^gs rows
// interleaved per kx, ld columns per group (CshPlan::gsh, CshPlan::gld).
// The groups follow Nx, which the x pass knows at compile time.  Nx = 4096, 2-row
// groups: a wave of the x pass reading two rows reads contiguous 32-byte pairs over
// consecutive kx.  Smaller Nx, 4-row groups.  Which columns an inverse y workgroup
// holds follows Ny (YiShape): at Ny = 4096 two, interleaved over the lanes, so that at
// 4096^2 their pairs of a row group are written together; else contiguous ones.
// Measured with the four fields themselves in G0..G3 and every column carried: 4096^2
// 0.195 ms inverse y + 0.276 ms x, against 0.186 + 0.311 ms with 4-row groups; 1024^2
// 0.0201 + 0.0186 ms, against 0.0236 + 0.0179 ms with 2-row groups and four interleaved
// columns.  (With one column per inverse-y workgroup at 4096^2, 4-row groups measured
// faster than 8-row (0.20, 0.39 ms), 2-row (0.25, 0.31) and plain row-major (0.34, 0.31).)
__device__ __forceinline__ size_t blkg(int i, int j, int ld, int gs)
{
    return ((size_t)(j >> gs) * ld + i) * (1 << gs) + (j & ((1 << gs) - 1));
}

// The state's support (CshPlan::band, hk): the dealiasing keeps the nonlinear
// term to kx < hk, and inside the circle imin; where a state is zero outside the
// circle (band flag of its run) it stays so, and the passes carry the circle only.
struct CshBand {
    static constexpr bool KNOWN = true;
    const int* band;   // per run; null: unknown
    const int* imin;
    int hk, nh;
    __device__ __forceinline__ bool limited(int run) const { return band && band[run] != 0; }
};

struct CshNoBand {
    static constexpr bool KNOWN = false;
};

inline CshBand csh_band(const CshPlan& p)
{
    return CshBand{csh_small(p) ? nullptr : p.band.as<int>(), p.imin.as<int>(), p.hk, p.nh};
}

// Tile of workgroup w of ntiles: the first nfirst tiles (those with more to do, or
// with anything to do) are spread over the XCDs first, the others after them.
__device__ __forceinline__ int csh_tile(int w, int nfirst, int ntiles)
{
    return w < nfirst ? xcd_remap(w, nfirst) : nfirst + xcd_remap(w - nfirst, ntiles - nfirst);
}

// derive2csh's ky: j-1 for j <= Ny/2, j-1-Ny above (exact integers, checked on the host).
template <int NY>
__device__ __forceinline__ double csh_ky(int j)
{
    return (double)(j < NY / 2 ? j : j - NY);
}

// Two real c2r transforms in one complex FFT: with X_a, X_b the Hermitian half
// spectra (kx = 0..M) of two real rows, Y[k] = X_a[k] + i X_b[k] over the full
// length Nx (X[Nx-k] = conj X[k]) transforms to y = x_a + i x_b.  The y passes
// store P = X_a + i X_b and Q = X_a - i X_b, so that Y[k] = P[k] up to M and
// conj Q[Nx-k] above: one load an element, where X_a and X_b themselves were each
// loaded at k and again at Nx-k.  At kx = 0 and M the imaginary parts of X_a and
// X_b are dropped, as FFTW's c2r does: Y = (P + conj Q)/2.  Columns kx >= lim are
// zero and not read.  Registers end with y at rf_final_idx<NX> positions.
// A pair shares its rounding error, so fields of like size are paired.
// sq: the row as the thread sees it (RfSeq, RfWide).  BAND false: lim is nh, and
// the loads go unguarded.
template <int NX, int EM, bool BAND, class SQ>
__device__ __forceinline__ void x_c2r_pair(const double2* gp, const double2* gq, int j, int lim, const SQ& sq,
                                           const double2* tw, double2 (&v)[RF<NX, EM>::E])
{
    constexpr int M = NX / 2, E = RF<NX, EM>::E;
    constexpr int LD = csh_gld(M + 1), GS = csh_gshift(M + 1);
    static_assert(rf_in_idx<NX, 1, EM>(1, E / 2) == 1 + M, "first pass of full radix");
    double2 q0 = make_double2(0.0, 0.0), pm = q0;
    if (sq.t == 0) {
        q0 = gq[blkg(0, j, LD, GS)];
        if (!BAND || M < lim) pm = gp[blkg(M, j, LD, GS)];
    }
#pragma unroll
    for (int e = 0; e < E; ++e) {
        const int k = rf_first_idx<NX, EM>(sq.t, e);
        const int kk = e < E / 2 ? k : NX - k;
        v[e] = make_double2(0.0, 0.0);
        if (!BAND || kk < lim) v[e] = (e < E / 2 ? gp : gq)[blkg(kk, j, LD, GS)];
        if (e >= E / 2) v[e].y = -v[e].y;
    }
    if (sq.t == 0) {
        v[0] = make_double2(0.5 * (v[0].x + q0.x), 0.5 * (v[0].y - q0.y));
        v[E / 2] = make_double2(0.5 * (v[E / 2].x + pm.x), 0.5 * (v[E / 2].y + pm.y));
    }
    sq.template fft<+1>(v, tw);
}

struct YfwdArgs {
    const double2* h;      // nonlinear term, x-transformed
    const double2* ws;     // stage input omega_s (viscous term)
    double2* base;         // AB2: state (in/out); RK4: omega_n (stage 4: out)
    double2* aux;          // AB2: history f_{n-1} (in/out); RK4: accumulator
    double2* next;         // RK4: next stage input (out); RHS mode: f (out)
    size_t si, sj;         // element (i, j) of ws, base, aux, next at i*si + j*sj (small grids; else ky-major)
    const int* imin;       // dealias: modes with i >= imin[j] drop the nonlinear term
    int nh;
    double nu, dt;
    double alpha, lam;     // screened form: alpha * NL, viscous term on k^2 ws/(k^2 + lam)
    int screened;
    size_t bs;             // batched runs: field stride per run (blockIdx.y)
    const double* nus;     // batched runs: viscosity per run (null: nu)
    int* bad;              // per run: set to 1 when a new state value is not finite (AB2, RK4 stage 4)
};

// The stage update of one mode: from the masked nonlinear term nl, the stage
// input ws and k^2, the value wn the stage produces (RHS: f; AB2, RK4 stage 4:
// the new state; other RK4 stages: the next stage's input) and, where the mode
// keeps one, the new auxiliary value av (AB2: f; RK4: the accumulator).
template <int MODE>
__device__ __forceinline__ void csh_update(const YfwdArgs& a, size_t q, bool origin, double2 nl, double2 ws, double k2,
                                           double2* wn, double2* av)
{
    const double vk = a.nu * k2;
    double2 f;
    if (a.screened) {
        // derive2css.f95:118-130: -(alpha (NLx + NLy) + nu k^2 omega_d)
        const double den = k2 + a.lam;
        const double2 wd = origin ? make_double2(0.0, 0.0) : make_double2(k2 * (ws.x / den), k2 * (ws.y / den));
        f = make_double2(-(a.alpha * nl.x + vk * wd.x), -(a.alpha * nl.y + vk * wd.y));
    } else {
        f = make_double2(-(nl.x + vk * ws.x), -(nl.y + vk * ws.y));
    }
    if (MODE == CSH_RHS) {
        *wn = f;
    } else if (MODE == CSH_AB2) {
        const double2 fo = a.aux[q];
        *wn = make_double2(ws.x + (1.5 * f.x - 0.5 * fo.x) * a.dt, ws.y + (1.5 * f.y - 0.5 * fo.y) * a.dt);
        *av = f;
    } else if (MODE == CSH_RK4_1) {
        const double c6 = a.dt / 6.0, c2 = 0.5 * a.dt;
        *wn = make_double2(ws.x + c2 * f.x, ws.y + c2 * f.y);
        *av = make_double2(ws.x + c6 * f.x, ws.y + c6 * f.y);
    } else if (MODE == CSH_RK4_2 || MODE == CSH_RK4_3) {
        const double c3 = a.dt / 3.0, cn = (MODE == CSH_RK4_2) ? 0.5 * a.dt : a.dt;
        const double2 w0 = a.base[q], acc = a.aux[q];
        *wn = make_double2(w0.x + cn * f.x, w0.y + cn * f.y);
        *av = make_double2(acc.x + c3 * f.x, acc.y + c3 * f.y);
    } else {  // CSH_RK4_4
        const double c6 = a.dt / 6.0;
        const double2 acc = a.aux[q];
        *wn = make_double2(acc.x + c6 * f.x, acc.y + c6 * f.y);
    }
}

// Stores what csh_update formed; false if a new state value is not finite.
template <int MODE>
__device__ __forceinline__ bool csh_store(const YfwdArgs& a, size_t q, double2 wn, double2 av)
{
    if (MODE == CSH_AB2 || MODE == CSH_RK4_4)
        a.base[q] = wn;
    else
        a.next[q] = wn;
    if (MODE != CSH_RHS && MODE != CSH_RK4_4) a.aux[q] = av;
    return (MODE != CSH_AB2 && MODE != CSH_RK4_4) || (isfinite(wn.x) && isfinite(wn.y));
}

}  // namespace tara
