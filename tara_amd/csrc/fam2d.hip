// 2D compressible families on gfx950: the right-hand sides of
// src/derive2coh.f95 (isothermal hydro: n, ux, uy) and src/derive2com.f95
// (compressible MHD with forcing: rho, rho ux, rho uy, E, Bx, By), their AB2
// updates (src/ab2coh.f95, src/ab2com.f95) and the Euler-type steppers of the
// coh family.
//
// Device layout: kx-fastest, row padded to ld (multiple of 8), element (i, j)
// at j*ld + i.  Grids of 16..256 a side, one at a time, never fill the chip: a
// pass takes as long as its longest chain of loads and transforms, so every
// transform has threads of its own and a step has as few passes as its data
// flow allows.  Sweeps per right-hand side:
//   coh: 1 k_f2_prep   per tile of 8 kx columns: spectral multiply (1, i ky,
//                      ky^2) of n, ux, uy and the backward y FFT -> A (8 fields)
//        2 k_coh_x     per x row: the 13 c2r of derive2coh.f95:92-129 as 7
//                      paired complex FFTs side by side (x derivatives i kx,
//                      kx^2 are applied here, where kx is constant along the
//                      completed y transform), the real-space terms of :131-167
//                      combined into three sums, 2 paired forward FFTs -> B
//        3 k_coh_yfwd  forward y FFT, circular dealias on every term
//                      (:201-242), negate (:246-258), RHS out, or AB2 in place
//                      and pass 1 of the new state
//      The reference transforms the nine real-space terms separately and sums
//      the masked spectra (:246-252); the sums are formed before one transform
//      each, which is the same linear map.
//   com: 1 k_f2_prep   backward y FFT of the 6 state fields -> A
//        2 k_com_x1    rho, rho u -> u = rho u/rho and the forcing
//                      (derive2com.f95:88-117), forward x -> C (4 fields)
//        3 k_com_mid   forward y of u, F -> K (ux_k, uy_k, Fx_k, Fy_k), and the
//                      backward y of i ky uy_k -> D (:124-168).  (i kx ux_k needs
//                      no y transform: back in y it is i kx C.)
//        4 k_com_x2    8 c2r (state + the two derivatives), the fluxes of
//                      :180-214, 7 distinct forward transforms -> B
//        5 k_com_yfwd  forward y, i k . flux, k^2 terms, dealias, forcing, assembly
//                      (:255-420), RHS out, or AB2 and pass 1 of the new state
// Pass 1 runs on its own once per advance call.
// Measured at 256^2 (AB2 step, kernel times): com 7 + 8.1 + 14.6 + 12.8 + 32.8 us
// with each pass's transforms one after another, now 4.6 + 6.7 + 6.5 + 12.5; coh
// 10.4 + 7.0.  What is left: of each pass about 2.2 us is what any kernel takes
// and 2 us its first loads and last stores, served past the L2 of another XCD;
// 4 instead of 8 elements per thread changed nothing (13.1 against 12.6 us for
// the last com pass).
#include <cmath>
#include <utility>
#include <vector>

#include "colpass.h"
#include "fam2d.h"

namespace tara {

// spectral multipliers of the prep pass
enum : int { MUL_1 = 0, MUL_IKY = 1, MUL_KY2 = 2, MUL_IKX = 3, MUL_KX2 = 4 };

// (0, 1) k z as the reference forms it: (-(k z.y), k z.x)
__device__ __forceinline__ double2 f2_ik(double k, double2 z) { return make_double2(-(k * z.y), k * z.x); }
__device__ __forceinline__ double2 f2_k2(double k, double2 z)
{
    const double kk = k * k;
    return make_double2(kk * z.x, kk * z.y);
}
// Without branches: a kind known only at run time must not stand between one
// element's load and the next (a switch here cost a load latency per element,
// 8.2 against 6.0 us for pass 1 at 256^2).
__device__ __forceinline__ double2 f2_mul(int kind, double kx, double ky, double2 z)
{
    const bool im = kind == MUL_IKY || kind == MUL_IKX;
    const double k = kind == MUL_IKY || kind == MUL_KY2 ? ky : kx;
    const double s = kind == MUL_1 ? 1.0 : im ? k : k * k;
    const double a = s * z.x, b = s * z.y;
    return im ? make_double2(-b, a) : make_double2(a, b);
}

// ------------------------------------------------------------ pass 1 (prep)
struct PrepArgs {
    const double2* src[8];
    double2* dst[8];
    int kind[8];
    const double* kx;
    const double* ky;
    int ld;
};

template <int NY>
__global__ __launch_bounds__(CShape<NY>::NT) void k_f2_prep(PrepArgs a, const double2* tw)
{
    using S = CShape<NY>;
    constexpr int E = RF<NY>::E;
    __shared__ double2 lds[8 * S::LP];
    const int c = threadIdx.x % 8, t = threadIdx.x / 8;
    const int i = xcd_remap(blockIdx.x, gridDim.x) * 8 + c;
    const int o = blockIdx.y;
    const double2* src = a.src[o] + i;
    const int kind = a.kind[o];
    const double kxv = a.kx[i];
    double2 v[E];
    double kyv[E];
#pragma unroll
    for (int e = 0; e < E; ++e) {
        const int j = rf_first_idx<NY>(t, e);
        v[e] = src[(size_t)j * a.ld];
        kyv[e] = a.ky[j];
    }
#pragma unroll
    for (int e = 0; e < E; ++e) v[e] = f2_mul(kind, kxv, kyv[e], v[e]);
    rf_fft<NY, +1>(v, t, lds + c * S::LP, tw);
    double2* dst = a.dst[o] + i;
#pragma unroll
    for (int e = 0; e < E; ++e) dst[(size_t)rf_final_idx<NY>(t, e) * a.ld] = v[e];
}

// ------------------------------------------------------------ x-pass helpers
// One x row per NG groups of T = NX/4 lanes (4 complex elements per lane): each
// group transforms one pair of fields, the real fields meet in LDS, and each
// group forms and transforms one pair of results.  A group sits in one
// wavefront, so the exchanges between FFT passes need only wave-level ordering.
template <int NX, int NG, int NR>
struct FXShape {
    static constexpr int E = RF<NX, 4>::E;
    static constexpr int T = RF<NX, 4>::T;
    static_assert(64 % T == 0, "a group must not straddle wavefronts");
    static constexpr int RB = NG * T >= 64 ? 1 : 64 / (NG * T);  // rows per workgroup
    static constexpr int NT = RB * NG * T;
    static constexpr int LP = RF<NX, 4>::LDS;                    // exchange buffer per group
    static constexpr int LDS = RB * NG * LP + RB * NR * NX / 2;  // and NR real rows
};

// Two real c2r rows in one complex FFT: Y = X_a + i X_b over the full length
// (X[Nx-k] = conj X[k]), with the x multipliers ka / kb applied to the stored
// half spectra first (row a also times sa) and the imaginary parts at kx = 0 and
// Nx/2 dropped as FFTW's c2r does.  fb may be null (second row zero).  The
// rows, times norm, go to ra and rb (null: not wanted).
template <int NX>
__device__ __forceinline__ void f2_c2r_pair(const double2* fa, int ka, double sa, const double2* fb, int kb,
                                            const double* kx, double norm, int t, double2* xl, const double2* tw,
                                            double* ra, double* rb)
{
    constexpr int M = NX / 2;
    double2 v[RF<NX, 4>::E];
#pragma unroll
    for (int e = 0; e < RF<NX, 4>::E; ++e) {
        const int k = rf_first_idx<NX, 4>(t, e);
        const int kk = k <= M ? k : NX - k;
        const double kxv = kx[kk];
        double2 u = f2_mul(ka, kxv, 0.0, fa[kk]);
        double2 w = fb ? f2_mul(kb, kxv, 0.0, fb[kk]) : make_double2(0.0, 0.0);
        u = make_double2(sa * u.x, sa * u.y);
        if (kk == 0 || kk == M) {
            u.y = 0.0;
            w.y = 0.0;
        }
        if (k > M) {
            u.y = -u.y;
            w.y = -w.y;
        }
        v[e] = make_double2(u.x - w.y, u.y + w.x);
    }
    rf_fft<NX, +1, 4, true>(v, t, xl, tw);
#pragma unroll
    for (int e = 0; e < RF<NX, 4>::E; ++e) {
        const int n = rf_final_idx<NX, 4>(t, e);
        ra[n] = v[e].x * norm;
        if (rb) rb[n] = v[e].y * norm;
    }
}

// Forward x transform of two real rows held at rf_first_idx positions
// (unnormalised r2c, FFTW's e^{-i}), split by the two-for-one identity
// A[k] = (Z[k] + conj Z[N-k])/2, B[k] = (Z[k] - conj Z[N-k])/(2i).
template <int NX>
__device__ __forceinline__ void f2_r2c_pair(double2* oa, double2* ob, double2 (&v)[RF<NX, 4>::E], int t, double2* xl,
                                            const double2* tw)
{
    constexpr int E = RF<NX, 4>::E, T = RF<NX, 4>::T, M = NX / 2;
    rf_fft<NX, -1, 4, true>(v, t, xl, tw);
#pragma unroll
    for (int e = 0; e < E; ++e) xl[rf_pad(rf_final_idx<NX, 4>(t, e))] = v[e];
    rf_sync<true>();
    for (int k = t; k <= M; k += T) {
        const double2 z = xl[rf_pad(k)], zm = xl[rf_pad(k == 0 ? 0 : NX - k)];
        oa[k] = make_double2(0.5 * (z.x + zm.x), 0.5 * (z.y - zm.y));
        if (ob) ob[k] = make_double2(0.5 * (z.y + zm.y), -0.5 * (z.x - zm.x));
    }
}

struct F2XArgs {
    const double2* a;  // input fields, field stride fs
    const double2* c;  // com: first-round x output
    const double2* d;  // com: i ky uy_k back in y
    double2* b;        // output fields
    size_t fs;
    const double* kx;
    int ld, ny;
    double norm;       // 1 / (Nx Ny)
    double p0, p1, p2;      // family constants
    const double* sines;    // com: k_com_sines
};

#define F2X_PROLOGUE(NX, NG, NR)                                                          \
    using S = FXShape<NX, NG, NR>;                                                        \
    constexpr int E = S::E;                                                               \
    __shared__ double2 lds[S::LDS];                                                       \
    const int t = threadIdx.x % S::T, g = (threadIdx.x / S::T) % NG;                      \
    const int rr = threadIdx.x / (S::T * NG);                                             \
    const int row = xcd_remap(blockIdx.x, gridDim.x) * S::RB + rr;                        \
    const size_t ro = (size_t)row * x.ld;                                                 \
    double2* xl = lds + (threadIdx.x / S::T) * S::LP;                                     \
    double* R = reinterpret_cast<double*>(lds + S::RB * NG * S::LP) + (size_t)rr * NR * NX; \
    auto F = [&](int f) { return x.a + (size_t)f * x.fs + ro; };

// ------------------------------------------------------------------ coh x pass
// A: 0 n, 1 ux, 2 uy, 3 i ky n, 4 i ky ux, 5 i ky uy, 6 ky^2 ux, 7 ky^2 uy.
// p0 = mux, p1 = muy, p2 = CS^2.  B: 0 NLn, 1 NLx + visc + CS^2 Px, 2 the y twin.
enum { RN, RNX, RUX, RUXX, RUY, RUYX, R2UXX, R2UYX, RNY, RUXY, RUYY, R2UXY, R2UYY, RCOH };
template <int NX>
__global__ __launch_bounds__((FXShape<NX, 7, RCOH>::NT)) void k_coh_x(F2XArgs x, const double2* tw)
{
    F2X_PROLOGUE(NX, 7, RCOH)
    // (n, dn/dx) (ux, dux/dx) (uy, duy/dx) (kx^2 ux, kx^2 uy) (dn/dy, dux/dy)
    // (duy/dy, ky^2 ux) (ky^2 uy, -)
    const double2* fa = F(g < 3 ? g : g == 3 ? 1 : 2 * g - 5);
    const double2* fb = g < 3 ? fa : g == 3 ? F(2) : g == 6 ? nullptr : F(2 * g - 4);
    f2_c2r_pair<NX>(fa, g == 3 ? MUL_KX2 : MUL_1, 1.0, fb, g < 3 ? MUL_IKX : g == 3 ? MUL_KX2 : MUL_1, x.kx, x.norm, t,
                    xl, tw, R + 2 * g * NX, g == 6 ? nullptr : R + (2 * g + 1) * NX);
    __syncthreads();
    if (g >= 2) return;  // no barrier follows
    double2 v[E];
#pragma unroll
    for (int e = 0; e < E; ++e) {
        const int q = rf_first_idx<NX, 4>(t, e);
        auto r = [&](int f) { return R[f * NX + q]; };
        const double n = r(RN), ux = r(RUX), uy = r(RUY), dnx = r(RNX), dny = r(RNY);
        // NLx + (mux Visc_xx + muy Visc_xy) + CS^2 Px, derive2coh.f95:248-249
        if (g == 0) {
            const double nln = (ux * dnx + uy * dny) + n * (r(RUXX) + r(RUYY));
            const double vis = x.p0 * (r(R2UXX) / n) + x.p1 * (r(R2UXY) / n);
            v[e] = make_double2(nln, ((ux * r(RUXX) + uy * r(RUXY)) + vis) + x.p2 * (dnx / n));
        } else {
            const double vis = x.p0 * (r(R2UYX) / n) + x.p1 * (r(R2UYY) / n);
            v[e] = make_double2(((ux * r(RUYX) + uy * r(RUYY)) + vis) + x.p2 * (dny / n), 0.0);
        }
    }
    double2* B0 = x.b + ro;
    f2_r2c_pair<NX>(g == 0 ? B0 : B0 + 2 * x.fs, g == 0 ? B0 + x.fs : nullptr, v, t, xl, tw);
}

// ------------------------------------------------------------------ com x passes
// sin(kf x(i)), i < nx, then sin(kf y(j)), j < ny: the forcing's factors, once per
// call (a sine in k_com_x1 costs each row about 1 us).
__global__ void k_com_sines(double* s, int nx, int ny, double kf, double dx, double dy)
{
    const int n = blockIdx.x * blockDim.x + threadIdx.x;
    if (n < nx + ny) s[n] = sin(kf * (n < nx ? (double)n * dx : (double)(n - nx) * dy));
}

// First round.  A: 0 rho, 1 rho ux, 2 rho uy.  p0 = A (forcing amplitude).
// C: 0 ux, 1 uy, 2 Fx, 3 Fy (x-transformed).
template <int NX>
__global__ __launch_bounds__((FXShape<NX, 2, 3>::NT)) void k_com_x1(F2XArgs x, const double2* tw)
{
    F2X_PROLOGUE(NX, 2, 3)
    if (g == 0)
        f2_c2r_pair<NX>(F(0), MUL_1, 1.0, F(1), MUL_1, x.kx, x.norm, t, xl, tw, R, R + NX);
    else
        f2_c2r_pair<NX>(F(2), MUL_1, 1.0, nullptr, MUL_1, x.kx, x.norm, t, xl, tw, R + 2 * NX, nullptr);
    const double sy = x.sines[NX + row];
    double sx[E];
#pragma unroll
    for (int e = 0; e < E; ++e) sx[e] = x.sines[rf_first_idx<NX, 4>(t, e)];
    __syncthreads();
    double2 v[E];
#pragma unroll
    for (int e = 0; e < E; ++e) {
        const int q = rf_first_idx<NX, 4>(t, e);
        const double rho = R[q];
        // Fx = -rho A sin(kf y), Fy = +rho A sin(kf x)  (derive2com.f95:109-110)
        if (g == 0)
            v[e] = make_double2(R[NX + q] / rho, R[2 * NX + q] / rho);
        else
            v[e] = make_double2(-(rho * x.p0 * sy), rho * x.p0 * sx[e]);
    }
    double2* C0 = x.b + (size_t)(2 * g) * x.fs + ro;
    f2_r2c_pair<NX>(C0, C0 + x.fs, v, t, xl, tw);
}

// Second round.  A: 0 rho, 1 rho ux, 2 rho uy, 3 E, 4 Bx, 5 By; C: 0 ux; D: i ky
// uy_k (y-inverted).  p0 = CS^2, p1 = eta.  B: 0 Mom_x_1, 1 Mom_x_2 (= Mom_y_1),
// 2 Mom_y_2, 3 Energy_x, 4 Energy_y, 5 E_Visc, 6 Mag_x (Mag_y = -Mag_x).
template <int NX>
__global__ __launch_bounds__((FXShape<NX, 4, 8>::NT)) void k_com_x2(F2XArgs x, const double2* tw)
{
    F2X_PROLOGUE(NX, 4, 8)
    // (rho, rho ux) (rho uy, E) (Bx, By) (dux/dx, duy/dy); i kx ux back in y is
    // i kx C times Ny, the y transforms' factor (exact: Ny is a power of two)
    if (g < 3)
        f2_c2r_pair<NX>(F(2 * g), MUL_1, 1.0, F(2 * g + 1), MUL_1, x.kx, x.norm, t, xl, tw, R + 2 * g * NX,
                        R + (2 * g + 1) * NX);
    else
        f2_c2r_pair<NX>(x.c + ro, MUL_IKX, (double)x.ny, x.d + ro, MUL_1, x.kx, x.norm, t, xl, tw, R + 6 * NX,
                        R + 7 * NX);
    __syncthreads();
    double2 v[E];
#pragma unroll
    for (int e = 0; e < E; ++e) {
        const int q = rf_first_idx<NX, 4>(t, e);
        const double rho = R[q], rux = R[NX + q], ruy = R[2 * NX + q], en = R[3 * NX + q], bx = R[4 * NX + q],
                     by = R[5 * NX + q], dudx = R[6 * NX + q], dvdy = R[7 * NX + q];
        const double ux = rux / rho, uy = ruy / rho;
        const double b2 = bx * bx + by * by;
        const double p = x.p0 * rho;
        // The reference sets d_Bx_dy and d_By_dx from the already normalised
        // d_ux_dx and d_uy_dy, divided by Nx*Ny once more (derive2com.f95:186-187).
        const double dbxdy = dudx * x.norm, dbydx = dvdy * x.norm;
        const double curl = dbydx - dbxdy;
        if (g == 0) {  // momentum fluxes (derive2com.f95:196-199)
            v[e] = make_double2(((rux * ux + p) + b2 / 2.0) - bx * bx, rux * uy - bx * by);
        } else if (g == 1) {
            const double ex = (((en + p) + b2 / 2.0) * ux - (ux * bx) * bx) - (uy * bx) * by;
            v[e] = make_double2(((ruy * uy + p) + b2 / 2.0) - by * by, ex - (x.p1 * by) * curl);
        } else if (g == 2) {
            const double ey = (((en + p) + b2 / 2.0) * uy - (ux * bx) * by) - (uy * by) * by;
            const double dv = dudx + dvdy;
            v[e] = make_double2(ey + (x.p1 * bx) * curl, dv * dv);
        } else {
            v[e] = make_double2(uy * bx - by * ux, 0.0);  // Mag_x (:208)
        }
    }
    double2* B0 = x.b + (size_t)(2 * g) * x.fs + ro;
    f2_r2c_pair<NX>(B0, g < 3 ? B0 + x.fs : nullptr, v, t, xl, tw);
}

// ------------------------------------------------------- y forward helpers
struct F2YArgs {
    const double2* b;      // x-pass output fields
    const double2* c;      // com: first-round x output (ux, uy, Fx, Fy)
    double2* d;            // com: i ky uy_k back in y (out of k_com_mid)
    double2* k;            // com: ux_k, uy_k, Fx_k, Fy_k
    double2* a;            // inverse-y-transformed fields of the new state (with INV)
    size_t fs;
    const double2* st[6];  // state
    double2* sn[6];        // F2_AB2: new state (coh, and com's momentum: other buffers than st)
    const double2* ho[6];  // F2_AB2: history f_{n-1}
    double2* out[6];       // RHS (F2_RHS) or new history f_n (coh: other buffers than ho)
    const double* kx;
    const double* ky;
    const int* imin;
    int ld;
    double dt, mu, eta;
    int* bad;              // set when an AB2 update stores a non-finite value
};

template <int NY>
__device__ __forceinline__ void f2_yfft_fwd(const double2* src, int i, int ld, int t, double2* xl, const double2* tw,
                                            double2 (&v)[RF<NY>::E])
{
#pragma unroll
    for (int e = 0; e < RF<NY>::E; ++e) v[e] = src[(size_t)rf_first_idx<NY>(t, e) * ld + i];
    rf_fft<NY, -1>(v, t, xl, tw);
}

// AB2: the new state from f and the history at q (which takes f).
__device__ __forceinline__ double2 f2_ab2(double2 w, double2 f, double2 fo, double dt)
{
    return make_double2(w.x + (1.5 * f.x - 0.5 * fo.x) * dt, w.y + (1.5 * f.y - 0.5 * fo.y) * dt);
}

// ------------------------------------------------------------ coh y forward
// One tile of 8 kx columns per workgroup: a state field's forward transform and
// update and, with INV, one backward transform of the new state (1, i ky, and
// for ux, uy ky^2: blockIdx.y as A's fields, the first three storing the
// update).  Several workgroups read a field's state and history: the new ones go
// to other buffers.  Stores come last: a twiddle load issued after a store would
// wait for it (one in-order counter).
template <int NY, int MODE, bool INV>
__global__ __launch_bounds__(CShape<NY>::NT) void k_coh_yfwd(F2YArgs a, const double2* tw)
{
    using S = CShape<NY>;
    constexpr int E = RF<NY>::E;
    __shared__ double2 lds[8 * S::LP];
    const int c = threadIdx.x % 8, t = threadIdx.x / 8;
    const int o = blockIdx.y, f = o < 6 ? o % 3 : o - 5;
    const int i = xcd_remap(blockIdx.x, gridDim.x) * 8 + c;
    double2* xl = lds + c * S::LP;
    double2 v[E], r[E], w[E], fo[E];
    double kyf[E];  // ky at the backward transform's inputs
    int im[E];
#pragma unroll
    for (int e = 0; e < E; ++e) {
        im[e] = a.imin[rf_final_idx<NY>(t, e)];
        kyf[e] = INV ? a.ky[rf_first_idx<NY>(t, e)] : 0.0;
    }
    if (MODE == F2_AB2) {  // fetched first: one latency with the transform's input
#pragma unroll
        for (int e = 0; e < E; ++e) {
            const size_t q = (size_t)rf_final_idx<NY>(t, e) * a.ld + i;
            w[e] = a.st[f][q];
            fo[e] = a.ho[f][q];
        }
    }
    f2_yfft_fwd<NY>(a.b + (size_t)f * a.fs, i, a.ld, t, xl, tw, v);
#pragma unroll
    for (int e = 0; e < E; ++e) {
        r[e] = i < im[e] ? make_double2(-v[e].x, -v[e].y) : make_double2(-0.0, -0.0);
        v[e] = w[e] = MODE == F2_RHS ? r[e] : f2_ab2(w[e], r[e], fo[e], a.dt);
    }
    if constexpr (INV) {
        rf_final_to_first<NY>(v, t, xl);
#pragma unroll
        for (int e = 0; e < E; ++e) v[e] = f2_mul(o < 3 ? MUL_1 : o < 6 ? MUL_IKY : MUL_KY2, 0.0, kyf[e], v[e]);
        rf_fft<NY, +1>(v, t, xl, tw);
        double2* d = a.a + (size_t)o * a.fs + i;
#pragma unroll
        for (int e = 0; e < E; ++e) d[(size_t)rf_final_idx<NY>(t, e) * a.ld] = v[e];
    }
    if (o >= 3) return;
#pragma unroll
    for (int e = 0; e < E; ++e) {
        const size_t q = (size_t)rf_final_idx<NY>(t, e) * a.ld + i;
        a.out[f][q] = r[e];
        if (MODE == F2_AB2) {
            a.sn[f][q] = w[e];
            if (!(isfinite(w[e].x) && isfinite(w[e].y))) *a.bad = 1;
        }
    }
}

// ------------------------------------------------------------ com middle pass
// Forward y of ux, uy, Fx, Fy (-> K, the reference's ux_k, uy_k, Fx_k, Fy_k), one
// field per workgroup; uy's goes on through the backward y of i ky uy_k (-> D).
template <int NY>
__global__ __launch_bounds__(CShape<NY>::NT) void k_com_mid(F2YArgs a, const double2* tw)
{
    using S = CShape<NY>;
    constexpr int E = RF<NY>::E;
    __shared__ double2 lds[8 * S::LP];
    const int c = threadIdx.x % 8, t = threadIdx.x / 8, f = blockIdx.y;
    const int i = xcd_remap(blockIdx.x, gridDim.x) * 8 + c;
    double2* xl = lds + c * S::LP;
    double2 v[E];
    double kyv[E];
#pragma unroll
    for (int e = 0; e < E; ++e) kyv[e] = a.ky[rf_final_idx<NY>(t, e)];
    f2_yfft_fwd<NY>(a.c + (size_t)f * a.fs, i, a.ld, t, xl, tw, v);
    double2 u[E];
#pragma unroll
    for (int e = 0; e < E; ++e) u[e] = v[e];
    if (f == 1) {  // the same for the whole workgroup
#pragma unroll
        for (int e = 0; e < E; ++e) v[e] = f2_ik(kyv[e], v[e]);
        rf_final_to_first<NY>(v, t, xl);
        rf_fft<NY, +1>(v, t, xl, tw);
#pragma unroll
        for (int e = 0; e < E; ++e) a.d[(size_t)rf_final_idx<NY>(t, e) * a.ld + i] = v[e];
    }
    double2* kf = a.k + (size_t)f * a.fs + i;
#pragma unroll
    for (int e = 0; e < E; ++e) kf[(size_t)rf_final_idx<NY>(t, e) * a.ld] = u[e];
}

// ------------------------------------------------------------ com y forward
// One state field of one tile of 8 kx columns per workgroup (the six fields of a
// tile next to each other on one XCD): its forward transforms, update and, with
// INV, the backward transform of the new field.  The density's right-hand side
// needs the momentum of the step's start: the new momentum goes to other buffers.
template <int NY, int MODE, bool INV>
__global__ __launch_bounds__(CShape<NY>::NT) void k_com_yfwd(F2YArgs a, const double2* tw)
{
    using S = CShape<NY>;
    constexpr int E = RF<NY>::E;
    __shared__ double2 lds[8 * S::LP];
    const int c = threadIdx.x % 8, t = threadIdx.x / 8;
    const int id = xcd_remap(blockIdx.x, gridDim.x), fld = id % 6;
    const int i = (id / 6) * 8 + c;
    double2* xl = lds + c * S::LP;
    const double kxv = a.kx[i];
    double2 v[E], r[E];
    auto pos = [&](int e) { return (size_t)rf_final_idx<NY>(t, e) * a.ld + i; };
    double kyv[E];
    bool keep[E];
#pragma unroll
    for (int e = 0; e < E; ++e) {
        kyv[e] = a.ky[rf_final_idx<NY>(t, e)];
        keep[e] = i < a.imin[rf_final_idx<NY>(t, e)];
    }
    auto msk = [&](int e, double2 z) { return keep[e] ? z : make_double2(0.0, 0.0); };
    // masked -(kx^2 + ky^2) w, summed as the reference does
    auto k2 = [&](int e, double2 w) {
        const double2 p = f2_k2(kxv, w), q = f2_k2(kyv[e], w);
        return msk(e, make_double2(p.x + q.x, p.y + q.y));
    };
    // r = -i k . flux: rho u: Mom_1, Mom_2; E: Energy_x, Energy_y and mu E_Visc;
    // Bx: i ky Mag_x; By: i kx Mag_y, Mag_y = -Mag_x.  Everything is fetched
    // first (one latency for all) and stored last (see k_coh_yfwd).
    const int first = fld == 1 || fld == 2 ? fld - 1 : fld == 3 ? 3 : 6;
    const int terms = fld == 0 ? 0 : fld < 3 ? 2 : fld == 3 ? 3 : 1;
    double2 fl[3][E], w[E], fo[E];
    double2* out = a.out[fld];
#pragma unroll
    for (int m = 0; m < 3; ++m) {
        if (m >= terms) continue;
        const double2* src = a.b + (size_t)(first + m) * a.fs + i;
#pragma unroll
        for (int e = 0; e < E; ++e) fl[m][e] = src[(size_t)rf_first_idx<NY>(t, e) * a.ld];
    }
#pragma unroll
    for (int e = 0; e < E; ++e) {
        if (MODE == F2_AB2 || fld >= 4) w[e] = a.st[fld][pos(e)];
        if (MODE == F2_AB2) fo[e] = a.ho[fld][pos(e)];
        r[e] = make_double2(0.0, 0.0);
    }
#pragma unroll
    for (int m = 0; m < 3; ++m) {
        if (m >= terms) continue;  // the same for the whole workgroup
        rf_fft<NY, -1>(fl[m], t, xl, tw);
        const bool along_x = m == 0 && fld != 4;
#pragma unroll
        for (int e = 0; e < E; ++e) {
            const double2 d = m == 2 ? make_double2(-a.mu * fl[m][e].x, -a.mu * fl[m][e].y)
                                     : f2_ik(fld == 5 ? -kxv : along_x ? kxv : kyv[e], fl[m][e]);
            r[e] = make_double2(r[e].x - d.x, r[e].y - d.y);
        }
    }
    if (fld == 0) {  // density: -(i kx rho ux + i ky rho uy) (derive2com.f95:267, 339, 402)
#pragma unroll
        for (int e = 0; e < E; ++e) {
            fl[0][e] = a.st[1][pos(e)];
            fl[1][e] = a.st[2][pos(e)];
        }
#pragma unroll
        for (int e = 0; e < E; ++e) {
            const double2 s1 = f2_ik(kxv, fl[0][e]), s2 = f2_ik(kyv[e], fl[1][e]);
            r[e] = msk(e, make_double2(-(s1.x + s2.x), -(s1.y + s2.y)));
        }
    } else if (fld < 3) {  // - mu (kx^2 u_k + ky^2 u_k) + F_k, the forcing unmasked
        const double2* uk = a.k + (size_t)(fld - 1) * a.fs;
#pragma unroll
        for (int e = 0; e < E; ++e) {
            fl[0][e] = uk[pos(e)];
            fl[1][e] = uk[2 * a.fs + pos(e)];
        }
#pragma unroll
        for (int e = 0; e < E; ++e) {
            const double2 d = k2(e, fl[0][e]), z = msk(e, r[e]);
            r[e] = make_double2((z.x - a.mu * d.x) + fl[1][e].x, (z.y - a.mu * d.y) + fl[1][e].y);
        }
    } else {  // E; B: - eta (kx^2 + ky^2) B
#pragma unroll
        for (int e = 0; e < E; ++e) {
            r[e] = msk(e, r[e]);
            if (fld >= 4) {
                const double2 d = k2(e, w[e]);
                r[e] = make_double2(r[e].x - a.eta * d.x, r[e].y - a.eta * d.y);
            }
        }
    }
    if constexpr (MODE == F2_AB2) {
#pragma unroll
        for (int e = 0; e < E; ++e) v[e] = w[e] = f2_ab2(w[e], r[e], fo[e], a.dt);
    }
    if constexpr (INV) {
        rf_final_to_first<NY>(v, t, xl);
        rf_fft<NY, +1>(v, t, xl, tw);
        double2* o = a.a + (size_t)fld * a.fs + i;
#pragma unroll
        for (int e = 0; e < E; ++e) o[(size_t)rf_final_idx<NY>(t, e) * a.ld] = v[e];
    }
#pragma unroll
    for (int e = 0; e < E; ++e) {
        if (MODE == F2_AB2) {
            a.sn[fld][pos(e)] = w[e];
            if (!(isfinite(w[e].x) && isfinite(w[e].y))) *a.bad = 1;
        }
        out[pos(e)] = r[e];
    }
}

// ------------------------------------------------------------ pointwise steppers
__global__ void k_f2_point(int kind, const double2* w, double2* __restrict__ wn, const double2* fo,
                           const double2* fn, double dt, size_t n)
{
    for (size_t q = blockIdx.x * (size_t)blockDim.x + threadIdx.x; q < n; q += (size_t)gridDim.x * blockDim.x) {
        const double2 a = w[q], f = fn[q];
        double2 r;
        if (kind == F2P_AB2) {
            const double2 o = fo[q];
            r = make_double2(a.x + (1.5 * f.x - 0.5 * o.x) * dt, a.y + (1.5 * f.y - 0.5 * o.y) * dt);
        } else if (kind == F2P_EULER) {
            r = make_double2(a.x + f.x * dt, a.y + f.y * dt);
        } else if (kind == F2P_RK4_DEGEN) {
            // all four stage slopes are the input slope (src/rk4nk2coh.f95:22-56)
            const double c = dt / 6.0;
            r = make_double2(a.x + c * (((f.x + 2.0 * f.x) + 2.0 * f.x) + f.x),
                             a.y + c * (((f.y + 2.0 * f.y) + 2.0 * f.y) + f.y));
        } else {
            // predictor and corrector slopes are both the input slope (src/pcnk2coh.f95:20-33)
            r = make_double2(a.x + ((f.x + f.x) * dt) / 2.0, a.y + ((f.y + f.y) * dt) / 2.0);
        }
        wn[q] = r;
    }
}

// ------------------------------------------------------------------ dispatch
#define TARA_F2_SWITCH(n, FN, ...)                  \
    switch (n) {                                    \
        case 16: return FN<16>(__VA_ARGS__);        \
        case 32: return FN<32>(__VA_ARGS__);        \
        case 64: return FN<64>(__VA_ARGS__);        \
        case 128: return FN<128>(__VA_ARGS__);      \
        case 256: return FN<256>(__VA_ARGS__);      \
        default: set_error("2D compressible: unsupported length %d (16..256)", n); return TARA_ERR_UNSUPPORTED; \
    }

template <int NY>
static int launch_prep(const F2Plan& p, const PrepArgs& a, int nfields, hipStream_t st)
{
    hipLaunchKernelGGL(k_f2_prep<NY>, dim3(p.ld / 8, nfields), dim3(CShape<NY>::NT), 0, st, a, p.tw_y);
    return TARA_OK;
}
static int prep(const F2Plan& p, const PrepArgs& a, int nfields, hipStream_t st)
{
    TARA_F2_SWITCH(p.ny, launch_prep, p, a, nfields, st)
}

template <int NX>
static int launch_x(const F2Plan& p, int which, const F2XArgs& x, hipStream_t st)
{
    if (which == 0) {
        using S = FXShape<NX, 7, RCOH>;
        hipLaunchKernelGGL(k_coh_x<NX>, dim3(p.ny / S::RB), dim3(S::NT), 0, st, x, p.tw_x);
    } else if (which == 1) {
        using S = FXShape<NX, 2, 3>;
        hipLaunchKernelGGL(k_com_x1<NX>, dim3(p.ny / S::RB), dim3(S::NT), 0, st, x, p.tw_x);
    } else {
        using S = FXShape<NX, 4, 8>;
        hipLaunchKernelGGL(k_com_x2<NX>, dim3(p.ny / S::RB), dim3(S::NT), 0, st, x, p.tw_x);
    }
    return TARA_OK;
}
static int xpass(const F2Plan& p, int which, const F2XArgs& x, hipStream_t st)
{
    TARA_F2_SWITCH(p.nx, launch_x, p, which, x, st)
}

template <int NY>
static int launch_coh_y(const F2Plan& p, int mode, bool inv, const F2YArgs& a, hipStream_t st)
{
    const dim3 g(p.ld / 8, 3), b(CShape<NY>::NT);
    if (mode == F2_RHS)
        hipLaunchKernelGGL((k_coh_yfwd<NY, F2_RHS, false>), g, b, 0, st, a, p.tw_y);
    else if (inv)
        hipLaunchKernelGGL((k_coh_yfwd<NY, F2_AB2, true>), dim3(p.ld / 8, 8), b, 0, st, a, p.tw_y);
    else
        hipLaunchKernelGGL((k_coh_yfwd<NY, F2_AB2, false>), g, b, 0, st, a, p.tw_y);
    return TARA_OK;
}

template <int NY>
static int launch_com_mid(const F2Plan& p, const F2YArgs& a, hipStream_t st)
{
    hipLaunchKernelGGL(k_com_mid<NY>, dim3(p.ld / 8, 4), dim3(CShape<NY>::NT), 0, st, a, p.tw_y);
    return TARA_OK;
}

template <int NY>
static int launch_com_y(const F2Plan& p, int mode, bool inv, const F2YArgs& a, hipStream_t st)
{
    const dim3 g(6 * (p.ld / 8)), b(CShape<NY>::NT);
    if (mode == F2_RHS)
        hipLaunchKernelGGL((k_com_yfwd<NY, F2_RHS, false>), g, b, 0, st, a, p.tw_y);
    else if (inv)
        hipLaunchKernelGGL((k_com_yfwd<NY, F2_AB2, true>), g, b, 0, st, a, p.tw_y);
    else
        hipLaunchKernelGGL((k_com_yfwd<NY, F2_AB2, false>), g, b, 0, st, a, p.tw_y);
    return TARA_OK;
}

static int coh_y(const F2Plan& p, int mode, bool inv, const F2YArgs& a, hipStream_t st)
{
    TARA_F2_SWITCH(p.ny, launch_coh_y, p, mode, inv, a, st)
}
static int com_mid(const F2Plan& p, const F2YArgs& a, hipStream_t st) { TARA_F2_SWITCH(p.ny, launch_com_mid, p, a, st) }
static int com_y(const F2Plan& p, int mode, bool inv, const F2YArgs& a, hipStream_t st)
{
    TARA_F2_SWITCH(p.ny, launch_com_y, p, mode, inv, a, st)
}

// ------------------------------------------------------------------ host side
int f2_plan_init(F2Plan& p, int family, int nx, int ny, double pi, double lx, double ly)
{
    TARA_CHECK(is_pow2(nx) && is_pow2(ny) && nx >= 16 && ny >= 16 && nx <= 256 && ny <= 256, TARA_ERR_UNSUPPORTED,
               "2D compressible: grid %dx%d unsupported (powers of two, 16..256)", nx, ny);
    TARA_CHECK(lx > 0 && ly > 0 && pi > 0, TARA_ERR_ARG, "2D compressible: pi and box lengths must be positive");
    p.nx = nx;
    p.ny = ny;
    p.nh = nx / 2 + 1;
    p.ld = (p.nh + 7) / 8 * 8;
    p.fsz = (size_t)p.ld * ny;
    p.pi = pi;
    p.lx = lx;
    p.ly = ly;
    const size_t fb = p.fsz * sizeof(double2);
    int rc;
    const int na = family == 0 ? 8 : 6, nb = family == 0 ? 3 : 7;
    if ((rc = p.a.alloc(na * fb)) || (rc = p.b.alloc(nb * fb))) return rc;
    TARA_HIP(hipMemset(p.a.p, 0, p.a.bytes));
    TARA_HIP(hipMemset(p.b.p, 0, p.b.bytes));
    if (family == 1) {
        if ((rc = p.c.alloc(4 * fb)) || (rc = p.d.alloc(fb)) || (rc = p.k.alloc(4 * fb)) ||
            (rc = p.sines.alloc((nx + ny) * sizeof(double))))
            return rc;
        TARA_HIP(hipMemset(p.c.p, 0, p.c.bytes));
        TARA_HIP(hipMemset(p.d.p, 0, p.d.bytes));
        TARA_HIP(hipMemset(p.k.p, 0, p.k.bytes));
    }
    // kx = 2 pi (i-1)/Lx, ky = 2 pi (j-1)/Ly or 2 pi ((j-1)-Ny)/Ly (derive2coh.f95:59-60, 74-75)
    std::vector<double> kx(p.ld, 0.0), ky(ny);
    for (int i = 0; i < p.nh; ++i) kx[i] = 2.0 * pi * (double)i / lx;
    for (int j = 0; j < ny; ++j) ky[j] = 2.0 * pi * (double)(j < ny / 2 ? j : j - ny) / ly;
    // circular dealias: sqrt(kx^2+ky^2) >= (Nx+Ny)/2/3 (derive2coh.f95:208)
    const double cut = ((double)(nx + ny) / 2.0) / 3.0 + 0;
    std::vector<int> imin(ny);
    for (int j = 0; j < ny; ++j) {
        int m = p.nh;
        for (int i = 0; i < p.nh; ++i)
            if (std::sqrt(kx[i] * kx[i] + ky[j] * ky[j]) >= cut) {
                m = i;
                break;
            }
        imin[j] = m;  // kx increases with i: every i >= m is cut
    }
    if ((rc = p.kx.alloc(p.ld * sizeof(double))) || (rc = p.ky.alloc(ny * sizeof(double))) ||
        (rc = p.imin.alloc(ny * sizeof(int))) || (rc = p.bad.alloc(sizeof(int))))
        return rc;
    TARA_HIP(hipMemset(p.bad.p, 0, sizeof(int)));
    TARA_HIP(hipMemcpy(p.kx.p, kx.data(), p.ld * sizeof(double), hipMemcpyHostToDevice));
    TARA_HIP(hipMemcpy(p.ky.p, ky.data(), ny * sizeof(double), hipMemcpyHostToDevice));
    TARA_HIP(hipMemcpy(p.imin.p, imin.data(), ny * sizeof(int), hipMemcpyHostToDevice));
    p.tw_y = twiddles(ny);
    p.tw_x = twiddles(nx, 4);
    TARA_CHECK(p.tw_y && p.tw_x, TARA_ERR_ALLOC, "twiddle table allocation failed");
    return TARA_OK;
}

namespace {

// Pass 1: the backward y transforms of st into A.
int coh_prep(const F2Plan& p, double2* const st[3], hipStream_t s)
{
    PrepArgs pa{};
    const int src[8] = {0, 1, 2, 0, 1, 2, 1, 2};
    const int kind[8] = {MUL_1, MUL_1, MUL_1, MUL_IKY, MUL_IKY, MUL_IKY, MUL_KY2, MUL_KY2};
    for (int o = 0; o < 8; ++o) {
        pa.src[o] = st[src[o]];
        pa.dst[o] = p.a.as<double2>() + o * p.fsz;
        pa.kind[o] = kind[o];
    }
    pa.kx = p.kx.as<double>();
    pa.ky = p.ky.as<double>();
    pa.ld = p.ld;
    return prep(p, pa, 8, s);
}

int com_prep(const F2Plan& p, const ComPhys& ph, double2* const st[6], hipStream_t s)
{
    // x(i) = (i-1) dx as src/main2com.f95:231 builds it
    hipLaunchKernelGGL(k_com_sines, dim3((p.nx + p.ny + 255) / 256), dim3(256), 0, s, p.sines.as<double>(), p.nx, p.ny,
                       ph.kf, p.lx / (double)p.nx, p.ly / (double)p.ny);
    PrepArgs pa{};
    for (int o = 0; o < 6; ++o) {
        pa.src[o] = st[o];
        pa.dst[o] = p.a.as<double2>() + o * p.fsz;
        pa.kind[o] = MUL_1;
    }
    pa.kx = p.kx.as<double>();
    pa.ky = p.ky.as<double>();
    pa.ld = p.ld;
    return prep(p, pa, 6, s);
}

F2XArgs xargs(const F2Plan& p)
{
    F2XArgs x{};
    x.a = p.a.as<double2>();
    x.c = p.c.as<double2>();
    x.d = p.d.as<double2>();
    x.b = p.b.as<double2>();
    x.fs = p.fsz;
    x.kx = p.kx.as<double>();
    x.ld = p.ld;
    x.ny = p.ny;
    x.norm = 1.0 / ((double)p.nx * (double)p.ny);
    return x;
}

F2YArgs yargs(const F2Plan& p, double dt)
{
    F2YArgs y{};
    y.b = p.b.as<double2>();
    y.c = p.c.as<double2>();
    y.d = p.d.as<double2>();
    y.k = p.k.as<double2>();
    y.a = p.a.as<double2>();
    y.fs = p.fsz;
    y.kx = p.kx.as<double>();
    y.ky = p.ky.as<double>();
    y.imin = p.imin.as<int>();
    y.ld = p.ld;
    y.dt = dt;
    y.bad = p.bad.as<int>();
    return y;
}

// Passes 2 and 3 of derive2coh, A holding pass 1 of st; AB2 takes the history ho
// and writes the new state to sn.
int coh_rest(const F2Plan& p, const CohPhys& ph, double2* const st[3], double2* const ho[3], double2* const sn[3],
             double2* const out[3], int mode, bool inv, double dt, hipStream_t s, EventTimer* tm)
{
    int rc;
    F2XArgs x = xargs(p);
    x.p0 = ph.mux;
    x.p1 = ph.muy;
    x.p2 = ph.cs * ph.cs;
    if (tm) tm->begin(1, s);
    if ((rc = xpass(p, 0, x, s))) return rc;
    if (tm) tm->end(1, s);
    F2YArgs y = yargs(p, dt);
    for (int f = 0; f < 3; ++f) {
        y.st[f] = st[f];
        y.ho[f] = ho[f];
        y.sn[f] = sn[f];
        y.out[f] = out[f];
    }
    if (tm) tm->begin(2, s);
    if ((rc = coh_y(p, mode, inv, y, s))) return rc;
    if (tm) tm->end(2, s);
    return TARA_OK;
}

// Passes 2 to 5 of derive2com, A holding pass 1 of st; AB2 writes the new state to sn.
int com_rest(const F2Plan& p, const ComPhys& ph, double2* const st[6], double2* const sn[6], double2* const out[6],
             int mode, bool inv, double dt, hipStream_t s, EventTimer* tm)
{
    int rc;
    F2XArgs x = xargs(p);
    x.b = p.c.as<double2>();
    x.p0 = ph.amp;
    x.sines = p.sines.as<double>();
    if (tm) tm->begin(1, s);
    if ((rc = xpass(p, 1, x, s))) return rc;
    F2YArgs y = yargs(p, dt);
    for (int f = 0; f < 6; ++f) {
        y.st[f] = st[f];
        y.sn[f] = sn[f];
        y.ho[f] = y.out[f] = out[f];
    }
    y.mu = ph.mu;
    y.eta = ph.eta;
    if ((rc = com_mid(p, y, s))) return rc;
    x.b = p.b.as<double2>();
    x.p0 = ph.cs * ph.cs;
    x.p1 = ph.eta;
    if ((rc = xpass(p, 2, x, s))) return rc;
    if (tm) tm->end(1, s);
    if (tm) tm->begin(2, s);
    if ((rc = com_y(p, mode, inv, y, s))) return rc;
    if (tm) tm->end(2, s);
    return TARA_OK;
}

}  // namespace

int coh_rhs(const F2Plan& p, const CohPhys& ph, double2* const st[3], double2* const out[3], hipStream_t s)
{
    int rc;
    if ((rc = coh_prep(p, st, s)) || (rc = coh_rest(p, ph, st, out, st, out, F2_RHS, false, 0.0, s, nullptr))) return rc;
    TARA_HIP(hipGetLastError());
    return TARA_OK;
}

int com_rhs(const F2Plan& p, const ComPhys& ph, double2* const st[6], double2* const out[6], hipStream_t s)
{
    int rc;
    if ((rc = com_prep(p, ph, st, s)) || (rc = com_rest(p, ph, st, st, out, F2_RHS, false, 0.0, s, nullptr))) return rc;
    TARA_HIP(hipGetLastError());
    return TARA_OK;
}

int coh_advance(const F2Plan& p, const CohPhys& ph, double2* st[3], double2* hist[3], double2* st2[3], double2* hist2[3],
                int nsteps, double dt, hipStream_t s, EventTimer* tm)
{
    if (nsteps <= 0) return TARA_OK;
    int rc;
    if (tm) tm->begin(0, s);
    if ((rc = coh_prep(p, st, s))) return rc;
    if (tm) tm->end(0, s);
    for (int k = 0; k < nsteps; ++k) {
        if ((rc = coh_rest(p, ph, st, hist, st2, hist2, F2_AB2, k + 1 < nsteps, dt, s, tm))) return rc;
        for (int f = 0; f < 3; ++f) {
            std::swap(st[f], st2[f]);
            std::swap(hist[f], hist2[f]);
        }
    }
    TARA_HIP(hipGetLastError());
    return TARA_OK;
}

int com_advance(const F2Plan& p, const ComPhys& ph, double2* st[6], double2* mom[2], double2* const hist[6], int nsteps,
                double dt, hipStream_t s, EventTimer* tm)
{
    if (nsteps <= 0) return TARA_OK;
    int rc;
    if (tm) tm->begin(0, s);
    if ((rc = com_prep(p, ph, st, s))) return rc;
    if (tm) tm->end(0, s);
    for (int k = 0; k < nsteps; ++k) {
        double2* sn[6];
        for (int f = 0; f < 6; ++f) sn[f] = f == 1 || f == 2 ? mom[f - 1] : st[f];
        if ((rc = com_rest(p, ph, st, sn, hist, F2_AB2, k + 1 < nsteps, dt, s, tm))) return rc;
        for (int f = 0; f < 2; ++f) std::swap(st[1 + f], mom[f]);
    }
    TARA_HIP(hipGetLastError());
    return TARA_OK;
}

int f2_pointwise(int kind, const double2* w, double2* wn, const double2* fo, const double2* fn, double dt, size_t n,
                 hipStream_t st)
{
    const int bs = 256;
    size_t nb = (n + bs - 1) / bs;
    if (nb > 65536) nb = 65536;
    if (nb == 0) return TARA_OK;
    hipLaunchKernelGGL(k_f2_point, dim3((unsigned)nb), dim3(bs), 0, st, kind, w, wn, fo, fn, dt, n);
    TARA_HIP(hipGetLastError());
    return TARA_OK;
}

}  // namespace tara
