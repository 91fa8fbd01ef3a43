// 3D compressible isothermal MHD on gfx950: the right-hand side of
// src/derive3com.f95 and the AB2 update of src/ab3com.f95.
//
// Only the live dataflow of derive3com is computed.  ab3com freezes the
// energy (src/ab3com.f95:51) and the pressure is P = CS^2 rho
// (src/derive3com.f95:395), so E, curl B, the energy fluxes and the
// (commented-out) forcing never reach rho, rho u or B; they are not formed.
//
// Five sweeps per right-hand side (device layout: kx-fastest, row length
// padded to ld = Nh rounded up to 8; element (i, j, k) at (k*Ny + j)*ld + i):
//   1 k_col_fft (z, backward)  state (7 fields) -> Az, tiles of 8 kx columns
//   2 k_col_fft (y, backward)  Az -> A
//   3 k_mhd_x                  per x row: 7 c2r as 4 paired complex FFTs,
//                              u = rho u / rho, P, B^2 and the 12 distinct live
//                              fluxes (derive3com.f95:176-186, 395-436), 6
//                              paired forward FFTs -> B (12 fields)
//   4 k_col_fft (y, forward)   B in place
//   5 k_mhd_zfwd               z forward of the 12 fields, i k . flux, k^2
//                              diffusion, spherical dealias on all terms
//                              (derive3com.f95:574-843), assembly
//                              (:1018-1037), then RHS out, or AB2 in place and
//                              the inverse z transform of the new state -> Az.
// The diffusion coefficients are parameters (the reference hard-wires 1/450,
// derive3com.f95:1023-1037).
//
// The dealiasing zeroes every term of every field outside the sphere
// k < (Nx+Ny+Nz)/9, so a mode outside it never changes: at 256^3 in a 2 pi box
// 14 % of the modes live, in 35 % of the z columns and 86 of 129 kx columns.
//   - Sweeps 3 to 5 carry only what a live mode reads: x writes the kx tiles that
//     hold one, y transforms them and stores the rows that hold one, z runs over
//     the tiles that hold one.
//   - Within one advance call the inverse transform of the rest is the same at
//     every step: sweep 1 runs once, sweep 5 replaces the live tiles of Az, and
//     sweep 2 redoes the kx tiles that hold a live mode (the others' A stays).
// Mom_x_3 = Mom_z_1 and Mom_y_3 = Mom_z_2 (the same products in another order)
// are formed once.  Per step, in half spectra of 16 Nh Ny Nz bytes at 256^3:
// 9.4 (y) + 15 (x) + 13.6 (y) + 14 (z) = 52, against 119 when every sweep carried
// every mode and 14 fluxes; 3.72 -> 1.65 ms (0.25 + 0.57 + 0.33 + 0.46 ms; the
// first step of a call adds 0.5 ms).
#include <algorithm>
#include <cmath>

#include "mhd3d.h"
#include "colpass.h"

namespace tara {

// ------------------------------------------------------------------ x pass
// One x row per wavefront group of T = NX/4 lanes (4 complex elements per
// lane), so the exchanges between FFT passes need only wave-level ordering.
template <int NX>
struct MXShape {
    static constexpr int E = RF<NX, 4>::E;
    static constexpr int T = RF<NX, 4>::T;
    static_assert(64 % T == 0, "x pass rows must not straddle wavefronts");
    static constexpr int RPW = 64 / T;      // rows per wavefront
    static constexpr int RPB = 4 * RPW;     // rows per 256-thread workgroup
    static constexpr int LP = RF<NX, 4>::LDS + 1;
};

struct XArgs {
    const double2* a;  // 7 inverse-transformed fields, field stride fs
    double2* b;        // 12 flux fields
    size_t fs;
    int ld;
    int nk;            // kx columns of the fluxes that are kept
    double norm;       // 1 / (Nx Ny Nz)
    double cs2;
};

// At most 168 VGPRs (three waves per SIMD): faster than two waves at 178 VGPRs
// and than four with spills.
template <int NX>
__global__ __launch_bounds__(256, 3) void k_mhd_x(XArgs x, const double2* tw)
{
    using S = MXShape<NX>;
    constexpr int E = S::E, T = S::T, M = NX / 2;
    __shared__ double2 lds[S::RPB * S::LP];
    const int lane = threadIdx.x % 64, wave = threadIdx.x / 64;
    const int rw = lane / T, t = lane % T;
    const int slot = wave * S::RPW + rw;
    const size_t row = (size_t)xcd_remap(blockIdx.x, gridDim.x) * S::RPB + slot;  // = k*Ny + j
    const size_t ro = row * x.ld;
    double2* xl = lds + slot * S::LP;

    // backward: pairs (rho, rho ux), (rho uy, rho uz), (Bx, By), (Bz, -)
    double pr[7][E];
#pragma unroll
    for (int p = 0; p < 4; ++p) {
        const double2* fa = x.a + (size_t)(2 * p) * x.fs + ro;
        const double2* fb = x.a + (size_t)(2 * p + 1) * x.fs + ro;
        double2 v[E];
#pragma unroll
        for (int e = 0; e < E; ++e) {
            const int k = rf_first_idx<NX, 4>(t, e);
            const int kk = k <= M ? k : NX - k;
            double2 u = fa[kk];
            double2 w = (p < 3) ? fb[kk] : make_double2(0.0, 0.0);
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
        for (int e = 0; e < E; ++e) {
            pr[2 * p][e] = v[e].x * x.norm;
            if (p < 3) pr[2 * p + 1][e] = v[e].y * x.norm;
        }
    }
    // real-space fluxes at this lane's positions (the reference's expressions)
    double ux[E], uy[E], uz[E], pp[E], hb2[E];
#pragma unroll
    for (int e = 0; e < E; ++e) {
        const double rho = pr[0][e];
        ux[e] = pr[1][e] / rho;
        uy[e] = pr[2][e] / rho;
        uz[e] = pr[3][e] / rho;
        pp[e] = x.cs2 * rho;
        hb2[e] = (pr[4][e] * pr[4][e] + pr[5][e] * pr[5][e] + pr[6][e] * pr[6][e]) / 2.0;
    }
    // forward pairs: (ux, uy) (uz, MXX) (MXY, MXZ) (MYY, MYZ) (MZZ, MG1) (MG2, MG3)
#pragma unroll 1
    for (int p = 0; p < 6; ++p) {
        double2 v[E];
#pragma unroll
        for (int e = 0; e < E; ++e) {
            const double rux = pr[1][e], ruy = pr[2][e], ruz = pr[3][e];
            const double bx = pr[4][e], by = pr[5][e], bz = pr[6][e];
            double f0, f1;
            switch (p) {
                case 0: f0 = ux[e]; f1 = uy[e]; break;
                case 1: f0 = uz[e]; f1 = rux * ux[e] + pp[e] + hb2[e] - bx * bx; break;
                case 2: f0 = rux * uy[e] - bx * by; f1 = rux * uz[e] - bx * bz; break;
                case 3: f0 = ruy * uy[e] + pp[e] + hb2[e] - by * by; f1 = ruy * uz[e] - by * bz; break;
                case 4: f0 = ruz * uz[e] + pp[e] + hb2[e] - bz * bz; f1 = ux[e] * by - uy[e] * bx; break;
                default: f0 = ux[e] * bz - uz[e] * bx; f1 = uy[e] * bz - uz[e] * by; break;
            }
            v[e] = make_double2(f0, f1);
        }
        rf_final_to_first<NX, 4, true>(v, t, xl);
        rf_fft<NX, -1, 4, true>(v, t, xl, tw);
#pragma unroll
        for (int e = 0; e < E; ++e) xl[rf_pad(rf_final_idx<NX, 4>(t, e))] = v[e];
        rf_sync<true>();
        double2* oa = x.b + (size_t)(2 * p) * x.fs + ro;
        double2* ob = x.b + (size_t)(2 * p + 1) * x.fs + ro;
        for (int k = t; k < x.nk; k += T) {
            const double2 z = xl[rf_pad(k)], zm = xl[rf_pad(k == 0 ? 0 : NX - k)];
            oa[k] = make_double2(0.5 * (z.x + zm.x), 0.5 * (z.y - zm.y));
            ob[k] = make_double2(0.5 * (z.y + zm.y), -0.5 * (z.x - zm.x));
        }
        rf_sync<true>();
    }
}

// ----------------------------------------------------- z forward + assembly
struct ZArgs {
    const double2* b;      // 12 flux fields after the y pass
    size_t fs;
    const double2* st[7];  // state (rho, rho ux, rho uy, rho uz, Bx, By, Bz)
    double2* sn[7];        // MHD_AB2: new state; for rho and B the same fields as st
    double2* out[7];       // RHS (MHD_RHS) or history f_{n-1} -> f_n (MHD_AB2)
    double2* az;           // with INV: 7 fields, the new state's inverse z transform
    const double* kx;
    const double* ky;
    const double* kz;
    const int* imin;       // per (k, j) row: modes with i >= imin are dealiased away
    const int* live;       // tiles j*(ld/8) + x that hold a live mode
    int ny, ld;
    double mu, eta, dt;
    int* bad;              // AB2: set to 1 when a new state value is not finite
};

// Flux fields of B, in the x pass's order.
enum MhdFlux { FUX, FUY, FUZ, FXX, FXY, FXZ, FYY, FYZ, FZZ, FG1, FG2, FG3 };

// One state field of one tile of 8 kx columns of one ky row per workgroup, 4
// elements per thread; the seven fields of a tile run next to each other on one
// XCD, which serves the fluxes that two of them read from its L2.
// Bound by its memory traffic: 1.9 GB in 0.46 ms at 256^3 (4.1 TB/s).  One
// workgroup for all seven fields of a tile reads each flux once, but needs three
// accumulators beside the density's and spilled 42-63 registers per lane at the
// 128 that four waves per SIMD allow; split by field nothing spills (123 at
// most), a thread's chain is at most 4 + 1 transforms instead of 12 + 7, and
// small grids fill the chip (64^3: 33.6 -> 13.0 us, with the inverse transform
// that was a kernel of its own before).
// The density's right-hand side needs the momentum of the step's start, which
// other workgroups update: the new momentum goes to other buffers (sn).
constexpr int kZfwdEM = 4;
template <int NZ, int MODE, bool INV, int EM>
__global__ __launch_bounds__((CShape<NZ, EM>::NT), 4) void k_mhd_zfwd(ZArgs a, const double2* tw)
{
    using S = CShape<NZ, EM>;
    constexpr int E = RF<NZ, EM>::E;
    __shared__ double2 lds[8 * S::LP];
    const int c = threadIdx.x % 8, t = threadIdx.x / 8;
    const int tpp = a.ld / 8;
    const int id = xcd_remap(blockIdx.x, gridDim.x);
    const int tile = a.live[id / 7], fld = id % 7;
    const int j = tile / tpp, i = (tile % tpp) * 8 + c;
    const size_t base = (size_t)j * a.ld + i, es = (size_t)a.ny * a.ld;
    double2* xl = lds + c * S::LP;
    const double kxv = a.kx[i], kyv = a.ky[j];
    double kzv[E], k2[E];
#pragma unroll
    for (int e = 0; e < E; ++e) {
        kzv[e] = a.kz[rf_final_idx<NZ, EM>(t, e)];
        k2[e] = (kxv * kxv + kyv * kyv) + kzv[e] * kzv[e];
    }
    // i k z = (-k z.y, k z.x)
    auto ik = [](double kk, double2 z) { return make_double2(-(kk * z.y), kk * z.x); };
    auto zk = [&](int e) { return base + (size_t)rf_final_idx<NZ, EM>(t, e) * es; };
    double2 acc[E];
    if (fld == 0) {
        // density: -(i kx rho ux + i ky rho uy + i kz rho uz) on the state spectra
#pragma unroll
        for (int e = 0; e < E; ++e) {
            const size_t q = zk(e);
            const double2 s1 = ik(kxv, a.st[1][q]), s2 = ik(kyv, a.st[2][q]), s3 = ik(kzv[e], a.st[3][q]);
            acc[e] = make_double2(-((s1.x + s2.x) + s3.x), -((s1.y + s2.y) + s3.y));
        }
    } else {
        // a sum of terms +-i k_d flux over directions d: momentum row r takes
        // -mu k^2 u_r - i k . (row r of the symmetric flux tensor); the induction
        // dBx = i ky MG1 + i kz MG2, dBy = -i kx MG1 + i kz MG3,
        // dBz = -i kx MG2 - i ky MG3 (src/derive3com.f95:1030-1037)
        const bool mom = fld < 4;
        const int r = (fld - 1) % 3;
#pragma unroll
        for (int e = 0; e < E; ++e) acc[e] = make_double2(0.0, 0.0);
#pragma unroll 1
        for (int m = mom ? -1 : 0; m < 3; ++m) {
            // induction: direction r has no term in row r; the flux of rows r and
            // m is MG(r + m), its sign minus below the diagonal
            if (!mom && m == r) continue;
            int f;
            if (m < 0)
                f = FUX + r;
            else if (mom)
                f = FXX + (r + m) + (r && m ? 1 : 0);
            else
                f = FG1 + r + m - 1;
            const double2* src = a.b + (size_t)f * a.fs + base;
            double2 v[E];
#pragma unroll
            for (int e = 0; e < E; ++e) v[e] = src[(size_t)rf_first_idx<NZ, EM>(t, e) * es];
            rf_fft<NZ, -1, EM>(v, t, xl, tw);
            const double sg = mom || m < r ? -1.0 : 1.0;
#pragma unroll
            for (int e = 0; e < E; ++e) {
                const double kd = sg * (m == 0 ? kxv : m == 1 ? kyv : kzv[e]);
                const double2 d = m < 0 ? make_double2(-(a.mu * k2[e] * v[e].x), -(a.mu * k2[e] * v[e].y)) : ik(kd, v[e]);
                acc[e] = make_double2(acc[e].x + d.x, acc[e].y + d.y);
            }
        }
    }
    // f = acc (- eta k^2 state for the components of B), masked; stored as the
    // RHS, or taken into the AB2 update, whose new state goes on through the
    // inverse z transform.  A masked mode's f and history are zero: its state is
    // read for the transform only.
    const double2* st = a.st[fld];
    double2* out = a.out[fld];
    bool finite = true;
#pragma unroll
    for (int e = 0; e < E; ++e) {
        const size_t q = zk(e);
        const bool keep = i < a.imin[(size_t)rf_final_idx<NZ, EM>(t, e) * a.ny + j];
        double2 f = acc[e], w = make_double2(0.0, 0.0);
        if (MODE == MHD_AB2 || fld >= 4) w = st[q];
        if (fld >= 4) f = make_double2(f.x - a.eta * k2[e] * w.x, f.y - a.eta * k2[e] * w.y);
        if (!keep) f = make_double2(0.0, 0.0);
        if (MODE == MHD_RHS) {
            out[q] = f;
        } else if (keep) {
            const double2 fo = out[q];
            w = make_double2(w.x + (1.5 * f.x - 0.5 * fo.x) * a.dt, w.y + (1.5 * f.y - 0.5 * fo.y) * a.dt);
            a.sn[fld][q] = w;
            out[q] = f;
            finite = finite && isfinite(w.x) && isfinite(w.y);
        }
        acc[e] = w;
    }
    if (MODE == MHD_AB2 && !finite && a.bad) a.bad[0] = 1;
    if constexpr (INV) {
        rf_final_to_first<NZ, EM>(acc, t, xl);
        rf_fft<NZ, +1, EM>(acc, t, xl, tw);
        double2* dst = a.az + (size_t)fld * a.fs;
#pragma unroll
        for (int e = 0; e < E; ++e) dst[zk(e)] = acc[e];
    }
}

// ------------------------------------------------------------------ dispatch
#define TARA_MHD_SWITCH(n, FN, ...)                 \
    switch (n) {                                    \
        case 16: return FN<16>(__VA_ARGS__);        \
        case 32: return FN<32>(__VA_ARGS__);        \
        case 64: return FN<64>(__VA_ARGS__);        \
        case 128: return FN<128>(__VA_ARGS__);      \
        case 256: return FN<256>(__VA_ARGS__);      \
        default: set_error("3D MHD: unsupported length %d (16..256)", n); return TARA_ERR_UNSUPPORTED; \
    }

template <int N>
static int launch_col(const ColArgs& a, int ntiles, int nfields, int dir, const double2* tw, hipStream_t st)
{
    dim3 g(ntiles, nfields), b(CShape<N>::NT);
    if (dir < 0)
        hipLaunchKernelGGL((k_col_fft<N, -1>), g, b, 0, st, a, tw);
    else
        hipLaunchKernelGGL((k_col_fft<N, +1>), g, b, 0, st, a, tw);
    return TARA_OK;
}
int col_fft_tiles(int n, const ColArgs& a, int ntiles, int nfields, int dir, const double2* tw, hipStream_t st)
{
    TARA_MHD_SWITCH(n, launch_col, a, ntiles, nfields, dir, tw, st)
}
static int col(int n, const ColArgs& a, int ntiles, int nfields, int dir, const double2* tw, hipStream_t st)
{
    return col_fft_tiles(n, a, ntiles, nfields, dir, tw, st);
}

template <int NX>
static int launch_x(const MhdPlan& p, const XArgs& x, hipStream_t st)
{
    using S = MXShape<NX>;
    const int nrows = p.ny * p.nz;
    TARA_CHECK(nrows % S::RPB == 0, TARA_ERR_UNSUPPORTED, "3D MHD: Ny*Nz=%d not a multiple of %d", nrows, S::RPB);
    hipLaunchKernelGGL(k_mhd_x<NX>, dim3(nrows / S::RPB), dim3(256), 0, st, x, p.tw_x);
    return TARA_OK;
}
static int xpass(const MhdPlan& p, const XArgs& x, hipStream_t st) { TARA_MHD_SWITCH(p.nx, launch_x, p, x, st) }

template <int NZ>
static int launch_z(const MhdPlan& p, int mode, bool inv, const ZArgs& z, hipStream_t st)
{
    constexpr int EM = kZfwdEM;
    dim3 g(7 * p.nlive), b(CShape<NZ, EM>::NT);
    if (mode == MHD_RHS)
        hipLaunchKernelGGL((k_mhd_zfwd<NZ, MHD_RHS, false, EM>), g, b, 0, st, z, p.tw_z4);
    else if (inv)
        hipLaunchKernelGGL((k_mhd_zfwd<NZ, MHD_AB2, true, EM>), g, b, 0, st, z, p.tw_z4);
    else
        hipLaunchKernelGGL((k_mhd_zfwd<NZ, MHD_AB2, false, EM>), g, b, 0, st, z, p.tw_z4);
    return TARA_OK;
}
static int zpass(const MhdPlan& p, int mode, bool inv, const ZArgs& z, hipStream_t st)
{
    TARA_MHD_SWITCH(p.nz, launch_z, p, mode, inv, z, st)
}

// ------------------------------------------------------------------ host side
int mhd_plan_init(MhdPlan& p, int nx, int ny, int nz, double lx, double ly, double lz, double mu, double eta,
                  double cs)
{
    TARA_CHECK(is_pow2(nx) && is_pow2(ny) && is_pow2(nz) && nx >= 16 && ny >= 16 && nz >= 16 && nx <= 256 &&
                   ny <= 256 && nz <= 256,
               TARA_ERR_UNSUPPORTED, "3D MHD: grid %dx%dx%d unsupported (powers of two, 16..256)", nx, ny, nz);
    TARA_CHECK(lx > 0 && ly > 0 && lz > 0, TARA_ERR_ARG, "3D MHD: box lengths must be positive");
    p.nx = nx;
    p.ny = ny;
    p.nz = nz;
    p.nh = nx / 2 + 1;
    p.ld = (p.nh + 7) / 8 * 8;
    p.lx = lx;
    p.ly = ly;
    p.lz = lz;
    p.mu = mu;
    p.eta = eta;
    p.cs = cs;
    p.fsz = (size_t)p.ld * ny * nz;
    int rc;
    if ((rc = p.a.alloc(7 * p.fsz * sizeof(double2))) || (rc = p.b.alloc(12 * p.fsz * sizeof(double2)))) return rc;
    TARA_HIP(hipMemset(p.a.p, 0, p.a.bytes));
    TARA_HIP(hipMemset(p.b.p, 0, p.b.bytes));
    // wavenumbers as derive3com forms them: 2 pi (i-1)/L with true pi
    // (src/derive3com.f95:245-247, 260-262), second halves of y and z negative
    const double pi = 3.14159265358979323846;
    std::vector<double> kx(p.ld, 0.0), ky(ny), kz(nz);
    for (int i = 0; i < p.nh; ++i) kx[i] = 2.0 * pi * (double)i / lx;
    for (int j = 0; j < ny; ++j) ky[j] = 2.0 * pi * (double)(j < ny / 2 ? j : j - ny) / ly;
    for (int k = 0; k < nz; ++k) kz[k] = 2.0 * pi * (double)(k < nz / 2 ? k : k - nz) / lz;
    // spherical dealias of derive3com.f95:802: sqrt(kx^2+ky^2+kz^2) >= (Nx+Ny+Nz)/3/3
    const double cut = ((double)(nx + ny + nz) / 3.0) / 3.0 + 0;
    std::vector<int> imin((size_t)ny * nz);
    for (int k = 0; k < nz; ++k)
        for (int j = 0; j < ny; ++j) {
            int m = p.nh;
            for (int i = 0; i < p.nh; ++i)
                if (std::sqrt(kx[i] * kx[i] + ky[j] * ky[j] + kz[k] * kz[k]) >= cut) {
                    m = i;
                    break;
                }
            imin[(size_t)k * ny + j] = m;  // kx increases with i: every i >= m is cut
        }
    if ((rc = p.kx.alloc(p.ld * sizeof(double))) || (rc = p.ky.alloc(ny * sizeof(double))) ||
        (rc = p.kz.alloc(nz * sizeof(double))) || (rc = p.imin.alloc(imin.size() * sizeof(int))) ||
        (rc = p.bad.alloc(sizeof(int))))
        return rc;
    // live tiles: imin is largest at the smallest |kz|, but every k is looked at
    const int tpp = p.ld / 8;
    std::vector<int> width(ny, 0), live;
    for (int k = 0; k < nz; ++k)
        for (int j = 0; j < ny; ++j) width[j] = std::max(width[j], imin[(size_t)k * ny + j]);
    for (int j = 0; j < ny; ++j) {
        const int nt = (width[j] + 7) / 8;
        p.ktiles = std::max(p.ktiles, nt);
        for (int x = 0; x < nt; ++x) live.push_back(j * tpp + x);
    }
    p.nlive = (int)live.size();  // at least the tile of k = 0, since the cut is positive
    // rows of a kx tile without a live mode: |ky| grows towards the middle, so
    // they are one run [lo, hi)
    std::vector<int2> yskip(p.ktiles);
    for (int x = 0; x < p.ktiles; ++x) {
        int lo = 0, hi = ny;
        while (lo < ny && width[lo] > 8 * x) ++lo;
        while (hi > lo && width[hi - 1] > 8 * x) --hi;
        yskip[x] = make_int2(lo, hi);
    }
    if ((rc = p.live.alloc(live.size() * sizeof(int))) || (rc = p.yskip.alloc(yskip.size() * sizeof(int2)))) return rc;
    TARA_HIP(hipMemcpy(p.live.p, live.data(), live.size() * sizeof(int), hipMemcpyHostToDevice));
    TARA_HIP(hipMemcpy(p.yskip.p, yskip.data(), yskip.size() * sizeof(int2), hipMemcpyHostToDevice));
    TARA_HIP(hipMemset(p.bad.p, 0, sizeof(int)));
    TARA_HIP(hipMemcpy(p.kx.p, kx.data(), p.ld * sizeof(double), hipMemcpyHostToDevice));
    TARA_HIP(hipMemcpy(p.ky.p, ky.data(), ny * sizeof(double), hipMemcpyHostToDevice));
    TARA_HIP(hipMemcpy(p.kz.p, kz.data(), nz * sizeof(double), hipMemcpyHostToDevice));
    TARA_HIP(hipMemcpy(p.imin.p, imin.data(), imin.size() * sizeof(int), hipMemcpyHostToDevice));
    p.tw_y = twiddles(ny);
    p.tw_z = twiddles(nz);
    p.tw_z4 = twiddles(nz, 4);
    p.tw_x = twiddles(nx, 4);
    TARA_CHECK(p.tw_y && p.tw_z && p.tw_z4 && p.tw_x, TARA_ERR_ALLOC, "twiddle table allocation failed");
    return TARA_OK;
}

int mhd_plan_stepping(MhdPlan& p) { return p.az.alloc(7 * p.fsz * sizeof(double2)); }

namespace {

// Backward z of every column: fields src -> dst (7 fields, stride fsz).
int inverse_z(const MhdPlan& p, double2* const src[7], double2* dst, hipStream_t s)
{
    ColArgs c{};
    for (int f = 0; f < 7; ++f) {
        c.src[f] = src[f];
        c.dst[f] = dst + f * p.fsz;
    }
    c.es = (long)p.ny * p.ld;
    c.pstride = p.ld;
    c.tpp = p.ld / 8;
    return col(p.nz, c, p.ny * c.tpp, 7, +1, p.tw_z, s);
}

// Backward y of the first ktiles kx tiles of every plane: 7 fields src -> dst.
int inverse_y(const MhdPlan& p, const double2* src, double2* dst, int ktiles, hipStream_t s)
{
    ColArgs c{};
    for (int f = 0; f < 7; ++f) {
        c.src[f] = src + f * p.fsz;
        c.dst[f] = dst + f * p.fsz;
    }
    c.es = p.ld;
    c.pstride = (long)p.ny * p.ld;
    c.tpp = ktiles;
    return col(p.ny, c, p.nz * ktiles, 7, +1, p.tw_y, s);
}

// x pass A -> B and the forward y transform of B's 12 fields.
int x_and_y(const MhdPlan& p, hipStream_t s, EventTimer* tm)
{
    int rc;
    double2* B = p.b.as<double2>();
    XArgs x{p.a.as<double2>(), B, p.fsz, p.ld, std::min(p.nh, 8 * p.ktiles),
            1.0 / ((double)p.nx * (double)p.ny * (double)p.nz), p.cs * p.cs};
    if (tm) tm->begin(1, s);
    if ((rc = xpass(p, x, s))) return rc;
    if (tm) tm->end(1, s);
    ColArgs c{};
    for (int f = 0; f < 12; ++f) c.src[f] = c.dst[f] = B + f * p.fsz;
    c.es = p.ld;
    c.pstride = (long)p.ny * p.ld;
    c.tpp = p.ktiles;
    c.skip = p.yskip.as<int2>();
    if (tm) tm->begin(2, s);
    if ((rc = col(p.ny, c, p.nz * p.ktiles, 12, -1, p.tw_y, s))) return rc;
    if (tm) tm->end(2, s);
    return TARA_OK;
}

ZArgs zargs(const MhdPlan& p, double2* const st[7], double2* const sn[7], double2* const out[7], double dt)
{
    ZArgs z{};
    z.b = p.b.as<double2>();
    z.fs = p.fsz;
    for (int f = 0; f < 7; ++f) {
        z.st[f] = st[f];
        z.sn[f] = sn[f];
        z.out[f] = out[f];
    }
    z.az = p.az.as<double2>();
    z.kx = p.kx.as<double>();
    z.ky = p.ky.as<double>();
    z.kz = p.kz.as<double>();
    z.imin = p.imin.as<int>();
    z.live = p.live.as<int>();
    z.ny = p.ny;
    z.ld = p.ld;
    z.mu = p.mu;
    z.eta = p.eta;
    z.dt = dt;
    z.bad = p.bad.as<int>();
    return z;
}

}  // namespace

int mhd_rhs_stage(const MhdPlan& p, double2* const st[7], double2* const out[7], hipStream_t s, EventTimer* tm)
{
    int rc;
    double2* A = p.a.as<double2>();
    if (tm) tm->begin(0, s);
    if ((rc = inverse_z(p, st, A, s)) || (rc = inverse_y(p, A, A, p.ld / 8, s))) return rc;
    if (tm) tm->end(0, s);
    if ((rc = x_and_y(p, s, tm))) return rc;
    if (tm) tm->begin(3, s);
    if ((rc = zpass(p, MHD_RHS, false, zargs(p, st, st, out, 0.0), s))) return rc;
    if (tm) tm->end(3, s);
    TARA_HIP(hipGetLastError());
    return TARA_OK;
}

int mhd_advance(const MhdPlan& p, double2* st[7], double2* mom[3], double2* const hist[7], int nsteps, double dt,
                hipStream_t s, EventTimer* tm)
{
    if (nsteps <= 0) return TARA_OK;
    int rc;
    TARA_CHECK(p.az.p, TARA_ERR_STATE, "3D MHD: plan without its stepping work space");
    for (int k = 0; k < nsteps; ++k) {
        if (tm) tm->begin(0, s);
        if (k == 0 && (rc = inverse_z(p, st, p.az.as<double2>(), s))) return rc;
        // the first step fills all of A; later only the kx tiles with a live mode change
        if ((rc = inverse_y(p, p.az.as<double2>(), p.a.as<double2>(), k == 0 ? p.ld / 8 : p.ktiles, s))) return rc;
        if (tm) tm->end(0, s);
        if ((rc = x_and_y(p, s, tm))) return rc;
        double2* sn[7];
        for (int f = 0; f < 7; ++f) sn[f] = f >= 1 && f <= 3 ? mom[f - 1] : st[f];
        if (tm) tm->begin(3, s);
        if ((rc = zpass(p, MHD_AB2, k + 1 < nsteps, zargs(p, st, sn, hist, dt), s))) return rc;
        if (tm) tm->end(3, s);
        for (int f = 0; f < 3; ++f) std::swap(st[1 + f], mom[f]);
    }
    TARA_HIP(hipGetLastError());
    return TARA_OK;
}

}  // namespace tara
