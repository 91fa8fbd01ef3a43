// 2D incompressible hydro in vorticity-streamfunction form on gfx950:
// the right-hand side of src/derive2csh.f95 and the AB2 / RK4 updates
// (src/ab2csh.f95; classic RK4), as three fused HBM sweeps per RHS.
//
// Device layout: the state half spectra are stored ky-major ("transposed"),
// element (kx = i, ky = j) at i*Ny + j, so a kx column (one y transform) is a
// contiguous Ny-element run.  The intermediates are stored in row groups
// interleaved per kx: G0..G3 in 2-row (Nx = 4096) or 4-row groups (blkg), H in
// 8-row groups (blk8, element (i, j) at ((j/8)*Nh + i)*8 + j%8): a y pass reads
// or writes a column as 32- to 128-byte runs, and an x-pass workgroup of fewer
// rows than a group reads pieces of those runs whose other pieces belong to the
// neighbouring workgroups, which the XCD-aware mapping runs next to it.  The
// reference's (Nh, Ny) kx-fastest arrays are converted on upload / download
// (layout.hip).
//
//   pass 1  k_csh_yinv : per kx column read omega_hat, form the four spectra of
//                        derive2csh.f95:29-71 (ux = i ky psi, uy = -i kx psi,
//                        psi = omega/k^2, psi(0,0) = 0; i kx omega, i ky omega)
//                        as the pairs ux +- i uy, dx omega +- i dy omega that the
//                        x pass transforms, run the backward y FFTs -> G0..G3.
//                        (4096^2 RK4 step 1.51 -> 1.44 ms, 512 runs of 128^2 ..
//                        512^2 6.04 -> 5.84, against the four fields themselves,
//                        each of which the x pass loaded twice.)
//   pass 2  k_csh_x    : per RB rows, four x c2r (two pairs),
//                        normalise by Nx*Ny and form ux*d_x omega + uy*d_y omega
//                        (derive2csh.f95:89-98), one x r2c -> H.  (The reference
//                        transforms the two products separately (:100-106); the
//                        sum is transformed once, which is the same linear map.)
//   pass 3  k_csh_yfwd : per kx column, forward y FFT of H, circular dealias
//                        sqrt(kx^2+ky^2) >= (Nx+Ny)/6 on the nonlinear part only
//                        (:108-125), add nu k^2 omega (:127-139), negate
//                        (:141-145), then the fused update (RHS / AB2 / RK4 stage).
//
// What the passes carry (CshPlan::hk, band): the nonlinear term is zero outside the
// dealiasing circle, so H is stored, read and transformed for kx < hk only (a
// third of its columns less), whatever the state; and a state that is zero
// outside the circle stays so, so its passes leave the columns kx >= hk of
// G0..G3 and the state's modes outside the circle alone (all but 35 % of them at
// Nx = Ny).  The passes' time at 1024^2 and above is that traffic and what it
// waits for: RK4 step 4096^2 2.30 -> 1.61 ms, 2048^2 0.58 -> 0.415, 1024^2 0.147
// -> 0.139 for such states; 1024^2 0.147 -> 0.143 for others.
//
// Wavenumbers: derive2csh uses pi = 3.1428 (a default-real literal) and
// Lx = Ly = 2 pi (:16-21), so kx = i-1 and ky = j-1 or j-1-Ny are exact integers;
// the host builds the tables with that exact expression (csh_plan_init).
#include <algorithm>
#include <type_traits>

#include "csh2d_dev.h"

namespace tara {

// --------------------------------------------------------------------- pass 1
// Shape of the inverse y pass.  At Ny = 4096 (512 threads per column) two
// columns share a workgroup with their lanes interleaved (column = lane parity):
// a wave's stores then cover both columns of each 2-row group of G0..G3
// together (64 B), where one column per workgroup wrote 32-byte pieces (two
// workgroups of one column a CU: 4096^2 RK4 step 1.81 against 1.51 ms).  They share
// one LDS buffer (rf_fft_w).  Other lengths, and the screened form (psi kept live, more
// registers), keep the contiguous shape of the y passes.
template <int NY, bool SCR>
struct YiShape {
    static constexpr int T = RY<NY>::T;
    static constexpr bool IL = csh_yinv_interleaved(NY, SCR);
    static constexpr int CB = csh_yinv_cols(NY, SCR);
    static_assert(IL || CB == YShape<NY>::CB, "contiguous shape differs from the y passes'");
    static constexpr int NT = CB * T;
    static constexpr int LDSC = IL ? NY : RY<NY>::LDS;  // per-column exchange buffer
    // Ny <= 512: at least 56 KB of LDS per workgroup, which holds the pass to
    // two 256-thread workgroups per CU.  Its registers would allow three, and
    // at three the ensemble step (128-512 grids) measured 6.67 against 6.42 ms.
    static constexpr int LDS_ELEMS = (!IL && NY <= 512 && CB * LDSC < 56 * 1024 / 16) ? 56 * 1024 / 16 : CB * LDSC;
};

// The inverse y pass of one kx column i given omega_hat (wv, at rf_first_idx
// positions): forms the four spectra of derive2csh.f95:29-71 (i kx omega,
// i ky omega, i ky psi, -i kx psi; psi = omega/k^2, psi(0,0) = 0), or of
// derive2css.f95:22-52 when SCR (screened), pairwise (x_c2r_pair), runs the backward y FFTs and writes
// G0..G3 (row-group stride ld).  sq: the column as the thread sees it.
template <int NY, bool SCR, int GS, class SQ>
__device__ __forceinline__ void csh_yinv_column(double2 (&wv)[RY<NY>::E], int i, bool live, const SQ& sq,
                                                const double2* tw, double lam, int ld,
                                                double2* __restrict__ g0, double2* __restrict__ g1,
                                                double2* __restrict__ g2, double2* __restrict__ g3)
{
    constexpr int E = RY<NY>::E;
    const double kxv = (double)i;  // derive2csh's kx = i-1 exactly (checked on the host)
    // screened: psi = omega/(k^2 + lambda) with psi(0,0) = 0, omega_d = k^2 psi;
    // the derivatives below act on omega_d, psi is kept in ps.
    double2 ps[SCR ? E : 1];
    if constexpr (SCR) {
#pragma unroll
        for (int e = 0; e < E; ++e) {
            const int j = rf_first_idx<NY, csh_yem(NY)>(sq.t, e);
            const double kyv = csh_ky<NY>(j);
            const double k2 = kxv * kxv + kyv * kyv;
            const double den = k2 + lam;
            ps[e] = (i == 0 && j == 0) ? make_double2(0.0, 0.0) : make_double2(wv[e].x / den, wv[e].y / den);
            wv[e] = make_double2(k2 * ps[e].x, k2 * ps[e].y);
        }
    }
    // i kx omega +- i (i ky omega) first; then omega -> psi in place; then
    // i ky psi +- i (-i kx psi).
#pragma unroll 1
    for (int f = 0; f < 4; ++f) {
        double2 v[E];
        // the slot, opaque per transform: the index arithmetic of the stores is
        // recomputed here rather than hoisted out of the loop and held in registers
        const int tt = rf_opaque(sq.t);
        if (f == 2) {
#pragma unroll
            for (int e = 0; e < E; ++e) {
                if constexpr (SCR) {
                    wv[e] = ps[e];
                } else {
                    const double kyv = csh_ky<NY>(rf_first_idx<NY, csh_yem(NY)>(tt, e));
                    const double k2 = kxv * kxv + kyv * kyv;
                    wv[e] = (k2 != 0.0) ? make_double2(wv[e].x / k2, wv[e].y / k2) : make_double2(0.0, 0.0);
                }
            }
        }
#pragma unroll
        for (int e = 0; e < E; ++e) {
            const double kyv = csh_ky<NY>(rf_first_idx<NY, csh_yem(NY)>(tt, e));
            const double cr = f == 0 ? -kyv : f == 1 ? kyv : f == 2 ? kxv : -kxv, ci = f < 2 ? kxv : kyv;
            const double2 z = wv[e];
            v[e] = make_double2(cr * z.x - ci * z.y, cr * z.y + ci * z.x);
        }
        sq.template fft<+1>(v, tw);
        // G0, G1 = ux +- i uy (f 2, 3), G2, G3 = d omega/dx +- i d omega/dy (f 0, 1)
        double2* o = f == 0 ? g2 : f == 1 ? g3 : f == 2 ? g0 : g1;
        if (live) {
#pragma unroll
            for (int e = 0; e < E; ++e) o[blkg(i, rf_final_idx<NY, csh_yem(NY)>(tt, e), ld, GS)] = v[e];
        }
    }
}

// The columns of a y pass's workgroup: CB side by side, of T threads each, or
// (IL) interleaved over its lanes.  Columns of several wavefronts at radix cap 8
// take rf_fft_w; columns of part of a wavefront exchange within it (171 runs of
// 256^2: 1.18 against 1.20 ms a step with workgroup barriers).  A column that is
// one whole wavefront (Ny = 512) keeps the barriers: its four columns write pieces
// of the same 64-byte groups, and let apart they measured 4.55 against 4.36 ms
// (171 runs of 512^2).
template <int NY, int CB, bool IL>
__device__ __forceinline__ auto csh_columns(double2* lds, int* c)
{
    constexpr int T = RY<NY>::T, EM = csh_yem(NY);
    if constexpr (EM == 8 && T >= 128) {
        if constexpr (IL) {
            const RfWide<NY, CB> sq((int)threadIdx.x, lds);
            *c = sq.c;
            return sq;
        } else {
            *c = (int)threadIdx.x / T;
            return RfWide<NY, 1>((int)threadIdx.x % T, lds + *c * RY<NY>::LDS);
        }
    } else {
        static_assert(!IL, "interleaved columns are those of rf_fft_w");
        *c = (int)threadIdx.x / T;
        return RfSeq<NY, EM, (T < 64)>{(int)threadIdx.x % T, lds + *c * RY<NY>::LDS};
    }
}

template <int NY, bool SCR, int GS>
__global__ __launch_bounds__((YiShape<NY, SCR>::NT), (YiShape<NY, SCR>::IL ? 4 : 1)) void k_csh_yinv(const double2* w, int nh,
                                                                    double2* __restrict__ g0, double2* __restrict__ g1,
                                                                    double2* __restrict__ g2, double2* __restrict__ g3,
                                                                    const double2* tw, double lam, int ld, size_t bs,
                                                                    CshBand bd)
{
    // batched runs: blockIdx.y selects the run, every field is strided by bs
    const size_t rb = blockIdx.y * bs;
    w += rb;
    g0 += rb;
    g1 += rb;
    g2 += rb;
    g3 += rb;
    using S = YiShape<NY, SCR>;
    constexpr int E = RY<NY>::E, T = S::T;
    __shared__ double2 lds[S::LDS_ELEMS];
    int c;
    const auto sq = csh_columns<NY, S::CB, S::IL>(lds, &c);
    const int t = sq.t;
    // a limited state: the kx columns that hold something, and of them the modes
    const bool lim = bd.limited(blockIdx.y);
    const int ncol = lim ? bd.hk : nh, ntile = (ncol + S::CB - 1) / S::CB;
    if ((int)blockIdx.x >= ntile) return;
    const int i = xcd_remap(blockIdx.x, ntile) * S::CB + c;
    const bool live = S::CB == 1 || i < ncol;
    const size_t col = (size_t)(live ? i : 0) * NY;
    double2 wv[E];
    // Separate loads: a test of the circle before each would put its latency between
    // every two loads of a state that holds everything.
    if (lim) {
#pragma unroll
        for (int e = 0; e < E; ++e) {
            const int j = rf_first_idx<NY, csh_yem(NY)>(t, e);
            wv[e] = make_double2(0.0, 0.0);
            if (live && i < bd.imin[j]) wv[e] = w[col + j];
        }
    } else {
#pragma unroll
        for (int e = 0; e < E; ++e)
            wv[e] = live ? w[col + rf_first_idx<NY, csh_yem(NY)>(t, e)] : make_double2(0.0, 0.0);
    }
    csh_yinv_column<NY, SCR, GS>(wv, i, live, sq, tw, lam, ld, g0, g1, g2, g3);
}

// --------------------------------------------------------------------- pass 2
// Shape of the x pass: EM complex elements per thread (4, 8, 16: radix-4, -8,
// -16 passes), RB rows per workgroup, SPLIT: the FFT exchanges go through LDS as
// doubles in two rounds (half the LDS, so that two workgroups share a CU).
template <int NX, int EM, int RB, bool SPLIT>
struct XShape {
    static constexpr int M = NX / 2;
    static constexpr int T = RF<NX, EM>::T;    // threads per row (backward transforms, length NX)
    static constexpr int TM = RF<M, EM>::T;    // of which active in the forward half-length transform
    static constexpr int NT = RB * T;
    // rows of several wavefronts take rf_fft_w, their half-length transform too
    static constexpr bool WIDE = EM == 8 && !SPLIT && T >= 128 && RB <= 8;
    static constexpr bool WIDEM = WIDE && TM >= 128;
    // Per-row exchange buffer (complex elements).  Rows are interleaved across
    // lanes, so successive row buffers are offset by 4 elements (64 B) to land
    // on different LDS banks.
    static constexpr int LDSR = (SPLIT ? RF<NX, EM>::LDS / 2 : RF<NX, EM>::LDS) + 4;
    // the forward half-length transform must use exactly half of the row's threads
    static constexpr bool OK = RB * LDSR * 16 <= 160 * 1024 && NT <= 1024 && NT >= 64 && 2 * TM == T;
};

template <int NX, int EM, int RB, bool SPLIT>
__global__ __launch_bounds__((XShape<NX, EM, RB, SPLIT>::NT), (XShape<NX, EM, RB, SPLIT>::WIDE ? 4 : 1)) void k_csh_x(
    const double2* g0, const double2* g1, const double2* g2, const double2* g3, double scale,
    double2* __restrict__ h, const double2* tw_n, const double2* tw_m, const double2* rctw, size_t bs, CshBand bd)
{
    const size_t rb = blockIdx.y * bs;  // batched runs
    const int lim = bd.limited(blockIdx.y) ? bd.hk : bd.nh;
    g0 += rb;
    g1 += rb;
    g2 += rb;
    g3 += rb;
    h += rb;
    using S = XShape<NX, EM, RB, SPLIT>;
    static_assert(S::OK, "x pass shape does not fit");
    constexpr int E = RF<NX, EM>::E, EH = RF<S::M, EM>::E, T = S::T, M = S::M;
    __shared__ double2 lds[RB * S::LDSR];
    const int r = threadIdx.x % RB, tk = threadIdx.x / RB;  // row fastest: RB-row chunks per kx
    const int j = xcd_remap(blockIdx.x, gridDim.x) * RB + r;
    double2* xl = lds + r * S::LDSR;
    const auto sq = [&] {
        if constexpr (S::WIDE)
            return RfWide<NX, RB>((int)threadIdx.x, lds);
        else
            return RfSeq<NX, EM, false, SPLIT>{tk, xl};
    }();
    const int t = sq.t;
    double nl[E];
    double2 u[E], v[E];
    x_c2r_pair<NX, EM, true>(g0, g1, j, lim, sq, tw_n, u);   // ux + i uy
    x_c2r_pair<NX, EM, true>(g2, g3, j, lim, sq, tw_n, v);   // d omega/dx + i d omega/dy
#pragma unroll
    for (int e = 0; e < E; ++e) nl[e] = (u[e].x * v[e].x + u[e].y * v[e].y) * scale;
    // forward x transform of the real product row: pack z[m] = nl[2m] + i nl[2m+1]
    // for the half-length FFT (threads t < TM carry it; the others only meet its
    // barriers where they fill whole waves, else run the same code on the
    // unused upper half of the row buffer so every barrier matches).
    double* xr = reinterpret_cast<double*>(xl);
    if constexpr (S::WIDE) __syncthreads();
#pragma unroll
    for (int e = 0; e < E; ++e) xr[rf_final_idx<NX, EM>(t, e)] = nl[e];
    __syncthreads();
    double2 z[EH];
    const bool half = tk < S::TM;  // threadIdx.x < TM RB
    int tm = tk % S::TM;
    if constexpr (S::WIDEM) tm = RfW<M, RB>((int)threadIdx.x % (S::TM * RB)).t;
#pragma unroll
    for (int e = 0; e < EH; ++e) {
        const int m = rf_first_idx<M, EM>(tm, e);
        z[e] = make_double2(xr[2 * m], xr[2 * m + 1]);
    }
    // The unpacking roots of this thread's kx = t + u T, fetched now, before
    // any store (loads and stores share one in-order counter: a root loaded
    // between the stores would also wait for the stores before it).  4096^2
    // x pass 0.274 against 0.278 ms.
    constexpr int NK = M / T;
    double2 wk[NK];
#pragma unroll
    for (int u = 0; u < NK; ++u) wk[u] = rctw[tk + u * T];
    __syncthreads();
    if constexpr (S::WIDEM) {
        if (half) {
            const RfWide<M, RB> sm((int)threadIdx.x, lds);
            sm.template fft<-1>(z, tw_m);
        } else {  // the barriers of rf_fft_w
            __syncthreads();
            __syncthreads();
        }
        __syncthreads();  // the waves' last exchanges
    } else if constexpr ((S::TM * RB) % 64 == 0) {
        // the threads t >= TM (threadIdx.x >= TM RB) fill whole waves: they meet
        // the transform's barriers without running it
        if (half)
            rf_fft<M, -1, EM, false, SPLIT>(z, tm, xl, tw_m);
        else
            rf_fft_barriers_only<M, EM, SPLIT>();
    } else {
        constexpr int HALF = SPLIT ? RF<M, EM>::LDS / 2 : RF<M, EM>::LDS;  // upper half, complex elements
        double2* zl = xl + (half ? 0 : HALF);
        rf_fft<M, -1, EM, false, SPLIT>(z, tm, zl, tw_m);
    }
    if (half) {
#pragma unroll
        for (int e = 0; e < EH; ++e) xl[rf_pad(rf_final_idx<M, EM>(tm, e))] = z[e];
    }
    __syncthreads();
#pragma unroll
    for (int u = 0; u < NK; ++u) {  // consecutive t -> consecutive kx
        const int k = tk + u * T;
        if (k >= bd.hk) continue;  // dealiased away at every ky
        const double2 zk = xl[rf_pad(k)];
        const double2 zmk = xl[rf_pad(k == 0 ? 0 : M - k)];
        double2 xm;
        h[blk8(k, j, M + 1)] = r2c_unpack_w(zk, zmk, k, wk[u], &xm);
        if (k == 0 && M < bd.hk) h[blk8(M, j, M + 1)] = xm;
    }
}

// --------------------------------------------------------------------- pass 3
template <int NY, int MODE>
__global__ __launch_bounds__(YShape<NY>::NT) void k_csh_yfwd(YfwdArgs a, CshBand bd, const double2* tw)
{
    const size_t rb = blockIdx.y * a.bs;
    a.h += rb;
    a.ws += rb;
    if (a.base) a.base += rb;
    if (a.aux) a.aux += rb;
    if (a.next) a.next += rb;
    if (a.nus) a.nu = a.nus[blockIdx.y];
    using S = YShape<NY>;
    constexpr int E = RY<NY>::E, T = S::T;
    __shared__ double2 lds[S::CB * RY<NY>::LDS];
    int c;
    const auto sq = csh_columns<NY, S::CB, false>(lds, &c);
    const int t = sq.t;
    // tiles below hk have a nonlinear term; the others only the viscous one, and a
    // limited state nothing
    const bool lim = bd.limited(blockIdx.y);
    const int nfwd = (bd.hk + S::CB - 1) / S::CB;
    if (lim && (int)blockIdx.x >= nfwd) return;
    const int tile = csh_tile(blockIdx.x, nfwd, gridDim.x);
    const int i = tile * S::CB + c;
    const bool live = S::CB == 1 || i < (lim ? bd.hk : a.nh);
    const size_t col = (size_t)(live ? i : 0) * NY;
    double2 v[E];
    if (tile < nfwd) {
#pragma unroll
        for (int e = 0; e < E; ++e)
            v[e] = S::CB == 1 || i < bd.hk ? a.h[blk8(i, rf_first_idx<NY, csh_yem(NY)>(t, e), a.nh)]
                                           : make_double2(0.0, 0.0);
        sq.template fft<-1>(v, tw);
    }
    if (!live) return;
    const double kxv = (double)i;
    bool finite = true;  // the new state's values (AB2, RK4 stage 4)
    auto update = [&](auto limited) {
#pragma unroll
        for (int e = 0; e < E; ++e) {
            const int j = rf_final_idx<NY, csh_yem(NY)>(t, e);
            const size_t q = col + j;
            double2 nl = v[e];
            if (i >= a.imin[j]) {
                if constexpr (limited.value) continue;  // zero, and stays so
                nl = make_double2(0.0, 0.0);
            }
            const double kyv = csh_ky<NY>(j);
            const double k2 = kxv * kxv + kyv * kyv;
            double2 wn, av;
            csh_update<MODE>(a, q, i == 0 && j == 0, nl, a.ws[q], k2, &wn, &av);
            finite = csh_store<MODE>(a, q, wn, av) && finite;
        }
    };
    // apart as in k_csh_yinv
    if (lim)
        update(std::true_type{});
    else
        update(std::false_type{});
    if (!finite && a.bad) a.bad[blockIdx.y] = 1;
}

// ------------------------------------------------------- passes 3 + 1 fused
// The forward y pass of one stage followed by the inverse y pass of the stage
// that comes next, per kx column (derive2csh only).  The update leaves the next
// stage's input (RK4: the stage field; AB2 and the last RK4 stage: the new
// state) in registers, and the four spectra of it are transformed and written
// to G0..G3 without reading it back: one field read less per stage.  Shape and
// LDS as the inverse y pass; the forward y pass of H uses the same lanes.
template <int NY, int MODE, int GS>
__global__ __launch_bounds__((YiShape<NY, false>::NT), (YiShape<NY, false>::IL ? 4 : 1)) void k_csh_yfwd_inv(
    YfwdArgs a, CshBand bd, const double2* tw, double2* __restrict__ g0, double2* __restrict__ g1, double2* __restrict__ g2,
    double2* __restrict__ g3, int ld)
{
    static_assert(MODE != CSH_RHS, "the fused pass needs a stage update");
    const size_t rb = blockIdx.y * a.bs;
    a.h += rb;
    a.ws += rb;
    a.base += rb;
    a.aux += rb;
    if (a.next) a.next += rb;
    g0 += rb;
    g1 += rb;
    g2 += rb;
    g3 += rb;
    if (a.nus) a.nu = a.nus[blockIdx.y];
    a.screened = 0;  // derive2csh only
    using S = YiShape<NY, false>;
    constexpr int E = RY<NY>::E, T = S::T;
    __shared__ double2 lds[S::LDS_ELEMS];
    int c;
    const auto sq = csh_columns<NY, S::CB, S::IL>(lds, &c);
    const int t = sq.t;
    // as k_csh_yfwd: tiles with a nonlinear term first, a limited state's only
    const bool lim = bd.limited(blockIdx.y);
    const int nfwd = (bd.hk + S::CB - 1) / S::CB;
    if (lim && (int)blockIdx.x >= nfwd) return;
    const int tile = csh_tile(blockIdx.x, nfwd, gridDim.x);
    const int i = tile * S::CB + c;
    const bool live = S::CB == 1 || i < (lim ? bd.hk : a.nh);
    const size_t col = (size_t)(live ? i : 0) * NY;
    double2 v[E];
    if (tile < nfwd) {
#pragma unroll
        for (int e = 0; e < E; ++e)
            v[e] = S::CB == 1 || i < bd.hk ? a.h[blk8(i, rf_first_idx<NY, csh_yem(NY)>(t, e), a.nh)]
                                           : make_double2(0.0, 0.0);
        sq.template fft<-1>(v, tw);
    }
    const double kxv = (double)i;
    bool finite = true;  // the new state's values (AB2, RK4 stage 4)
    auto update = [&](auto limited) {
#pragma unroll
        for (int e = 0; e < E; ++e) {
            const int j = rf_final_idx<NY, csh_yem(NY)>(t, e);
            const size_t q = col + j;
            const bool in = live && i < a.imin[j];
            if (!in && (limited || !live)) {
                v[e] = make_double2(0.0, 0.0);
                continue;
            }
            const double2 nl = in ? v[e] : make_double2(0.0, 0.0);
            const double kyv = csh_ky<NY>(j);
            double2 wn, av;  // wn: the next stage's input
            csh_update<MODE>(a, q, false, nl, a.ws[q], kxv * kxv + kyv * kyv, &wn, &av);
            finite = csh_store<MODE>(a, q, wn, av) && finite;
            v[e] = wn;
        }
    };
    // apart as in k_csh_yinv; with one workgroup of 16 wavefronts a CU (IL) the other
    // waves cover the latency, and together they are faster (4096^2 RK4 step of a
    // general state 2.161 against 2.177 ms)
    if constexpr (S::IL)
        update(lim);
    else if (lim)
        update(std::true_type{});
    else
        update(std::false_type{});
    if (!finite && a.bad) a.bad[blockIdx.y] = 1;
    sq.final_to_first(v);
    csh_yinv_column<NY, false, GS>(v, i, live, sq, tw, 0.0, ld, g0, g1, g2, g3);
}

// ------------------------------------------------------------ pointwise AB2
__global__ void k_ab2(const double2* w, double2* __restrict__ wn, const double2* fo,
                      const double2* fn, double dt, size_t n)
{
    for (size_t q = blockIdx.x * (size_t)blockDim.x + threadIdx.x; q < n; q += (size_t)gridDim.x * blockDim.x) {
        const double2 a = w[q], o = fo[q], f = fn[q];
        wn[q] = make_double2(a.x + (1.5 * f.x - 0.5 * o.x) * dt, a.y + (1.5 * f.y - 0.5 * o.y) * dt);
    }
}

// ------------------------------------------------------------ a state set anew
// Zeroes a run's history (naux elements) and, with band, clears *band if the state w
// has a mode outside the dealiasing circle.  As launches of their own beside memsets of
// history and flag, finding the support took 15 to 25 us more of a call of 50 us
// (tara_ens_set_omega, batches on the large grids' passes); as one launch whose last
// workgroup sets the flag, 45 more at 1024^2, for the counting and its fences.
__global__ __launch_bounds__(256) void k_csh_state_set(const double2* w, const int* imin, int nh, int ny, double2* aux,
                                                       size_t naux, int* band)
{
    const size_t first = blockIdx.x * (size_t)blockDim.x + threadIdx.x, step = (size_t)gridDim.x * blockDim.x;
    for (size_t q = first; q < naux; q += step) aux[q] = make_double2(0.0, 0.0);
    if (!band) return;
    bool any = false;
    for (size_t q = first; q < (size_t)nh * ny; q += step) {
        const int i = (int)(q / ny), j = (int)(q % ny);
        if (i < imin[j]) continue;
        const double2 z = w[q];
        any = any || !(z.x == 0.0 && z.y == 0.0);
    }
    if (any) *band = 0;
}

__global__ void k_csh_state_flags(int* bad, int* band)
{
    *bad = 0;
    *band = 1;
}

// ------------------------------------------------------------------ dispatch
template <int NY, bool SCR, int GS>
static int launch_yinv_t(const CshPlan& p, const double2* w, const CshPhys& ph, hipStream_t st)
{
    using S = YiShape<NY, SCR>;
    hipLaunchKernelGGL((k_csh_yinv<NY, SCR, GS>), dim3((p.nh + S::CB - 1) / S::CB, p.batch), dim3(S::NT), 0, st, w,
                       p.nh, p.g[0].as<double2>(), p.g[1].as<double2>(), p.g[2].as<double2>(), p.g[3].as<double2>(),
                       p.tw_y, ph.lambda, p.gld, p.bstride, csh_band(p));
    return TARA_OK;
}

// Below Ny = 256 only batches come here (csh_small): square grids of derive2csh.
template <int NY>
static int launch_yinv(const CshPlan& p, const double2* w, const CshPhys& ph, hipStream_t st)
{
    if constexpr (NY >= 256) {
        if (p.gsh == 1)
            return ph.screened ? launch_yinv_t<NY, true, 1>(p, w, ph, st) : launch_yinv_t<NY, false, 1>(p, w, ph, st);
        if (ph.screened) return launch_yinv_t<NY, true, 2>(p, w, ph, st);
    }
    TARA_CHECK(p.gsh == 2 && !ph.screened, TARA_ERR_UNSUPPORTED, "inverse y pass of large grids at %dx%d", p.nx, p.ny);
    return launch_yinv_t<NY, false, 2>(p, w, ph, st);
}

// x-pass shapes the autotuner chooses among (launch_x).  Shape 0 is
// RB = min(8, 512 / T) at EM = 8 without splitting: two workgroups a CU, one in
// memory while the other transforms (RK4 step, one workgroup of twice the rows ->
// two: 1024^2 0.172 -> 0.145 ms, 2048^2 0.303 -> 0.297, 2048 x 512 0.166 -> 0.151).
// Nx = 4096 keeps two rows and one workgroup: of its 2-row groups a single row
// reads half of every line (4096^2 1.51 ms, single rows 1.60).
// Shape kXPairs runs a row's two field pairs side by side (csh2d_pairs.hip).
constexpr int kNumXCands = 10;

template <int NX, int EM>
constexpr int default_rb()
{
    return NX == 4096 && EM == 8 ? 2 : (512 / RF<NX, EM>::T) < 1 ? 1 : (512 / RF<NX, EM>::T) > 8 ? 8 : (512 / RF<NX, EM>::T);
}

template <int NX, int EM, int RB, bool SPLIT>
static int launch_x_shape(const CshPlan& p, hipStream_t st)
{
    using S = XShape<NX, EM, RB, SPLIT>;
    if constexpr (!S::OK) {
        set_error("x pass shape unsupported at Nx=%d", NX);
        return TARA_ERR_UNSUPPORTED;
    } else {
        TARA_CHECK(p.ny % RB == 0, TARA_ERR_UNSUPPORTED, "Ny=%d not a multiple of %d", p.ny, RB);
        const double scale = 1.0 / ((double)p.nx * (double)p.ny * (double)p.nx * (double)p.ny);
        const double2* twn = EM == 16 ? p.tw_xn16 : EM == 4 ? p.tw_xn4 : p.tw_xn;
        const double2* twm = EM == 16 ? p.tw_x16 : EM == 4 ? p.tw_x4 : p.tw_x;
        TARA_CHECK(twn && twm, TARA_ERR_UNSUPPORTED, "x pass shape without its twiddle tables");
        hipLaunchKernelGGL((k_csh_x<NX, EM, RB, SPLIT>), dim3(p.ny / RB, p.batch), dim3(S::NT), 0, st,
                           p.g[0].as<double2>(), p.g[1].as<double2>(), p.g[2].as<double2>(), p.g[3].as<double2>(),
                           scale, p.h.as<double2>(), twn, twm, p.rctw, p.bstride, csh_band(p));
        return TARA_OK;
    }
}

template <int NX>
static int launch_x(const CshPlan& p, hipStream_t st)
{
    switch (p.xcfg) {
        case 0: return launch_x_shape<NX, 8, default_rb<NX, 8>(), false>(p, st);
        case 1: return launch_x_shape<NX, 16, 2, true>(p, st);
        case 2: return launch_x_shape<NX, 8, 1, true>(p, st);
        case 3: return launch_x_shape<NX, 16, 4, true>(p, st);
        case 4: return launch_x_shape<NX, 8, 2, true>(p, st);
        case 5: return launch_x_shape<NX, 16, 1, false>(p, st);
        case 6: return launch_x_shape<NX, 4, 1, false>(p, st);
        case 7: return launch_x_shape<NX, 4, 2, false>(p, st);
        case 8: return launch_x_shape<NX, 4, 4, true>(p, st);
        case kXPairs: return csh_x_pairs(p, st);
        default: set_error("x pass shape %d unknown", p.xcfg); return TARA_ERR_ARG;
    }
}

template <int NX>
static bool x_shape_ok(int c, int ny)
{
    switch (c) {
        case 0: return XShape<NX, 8, default_rb<NX, 8>(), false>::OK && ny % default_rb<NX, 8>() == 0;
        case 1: return XShape<NX, 16, 2, true>::OK && ny % 2 == 0;
        case 2: return XShape<NX, 8, 1, true>::OK;
        case 3: return XShape<NX, 16, 4, true>::OK && ny % 4 == 0;
        case 4: return XShape<NX, 8, 2, true>::OK && ny % 2 == 0;
        case 5: return XShape<NX, 16, 1, false>::OK;
        case 6: return XShape<NX, 4, 1, false>::OK;
        case 7: return XShape<NX, 4, 2, false>::OK && ny % 2 == 0;
        case 8: return XShape<NX, 4, 4, true>::OK && ny % 4 == 0;
        case kXPairs: return csh_x_pairs_ok(NX, ny);
        default: return false;
    }
}

template <int NY>
static int launch_yfwd(const CshPlan& p, int mode, const YfwdArgs& a, hipStream_t st)
{
    using S = YShape<NY>;
    dim3 g((p.nh + S::CB - 1) / S::CB, p.batch), b(S::NT);
    switch (mode) {
        case CSH_RHS: hipLaunchKernelGGL((k_csh_yfwd<NY, CSH_RHS>), g, b, 0, st, a, csh_band(p), p.tw_y); break;
        case CSH_AB2: hipLaunchKernelGGL((k_csh_yfwd<NY, CSH_AB2>), g, b, 0, st, a, csh_band(p), p.tw_y); break;
        case CSH_RK4_1: hipLaunchKernelGGL((k_csh_yfwd<NY, CSH_RK4_1>), g, b, 0, st, a, csh_band(p), p.tw_y); break;
        case CSH_RK4_2: hipLaunchKernelGGL((k_csh_yfwd<NY, CSH_RK4_2>), g, b, 0, st, a, csh_band(p), p.tw_y); break;
        case CSH_RK4_3: hipLaunchKernelGGL((k_csh_yfwd<NY, CSH_RK4_3>), g, b, 0, st, a, csh_band(p), p.tw_y); break;
        case CSH_RK4_4: hipLaunchKernelGGL((k_csh_yfwd<NY, CSH_RK4_4>), g, b, 0, st, a, csh_band(p), p.tw_y); break;
        default: set_error("bad mode %d", mode); return TARA_ERR_ARG;
    }
    return TARA_OK;
}

#define TARA_CSH_SWITCH(n, FN, ...)                 \
    switch (n) {                                    \
        case 32: return FN<32>(__VA_ARGS__);        \
        case 64: return FN<64>(__VA_ARGS__);        \
        case 128: return FN<128>(__VA_ARGS__);      \
        case 256: return FN<256>(__VA_ARGS__);      \
        case 512: return FN<512>(__VA_ARGS__);      \
        case 1024: return FN<1024>(__VA_ARGS__);    \
        case 2048: return FN<2048>(__VA_ARGS__);    \
        case 4096: return FN<4096>(__VA_ARGS__);    \
        default: set_error("unsupported transform length %d", n); return TARA_ERR_UNSUPPORTED; \
    }

static int yinv(const CshPlan& p, const double2* w, const CshPhys& ph, hipStream_t st)
{
    TARA_CSH_SWITCH(p.ny, launch_yinv, p, w, ph, st)
}
static int xpass(const CshPlan& p, hipStream_t st) { TARA_CSH_SWITCH(p.nx, launch_x, p, st) }
template <int NX>
static int shape_ok_n(int c, int ny)
{
    return x_shape_ok<NX>(c, ny) ? 1 : 0;
}
static int shape_ok(const CshPlan& p, int c) { TARA_CSH_SWITCH(p.nx, shape_ok_n, c, p.ny) }
template <int NY, int GS>
static int launch_yfwd_inv_g(const CshPlan& p, int mode, const YfwdArgs& a, hipStream_t st)
{
    using S = YiShape<NY, false>;
    const dim3 g((p.nh + S::CB - 1) / S::CB, p.batch), b(S::NT);
    double2* const g0 = p.g[0].as<double2>();
    double2* const g1 = p.g[1].as<double2>();
    double2* const g2 = p.g[2].as<double2>();
    double2* const g3 = p.g[3].as<double2>();
    switch (mode) {
        case CSH_AB2: hipLaunchKernelGGL((k_csh_yfwd_inv<NY, CSH_AB2, GS>), g, b, 0, st, a, csh_band(p), p.tw_y, g0, g1, g2, g3, p.gld); break;
        case CSH_RK4_1: hipLaunchKernelGGL((k_csh_yfwd_inv<NY, CSH_RK4_1, GS>), g, b, 0, st, a, csh_band(p), p.tw_y, g0, g1, g2, g3, p.gld); break;
        case CSH_RK4_2: hipLaunchKernelGGL((k_csh_yfwd_inv<NY, CSH_RK4_2, GS>), g, b, 0, st, a, csh_band(p), p.tw_y, g0, g1, g2, g3, p.gld); break;
        case CSH_RK4_3: hipLaunchKernelGGL((k_csh_yfwd_inv<NY, CSH_RK4_3, GS>), g, b, 0, st, a, csh_band(p), p.tw_y, g0, g1, g2, g3, p.gld); break;
        case CSH_RK4_4: hipLaunchKernelGGL((k_csh_yfwd_inv<NY, CSH_RK4_4, GS>), g, b, 0, st, a, csh_band(p), p.tw_y, g0, g1, g2, g3, p.gld); break;
        default: set_error("fused y pass: mode %d has no stage update", mode); return TARA_ERR_ARG;
    }
    return TARA_OK;
}

template <int NY>
static int launch_yfwd_inv(const CshPlan& p, int mode, const YfwdArgs& a, hipStream_t st)
{
    return p.gsh == 1 ? launch_yfwd_inv_g<NY, 1>(p, mode, a, st) : launch_yfwd_inv_g<NY, 2>(p, mode, a, st);
}

static int yfwd_inv(const CshPlan& p, int mode, const YfwdArgs& a, hipStream_t st)
{
    switch (p.ny) {  // csh_fuses_y: from Ny = 1024
        case 1024: return launch_yfwd_inv<1024>(p, mode, a, st);
        case 2048: return launch_yfwd_inv<2048>(p, mode, a, st);
        case 4096: return launch_yfwd_inv<4096>(p, mode, a, st);
        default: set_error("fused y pass of large grids at Ny=%d", p.ny); return TARA_ERR_UNSUPPORTED;
    }
}

static int yfwd(const CshPlan& p, int mode, const YfwdArgs& a, hipStream_t st)
{
    TARA_CSH_SWITCH(p.ny, launch_yfwd, p, mode, a, st)
}

// ------------------------------------------------------------------ host side
int csh_host_tables(int nx, int ny, std::vector<double>& kx, std::vector<double>& ky, std::vector<int>& imin)
{
    // wavenumber and dealias tables, with derive2csh's own expressions
    const int nh = nx / 2 + 1;
    kx.resize(nh);
    ky.resize(ny);
    imin.resize(ny);
    const double pi_s = (double)3.1428f;  // real(8), parameter :: pi = 3.1428 (default-real literal)
    const double L = 2.0 * pi_s;
    for (int i = 0; i < nh; ++i) kx[i] = 2.0 * pi_s * (double)i / L;
    for (int j = 0; j < ny; ++j) ky[j] = (j < ny / 2) ? 2.0 * pi_s * (double)j / L : 2.0 * pi_s * ((double)j - ny) / L;
    for (int i = 0; i < nh; ++i)
        TARA_CHECK(kx[i] == (double)i, TARA_ERR_UNSUPPORTED, "derive2csh kx(%d) is not an integer", i);
    for (int j = 0; j < ny; ++j)
        TARA_CHECK(ky[j] == (double)(j < ny / 2 ? j : j - ny), TARA_ERR_UNSUPPORTED, "derive2csh ky(%d) not an integer", j);
    const double cut = ((double)(nx + ny) / 2.0) / 3.0;
    for (int j = 0; j < ny; ++j) {
        int m = nh;
        for (int i = 0; i < nh; ++i)
            if (std::sqrt(kx[i] * kx[i] + ky[j] * ky[j]) >= cut) {
                m = i;
                break;
            }
        imin[j] = m;  // kx increases with i, so every i >= m is cut as well
    }
    return TARA_OK;
}

int csh_live_columns(int nx, int ny)
{
    const double cut = ((double)(nx + ny) / 2.0) / 3.0;
    int i = 0;
    while (i < nx / 2 + 1 && !((double)i >= cut)) ++i;  // imin at ky = 0, its largest
    return i;
}

int csh_state_set(const CshPlan& p, const double2* w, double2* aux, size_t naux, int run, bool flags, hipStream_t st)
{
    int* band = p.band.as<int>() + run;
    const size_t n = std::max(naux, (size_t)p.nh * p.ny), nb = (n + 255) / 256;
    if (flags) hipLaunchKernelGGL(k_csh_state_flags, dim3(1), dim3(1), 0, st, p.bad.as<int>() + run, band);
    hipLaunchKernelGGL(k_csh_state_set, dim3((unsigned)(nb < 2048 ? nb : 2048)), dim3(256), 0, st, w, p.imin.as<int>(),
                       p.nh, p.ny, aux, naux, csh_small(p) ? nullptr : band);
    TARA_HIP(hipGetLastError());
    return TARA_OK;
}

int csh_plan_init(CshPlan& p, int nx, int ny, int batch)
{
    TARA_CHECK(batch >= 1 && batch <= 65535, TARA_ERR_ARG, "batch %d out of range", batch);
    TARA_CHECK(is_pow2(nx) && is_pow2(ny) && nx >= 32 && ny >= 16 && nx <= 4096 && ny <= 4096,
               TARA_ERR_UNSUPPORTED, "derive2csh: grid %dx%d unsupported (powers of two, 32..4096 x 16..4096)",
               nx, ny);
    p.nx = nx;
    p.ny = ny;
    p.nh = nx / 2 + 1;
    p.gld = csh_gld(p.nh);
    p.gsh = csh_gshift(p.nh);
    p.hk = csh_live_columns(nx, ny);
    const size_t ns = (size_t)p.gld * ny;  // G0..G3 hold gld columns per row group
    p.batch = batch;
    p.bstride = ns;
    int rc;
    for (int f = 0; f < 4; ++f) {
        if ((rc = p.g[f].alloc(batch * ns * sizeof(double2)))) return rc;
        TARA_HIP(hipMemset(p.g[f].p, 0, batch * ns * sizeof(double2)));
    }
    if ((rc = p.h.alloc(batch * ns * sizeof(double2)))) return rc;
    if ((rc = p.bad.alloc(batch * sizeof(int))) || (rc = p.band.alloc(batch * sizeof(int)))) return rc;
    TARA_HIP(hipMemset(p.band.p, 0, batch * sizeof(int)));
    TARA_HIP(hipMemset(p.bad.p, 0, batch * sizeof(int)));
    std::vector<double> kx, ky;
    std::vector<int> imin;
    if ((rc = csh_host_tables(nx, ny, kx, ky, imin))) return rc;
    if ((rc = p.kx.alloc(p.nh * sizeof(double)))) return rc;
    if ((rc = p.ky.alloc(ny * sizeof(double)))) return rc;
    if ((rc = p.imin.alloc(ny * sizeof(int)))) return rc;
    TARA_HIP(hipMemcpy(p.kx.p, kx.data(), p.nh * sizeof(double), hipMemcpyHostToDevice));
    TARA_HIP(hipMemcpy(p.ky.p, ky.data(), ny * sizeof(double), hipMemcpyHostToDevice));
    TARA_HIP(hipMemcpy(p.imin.p, imin.data(), ny * sizeof(int), hipMemcpyHostToDevice));
    p.tw_y = twiddles(ny, csh_yem(ny));
    p.tw_x = twiddles(nx / 2);
    p.tw_xn = twiddles(nx);
    p.tw_x16 = twiddles(nx / 2, 16);
    p.tw_xn16 = twiddles(nx, 16);
    p.tw_x4 = twiddles(nx / 2, 4);
    p.tw_xn4 = twiddles(nx, 4);
    p.rctw = rc_twiddles(nx);
    TARA_CHECK(p.tw_y && p.tw_x && p.tw_xn && p.tw_x16 && p.tw_xn16 && p.tw_x4 && p.tw_xn4 && p.rctw, TARA_ERR_ALLOC,
               "twiddle table allocation failed");
    p.xcfg = csh_default_xshape(p);
    TARA_CHECK(csh_xshape_ok(p, p.xcfg), TARA_ERR_UNSUPPORTED, "derive2csh: no x pass for %dx%d", nx, ny);
    return TARA_OK;
}

// Nx = 32 has the paired pass only: eight rows of the others are half a wavefront.
int csh_default_xshape(const CshPlan& p)
{
    const bool pairs = shape_ok(p, kXPairs) == 1;
    return pairs && (csh_small_xrows(p) || shape_ok(p, 0) != 1) ? kXPairs : 0;
}

int csh_num_xshapes() { return kNumXCands; }

int csh_xshape_ok(const CshPlan& p, int c) { return c >= 0 && c < kNumXCands && shape_ok(p, c) == 1; }

int csh_xpass(const CshPlan& p, hipStream_t st) { return xpass(p, st); }

int csh_nonfinite(const CshPlan& p, int* flags, hipStream_t st)
{
    std::vector<int> f(p.batch, 0);
    TARA_HIP(hipMemcpyAsync(f.data(), p.bad.p, p.batch * sizeof(int), hipMemcpyDeviceToHost, st));
    TARA_HIP(hipStreamSynchronize(st));
    int n = 0;
    for (int r = 0; r < p.batch; ++r) {
        n += f[r] != 0;
        if (flags) flags[r] = f[r] != 0;
    }
    return n;
}

// The arguments of a forward y pass whose stage input, base, accumulator and
// output are set by the caller.
static YfwdArgs yargs(const CshPlan& p, const CshPhys& ph, double dt)
{
    YfwdArgs a{};
    a.h = p.h.as<double2>();
    a.imin = p.imin.as<int>();
    a.nh = p.nh;
    a.nu = ph.nu;
    a.dt = dt;
    a.alpha = ph.alpha;
    a.lam = ph.lambda;
    a.screened = ph.screened;
    a.bs = p.bstride;
    a.nus = ph.nus;
    a.bad = p.bad.as<int>();
    a.si = p.ny;
    a.sj = 1;
    return a;
}

int csh_rhs_stage(const CshPlan& p, const double2* ws, int mode, const CshPhys& ph, double dt, double2* base,
                  double2* aux, double2* next, hipStream_t st, EventTimer* tm)
{
    int rc;
    const bool small = csh_small(p);
    YfwdArgs a = yargs(p, ph, dt);
    a.ws = ws;
    a.base = base;
    a.aux = aux;
    a.next = next;
    if (tm) tm->begin(0, st);
    if ((rc = small ? csh_small_yinv(p, ws, ph, p.ny, 1, st) : yinv(p, ws, ph, st))) return rc;
    if (tm) tm->end(0, st);
    if (tm) tm->begin(1, st);
    if ((rc = xpass(p, st))) return rc;
    if (tm) tm->end(1, st);
    if (tm) tm->begin(2, st);
    if ((rc = small ? csh_small_yfwd(p, mode, a, false, st) : yfwd(p, mode, a, st))) return rc;
    if (tm) tm->end(2, st);
    TARA_HIP(hipGetLastError());
    return TARA_OK;
}

int csh_rhs_direct(const CshPlan& p, const double2* w, double2* f, const CshPhys& ph, hipStream_t st)
{
    int rc;
    YfwdArgs a = yargs(p, ph, 0.0);
    a.ws = w;
    a.next = f;
    a.si = 1;
    a.sj = p.nh;
    if ((rc = csh_small_yinv(p, w, ph, 1, p.nh, st)) || (rc = xpass(p, st)) ||
        (rc = csh_small_yfwd(p, CSH_RHS, a, false, st)))
        return rc;
    TARA_HIP(hipGetLastError());
    return TARA_OK;
}

// Fusing the forward y pass with the next inverse y pass pays at Ny = 1024 and 2048
// (RK4 step apart -> fused, general / limited state: 1024^2 0.154 -> 0.138 / 0.151 ->
// 0.138 ms, 2048^2 0.406 -> 0.391 / 0.301 -> 0.271) and on grids too small to fill the
// chip (csh2d_small.hip).  At 4096^2 it did with the four fields in G0..G3 (2.41 ->
// 2.36); with the pairs the passes apart are faster (2.06 against 2.16 / 1.403 against
// 1.427), not taken up yet.  Below 1024 the fused pass holds fewer waves per CU than the
// separate forward y pass: the 128-512 ensemble step measured 6.65 ms fused against 6.43
// separate, with the four fields in G0..G3.
bool csh_fuses_y(const CshPlan& p) { return p.ny >= 1024 || csh_small(p); }

int csh_yinv_pass(const CshPlan& p, const double2* w, const CshPhys& ph, hipStream_t st)
{
    if (!csh_fuses_y(p)) return TARA_OK;  // the unfused step runs its own inverse y passes
    int rc = csh_small(p) ? csh_small_yinv(p, w, ph, p.ny, 1, st) : yinv(p, w, ph, st);
    if (rc) return rc;
    TARA_HIP(hipGetLastError());
    return TARA_OK;
}

int csh_fused_step(const CshPlan& p, int scheme, const CshPhys& ph, double dt, double2* w, double2* aux,
                   double2* next, bool plain_last, hipStream_t st, EventTimer* tm)
{
    const bool small = csh_small(p);
    TARA_CHECK(!ph.screened || small, TARA_ERR_ARG, "the fused step of large grids covers derive2csh only");
    int rc;
    if (!csh_fuses_y(p)) {
        if (scheme == TARA_SCHEME_AB2) return csh_rhs_stage(p, w, CSH_AB2, ph, dt, w, aux, nullptr, st, tm);
        for (int k = 0; k < 4; ++k)
            if ((rc = csh_rhs_stage(p, k == 0 ? w : next, CSH_RK4_1 + k, ph, dt, w, aux, next, st, tm))) return rc;
        return TARA_OK;
    }
    YfwdArgs a = yargs(p, ph, dt);
    a.base = w;
    a.aux = aux;
    const int nst = scheme == TARA_SCHEME_AB2 ? 1 : 4;
    for (int k = 0; k < nst; ++k) {
        const int mode = scheme == TARA_SCHEME_AB2 ? CSH_AB2 : CSH_RK4_1 + k;
        a.ws = (scheme == TARA_SCHEME_AB2 || k == 0) ? w : next;
        a.next = (scheme == TARA_SCHEME_AB2 || k == 3) ? nullptr : next;
        if (tm) tm->begin(1, st);
        if ((rc = xpass(p, st))) return rc;
        if (tm) tm->end(1, st);
        const bool plain = plain_last && k == nst - 1;
        if (tm) tm->begin(2, st);
        if ((rc = small ? csh_small_yfwd(p, mode, a, !plain, st) : plain ? yfwd(p, mode, a, st) : yfwd_inv(p, mode, a, st)))
            return rc;
        if (tm) tm->end(2, st);
    }
    TARA_HIP(hipGetLastError());
    return TARA_OK;
}

bool csh_fused(const CshPlan& p, const CshPhys& ph) { return !ph.screened || csh_small(p); }

int csh_advance(const CshPlan& p, int scheme, int nsteps, const CshPhys& ph, double dt, double2* w,
                double2* aux, double2* next, hipStream_t st, EventTimer* tm)
{
    TARA_CHECK(csh_fused(p, ph), TARA_ERR_ARG, "the fused advance of large grids covers derive2csh only");
    if (nsteps <= 0) return TARA_OK;
    int rc;
    if (tm) tm->begin(0, st);
    if ((rc = csh_yinv_pass(p, w, ph, st))) return rc;  // the only stand-alone inverse y pass of the call
    if (tm) tm->end(0, st);
    for (int s = 0; s < nsteps; ++s)
        if ((rc = csh_fused_step(p, scheme, ph, dt, w, aux, next, s == nsteps - 1, st, tm))) return rc;
    return TARA_OK;
}

int launch_ab2(const double2* w, double2* wn, const double2* fo, const double2* fn, double dt, size_t n,
               hipStream_t st)
{
    const int bs = 256;
    size_t nb = (n + bs - 1) / bs;
    if (nb > 65536) nb = 65536;
    hipLaunchKernelGGL(k_ab2, dim3((unsigned)nb), dim3(bs), 0, st, w, wn, fo, fn, dt, n);
    TARA_HIP(hipGetLastError());
    return TARA_OK;
}

}  // namespace tara
