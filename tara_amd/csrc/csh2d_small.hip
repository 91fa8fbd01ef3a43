// The 2D incompressible passes for grids too small to fill the chip (csh2d.hip
// holds those of large grids and batches).  There a pass's time is the latency
// of one thread's chain of loads and transforms, not bandwidth: at 64^2 the
// inverse y pass ran four transforms one after another in 6.9 us, the forward y
// and x passes 4.8 and 4.7 us, against about 2.2 us for a kernel that does
// nothing.  So the chains are cut: every transform of a pass gets its own
// threads, sequences of at most 64 threads exchange within their wavefront, and
// a stage is two kernels (x, csh2d_pairs.hip, and forward y + next inverse y) instead
// of three.
// RK4 step, three kernels a stage -> two, default x shapes: 64^2 65.4 -> 39.8 us,
// 256^2 98.7 -> 47.2, 512^2 131.8 -> 72.5, 1024 x 512 201 -> 118; 512 x 256 screened
// 122 -> 60; one right-hand side on device arrays at 256^2 30.1 -> 14.5 us.  What
// is left is the chain itself: about 5 us a kernel at 64^2, of which 2.2 us is
// what any kernel takes.
#include "csh2d_dev.h"

namespace tara {

// --------------------------------------------------------------------- y pass
// One kx column per NG T threads, NG = 4 or 2: group g transforms fields g, g + NG
// of the inverse pass (G0, G1 = ux +- i uy, G2, G3 = d omega/dx +- i d omega/dy).
// The forward transform and the update before it (FWD) are done by every group, so
// that each holds the next stage's input in registers; group 0 stores it.
template <int NY, int NG>
struct SYShape {
    static constexpr int T = RY<NY>::T;                      // threads per sequence
    static constexpr bool WAVE = T <= 64;                    // a sequence sits in one wavefront
    static constexpr int CB = NG * T >= 64 ? 1 : 64 / (NG * T);  // columns per workgroup
    static constexpr int NT = CB * NG * T;
    static constexpr bool OK = NT <= 1024;
};

struct SYInv {
    double2 *g0, *g1, *g2, *g3;
    int ld;
};

template <int NY, int MODE, int GS, bool FWD, int NG>
__global__ __launch_bounds__((SYShape<NY, NG>::NT)) void k_csh_small_y(YfwdArgs a, SYInv o, const double2* tw)
{
    constexpr bool INV = NG > 1;
    using S = SYShape<NY, NG>;
    constexpr int E = RY<NY>::E, T = S::T, EM = csh_yem(NY);
    __shared__ double2 lds[S::CB * NG * RY<NY>::LDS];
    const size_t rb = blockIdx.y * a.bs;  // batched runs
    a.ws += rb;
    const int t = threadIdx.x % T, seq = threadIdx.x / T, g = seq % NG;
    const int i0 = xcd_remap(blockIdx.x, gridDim.x) * S::CB, i = i0 + seq / NG;
    const bool live = i < a.nh;
    // dead columns recompute the workgroup's first column and store nothing: one that
    // no other workgroup writes
    const int ic = live ? i : i0;
    double2* xl = lds + seq * RY<NY>::LDS;
    const double kxv = (double)ic;
    double2 v[E];
    if constexpr (FWD) {
        a.h += rb;
        if (a.base) a.base += rb;
        if (a.aux) a.aux += rb;
        if (a.next) a.next += rb;
        if (a.nus) a.nu = a.nus[blockIdx.y];
#pragma unroll
        for (int e = 0; e < E; ++e) v[e] = a.h[blk8(ic, rf_first_idx<NY, EM>(t, e), a.nh)];
        rf_fft<NY, -1, EM, S::WAVE>(v, t, xl, tw);
        double2 av[E];
#pragma unroll
        for (int e = 0; e < E; ++e) {
            const int j = rf_final_idx<NY, EM>(t, e);
            const size_t q = (size_t)ic * a.si + (size_t)j * a.sj;
            const double2 nl = ic >= a.imin[j] ? make_double2(0.0, 0.0) : v[e];
            const double kyv = csh_ky<NY>(j);
            csh_update<MODE>(a, q, ic == 0 && j == 0, nl, a.ws[q], kxv * kxv + kyv * kyv, &v[e], &av[e]);
        }
        // every group and dead column has read the column before its group 0 writes it
        if constexpr (NG > 1 || S::CB > 1) __syncthreads();
        if (live && g == 0) {
            bool finite = true;
#pragma unroll
            for (int e = 0; e < E; ++e) {
                const size_t q = (size_t)ic * a.si + (size_t)rf_final_idx<NY, EM>(t, e) * a.sj;
                finite = csh_store<MODE>(a, q, v[e], av[e]) && finite;
            }
            if (!finite && a.bad) a.bad[blockIdx.y] = 1;
        }
        if constexpr (INV) rf_final_to_first<NY, EM, S::WAVE>(v, t, xl);
    } else {
#pragma unroll
        for (int e = 0; e < E; ++e) v[e] = a.ws[(size_t)ic * a.si + (size_t)rf_first_idx<NY, EM>(t, e) * a.sj];
    }
    if constexpr (INV) {
        // derive2csh.f95:29-71: ux, uy = i ky psi, -i kx psi with psi = omega/k^2,
        // psi(0,0) = 0; fields 0, 1 ux +- i uy, 2, 3 i kx omega +- i (i ky omega)
        // (x_c2r_pair).  Screened (derive2css.f95:22-52): psi = omega/(k^2 +
        // lambda), omega_d = k^2 psi.
        double2 w[E];
#pragma unroll
        for (int e = 0; e < E; ++e) w[e] = v[e];
#pragma unroll 1
        for (int f = g; f < 4; f += NG) {
#pragma unroll
            for (int e = 0; e < E; ++e) {
                const int j = rf_first_idx<NY, EM>(t, e);
                const double kyv = csh_ky<NY>(j);
                const double k2 = kxv * kxv + kyv * kyv;
                const double den = a.screened ? k2 + a.lam : k2;
                const bool zero = a.screened ? ic == 0 && j == 0 : k2 == 0.0;
                double2 z = w[e];
                if (f < 2 || a.screened) z = zero ? make_double2(0.0, 0.0) : make_double2(z.x / den, z.y / den);
                if (f >= 2 && a.screened) z = make_double2(k2 * z.x, k2 * z.y);
                const double cr = f == 0 ? kxv : f == 1 ? -kxv : f == 2 ? -kyv : kyv, ci = f < 2 ? kyv : kxv;
                v[e] = make_double2(cr * z.x - ci * z.y, cr * z.y + ci * z.x);
            }
            rf_fft<NY, +1, EM, S::WAVE>(v, t, xl, tw);
            double2* out = (f == 0 ? o.g0 : f == 1 ? o.g1 : f == 2 ? o.g2 : o.g3) + rb;
            if (live) {
#pragma unroll
                for (int e = 0; e < E; ++e) out[blkg(i, rf_final_idx<NY, EM>(t, e), o.ld, GS)] = v[e];
            }
            if (NG == 4) break;
        }
    }
}

// ------------------------------------------------------------------- dispatch
// The y passes run here with four groups a column while their threads come to at
// most 2112 wavefronts, two per SIMD and the odd column of Nh.  RK4 step (tuned x
// shape) here against the larger grids' passes: 1024 x 512 (2052 wavefronts) 117 /
// 146 us, 256 x 1024 (2064) 91.7 / 93.9; beyond, the repeated forward transform
// costs more than the shorter chain gives: 512 x 1024 (4112) 139 / 112, 1024^2
// (8208) 203 / 147.
// Up to Ny = 512 and 6000 wavefronts two groups, two fields each, repeat it once
// only.  A step here against the larger grids' passes: 64 runs of 128^2 (2080) 144
// / 164 us, 200 of 64^2 (1650) 110 / 146, 512 of 64^2 (4224) 210 / 250, 32 of 256^2
// (4128) 219 / 238, 8 of 512^2 (4112) 234 / 256, 2048 x 512 (4100) 150 / 159;
// beyond, 64 of 256^2 (8256) 454 / 428, 16 of 512^2 (8224) 435 / 423.  Not at Nx =
// 4096, whose 2-row groups one column a workgroup writes in pieces: 4096 x 512 234
// / 190, 4096 x 256 165 / 161; and not at Ny = 1024: 512 x 1024 132 / 127.
constexpr size_t kSmallWaves = 2112, kPairWaves = 6000;

// Thread groups a column, 0 for the larger grids' passes.
static int small_groups(const CshPlan& p)
{
    const size_t threads = (size_t)p.nh * (p.ny / csh_yem(p.ny)) * p.batch;
    if (p.ny <= 1024 && 4 * threads <= 64 * kSmallWaves) return 4;
    return p.nx <= 2048 && p.ny <= 512 && 2 * threads <= 64 * kPairWaves ? 2 : 0;
}

bool csh_small(const CshPlan& p) { return small_groups(p) > 0; }

template <int NY, int MODE, bool FWD, int NG>
static int launch_small_y(const CshPlan& p, const YfwdArgs& a, hipStream_t st)
{
    using S = SYShape<NY, NG>;
    if constexpr (!S::OK) {
        set_error("small y pass at Ny=%d", NY);
        return TARA_ERR_UNSUPPORTED;
    } else {
        const SYInv o{p.g[0].as<double2>(), p.g[1].as<double2>(), p.g[2].as<double2>(), p.g[3].as<double2>(), p.gld};
        const dim3 grid((p.nh + S::CB - 1) / S::CB, p.batch), b(S::NT);
        if (p.gsh == 1)
            hipLaunchKernelGGL((k_csh_small_y<NY, MODE, 1, FWD, NG>), grid, b, 0, st, a, o, p.tw_y);
        else
            hipLaunchKernelGGL((k_csh_small_y<NY, MODE, 2, FWD, NG>), grid, b, 0, st, a, o, p.tw_y);
        return TARA_OK;
    }
}

// Two groups exist up to Ny = 512 (small_groups).
template <int NY, int MODE, bool FWD>
static int launch_small_inv(const CshPlan& p, const YfwdArgs& a, hipStream_t st)
{
    if constexpr (NY <= 512)
        if (small_groups(p) == 2) return launch_small_y<NY, MODE, FWD, 2>(p, a, st);
    return launch_small_y<NY, MODE, FWD, 4>(p, a, st);
}

template <int NY>
static int launch_small_yinv(const CshPlan& p, const YfwdArgs& a, hipStream_t st)
{
    return launch_small_inv<NY, CSH_RHS, false>(p, a, st);
}

template <int NY>
static int launch_small_yfwd(const CshPlan& p, int mode, const YfwdArgs& a, bool inv, hipStream_t st)
{
#define TARA_SMALL_MODE(M) \
    case M: return inv ? launch_small_inv<NY, M, true>(p, a, st) : launch_small_y<NY, M, true, 1>(p, a, st);
    switch (mode) {
        case CSH_RHS: return launch_small_y<NY, CSH_RHS, true, 1>(p, a, st);
        TARA_SMALL_MODE(CSH_AB2)
        TARA_SMALL_MODE(CSH_RK4_1)
        TARA_SMALL_MODE(CSH_RK4_2)
        TARA_SMALL_MODE(CSH_RK4_3)
        TARA_SMALL_MODE(CSH_RK4_4)
        default: set_error("bad mode %d", mode); return TARA_ERR_ARG;
    }
#undef TARA_SMALL_MODE
}

#define TARA_SMALL_Y_SWITCH(n, FN, ...)             \
    switch (n) {                                    \
        case 16: return FN<16>(__VA_ARGS__);        \
        case 32: return FN<32>(__VA_ARGS__);        \
        case 64: return FN<64>(__VA_ARGS__);        \
        case 128: return FN<128>(__VA_ARGS__);      \
        case 256: return FN<256>(__VA_ARGS__);      \
        case 512: return FN<512>(__VA_ARGS__);      \
        case 1024: return FN<1024>(__VA_ARGS__);    \
        default: set_error("small y pass: unsupported length %d", n); return TARA_ERR_UNSUPPORTED; \
    }

int csh_small_yinv(const CshPlan& p, const double2* w, const CshPhys& ph, size_t si, size_t sj, hipStream_t st)
{
    YfwdArgs a{};
    a.ws = w;
    a.nh = p.nh;
    a.lam = ph.lambda;
    a.screened = ph.screened;
    a.bs = p.bstride;
    a.si = si;
    a.sj = sj;
    TARA_SMALL_Y_SWITCH(p.ny, launch_small_yinv, p, a, st)
}

int csh_small_yfwd(const CshPlan& p, int mode, const YfwdArgs& a, bool inv, hipStream_t st)
{
    TARA_SMALL_Y_SWITCH(p.ny, launch_small_yfwd, p, mode, a, inv, st)
}

}  // namespace tara
