// The paired x pass of the 2D incompressible right-hand side: a row's two field pairs
// side by side (csh2d_small.hip: why).  It is one of the x-pass shapes on any grid, so
// it has a code object of its own: a code object is loaded whole when its first kernel
// runs, and a large grid's autotuner would load the small grids' y passes with it.
#include "csh2d_dev.h"

namespace tara {

// One y row per 2 T threads: the first T transform ux + i uy, the others
// d omega/dx + i d omega/dy; they meet in LDS, where the first T/2 threads form
// ux d omega/dx + uy d omega/dy and run its forward half-length transform.
template <int NX>
struct SXShape {
    static constexpr int M = NX / 2;
    static constexpr int T = RF<NX>::T, TM = RF<M>::T;
    static constexpr bool WAVE = T <= 64;
    static constexpr int RB = 2 * T >= 64 ? 1 : 64 / (2 * T);  // rows per workgroup
    static constexpr int NT = 2 * T * RB;
    static constexpr bool OK = NT <= 1024 && 2 * TM == T && 2 * RB * RF<NX>::LDS * 16 <= 160 * 1024;
};

template <int NX, typename Band>
__global__ __launch_bounds__((SXShape<NX>::NT)) void k_csh_x_pairs(const double2* g0, const double2* g1,
                                                                   const double2* g2, const double2* g3, double scale,
                                                                   double2* __restrict__ h, const double2* tw_n,
                                                                   const double2* tw_m, const double2* rctw, size_t bs,
                                                                   Band bd)
{
    constexpr bool BAND = Band::KNOWN;
    using S = SXShape<NX>;
    static_assert(S::OK, "paired x pass does not fit");
    constexpr int E = RF<NX>::E, EH = RF<S::M>::E, T = S::T, M = S::M;
    __shared__ double2 lds[2 * S::RB * RF<NX>::LDS];
    const size_t rb = blockIdx.y * bs;  // batched runs
    const int t = threadIdx.x % T, seq = threadIdx.x / T, p = seq % 2, r = seq / 2;
    const int j = xcd_remap(blockIdx.x, gridDim.x) * S::RB + r;
    double2* xl = lds + seq * RF<NX>::LDS;
    double2* x0 = lds + 2 * r * RF<NX>::LDS;  // the row's first buffer
    double2 v[E];
    int lim = M + 1;
    if constexpr (BAND)
        if (bd.limited(blockIdx.y)) lim = bd.hk;
    x_c2r_pair<NX, 8, BAND>((p ? g2 : g0) + rb, (p ? g3 : g1) + rb, j, lim, RfSeq<NX, 8, S::WAVE>{t, xl}, tw_n, v);
#pragma unroll
    for (int e = 0; e < E; ++e) xl[rf_pad(rf_final_idx<NX>(t, e))] = v[e];
    // the unpacking roots of this thread's kx, fetched before the stores
    constexpr int NK = M / (2 * T);
    const int tt = p * T + t;
    double2 wk[NK];
#pragma unroll
    for (int u = 0; u < NK; ++u) wk[u] = rctw[tt + u * 2 * T];
    __syncthreads();
    const bool fwd = p == 0 && t < S::TM;
    double2 z[EH];
    if (fwd) {
        const double2* x1 = x0 + RF<NX>::LDS;
        auto nl = [&](int n) {
            const double2 u = x0[rf_pad(n)], w = x1[rf_pad(n)];
            return (u.x * w.x + u.y * w.y) * scale;
        };
#pragma unroll
        for (int e = 0; e < EH; ++e) {
            const int m = rf_first_idx<M>(t, e);
            z[e] = make_double2(nl(2 * m), nl(2 * m + 1));
        }
    }
    __syncthreads();
    if (fwd) {
        rf_fft<M, -1, 8, S::WAVE>(z, t, x0, tw_m);
#pragma unroll
        for (int e = 0; e < EH; ++e) x0[rf_pad(rf_final_idx<M>(t, e))] = z[e];
    } else if constexpr (!S::WAVE) {
        rf_fft_barriers_only<M>();  // TM >= 64: whole waves
    }
    __syncthreads();
    h += rb;
#pragma unroll
    for (int u = 0; u < NK; ++u) {
        const int k = tt + u * 2 * T;
        if constexpr (BAND)
            if (k >= bd.hk) continue;  // dealiased away at every ky
        const double2 zk = x0[rf_pad(k)];
        const double2 zmk = x0[rf_pad(k == 0 ? 0 : M - k)];
        double2 xm;
        h[blk8(k, j, M + 1)] = r2c_unpack_w(zk, zmk, k, wk[u], &xm);
        if (k == 0) h[blk8(M, j, M + 1)] = xm;
    }
}

// ------------------------------------------------------------------- dispatch
// The paired x pass is the default up to 2^19 points and Ny = 2048, against
// shape 0 there: RK4 step 512^2 70.1 / 92.6 us, 1024 x 512 118 / 123, 512 x 1024
// 118 / 134, 2048 x 256 114.5 / 116, 64^2 40 / 44; beyond, 1024^2 145 / 142, 2048 x
// 512 153 / 148, 2048^2 315 / 292.  (The autotuner times it among the other shapes.)
constexpr size_t kSmallX = 1 << 19;

bool csh_small_xrows(const CshPlan& p) { return p.ny <= 2048 && (size_t)p.nx * p.ny * p.batch <= kSmallX; }

template <int NX, typename Band>
static int launch_x_pairs_t(const CshPlan& p, Band bd, hipStream_t st)
{
    using S = SXShape<NX>;
    const double scale = 1.0 / ((double)p.nx * (double)p.ny * (double)p.nx * (double)p.ny);
    hipLaunchKernelGGL((k_csh_x_pairs<NX, Band>), dim3(p.ny / S::RB, p.batch), dim3(S::NT), 0, st,
                       p.g[0].as<double2>(), p.g[1].as<double2>(), p.g[2].as<double2>(), p.g[3].as<double2>(), scale,
                       p.h.as<double2>(), p.tw_xn, p.tw_x, p.rctw, p.bstride, bd);
    return TARA_OK;
}

// The small grids' y passes write and read every column: guarding the loads and
// stores by the support cost a 64^2 AB2 step 12 % there (and two more kernel
// arguments alone 2.5 %).
template <int NX>
static int launch_x_pairs(const CshPlan& p, hipStream_t st)
{
    return csh_small(p) ? launch_x_pairs_t<NX>(p, CshNoBand{}, st) : launch_x_pairs_t<NX>(p, csh_band(p), st);
}

#define TARA_X_PAIRS_SWITCH(n, FN, ...)             \
    switch (n) {                                    \
        case 32: return FN<32>(__VA_ARGS__);        \
        case 64: return FN<64>(__VA_ARGS__);        \
        case 128: return FN<128>(__VA_ARGS__);      \
        case 256: return FN<256>(__VA_ARGS__);      \
        case 512: return FN<512>(__VA_ARGS__);      \
        case 1024: return FN<1024>(__VA_ARGS__);    \
        case 2048: return FN<2048>(__VA_ARGS__);    \
        case 4096: return FN<4096>(__VA_ARGS__);    \
        default: return 0;                          \
    }

template <int NX>
static int x_pairs_rows(int)
{
    return SXShape<NX>::RB;
}

// Rows per workgroup of the paired x pass, 0 where it has no kernel.
static int pairs_rows(int nx) { TARA_X_PAIRS_SWITCH(nx, x_pairs_rows, 0) }

bool csh_x_pairs_ok(int nx, int ny) { return pairs_rows(nx) > 0 && ny % pairs_rows(nx) == 0; }

int csh_x_pairs(const CshPlan& p, hipStream_t st)
{
    TARA_CHECK(csh_x_pairs_ok(p.nx, p.ny), TARA_ERR_UNSUPPORTED, "x pass shape %d does not run on %dx%d", kXPairs, p.nx,
               p.ny);
    TARA_X_PAIRS_SWITCH(p.nx, launch_x_pairs, p, st)
}

}  // namespace tara
