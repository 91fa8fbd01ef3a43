// Transforms of any length: the fallback behind col_fft / row_r2c / row_c2r
// for lengths the register-resident kernels do not cover (FFTW accepts any
// size; a kept main may ask for Nx = 96 or 100).
//
// A complex transform of length n = r1 r2 ... rs runs as s Stockham
// (autosort, decimation in frequency) passes between two device buffers.
// The pass with radix r on the current sub-length L (stride s0 = n / L) maps
//   y[q + s0 (r p + u)] = w_L^{p u} * sum_j x[q + s0 (p + j m)] w_r^{j u},
//   m = L / r, p < m, q < s0, u < r,
// and the output of the last pass is in natural order.  One thread computes
// one output (O(r) work), so large prime factors still spread over the
// device (in LDS radices 2 to 5 take a butterfly a thread).  Roots come from one table of e^{-2 pi i k/n} (long double, rounded
// once).  Radices: 4 while possible, then 2, 3, 5, 7, then the remaining
// primes.
//
// Real transforms keep FFTW's semantics: r2c is the complex transform of the
// real row, of which entries 0..n/2 are kept; c2r builds the Hermitian row
// from entries 0..n/2 with the imaginary parts of entry 0 and (even n) entry
// n/2 taken as zero, which is what FFTW's c2r reads, and keeps the real part.
//
// Up to kAnyLds elements a workgroup runs whole sequences through all passes in
// LDS, from and to the caller's arrays (k_any_lds): one launch per transform, no
// work space, no synchronisation.  Longer sequences, and few sequences of a large
// prime (any_lds), take one launch per pass over two global buffers, allocated per
// call, and the stream is synchronised before the call returns.
#include <algorithm>
#include <vector>

#include "common.h"
#include "fft_api.h"

namespace tara {

namespace {

std::vector<int> radices(int n)
{
    std::vector<int> r;
    while (n % 4 == 0) {
        r.push_back(4);
        n /= 4;
    }
    for (int p = 2; p <= n; ++p)
        while (n % p == 0) {
            r.push_back(p);
            n /= p;
        }
    return r;
}

__device__ __forceinline__ double2 root(const double2* tw, long k, int dir)
{
    const double2 w = tw[k];
    return dir < 0 ? w : make_double2(w.x, -w.y);
}

__device__ __forceinline__ double2 cmul(double2 a, double2 b)
{
    return make_double2(a.x * b.x - a.y * b.y, a.x * b.y + a.y * b.x);
}

// One pass over ntrans transforms; element e of transform t at
// buf[e * es + t * ts].  tfast: consecutive threads take consecutive t.
__global__ void k_any_pass(const double2* __restrict__ x, double2* __restrict__ y, int n, int L, int r, long ntrans,
                           long es, long ts, int tfast, const double2* __restrict__ tw, int dir)
{
    const long total = ntrans * n;
    const int s0 = n / L, m = L / r;
    const long nr = n / r, nl = n / L;
    for (long idx = blockIdx.x * (long)blockDim.x + threadIdx.x; idx < total; idx += (long)gridDim.x * blockDim.x) {
        long t, e;
        if (tfast) {
            t = idx % ntrans;
            e = idx / ntrans;
        } else {
            t = idx / n;
            e = idx % n;
        }
        const long q = e % s0, rest = e / s0;
        const long u = rest % r, p = rest / r;
        const double2* xt = x + t * ts;
        double2 acc = make_double2(0.0, 0.0);
        for (int j = 0; j < r; ++j) {
            const double2 a = xt[(q + s0 * (p + (long)j * m)) * es];
            const double2 w = root(tw, ((j * u) % r) * nr, dir);
            acc.x += a.x * w.x - a.y * w.y;
            acc.y += a.x * w.y + a.y * w.x;
        }
        y[t * ts + e * es] = (p * u == 0) ? acc : cmul(acc, root(tw, (p * u) * nl, dir));
    }
}

// Strided columns <-> transform-fastest workspace: element j of column c of
// plane pl at a[pl * pstride + j * es + c] <-> W[j * ntrans + pl * ncols + c].
__global__ void k_any_gather(const double2* __restrict__ a, double2* __restrict__ w, int n, int ncols, long es,
                             long pstride, long ntrans)
{
    for (long idx = blockIdx.x * (long)blockDim.x + threadIdx.x; idx < ntrans * n; idx += (long)gridDim.x * blockDim.x) {
        const long t = idx % ntrans, j = idx / ntrans, c = t % ncols, pl = t / ncols;
        w[idx] = a[pl * pstride + j * es + c];
    }
}

__global__ void k_any_scatter(const double2* __restrict__ w, double2* __restrict__ a, int n, int ncols, long es,
                              long pstride, long ntrans)
{
    for (long idx = blockIdx.x * (long)blockDim.x + threadIdx.x; idx < ntrans * n; idx += (long)gridDim.x * blockDim.x) {
        const long t = idx % ntrans, j = idx / ntrans, c = t % ncols, pl = t / ncols;
        a[pl * pstride + j * es + c] = w[idx];
    }
}

// Real rows (pitch nx) -> complex rows (pitch nx).
__global__ void k_any_real_in(const double* __restrict__ x, double2* __restrict__ w, long total)
{
    for (long idx = blockIdx.x * (long)blockDim.x + threadIdx.x; idx < total; idx += (long)gridDim.x * blockDim.x)
        w[idx] = make_double2(x[idx], 0.0);
}

// Complex rows (pitch nx) -> half spectra (pitch ld), entries nh..ld-1 zeroed.
__global__ void k_any_half_out(const double2* __restrict__ w, double2* __restrict__ X, int nx, int ld, long nrows)
{
    const int nh = nx / 2 + 1;
    for (long idx = blockIdx.x * (long)blockDim.x + threadIdx.x; idx < nrows * ld; idx += (long)gridDim.x * blockDim.x) {
        const long row = idx / ld, k = idx % ld;
        X[idx] = k < nh ? w[row * nx + k] : make_double2(0.0, 0.0);
    }
}

// Half spectra (pitch ld) -> Hermitian complex rows (pitch nx).
__global__ void k_any_herm_in(const double2* __restrict__ X, double2* __restrict__ w, int nx, int ld, long nrows)
{
    const int nh = nx / 2 + 1;
    for (long idx = blockIdx.x * (long)blockDim.x + threadIdx.x; idx < nrows * nx; idx += (long)gridDim.x * blockDim.x) {
        const long row = idx / nx, k = idx % nx;
        const double2* src = X + row * ld;
        double2 v;
        if (k == 0 || 2 * k == nx)
            v = make_double2(src[k].x, 0.0);
        else if (k < nh)
            v = src[k];
        else {
            const double2 c = src[nx - k];
            v = make_double2(c.x, -c.y);
        }
        w[idx] = v;
    }
}

// Real part of complex rows (pitch nx), times s.
__global__ void k_any_real_out(const double2* __restrict__ w, double* __restrict__ x, double s, long total)
{
    for (long idx = blockIdx.x * (long)blockDim.x + threadIdx.x; idx < total; idx += (long)gridDim.x * blockDim.x)
        x[idx] = w[idx].x * s;
}

// ------------------------------------------------------------ passes in LDS
constexpr int kAnyLds = 2048;         // two buffers of 16-byte elements in 64 KB
constexpr int kAnyPasses = 12;        // 2048 = 4^5 2 takes 6; at most 11 (2^11) for any schedule

enum AnyKind { ANY_COL, ANY_R2C, ANY_C2R };

struct AnyArgs {
    const void* src;
    void* dst;
    int n, dir;
    int seqs;                 // sequences per workgroup
    long ntrans;
    long es, pstride;         // columns: element stride, plane stride
    int ncols;
    int ld;                   // rows: pitch of the half spectra
    double scale;             // c2r
    int npass;
    int radix[kAnyPasses];
};

// Butterflies of radix R of one pass (span s0 done): sequence c, output
// position group t (see k_any_lds).  x, y: this sequence's buffers.
template <int R>
__device__ __forceinline__ void any_butterfly(const double2* x, double2* y, int n, int s0, unsigned t, int nl,
                                              const double2* tw, int dir)
{
    const int nr = n / R;
    const unsigned p = t / (unsigned)s0, q = t - p * s0;
    double2 a[R];
#pragma unroll
    for (int j = 0; j < R; ++j) a[j] = x[t + j * nr];
    double2 y_[R];
    if constexpr (R == 2) {
        y_[0] = make_double2(a[0].x + a[1].x, a[0].y + a[1].y);
        y_[1] = make_double2(a[0].x - a[1].x, a[0].y - a[1].y);
    } else if constexpr (R == 4) {
        const double2 s02 = make_double2(a[0].x + a[2].x, a[0].y + a[2].y), d02 = make_double2(a[0].x - a[2].x, a[0].y - a[2].y);
        const double2 s13 = make_double2(a[1].x + a[3].x, a[1].y + a[3].y), d13 = make_double2(a[1].x - a[3].x, a[1].y - a[3].y);
        const double2 r = dir < 0 ? make_double2(d13.y, -d13.x) : make_double2(-d13.y, d13.x);  // -+i d13
        y_[0] = make_double2(s02.x + s13.x, s02.y + s13.y);
        y_[1] = make_double2(d02.x + r.x, d02.y + r.y);
        y_[2] = make_double2(s02.x - s13.x, s02.y - s13.y);
        y_[3] = make_double2(d02.x - r.x, d02.y - r.y);
    } else {
        double2 w[R];
#pragma unroll
        for (int k = 1; k < R; ++k) w[k] = root(tw, (long)k * nr, dir);
#pragma unroll
        for (int u = 0; u < R; ++u) {
            y_[u] = a[0];
#pragma unroll
            for (int j = 1; j < R; ++j) {
                const int k = (j * u) % R;
                if (k == 0) {
                    y_[u].x += a[j].x;
                    y_[u].y += a[j].y;
                } else {
                    y_[u].x += a[j].x * w[k].x - a[j].y * w[k].y;
                    y_[u].y += a[j].x * w[k].y + a[j].y * w[k].x;
                }
            }
        }
    }
#pragma unroll
    for (int u = 0; u < R; ++u)
        y[q + s0 * (R * p + u)] = (u == 0 || p == 0) ? y_[u] : cmul(y_[u], root(tw, (long)p * u * nl, dir));
}

// Whole transforms of a.seqs sequences.  Bound by latency on the grids that come
// here (a 96 x 80 right-hand side is a few hundred KB): the passes of a transform
// were a launch each, with two buffers allocated, a copy in and out and a
// synchronisation around them, 1.5 ms for the six transforms of a derive2csh
// call at 96 x 80 against 0.02 ms here (four launches of 6 us).
template <AnyKind KIND>
__global__ __launch_bounds__(1024) void k_any_lds(AnyArgs a, const double2* __restrict__ tw)
{
    extern __shared__ double2 lds[];
    const unsigned n = a.n, S = a.seqs, tid = threadIdx.x, nt = blockDim.x;
    double2* x = lds;
    double2* y = lds + S * n;
    const long t0 = (long)blockIdx.x * S;
    const unsigned live = (unsigned)(a.ntrans - t0 < (long)S ? a.ntrans - t0 : S);
    if constexpr (KIND == ANY_COL) {
        // sequences fastest: neighbouring columns are contiguous
        const double2* src = static_cast<const double2*>(a.src);
        for (unsigned b = tid; b < S * n; b += nt) {
            const unsigned c = b % S, e = b / S;
            const long t = t0 + (c < live ? c : 0), pl = t / a.ncols;
            x[c * n + e] = src[pl * a.pstride + (long)e * a.es + (t - pl * a.ncols)];
        }
    } else if constexpr (KIND == ANY_R2C) {
        const double* src = static_cast<const double*>(a.src) + t0 * n;
        for (unsigned b = tid; b < live * n; b += nt) x[b] = make_double2(src[b], 0.0);
    } else {
        const double2* src = static_cast<const double2*>(a.src) + t0 * a.ld;
        for (unsigned b = tid; b < live * n; b += nt) {
            const unsigned c = b / n, k = b - c * n;
            double2 v = src[(long)c * a.ld + (2 * k <= n ? k : n - k)];
            if (k == 0 || 2 * k == n) v.y = 0.0;
            if (2 * k > n) v.y = -v.y;
            x[b] = v;
        }
    }
    __syncthreads();
    int s0 = 1;  // n / L: spans done
    for (int ip = 0; ip < a.npass; ++ip) {
        const int r = a.radix[ip], nr = n / r;
        if (r <= 5) {
            for (unsigned b = tid; b < S * nr; b += nt) {
                const unsigned c = b / nr, t = b - c * nr;
                const double2* xs = x + c * n;
                double2* ys = y + c * n;
                switch (r) {
                    case 2: any_butterfly<2>(xs, ys, n, s0, t, s0, tw, a.dir); break;
                    case 3: any_butterfly<3>(xs, ys, n, s0, t, s0, tw, a.dir); break;
                    case 4: any_butterfly<4>(xs, ys, n, s0, t, s0, tw, a.dir); break;
                    default: any_butterfly<5>(xs, ys, n, s0, t, s0, tw, a.dir); break;
                }
            }
        } else {
            // one output per thread: a large prime spreads over the workgroup, which
            // has a thread for every one (launch_any_lds); four terms' loads in flight
            for (unsigned b = tid; b < S * n; b += nt) {
                const unsigned c = b / n, e = b - c * n;
                const unsigned rest = e / (unsigned)s0, q = e - rest * s0, p = rest / (unsigned)r, u = rest - p * r;
                const double2* xs = x + c * n + q + s0 * p;
                double2 acc = make_double2(0.0, 0.0);
                unsigned k = 0;  // j u mod r
#pragma unroll 4
                for (int j = 0; j < r; ++j) {
                    const double2 v = xs[j * nr], w = root(tw, (long)k * nr, a.dir);
                    acc.x += v.x * w.x - v.y * w.y;
                    acc.y += v.x * w.y + v.y * w.x;
                    k += u;
                    if (k >= (unsigned)r) k -= r;
                }
                y[c * n + e] = p * u == 0 ? acc : cmul(acc, root(tw, (long)p * u * s0, a.dir));
            }
        }
        __syncthreads();
        s0 *= r;
        double2* z = x;
        x = y;
        y = z;
    }
    if constexpr (KIND == ANY_COL) {
        double2* dst = static_cast<double2*>(a.dst);
        for (unsigned b = tid; b < S * n; b += nt) {
            const unsigned c = b % S, e = b / S;
            const long t = t0 + c, pl = t / a.ncols;
            if (c < live) dst[pl * a.pstride + (long)e * a.es + (t - pl * a.ncols)] = x[c * n + e];
        }
    } else if constexpr (KIND == ANY_R2C) {
        double2* dst = static_cast<double2*>(a.dst) + t0 * a.ld;
        const unsigned nh = n / 2 + 1;
        for (unsigned b = tid; b < live * a.ld; b += nt) {
            const unsigned c = b / a.ld, k = b - c * a.ld;
            dst[b] = k < nh ? x[c * n + k] : make_double2(0.0, 0.0);
        }
    } else {
        double* dst = static_cast<double*>(a.dst) + t0 * n;
        for (unsigned b = tid; b < live * n; b += nt) dst[b] = x[b].x * a.scale;
    }
}

// Whether length n runs in LDS; if so, the pass schedule and how many sequences
// share a workgroup: up to 8 (columns: a 128-byte line) that fit 64 KB and still
// leave 256 workgroups.  A prime factor above 1000 sums n r terms a sequence, each
// with a gathered root, which its one CU bounds: such sequences run here only if
// there are enough of them, r / 12, to fill the chip.  Host r2c of n x rows here
// against the passes over the whole chip: 2039 x 1 1178 / 545 us, x 128 1375 / 1202, x
// 256 1628 / 2282; 1499 x 64 709 / 506, x 128 804 / 788; 1021 x 64 352 / 325, x 128 401
// / 424; 1994 (2 x 997) x 1 327 / 310, x 64 418 / 436; 761 x 1 182 / 221.
bool any_lds(int n, long ntrans, AnyArgs& a)
{
    if (n > kAnyLds) return false;
    const std::vector<int> rs = radices(n);  // ascending past the fours
    if (!rs.empty() && rs.back() > 1000 && ntrans * 12 < rs.back()) return false;
    a = AnyArgs{};
    a.n = n;
    a.ntrans = ntrans;
    for (int r : rs) a.radix[a.npass++] = r;
    a.seqs = 8;
    while (a.seqs > 1 && (2L * a.seqs * n * 16 > 65536 || ntrans / a.seqs < 256)) a.seqs /= 2;
    return true;
}

template <AnyKind KIND>
int launch_any_lds(const AnyArgs& a, hipStream_t st)
{
    const double2* tw = unit_roots(a.n);
    TARA_CHECK(tw, TARA_ERR_ALLOC, "root table allocation failed (n = %d)", a.n);
    const int work = a.seqs * a.n / 4;  // butterflies of a pass
    int nt = work >= 192 ? 256 : work >= 96 ? 128 : 64;
    // a large prime: a thread per output, whose sum is a chain of r gathers (64 to
    // 256 threads, one term after another / as here: 251 x 1 140 / 55 us, 509 x 1 243 /
    // 98, 2036 x 1 572 / 167, 1021 x 512 1250 / 988)
    if (a.npass && a.radix[a.npass - 1] > 64) nt = std::min(1024, (a.seqs * a.n + 63) / 64 * 64);
    const long blocks = (a.ntrans + a.seqs - 1) / a.seqs;
    TARA_CHECK(blocks <= 0x7fffffffL, TARA_ERR_UNSUPPORTED, "transform batch too large");
    hipLaunchKernelGGL(k_any_lds<KIND>, dim3((unsigned)blocks), dim3(nt), 2 * (size_t)a.seqs * a.n * sizeof(double2), st,
                       a, tw);
    TARA_HIP(hipGetLastError());
    return TARA_OK;
}

unsigned blocks_for(long n)
{
    long b = (n + 255) / 256;
    return (unsigned)(b > 16384 ? 16384 : (b < 1 ? 1 : b));
}

// Runs the passes over w0 (w1: scratch of the same size); returns the buffer
// that holds the result.
int run_passes(double2* w0, double2* w1, int n, long ntrans, long es, long ts, int tfast, int dir, hipStream_t st,
               double2** result)
{
    *result = w0;
    if (n == 1) return TARA_OK;
    const double2* tw = unit_roots(n);
    TARA_CHECK(tw, TARA_ERR_ALLOC, "root table allocation failed (n = %d)", n);
    double2 *x = w0, *y = w1;
    int L = n;
    for (int r : radices(n)) {
        hipLaunchKernelGGL(k_any_pass, dim3(blocks_for(ntrans * n)), dim3(256), 0, st, x, y, n, L, r, ntrans, es, ts,
                           tfast, tw, dir);
        TARA_HIP(hipGetLastError());
        L /= r;
        std::swap(x, y);
    }
    *result = x;
    return TARA_OK;
}

}  // namespace

int any_col_fft(double2* a, int n, int ncols, long es, long pstride, int nplanes, int dir, hipStream_t st)
{
    TARA_CHECK(n >= 1 && ncols >= 1 && nplanes >= 1, TARA_ERR_ARG, "any_col_fft: bad shape");
    if (n == 1) return TARA_OK;
    const long ntrans = (long)ncols * nplanes;
    AnyArgs q;
    if (any_lds(n, ntrans, q)) {
        q.src = q.dst = a;
        q.dir = dir;
        q.es = es;
        q.pstride = pstride;
        q.ncols = ncols;
        return launch_any_lds<ANY_COL>(q, st);
    }
    DevBuf b0, b1;
    int rc;
    if ((rc = b0.alloc((size_t)ntrans * n * sizeof(double2))) || (rc = b1.alloc((size_t)ntrans * n * sizeof(double2))))
        return rc;
    hipLaunchKernelGGL(k_any_gather, dim3(blocks_for(ntrans * n)), dim3(256), 0, st, a, b0.as<double2>(), n, ncols, es,
                       pstride, ntrans);
    TARA_HIP(hipGetLastError());
    double2* res = nullptr;
    if ((rc = run_passes(b0.as<double2>(), b1.as<double2>(), n, ntrans, ntrans, 1, 1, dir, st, &res))) return rc;
    hipLaunchKernelGGL(k_any_scatter, dim3(blocks_for(ntrans * n)), dim3(256), 0, st, res, a, n, ncols, es, pstride,
                       ntrans);
    TARA_HIP(hipGetLastError());
    TARA_HIP(hipStreamSynchronize(st));
    return TARA_OK;
}

int any_row_r2c(const double* x, double2* X, int nx, int ld, int nrows, hipStream_t st)
{
    TARA_CHECK(nx >= 1 && nrows >= 1 && ld >= nx / 2 + 1, TARA_ERR_ARG, "any_row_r2c: bad shape");
    AnyArgs q;
    if (any_lds(nx, nrows, q)) {
        q.src = x;
        q.dst = X;
        q.dir = -1;
        q.ld = ld;
        return launch_any_lds<ANY_R2C>(q, st);
    }
    const long total = (long)nrows * nx;
    DevBuf b0, b1;
    int rc;
    if ((rc = b0.alloc((size_t)total * sizeof(double2))) || (rc = b1.alloc((size_t)total * sizeof(double2)))) return rc;
    hipLaunchKernelGGL(k_any_real_in, dim3(blocks_for(total)), dim3(256), 0, st, x, b0.as<double2>(), total);
    TARA_HIP(hipGetLastError());
    double2* res = nullptr;
    if ((rc = run_passes(b0.as<double2>(), b1.as<double2>(), nx, nrows, 1, nx, 0, -1, st, &res))) return rc;
    hipLaunchKernelGGL(k_any_half_out, dim3(blocks_for((long)nrows * ld)), dim3(256), 0, st, res, X, nx, ld,
                       (long)nrows);
    TARA_HIP(hipGetLastError());
    TARA_HIP(hipStreamSynchronize(st));
    return TARA_OK;
}

int any_row_c2r(const double2* X, double* x, int nx, int ld, int nrows, double s, hipStream_t st)
{
    TARA_CHECK(nx >= 1 && nrows >= 1 && ld >= nx / 2 + 1, TARA_ERR_ARG, "any_row_c2r: bad shape");
    AnyArgs q;
    if (any_lds(nx, nrows, q)) {
        q.src = X;
        q.dst = x;
        q.dir = +1;
        q.ld = ld;
        q.scale = s;
        return launch_any_lds<ANY_C2R>(q, st);
    }
    const long total = (long)nrows * nx;
    DevBuf b0, b1;
    int rc;
    if ((rc = b0.alloc((size_t)total * sizeof(double2))) || (rc = b1.alloc((size_t)total * sizeof(double2)))) return rc;
    hipLaunchKernelGGL(k_any_herm_in, dim3(blocks_for(total)), dim3(256), 0, st, X, b0.as<double2>(), nx, ld,
                       (long)nrows);
    TARA_HIP(hipGetLastError());
    double2* res = nullptr;
    if ((rc = run_passes(b0.as<double2>(), b1.as<double2>(), nx, nrows, 1, nx, 0, +1, st, &res))) return rc;
    hipLaunchKernelGGL(k_any_real_out, dim3(blocks_for(total)), dim3(256), 0, st, res, x, s, total);
    TARA_HIP(hipGetLastError());
    TARA_HIP(hipStreamSynchronize(st));
    return TARA_OK;
}

}  // namespace tara
