// Tiled transposes through LDS (32 x 32 complex tiles, one padding column) for
// the kx-fastest <-> ky-major conversions at the host boundary, and the packing
// of padded rows for host copies.
#include "layout.h"

namespace tara {

// out[c*rows + r] = in[r*cols + c] within each plane (rows x cols, row-major in).
__global__ __launch_bounds__(256) void k_transpose(const double2* __restrict__ in, double2* __restrict__ out,
                                                   int rows, int cols, int* zero, int* one)
{
    if (threadIdx.x == 0 && blockIdx.x + blockIdx.y + blockIdx.z == 0) {
        if (zero) *zero = 0;
        if (one) *one = 1;
    }
    __shared__ double2 tile[32][33];
    const size_t plane = (size_t)blockIdx.z * rows * cols;
    const int c0 = blockIdx.x * 32, r0 = blockIdx.y * 32;
    const int tx = threadIdx.x % 32, ty = threadIdx.x / 32;  // 32 x 8
    for (int k = ty; k < 32; k += 8) {
        const int r = r0 + k, c = c0 + tx;
        if (r < rows && c < cols) tile[k][tx] = in[plane + (size_t)r * cols + c];
    }
    __syncthreads();
    for (int k = ty; k < 32; k += 8) {
        const int c = c0 + k, r = r0 + tx;
        if (r < rows && c < cols) out[plane + (size_t)c * rows + r] = tile[tx][k];
    }
}

static int transpose(const double2* in, double2* out, int rows, int cols, int nplanes, hipStream_t st,
                     int* zero = nullptr, int* one = nullptr)
{
    dim3 g((cols + 31) / 32, (rows + 31) / 32, nplanes);
    hipLaunchKernelGGL(k_transpose, g, dim3(256), 0, st, in, out, rows, cols, zero, one);
    TARA_HIP(hipGetLastError());
    return TARA_OK;
}

int to_kymajor(const double2* src, double2* dst, int nh, int ny, int nplanes, hipStream_t st, int* zero, int* one)
{
    return transpose(src, dst, ny, nh, nplanes, st, zero, one);
}

int from_kymajor(const double2* src, double2* dst, int nh, int ny, int nplanes, hipStream_t st)
{
    return transpose(src, dst, nh, ny, nplanes, st);
}

// One thread per element of the padded or packed rows; both streams are read
// and written contiguously, so the kernel runs at the copy rate (0.1 ms for
// the 270 MB above) and the host link bounds the transfer.
template <bool PACK>
__global__ __launch_bounds__(256) void k_rows(RowFields f, int nh, int ld, size_t rows)
{
    const double2* src = f.src[blockIdx.y];
    double2* dst = f.dst[blockIdx.y];
    const int w = PACK ? nh : ld;
    for (size_t q = blockIdx.x * (size_t)blockDim.x + threadIdx.x; q < rows * w; q += (size_t)gridDim.x * blockDim.x) {
        const size_t r = q / w;
        const int i = (int)(q - r * w);
        if (PACK)
            dst[q] = src[r * ld + i];
        else
            dst[q] = i < nh ? src[r * nh + i] : make_double2(0.0, 0.0);
    }
}

template <bool PACK>
static int launch_rows(const RowFields& f, int nfields, int nh, int ld, size_t rows, hipStream_t st)
{
    TARA_CHECK(nfields >= 1 && nfields <= 8 && nh <= ld, TARA_ERR_ARG, "row packing: bad shape");
    const size_t n = rows * (PACK ? nh : ld), nb = (n + 255) / 256;
    hipLaunchKernelGGL(k_rows<PACK>, dim3((unsigned)(nb < 16384 ? nb : 16384), nfields), dim3(256), 0, st, f, nh, ld,
                       rows);
    TARA_HIP(hipGetLastError());
    return TARA_OK;
}

int pack_rows(const RowFields& f, int nfields, int nh, int ld, size_t rows, hipStream_t st)
{
    return launch_rows<true>(f, nfields, nh, ld, rows, st);
}

int unpack_rows(const RowFields& f, int nfields, int nh, int ld, size_t rows, hipStream_t st)
{
    return launch_rows<false>(f, nfields, nh, ld, rows, st);
}

int rows_from_host(double2* const dev[], const double* const host[], int nfields, int nh, int ld, size_t rows,
                   const DevBuf& pack, hipStream_t st)
{
    const size_t n = rows * nh;
    TARA_CHECK(nfields >= 1 && nfields <= 8 && pack.bytes >= nfields * n * sizeof(double2), TARA_ERR_STATE,
               "row transfer: work space too small");
    RowFields f{};
    for (int k = 0; k < nfields; ++k) {
        f.src[k] = pack.as<double2>() + k * n;
        f.dst[k] = dev[k];
        TARA_HIP(hipMemcpyAsync(pack.as<double2>() + k * n, host[k], n * sizeof(double2), hipMemcpyHostToDevice, st));
    }
    return unpack_rows(f, nfields, nh, ld, rows, st);
}

int rows_to_host(double* const host[], const double2* const dev[], int nfields, int nh, int ld, size_t rows,
                 const DevBuf& pack, hipStream_t st)
{
    const size_t n = rows * nh;
    TARA_CHECK(nfields >= 1 && nfields <= 8 && pack.bytes >= nfields * n * sizeof(double2), TARA_ERR_STATE,
               "row transfer: work space too small");
    RowFields f{};
    for (int k = 0; k < nfields; ++k) {
        f.src[k] = dev[k];
        f.dst[k] = pack.as<double2>() + k * n;
    }
    int rc = pack_rows(f, nfields, nh, ld, rows, st);
    if (rc) return rc;
    for (int k = 0; k < nfields; ++k)
        TARA_HIP(hipMemcpyAsync(host[k], pack.as<double2>() + k * n, n * sizeof(double2), hipMemcpyDeviceToHost, st));
    return TARA_OK;
}

}  // namespace tara
