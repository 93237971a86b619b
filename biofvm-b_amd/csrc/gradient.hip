// gradient.hip -- density gradients of the device-resident field.
//
// Microenvironment::compute_all_gradient_vectors (BioFVM_microenvironment.cpp:1243-1386) and
// compute_gradient_vector (:1388-1533), per voxel, substrate and axis:
//   interior  (rho[+1] - rho[-1]) / (2*dx),   first  (rho[1] - rho[0]) / dx,
//   last      (rho[n-1] - rho[n-2]) / dx,
// every subtraction and division rounded on its own (FP64 arithmetic on both storage
// paths).  An axis of length 1 gives 0: the reference leaves z at its initial 0 then and
// reads outside the field for x or y.
//
// The full field is written as [substrate*3 + axis][z][y][x] in the field's precision, so
// that the voxel-major download ([voxel][substrate][axis], gradient_vectors' layout) is the
// field transpose with 3*nsub components.
#include <algorithm>

#include "bfvmb_internal.hpp"

namespace bfvmb {
namespace {

__device__ __forceinline__ double axis_diff(const double lo, const double mid, const double hi, int i, int n,
                                            double dx, double two_dx)
{
    if (n == 1)
        return 0.0;
    if (i == 0)
        return (hi - mid) / dx;
    if (i == n - 1)
        return (mid - lo) / dx;
    return (hi - lo) / two_dx;
}

// RN(a / d) for the divisor d whose certified reciprocal pair is (hi, lo); `odd` is set where the
// pair does not apply: -0, values whose product with lo is not normal, infinities and NaN.
__device__ __forceinline__ double pair_quotient(double a, double hi, double lo, bool &odd)
{
    const double m = fabs(a);
    odd |= !(m >= 0x1p-900 && m <= 0x1p960) && __double_as_longlong(a) != 0;
    return fma(a, hi, a * lo);
}

constexpr int kGradBlock = 256;

// One thread per voxel column piece: (substrate, x, y) and zlen planes, its z neighbours carried
// in registers, ROWS planes' loads in flight at a time; the neighbours along x and y hit the L1.
// Blocks take consecutive pieces of a plane, and each XCD a contiguous range of blocks, so that
// neighbouring rows share its L2.  What bounds it is HBM, three results per value read; what
// bounded one thread per voxel was arithmetic, of which the voxel's coordinates (64-bit
// divisions) were the larger part, here once per piece in 32 bits, and three FP64 divisions by
// dx or 2 dx the rest.  Those are products with a certified reciprocal pair (PAIR; 2 dx takes
// half of dx's pair), a voxel whose differences the pair does not cover divides.
// Microseconds, one thread per voxel -> this: FP32 97 x 61 x 83 x 3 14 -> 9.5, 190 x 161 x 177
// x 3 121 -> 55 (4.7 TB/s; 61 with divisions), 400^3 550 -> 280; FP64 128^3 x 2 31 -> 24 (5.5
// TB/s), 400^3 x 2 1190 -> 1060; 250 x 230 x 210 x 2 FP64 stays at 230.  32 planes per thread
// or non-temporal stores: no gain; 8 planes: 58 instead of 55, 400^3 the same.

template <class T, bool PAIR, int ROWS>
__global__ __launch_bounds__(kGradBlock) void k_gradients(const T *__restrict__ f, int nx, int ny, int nz,
                                                          unsigned blocks, int zlen, unsigned items, double dx,
                                                          double inv_hi, double inv_lo, T *__restrict__ grad)
{
    const unsigned nxy = (unsigned)nx * (unsigned)ny;
    const size_t nvox = (size_t)nxy * nz;
    const unsigned b = blockIdx.x, share = gridDim.x / 8, more = gridDim.x % 8;
    const unsigned t = b % 8 * share + min(b % 8, more) + b / 8;
    const unsigned s = t / blocks, item = (t - s * blocks) * kGradBlock + threadIdx.x;
    if (item >= items)
        return;
    const unsigned chunk = item / nxy, p = item - chunk * nxy;
    const int z0 = (int)chunk * zlen, z1 = min(z0 + zlen, nz);
    const int y = (int)(p / (unsigned)nx), x = (int)(p - (unsigned)y * (unsigned)nx);
    // (f[hi] - f[lo]) / d on every axis: one-sided ends have lo or hi at the voxel itself
    const int xl = x > 0 ? -1 : 0, xh = x < nx - 1 ? 1 : 0;
    const ptrdiff_t yl = y > 0 ? -(ptrdiff_t)nx : 0, yh = y < ny - 1 ? nx : 0;
    const double sx = xh - xl == 2 ? 2.0 : 1.0, sy = y > 0 && y < ny - 1 ? 2.0 : 1.0;
    const double hx = inv_hi / sx, lx = inv_lo / sx, hy = inv_hi / sy, ly = inv_lo / sy;
    const T *q = f + (size_t)s * nvox + p;
    T *g = grad + (size_t)s * 3 * nvox + p;
    double below = (double)q[(size_t)max(z0 - 1, 0) * nxy], mid = (double)q[(size_t)z0 * nxy];
    for (int z = z0; z < z1; z += ROWS) {
        T vx[ROWS][2], vy[ROWS][2], vz[ROWS];
#pragma unroll
        for (int r = 0; r < ROWS; ++r) {
            const T *c = q + (size_t)min(z + r, z1 - 1) * nxy;
            vx[r][0] = c[xl], vx[r][1] = c[xh];
            vy[r][0] = c[yl], vy[r][1] = c[yh];
            vz[r] = q[(size_t)min(z + r + 1, nz - 1) * nxy];
        }
#pragma unroll
        for (int r = 0; r < ROWS; ++r) {
            if (z + r >= z1)
                break;
            const double above = (double)vz[r];
            const double ax = (double)vx[r][1] - (double)vx[r][0], ay = (double)vy[r][1] - (double)vy[r][0];
            const double az = above - below;
            const double sz = z + r > 0 && z + r < nz - 1 ? 2.0 : 1.0;
            double gx, gy, gz;
            bool odd = !PAIR;
            if (PAIR) {
                gx = pair_quotient(ax, hx, lx, odd);
                gy = pair_quotient(ay, hy, ly, odd);
                gz = pair_quotient(az, inv_hi * (1.0 / sz), inv_lo * (1.0 / sz), odd);
            }
            if (odd) {
                gx = ax / (dx * sx);
                gy = ay / (dx * sy);
                gz = az / (dx * sz);
            }
            T *o = g + (size_t)(z + r) * nxy;
            o[0] = (T)(nx == 1 ? 0.0 : gx);
            o[nvox] = (T)(ny == 1 ? 0.0 : gy);
            o[2 * nvox] = (T)(nz == 1 ? 0.0 : gz);
            below = mid;
            mid = above;
        }
    }
}

// gradients at listed voxels (reference numbering), out[k][substrate][axis] in FP64
template <class T>
__global__ __launch_bounds__(256) void k_gradients_at(const T *__restrict__ f, int nx, int ny, int nz, int nsub,
                                                      double dx, const int *__restrict__ voxel, int n,
                                                      double *__restrict__ out)
{
    const long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= (long long)n * nsub)
        return;
    const int k = (int)(i / nsub), s = (int)(i - (long long)k * nsub);
    const int v = voxel[k];
    const int x = v / (ny * nz), rem = v - x * ny * nz, y = rem / nz, z = rem - y * nz;
    const size_t nxy = (size_t)nx * ny;
    const T *p = f + (size_t)s * nxy * nz + (size_t)z * nxy + (size_t)y * nx + x;
    const double two_dx = dx * 2.0;
    const double c = (double)p[0];
    const double xm = x > 0 ? (double)p[-1] : c, xp = x < nx - 1 ? (double)p[1] : c;
    const double ym = y > 0 ? (double)p[-(ptrdiff_t)nx] : c, yp = y < ny - 1 ? (double)p[nx] : c;
    const double zm = z > 0 ? (double)p[-(ptrdiff_t)nxy] : c, zp = z < nz - 1 ? (double)p[nxy] : c;
    double *o = out + (size_t)i * 3;
    o[0] = axis_diff(xm, c, xp, x, nx, dx, two_dx);
    o[1] = axis_diff(ym, c, yp, y, ny, dx, two_dx);
    o[2] = axis_diff(zm, c, zp, z, nz, dx, two_dx);
}

template <class T>
int compute_t(Group *g, Domain &d)
{
    const size_t n = d.nvox * d.nsub;
    if (!d.grad && hip_check(g, hipMalloc(&d.grad, 3 * n * sizeof(T)), "gradient buffer"))
        return BFVMB_ERR_NOMEM;
    const size_t nxy = d.nvox / d.nz;
    // Planes per thread: 16 where that leaves threads enough to fill the chip, 4 at least; a
    // tiny field (one wavefront per SIMD or two) is all latency, and one plane per thread is
    // the shorter chain: 50^3 FP64 3.2 against 3.6 us, 64^3 FP32 4.2 against 3.5.
    const bool tiny = n <= (1u << 17);
    int zlen = tiny ? 1 : 16;
    while (zlen > 4 && nxy * d.nsub * ((d.nz + zlen - 1) / zlen) < 256 * 2048)
        zlen /= 2;
    const unsigned items = (unsigned)(nxy * ((d.nz + zlen - 1) / zlen));
    const unsigned blocks = (items + kGradBlock - 1) / kGradBlock;
    double hi, lo;
    const bool pair = reciprocal_pair(d.dx, &hi, &lo);
    hipLaunchKernelGGL((!pair ? k_gradients<T, false, 4> : tiny ? k_gradients<T, true, 1> : k_gradients<T, true, 4>),
                       dim3(blocks * (unsigned)d.nsub), dim3(kGradBlock), 0, g->stream,
                       static_cast<const T *>(d.field[g->cur]), d.nx, d.ny, d.nz, blocks, zlen, items, d.dx, hi,
                       lo, static_cast<T *>(d.grad));
    return hip_check(g, hipGetLastError(), "gradient launch");
}

}  // namespace

int domain_compute_gradients(Group *g)
{
    if (g->doms.size() != 1)
        return set_error(g, BFVMB_ERR_ARG, "compute_gradients: single microenvironment only");
    Domain &d = g->doms[0];
    if (d.nvox * d.nsub >= (size_t)UINT32_MAX * 256)
        return set_error(g, BFVMB_ERR_ARG, "compute_gradients: field too large");
    const int rc = g->precision == BFVMB_FP64 ? compute_t<double>(g, d) : compute_t<float>(g, d);
    if (rc)
        return rc;
    d.grad_valid = true;
    return BFVMB_OK;
}

int domain_download_gradients(Group *g, double *out)
{
    if (g->doms.size() != 1 || !out)
        return set_error(g, BFVMB_ERR_ARG, "download_gradients: bad argument");
    Domain &d = g->doms[0];
    if (!d.grad || !d.grad_valid)
        return set_error(g, BFVMB_ERR_STATE, "download_gradients: compute_gradients has not been called");
    // the transpose with 3*nsub components maps [s*3+a][z][y][x] to [voxel][s][a]
    Domain view;
    view.nx = d.nx;
    view.ny = d.ny;
    view.nz = d.nz;
    view.nsub = 3 * d.nsub;
    const size_t bytes = d.nvox * view.nsub * sizeof(double);
    double *stage = nullptr;
    int rc;
    if ((rc = hip_check(g, hipMalloc((void **)&stage, bytes), "gradient staging")))
        return rc;
    if (!(rc = launch_soa_to_aos(g, view, d.grad, stage)))
        rc = hip_check(g, hipMemcpyAsync(out, stage, bytes, hipMemcpyDeviceToHost, g->stream), "gradient download");
    if (!rc)
        rc = hip_check(g, hipStreamSynchronize(g->stream), "gradient sync");
    (void)hipFree(stage);
    return rc;
}

int domain_gradients_at(Group *g, int n, const int *voxel, double *out)
{
    if (g->doms.size() != 1 || n < 0 || (n > 0 && (!voxel || !out)))
        return set_error(g, BFVMB_ERR_ARG, "gradients_at: bad argument");
    Domain &d = g->doms[0];
    for (int k = 0; k < n; ++k)
        if (voxel[k] < 0 || (size_t)voxel[k] >= d.nvox)
            return set_error(g, BFVMB_ERR_ARG, "gradients_at: voxel index out of range");
    if (n == 0)
        return BFVMB_OK;
    int *dv = nullptr;
    double *dout = nullptr;
    const size_t obytes = (size_t)n * d.nsub * 3 * sizeof(double);
    int rc;
    if (!(rc = hip_check(g, hipMalloc((void **)&dv, n * sizeof(int)), "gradient voxels")) &&
        !(rc = hip_check(g, hipMalloc((void **)&dout, obytes), "gradient output")) &&
        !(rc = hip_check(g, hipMemcpyAsync(dv, voxel, n * sizeof(int), hipMemcpyHostToDevice, g->stream), "voxels"))) {
        const unsigned grid = (unsigned)(((long long)n * d.nsub + 255) / 256);
        if (g->precision == BFVMB_FP64)
            hipLaunchKernelGGL(k_gradients_at<double>, dim3(grid), dim3(256), 0, g->stream,
                               static_cast<const double *>(d.field[g->cur]), d.nx, d.ny, d.nz, d.nsub, d.dx, dv, n,
                               dout);
        else
            hipLaunchKernelGGL(k_gradients_at<float>, dim3(grid), dim3(256), 0, g->stream,
                               static_cast<const float *>(d.field[g->cur]), d.nx, d.ny, d.nz, d.nsub, d.dx, dv, n,
                               dout);
        if (!(rc = hip_check(g, hipGetLastError(), "gradient launch")) &&
            !(rc = hip_check(g, hipMemcpyAsync(out, dout, obytes, hipMemcpyDeviceToHost, g->stream), "gradients")))
            rc = hip_check(g, hipStreamSynchronize(g->stream), "gradient sync");
    }
    (void)hipFree(dv);
    (void)hipFree(dout);
    return rc;
}

}  // namespace bfvmb

extern "C" int bfvmb_compute_gradients(bfvmb_ctx *ctx)
{
    return ctx ? bfvmb::domain_compute_gradients(ctx) : BFVMB_ERR_ARG;
}

extern "C" int bfvmb_download_gradients(bfvmb_ctx *ctx, double *grad_voxel_major)
{
    return ctx ? bfvmb::domain_download_gradients(ctx, grad_voxel_major) : BFVMB_ERR_ARG;
}

extern "C" int bfvmb_gradients_at(bfvmb_ctx *ctx, int n, const int *voxel, double *grad)
{
    return ctx ? bfvmb::domain_gradients_at(ctx, n, voxel, grad) : BFVMB_ERR_ARG;
}

extern "C" int bfvmb_gradient_device_ptr(bfvmb_ctx *ctx, void **ptr)
{
    if (!ctx || !ptr || ctx->doms.size() != 1)
        return BFVMB_ERR_ARG;
    *ptr = ctx->doms[0].grad;
    return BFVMB_OK;
}
