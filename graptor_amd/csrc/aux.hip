// Auxiliary device work: the FP64 operator-norm power iteration
// (radon_normest, radon_tgv_primal_dual_2d.py 2D:576-588) and the
// feasibility mask (Make_function_feasible, 2D:476-486).
#include "common.h"

#include <algorithm>
#include <cmath>
#include <vector>

namespace gr {

namespace {

// The FP64 pair of the power iteration works on one slice, so there is little
// of everything: the kernels split their sums over the waves of a work-group
// to fill the chip, and normalisation and sums ride along (two launches a
// round).  256 x 256, 60 angles, per round: 225 us with a thread per bin, one
// per pixel and sums in one work-group; 26 us so (projection 13.5,
// backprojection 12).  What is left is the latency of the candidates' loads
// and of the launches.
constexpr int T64 = 1024;             // threads
constexpr int W64 = T64 / 64;         // waves: shares of the lines of 64 bins
constexpr int TILE64 = 16;            // pixels of a tile's side, T64 / 256 shares of the angles
constexpr int PARTS64 = 1024;         // work-groups, and so partial sums, of the backprojection

// Sum of a value over the work-group, in a fixed order.
__device__ __forceinline__ double block_sum64(double v, double* red)
{
    for (int w = 32; w > 0; w >>= 1) v += __shfl_xor(v, w);
    __syncthreads();
    if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = v;
    __syncthreads();
    double s = 0.0;
    for (int w = 0; w < W64; ++w) s += red[w];
    return s;
}

// Forward projection of img / n, n the sum of the partial sums (root: its
// square root), for 64 bins of an angle; the same hat-weight gather as the
// FP32 kernel, with four candidates so that any rounding of the float
// constants is tolerated (WIDE: bins of more pixels, as many as their hats
// reach over).  Candidates are contiguous: rows of the image, or of its
// transpose where the lines are columns.
template <bool WIDE>
__global__ __launch_bounds__(T64) void fwd64_kernel(const double* __restrict__ img,
                                                    const double* __restrict__ imgt,
                                                    double* __restrict__ sino,
                                                    const FwdAngle* __restrict__ angs, int nx,
                                                    int ny, int nd, const double* parts,
                                                    int nparts, int root, double* norm)
{
    __shared__ double red[W64], sums[W64][64];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int groups = (nd + 63) / 64, aa = blockIdx.x / groups;
    const int i = (blockIdx.x - aa * groups) * 64 + lane;
    const FwdAngle A = angs[aa];
    const int len_step = A.cls == 0 ? nx : ny;
    const int len_cand = A.cls == 0 ? ny : nx;
    const double* __restrict__ src = A.cls == 0 ? imgt : img;
    const double ms = A.mstep, mc = A.mcand, inv = 1.0 / mc, half = fabs(inv);
    const double ro = (double)A.off - (double)i;
    double acc = 0.0;
#pragma unroll 2
    for (int l = wave; l < len_step; l += W64) {
        const double r = (double)l * ms + ro;
        if constexpr (WIDE) {
            const double* __restrict__ line = src + (size_t)l * len_cand;
            const double hi = (double)len_cand;
            const int b = (int)fmin(fmax(ceil(-r * inv - half) - 1.0, 0.0), hi);
            const int e = (int)fmin(fmax(floor(-r * inv + half) + 2.0, 0.0), hi);
            for (int c = b; c < e; ++c)
                acc += fmax(1.0 - fabs((double)c * mc + r), 0.0) * line[c];
            continue;
        }
        const double first = fmin(fmax(ceil(-r * inv - half) - 1.0, -4.0), (double)len_cand);
        const int b = (int)first;
        const double* __restrict__ line = src + (size_t)l * len_cand;
#pragma unroll
        for (int k = 0; k < 4; ++k) {
            const bool in = b + k >= 0 && b + k < len_cand;
            const double v = line[in ? b + k : 0];
            const double wgt = fmax(1.0 - fabs((first + k) * mc + r), 0.0);
            acc += in && wgt > 0.0 ? wgt * v : 0.0;
        }
    }
    double part = 0.0;
    for (int e = threadIdx.x; e < nparts; e += T64) part += parts[e];
    double n = block_sum64(part, red);
    if (root) n = sqrt(n);
    if (blockIdx.x == 0 && threadIdx.x == 0) *norm = n;
    sums[wave][lane] = acc;
    __syncthreads();
    if (wave == 0 && i < nd) {
        double s = 0.0;
        for (int w = 0; w < W64; ++w) s += sums[w][lane];
        sino[(size_t)A.id * nd + i] = s / n;
    }
}

// A round's new image: the backprojection of one slice (2D:436-462), or with
// no sinogram the image itself; its transpose; and the partial sums of its
// values (square: of their squares) and, if asked for, of their products with
// the values they replace.
__global__ __launch_bounds__(T64) void adj64_kernel(const double* __restrict__ sino,
                                                    double* __restrict__ img,
                                                    double* __restrict__ imgt,
                                                    const float4* __restrict__ ofs, int nx,
                                                    int ny, int nd, int na, int square,
                                                    double* parts, double* dots)
{
    constexpr int NP = TILE64 * TILE64, SH = T64 / NP;
    __shared__ double red[W64], sums[SH][NP], tile[TILE64][TILE64 + 1];
    const int px = threadIdx.x % NP, share = threadIdx.x / NP;
    const int tx = px % TILE64, ty = px / TILE64;
    const int tiles_x = (nx + TILE64 - 1) / TILE64, tiles_y = (ny + TILE64 - 1) / TILE64;
    double part = 0.0, dot = 0.0;
    for (int t = blockIdx.x; t < tiles_x * tiles_y; t += gridDim.x) {
        const int x0 = t % tiles_x * TILE64, y0 = t / tiles_x * TILE64;
        const int x = x0 + tx, y = y0 + ty;
        const bool in = x < nx && y < ny;
        const size_t at = (size_t)min(y, ny - 1) * nx + min(x, nx - 1);
        double acc = 0.0;
        if (sino) {
#pragma unroll 4
            for (int j = share; j < na; j += SH) {
                const float4 o = ofs[j];
                const double d = (double)x * o.x + (double)y * o.y + (double)o.z;
                const double fl = fmin(fmax(floor(d), -2.0), (double)nd);
                const double p = d - fl;
                const int i0 = (int)fl;
                const bool lo = i0 >= 0 && i0 < nd, hi = i0 >= -1 && i0 <= nd - 2 && p > 0.0;
                const double* __restrict__ row = sino + (size_t)j * nd;
                const double a = row[lo ? i0 : 0], b = row[hi ? i0 + 1 : 0];
                acc += lo ? (1.0 - p) * a : 0.0;
                acc += hi ? p * b : 0.0;
            }
        } else if (share == 0) {
            acc = img[at];
        }
        sums[share][px] = acc;
        __syncthreads();
        if (share == 0) {
            double v = sums[0][px];
            for (int k = 1; k < SH; ++k) v += sums[k][px];
            if (in) {
                part += square ? v * v : v;
                if (dots) dot += img[at] * v;
                img[at] = v;
            }
            tile[ty][tx] = v;
        }
        __syncthreads();
        if (share == 0 && x0 + ty < nx && y0 + tx < ny)
            imgt[(size_t)(x0 + ty) * ny + y0 + tx] = tile[tx][ty];
    }
    part = block_sum64(part, red);
    if (threadIdx.x == 0) parts[blockIdx.x] = part;
    if (dots) {
        dot = block_sum64(dot, red);
        if (threadIdx.x == 0) dots[blockIdx.x] = dot;
    }
}

__global__ __launch_bounds__(T64) void sum64_kernel(const double* parts, int n, double* out)
{
    __shared__ double red[W64];
    double v = 0.0;
    for (int e = threadIdx.x; e < n; e += T64) v += parts[e];
    v = block_sum64(v, red);
    if (threadIdx.x == 0) *out = v;
}

__global__ void feasible_kernel(float* f, const float* r1, size_t per_slice, size_t total)
{
    const size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= total) return;
    if (r1[i % per_slice] <= 0.f) f[i] = 0.f;
}

__global__ void fill_kernel(float* x, size_t n, float v)
{
    const size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) x[i] = v;
}

}  // namespace

int launch_normest(const Geometry& g, const double* x0_host, int iters, int mode, double tol,
                   double* out, hipStream_t st)
{
    const size_t npx = (size_t)g.nx * g.ny, nsb = (size_t)g.nd * g.na;
    // image, its transpose, sinogram, two sets of partial sums, norm and dot
    double* x = nullptr;
    if (hipMalloc(&x, sizeof(double) * (2 * npx + nsb + 2 * PARTS64 + 2)) != hipSuccess) {
        set_error("normest: device allocation failed");
        return GR_ERR_OOM;
    }
    double *xt = x + npx, *s = xt + npx, *parts = s + nsb, *dots = parts + PARTS64;
    double* red = dots + PARTS64;
    std::vector<double> h0;
    if (!x0_host) {
        h0.resize(npx);
        for (size_t i = 0; i < npx; ++i) h0[i] = 1.0 + 0.25 * std::sin(0.37 * (int)i);
        x0_host = h0.data();
    }
    int rc = GR_OK;
    auto chk = [&](hipError_t e, const char* w) {
        if (e != hipSuccess && rc == GR_OK) rc = hip_status(e, w);
    };
    chk(hipMemcpyAsync(x, x0_host, sizeof(double) * npx, hipMemcpyHostToDevice, st),
        "normest copy");
    const float4* ofs = reinterpret_cast<const float4*>(g.ofs_dev);
    const bool power = mode != GR_NORMEST_REFERENCE;
    const long long tiles = (long long)((g.nx + TILE64 - 1) / TILE64) *
                            ((g.ny + TILE64 - 1) / TILE64);
    const int np = (int)std::min<long long>(tiles, PARTS64);
    const unsigned fb = (unsigned)((g.nd + 63) / 64) * (unsigned)g.na;
    auto image = [&](const double* sino, double* dot) {
        hipLaunchKernelGGL(adj64_kernel, dim3(np), dim3(T64), 0, st, sino, x, xt, ofs, g.nx, g.ny,
                           g.nd, g.na, power ? 1 : 0, parts, dot);
    };
    if (rc == GR_OK) image(nullptr, nullptr);
    double result = 0.0, prev = 0.0, h[2] = {0.0, 0.0};  // norm, dot
    for (int it = 0; it < iters && rc == GR_OK; ++it) {
        hipLaunchKernelGGL(g.wide_bins ? fwd64_kernel<true> : fwd64_kernel<false>, dim3(fb),
                           dim3(T64), 0, st, x, xt, s, g.fwd_dev, g.nx, g.ny, g.nd, parts, np,
                           power ? 1 : 0, red);
        image(s, power ? dots : nullptr);
        chk(hipGetLastError(), "normest launch");
        if (!power && it + 1 < iters) continue;
        if (power) {
            hipLaunchKernelGGL(sum64_kernel, dim3(1), dim3(T64), 0, st, dots, np, red + 1);
            chk(hipGetLastError(), "normest launch");
        }
        chk(hipMemcpyAsync(h, red, sizeof(double) * (power ? 2 : 1), hipMemcpyDeviceToHost, st),
            "normest read");
        chk(hipStreamSynchronize(st), "normest sync");
        if (!power) {
            result = std::sqrt(h[0]);
            break;
        }
        const double lam = h[1] / h[0];  // of the normalised image
        result = std::sqrt(std::max(lam, 0.0));
        if (it > 0 && std::fabs(lam - prev) <= tol * std::fabs(lam)) break;
        prev = lam;
    }
    (void)hipFree(x);
    if (rc != GR_OK) return rc;
    *out = result;
    return GR_OK;
}

int launch_feasible(const Geometry& g, float* f, int nslices, hipStream_t st)
{
    const size_t npx = (size_t)g.nx * g.ny, per = (size_t)g.nd * g.na;
    float *ones = nullptr, *r1 = nullptr;
    if (hipMalloc(&ones, npx * 4) != hipSuccess || hipMalloc(&r1, per * 4) != hipSuccess) {
        if (ones) (void)hipFree(ones);
        set_error("make_feasible: device allocation failed");
        return GR_ERR_OOM;
    }
    const int tb = 256;
    hipLaunchKernelGGL(fill_kernel, dim3((unsigned)((npx + tb - 1) / tb)), dim3(tb), 0, st, ones,
                       npx, 1.0f);
    ProbDev P{};
    P.dim = 2; P.nx = g.nx; P.ny = g.ny; P.nz = 1; P.nch = 1; P.nd = g.nd; P.na = g.na;
    P.ofs = reinterpret_cast<const float4*>(g.ofs_dev);
    P.fwd = g.fwd_dev;
    P.fwd_band = g.fwd_band;
    P.ubar = ones;
    P.ku = r1;
    int rc = launch_fwd(P, g, 1, FWD_WRITE, st);
    if (rc == GR_OK) {
        const size_t total = per * (size_t)nslices;
        hipLaunchKernelGGL(feasible_kernel, dim3((unsigned)((total + tb - 1) / tb)), dim3(tb), 0,
                           st, f, r1, per, total);
        hipError_t e = hipGetLastError();
        if (e == hipSuccess) e = hipStreamSynchronize(st);
        if (e != hipSuccess) rc = hip_status(e, "make_feasible");
    }
    (void)hipFree(ones);
    (void)hipFree(r1);
    return rc;
}

}  // namespace gr
