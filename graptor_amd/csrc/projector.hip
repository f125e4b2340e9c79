// Parallel-beam projector pair for gfx950.
//
// Forward projection: ray gather through LDS bands, fused with the KL/L2
// sinogram prox.  Backprojection: pixel tiles gathering from LDS-staged
// sinogram segments, optionally fused with the primal step of the
// primal-dual iteration (u, p updates and their extrapolations), so that
// K^T lam never goes through HBM.
//
// Discretisation (radon_tgv_primal_dual_2d.py 2D:391-462): with detector
// coordinate t(x, y) = x*cos + y*sin + off, bin i of the forward projection
// sums hat(t - i) * img over pixels, hat(d) = max(0, 1 - |d|), and the
// backprojection interpolates the sinogram linearly at t.  The two are exact
// transposes of each other.
#include "common.h"
#include "stencil.h"

#include <algorithm>
#include <cmath>
#include <cstdlib>

namespace gr {

namespace {

template <int K>
struct Pack {
    float v[K];
};

// LDS entries of K slices at a position: K <= 4 interleaved (one read of
// 4K bytes); K = 8 as two planes of four, hs floats apart, so that a
// 16-byte read per plane keeps the bank pattern of four slices.
template <int K>
__device__ __forceinline__ Pack<K> lds_load(const float* sh, int pos, int hs = 0)
{
    Pack<K> r;
    if constexpr (K == 8) {
        const float4 t = *reinterpret_cast<const float4*>(sh + 4 * pos);
        const float4 u = *reinterpret_cast<const float4*>(sh + 4 * pos + hs);
        r.v[0] = t.x; r.v[1] = t.y; r.v[2] = t.z; r.v[3] = t.w;
        r.v[4] = u.x; r.v[5] = u.y; r.v[6] = u.z; r.v[7] = u.w;
    } else if constexpr (K == 4) {
        const float4 t = *reinterpret_cast<const float4*>(sh + 4 * pos);
        r.v[0] = t.x; r.v[1] = t.y; r.v[2] = t.z; r.v[3] = t.w;
    } else if constexpr (K == 2) {
        const float2 t = *reinterpret_cast<const float2*>(sh + 2 * pos);
        r.v[0] = t.x; r.v[1] = t.y;
    } else {
        r.v[0] = sh[pos];
    }
    return r;
}

template <int K>
__device__ __forceinline__ void lds_store(float* sh, int pos, const float (&v)[K], int hs = 0)
{
    if constexpr (K == 8) {
        *reinterpret_cast<float4*>(sh + 4 * pos) = make_float4(v[0], v[1], v[2], v[3]);
        *reinterpret_cast<float4*>(sh + 4 * pos + hs) = make_float4(v[4], v[5], v[6], v[7]);
    } else if constexpr (K == 4) {
        *reinterpret_cast<float4*>(sh + 4 * pos) = make_float4(v[0], v[1], v[2], v[3]);
    } else if constexpr (K == 2) {
        *reinterpret_cast<float2*>(sh + 2 * pos) = make_float2(v[0], v[1]);
    } else {
        sh[pos] = v[0];
    }
}

// Sinogram epilogue of the projection by lines, K slices s0.. at (angle id,
// bin i): store and/or apply the prox (2D:316-338).  The gather has its own
// copy: called from there, this costs its schedule 3%.
template <int K>
__device__ __forceinline__ void fwd_epilogue(const ProbDev& P, int mode, int s0, int id, int i,
                                             const float (&val)[K])
{
    const int nslices = P.nz * P.nch;
#pragma unroll
    for (int k = 0; k < K; ++k) {
        const int s = s0 + k;
        if (s >= nslices) continue;
        const size_t idx = ((size_t)s * P.na + id) * P.nd + i;
        if (mode & FWD_WRITE) P.ku[idx] = val[k];
        if (mode & FWD_KL) {
            const float m = P.mfac[s / P.nz];
            const float sv = P.lam[idx] + P.sigma_p * val[k];
            const float z = sv - m;
            const float d = z * z + 4.f * P.sigma_p * P.f[idx] * m;
            P.lam[idx] = sv - 0.5f * (z + sqrtf(d));
        } else if (mode & FWD_L2) {
            const float m = P.mfac[s / P.nz];
            P.lam[idx] = (P.lam[idx] + P.sigma_p * (val[k] - P.f[idx])) * m;
        }
    }
}

// --------------------------------------------------------------------------
// Sheared forward projection (unit detector bins).  At line l of the stepping
// axis, candidate c = j + s(l) has detector coordinate
//   t = l mstep + c mcand + off = (j mcand + off) + d(l),  |d| <= |mcand| / 2,
// so along a fixed j the coordinate stays within one bin of the integer m
// nearest to j mcand + off.  An item (one lane) follows one j through the
// lines and, with v = t - m in [-1, 1], sums its hat-weighted contributions
// max(-v, 0) img to bin m - 1, (1 - |v|) img to m and max(v, 0) img to m + 1.
// (Sums of img, v img and |v| img, combined at the end, save two operations
// an item and line and no time, and cost a bit of precision.)  Neighbouring lanes read neighbouring
// pixels of a line, and s(l), d(l) are scalars of the wave, so lines are read
// from memory directly (no LDS, no barriers): rows of the image for class 1,
// rows of its transpose (P.ktl) for class 0.
//
// A work-group holds angles [a0, a0 + count) of K slices: for each J waves of
// items, times ns = 1 or 2: one wave for both halves of the lines, or one for
// each.  At the end the items' sums go through LDS, the halves are added, and
// every bin adds its items in the order of j; so neither K, ns nor a batch
// changes a value.
//
// What it replaces for stacks of few slices (the gather below) stages bands
// of lines in LDS behind barriers and finds each ray's candidates from the
// ray, 5 operations and a read for each of 3 candidates; with a work-group or
// less per CU its time is that chain's latency.  Here a line costs an item
// one read and 3 operations a slice and 5 for the weights, 8 lines in flight.  Bound by the L1's rate
// (about 8 cycles a wave's read) and, for single slices, by latency; two
// halves give single slices twice the waves (317 x 317 x 3, 71 angles, 10
// iterations: 1000 us with one wave, 898 with two; 183 x 183: 680, 630).
// --------------------------------------------------------------------------
typedef int ShearOct __attribute__((ext_vector_type(2 * SHEAR_BLOCK), aligned(4)));
typedef const __attribute__((address_space(4))) ShearOct* ShearOctPtr;

template <int K>
__device__ __forceinline__ void fwd_line_body(const ProbDev& P, int a0, int count, int s0, int J,
                                              int ns, int mode, float* sh)
{
    if (mode & FWD_PROX) mode |= P.disc == GR_DISC_KL ? FWD_KL : FWD_L2;
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int job = wave % J, run = wave / J % ns, al = wave / (J * ns);
    const int a = a0 + min(al, count - 1);
    const FwdAngle A = P.fwd[a];
    const int first = P.line0[a], n = P.line0[a + 1] - first;
    const int nline = A.cls == 0 ? P.nx : P.ny, ncand = A.cls == 0 ? P.ny : P.nx;
    const int last = P.nz * P.nch - 1;
    const float* __restrict__ img[K];
#pragma unroll
    for (int k = 0; k < K; ++k)
        img[k] = (A.cls == 0 ? P.ktl : P.ubar) + (size_t)min(s0 + k, last) * ((size_t)nline * ncand);

    // sums of the first and the second half of the lines, in this order
    // whichever waves take them; `part` is [angle][3][K][item]
    const int items = J * 64, i = job * 64 + lane;
    float* part = sh + (size_t)al * 3 * K * items;
    float acc[3][K];
    for (int half = run; half < 2; half += ns) {
#pragma unroll
        for (int m = 0; m < 3; ++m)
#pragma unroll
            for (int k = 0; k < K; ++k) acc[m][k] = 0.f;
        if (job * 64 < n && al < count) {
            const FwdLine L = P.lines[first + min(job * 64 + lane, n - 1)];
            const int jf = __builtin_amdgcn_readfirstlane(L.j), jl = __builtin_amdgcn_readlane(L.j, 63);
            const int blocks = (nline + SHEAR_BLOCK - 1) / SHEAR_BLOCK;
            const int b0 = blocks * half / 2, b1 = blocks * (half + 1) / 2;
            const ShearOctPtr table = (ShearOctPtr)(P.shear + (size_t)a * P.shear_stride);
            ShearOct next = table[b0];
            for (int b = b0; b < b1; ++b) {
                const ShearOct q = next;
                if (b + 1 < b1) next = table[b + 1];
                const int l0 = b * SHEAR_BLOCK;
                // candidates of the block's lines (s is monotonic along them)
                const int lo = jf + min(q[1], q[2 * SHEAR_BLOCK - 1]);
                const int hi = jl + max(q[1], q[2 * SHEAR_BLOCK - 1]);
                if (hi < 0 || lo >= ncand) continue;
                float p[SHEAR_BLOCK][K];
                if (lo >= 0 && hi < ncand && l0 + SHEAR_BLOCK <= nline) {
#pragma unroll
                    for (int l = 0; l < SHEAR_BLOCK; ++l) {
                        const unsigned at = (unsigned)(L.j + ((l0 + l) * ncand + q[2 * l + 1]));
#pragma unroll
                        for (int k = 0; k < K; ++k) p[l][k] = img[k][at];
                    }
                } else {  // zero beyond the image
#pragma unroll
                    for (int l = 0; l < SHEAR_BLOCK; ++l) {
                        const int c = L.j + q[2 * l + 1];
                        const bool in = c >= 0 && c < ncand && l0 + l < nline;
                        const unsigned at = in ? (unsigned)((l0 + l) * ncand + c) : 0u;
#pragma unroll
                        for (int k = 0; k < K; ++k) {
                            const float v = img[k][at];
                            p[l][k] = in ? v : 0.f;
                        }
                    }
                }
#pragma unroll
                for (int l = 0; l < SHEAR_BLOCK; ++l) {
                    const float v = L.rel + __int_as_float(q[2 * l]);
                    const float hi1 = fmaxf(v, 0.f), lo1 = hi1 - v, mid = 1.f - fabsf(v);
#pragma unroll
                    for (int k = 0; k < K; ++k) {
                        acc[0][k] = fmaf(lo1, p[l][k], acc[0][k]);
                        acc[1][k] = fmaf(mid, p[l][k], acc[1][k]);
                        acc[2][k] = fmaf(hi1, p[l][k], acc[2][k]);
                    }
                }
            }
        }
        if (half == 0 && al < count) {
#pragma unroll
            for (int m = 0; m < 3; ++m)
#pragma unroll
                for (int k = 0; k < K; ++k) part[(m * K + k) * items + i] = acc[m][k];
        }
    }
    if (ns > 1) __syncthreads();
    if (run == ns - 1 && al < count) {
#pragma unroll
        for (int m = 0; m < 3; ++m)
#pragma unroll
            for (int k = 0; k < K; ++k) part[(m * K + k) * items + i] += acc[m][k];
    }
    __syncthreads();
    if (al >= count) return;
    // the angle's bins, by its J ns waves
    for (int b = (run * J + job) * 64 + lane; b < P.nd; b += J * ns * 64) {
        const FwdBin B = P.bins[(size_t)a * P.nd + b];
        float val[K];
#pragma unroll
        for (int k = 0; k < K; ++k) val[k] = 0.f;
#pragma unroll
        for (int r = 0; r < FWD_BIN_ITEMS; ++r) {
            const int c = ((B.code >> (3 * r)) & 7) - 1;
            if (c < 0) continue;
#pragma unroll
            for (int k = 0; k < K; ++k) val[k] += part[(c * K + k) * items + B.first + r];
        }
        fwd_epilogue<K>(P, mode, s0, A.id, b, val);
    }
}

template <int K>
__global__ __launch_bounds__(1024) void fwd_line_kernel(ProbDev P, int J, int ns, int mode)
{
    extern __shared__ float sh[];
    const int work = xcd_work_id(blockIdx.x, gridDim.x);
    fwd_line_body<K>(P, work % P.na, 1, (work / P.na) * K, J, ns, mode, sh);
}

// An item by lines of a batch, of K slices, or (K = 0) as many as it says.
template <int K>
__device__ __forceinline__ void fwd_line_item(const ProbDev& P, const FwdItem& I, int mode,
                                              float* sh)
{
    if constexpr (K > 0) {
        fwd_line_body<K>(P, I.a0, I.na, I.s0, I.cls, 1, mode, sh);
    } else {
        switch (I.k) {
        case 4: fwd_line_body<4>(P, I.a0, I.na, I.s0, I.cls, 1, mode, sh); break;
        case 2: fwd_line_body<2>(P, I.a0, I.na, I.s0, I.cls, 1, mode, sh); break;
        default: fwd_line_body<1>(P, I.a0, I.na, I.s0, I.cls, 1, mode, sh);
        }
    }
}

template <int K>
__global__ __launch_bounds__(1024) void fwd_line_batch_kernel(const ProbDev* __restrict__ probs,
                                                              const FwdItem* __restrict__ items,
                                                              int mode)
{
    extern __shared__ float sh[];
    const FwdItem I = items[xcd_work_id(blockIdx.x, gridDim.x)];
    fwd_line_item<K>(load_prob(probs, I.prob), I, mode, sh);
}

// Tables of the sheared projection, a work-group per angle.  In 64 bits the
// products of an angle's floats and an item's or line's number are exact, so
// only sums and the quotient round; contraction would skip one rounding.
// Filled here because a geometry is made far more often than its tables are
// large: on the host they took 0.13 / 0.58 ms of 0.15 / 0.60 (256 x 256, 60 angles;
// 512 x 512, 120), with the copy, of every geometry's creation.
__device__ __forceinline__ int nearest_int(double x) { return (int)(x + (x < 0 ? -0.5 : 0.5)); }

__global__ __launch_bounds__(256) void line_tables_kernel(const FwdAngle* __restrict__ angs,
                                                          const int* __restrict__ line0,
                                                          const int* __restrict__ first, int nd,
                                                          int stride, Shear* __restrict__ shear,
                                                          FwdLine* __restrict__ lines,
                                                          FwdBin* __restrict__ bins)
{
#pragma clang fp contract(off)
    const int a = blockIdx.x, tid = threadIdx.x;
    const FwdAngle A = angs[a];
    const double ms = A.mstep, mc = A.mcand, off = A.off, inv = 1.0 / mc;
    const int i0 = line0[a], n = line0[a + 1] - i0, j0 = first[a];
    auto at = [&](int i) { return (double)(j0 + i) * mc + off; };
    for (int l = tid; l < stride; l += 256) {
        const int s = nearest_int(-l * ms * inv);
        shear[(size_t)a * stride + l] = Shear{(float)(l * ms + (double)s * mc), s};
    }
    for (int i = tid; i < n; i += 256) {
        const double t = at(i);
        lines[i0 + i] = FwdLine{j0 + i, (float)(t - (double)nearest_int(t))};
    }
    for (int b = tid; b < nd; b += 256) {
        // from an item before the bin's first on: its items follow each other
        const double edge = ((mc > 0 ? b - 1.5 : b + 1.5) - off) * inv;
        int i = min(max((int)floor(edge) - 2 - j0, 0), n);
        while (i < n && abs(nearest_int(at(i)) - b) > 1) ++i;
        FwdBin B{i < n ? i : 0, 0};
        for (int k = 0; k < FWD_BIN_ITEMS && i < n; ++k, ++i) {
            const int m = nearest_int(at(i));
            if (abs(m - b) > 1) break;
            B.code |= (b - m + 2) << (3 * k);
        }
        bins[(size_t)a * nd + b] = B;
    }
}

__global__ __launch_bounds__(256) void transpose_kernel(ProbDev P, int tiles_x, int tiles_y)
{
    __shared__ float tile[TRANSPOSE_FLOATS];
    const int tiles = tiles_x * tiles_y, t = blockIdx.x % tiles;
    transpose_tile(tile, P, blockIdx.x / tiles, 32 * (t % tiles_x), 32 * (t / tiles_x));
}

__global__ __launch_bounds__(256) void transpose_batch_kernel(const ProbDev* __restrict__ probs,
                                                              const DualItem* __restrict__ items)
{
    __shared__ float tile[TRANSPOSE_FLOATS];
    const DualItem I = items[blockIdx.x];
    const ProbDev P = load_prob(probs, I.prob);
    transpose_tile(tile, P, I.z, I.x0, I.y0);
}

// --------------------------------------------------------------------------
// Forward projection of one work item: K slices s0.. (sharing all geometry)
// times a chunk of (angle, bin) items whose angles step along the same axis.
// The K slices stream through LDS in bands of `band` lines of that axis; per
// line every item reads the <= 3 candidates on the other axis whose hat
// weight can be positive.  After the last band each item holds its complete
// ray sum and applies the sinogram epilogue.  WIDE: detector bins of more than
// 1.06 pixels, whose hats reach over more candidates (2 / |mcand|): a loop over
// those that lie in the image.
// --------------------------------------------------------------------------
template <int K, int MI, bool WIDE>
__device__ __forceinline__ void fwd_body(const ProbDev& P, const FwdItem& I, int mode,
                                         float* sh)
{
    if (mode & FWD_PROX) mode |= P.disc == GR_DISC_KL ? FWD_KL : FWD_L2;
    const int tid = threadIdx.x;
    const int nx = P.nx, ny = P.ny, nd = P.nd, na = P.na;
    const int nslices = P.nz * P.nch;
    const int band = P.fwd_band, pitch = P.fwd_pitch;
    const int len_step = I.cls == 0 ? nx : ny;
    const int len_cand = I.cls == 0 ? ny : nx;
    const int nitems = I.na * I.nb;
    const int s0 = I.s0;
    const float* __restrict__ img = P.ubar;

    // Per item, along the ray at stepping coordinate xs: the offset of the
    // candidate-axis origin from bin i is r = xs * mstep + (off - i); the
    // first candidate whose hat weight can be positive is
    // ceil(-r / mcand - hc) = ceil(xs * ta + tb).
    float acc[MI][K];
    float ms[MI], mc[MI], ro[MI], ta[MI], tb[MI];
    float reach[WIDE ? MI : 1];  // candidates of a hat
#pragma unroll
    for (int it = 0; it < MI; ++it) {
        const int item = tid + it * FWD_THREADS;
        const int a = item < nitems ? item / I.nb : 0;
        const FwdAngle A = P.fwd[I.a0 + a];
        const float fi = (float)(I.b0 + (item < nitems ? item - a * I.nb : 0));
        ms[it] = A.mstep;
        mc[it] = A.mcand;
        ro[it] = A.off - fi;
        ta[it] = -A.mstep * A.invc;
        tb[it] = fmaf(-ro[it], A.invc, -A.hc);
        if constexpr (WIDE) reach[it] = 2.f * A.hc;
#pragma unroll
        for (int k = 0; k < K; ++k) acc[it][k] = 0.f;
    }

    const int lds_floats = band * pitch * K;
    for (int e = tid; e < lds_floats; e += FWD_THREADS) sh[e] = 0.f;

    const float cand_hi = (float)len_cand;
    const size_t slice_stride = (size_t)nx * ny;
    // staging walk: element e = tid + j * FWD_THREADS of a band, split into
    // (outer, inner) = (e / n_in, e % n_in) by stepping rather than dividing
    // (n_in = candidates per line for rows, band for columns)
    const int n_in = I.cls == 1 ? len_cand : band;
    const int n_out = I.cls == 1 ? band : len_cand;
    const int st_out0 = tid / n_in, st_in0 = tid - st_out0 * n_in;
    const int st_dout = FWD_THREADS / n_in, st_din = FWD_THREADS - st_dout * n_in;
    for (int l0 = 0; l0 < len_step; l0 += band) {
        __syncthreads();
        // stage lines [l0, l0+band) of K slices, candidates contiguous
        if (I.cls == 1) {  // lines are rows, candidates are x
            for (int li = st_out0, x = st_in0; li < n_out;) {
                const int y = l0 + li;
                float v[K];
#pragma unroll
                for (int k = 0; k < K; ++k) {
                    const int s = s0 + k;
                    v[k] = (y < ny && s < nslices)
                               ? img[(size_t)s * slice_stride + (size_t)y * nx + x]
                               : 0.f;
                }
                lds_store<K>(sh, li * pitch + FWD_PADL + x, v);
                x += st_din;
                li += st_dout;
                if (x >= n_in) {
                    x -= n_in;
                    ++li;
                }
            }
        } else {  // lines are columns, candidates are y
            for (int y = st_out0, li = st_in0; y < n_out;) {
                const int x = l0 + li;
                float v[K];
#pragma unroll
                for (int k = 0; k < K; ++k) {
                    const int s = s0 + k;
                    v[k] = (x < nx && s < nslices)
                               ? img[(size_t)s * slice_stride + (size_t)y * nx + x]
                               : 0.f;
                }
                lds_store<K>(sh, li * pitch + FWD_PADL + y, v);
                li += st_din;
                y += st_dout;
                if (li >= n_in) {
                    li -= n_in;
                    ++y;
                }
            }
        }
        __syncthreads();

#pragma unroll
        for (int it = 0; it < MI; ++it) {
            if (tid + it * FWD_THREADS >= nitems) continue;
            float xs = (float)l0;  // exact integer-valued step coordinate
            for (int st = 0; st < band; ++st, xs += 1.f) {
                const float r = fmaf(xs, ms[it], ro[it]);
                if constexpr (WIDE) {
                    // one more on either side, for the rounding of the bounds
                    const float at = fmaf(xs, ta[it], tb[it]);
                    const int first = (int)__builtin_amdgcn_fmed3f(ceilf(at) - 1.f, 0.f, cand_hi);
                    const int end = (int)__builtin_amdgcn_fmed3f(floorf(at + reach[it]) + 2.f,
                                                                 0.f, cand_hi);
                    const float* line = sh + K * (st * pitch + FWD_PADL);
                    for (int c = first; c < end; ++c) {
                        const float d = fmaf((float)c, mc[it], r);
                        const float w = __builtin_amdgcn_fmed3f(1.f - fabsf(d), 0.f, 1.f);
                        const Pack<K> v = lds_load<K>(line, c);
#pragma unroll
                        for (int k = 0; k < K; ++k) acc[it][k] = fmaf(w, v.v[k], acc[it][k]);
                    }
                    continue;
                }
                float bf = ceilf(fmaf(xs, ta[it], tb[it]));
                // clamp into [-3, len_cand] (bf is never NaN: finite operands)
                bf = __builtin_amdgcn_fmed3f(bf, -3.f, cand_hi);
                const float d0 = fmaf(bf, mc[it], r);
                const float d1 = d0 + mc[it];
                const float d2 = d1 + mc[it];
                // hat weights max(0, 1 - |d|) (1 - |d| <= 1, so a clamp to [0, 1])
                const float w0 = __builtin_amdgcn_fmed3f(1.f - fabsf(d0), 0.f, 1.f);
                const float w1 = __builtin_amdgcn_fmed3f(1.f - fabsf(d1), 0.f, 1.f);
                const float w2 = __builtin_amdgcn_fmed3f(1.f - fabsf(d2), 0.f, 1.f);
                // line base is uniform across the wave; the candidate offset is per lane
                const float* line = sh + K * (st * pitch + FWD_PADL);
                const int c0 = (int)bf;
                const Pack<K> v0 = lds_load<K>(line, c0);
                const Pack<K> v1 = lds_load<K>(line, c0 + 1);
                const Pack<K> v2 = lds_load<K>(line, c0 + 2);
#pragma unroll
                for (int k = 0; k < K; ++k) {
                    float a = fmaf(w0, v0.v[k], acc[it][k]);
                    a = fmaf(w1, v1.v[k], a);
                    acc[it][k] = fmaf(w2, v2.v[k], a);
                }
            }
        }
    }

    // epilogue: store and/or apply the sinogram prox (2D:316-338)
#pragma unroll
    for (int it = 0; it < MI; ++it) {
        const int item = tid + it * FWD_THREADS;
        if (item >= nitems) continue;
        const int a = item / I.nb;
        const int i = I.b0 + item - a * I.nb;
        const int id = P.fwd[I.a0 + a].id;
#pragma unroll
        for (int k = 0; k < K; ++k) {
            const int s = s0 + k;
            if (s >= nslices) continue;
            const size_t idx = ((size_t)s * na + id) * nd + i;
            const float val = acc[it][k];
            if (mode & FWD_WRITE) P.ku[idx] = val;
            if (mode & FWD_KL) {
                const float m = P.mfac[s / P.nz];
                const float sv = P.lam[idx] + P.sigma_p * val;
                const float z = sv - m;
                const float d = z * z + 4.f * P.sigma_p * P.f[idx] * m;
                P.lam[idx] = sv - 0.5f * (z + sqrtf(d));
            } else if (mode & FWD_L2) {
                const float m = P.mfac[s / P.nz];
                P.lam[idx] = (P.lam[idx] + P.sigma_p * (val - P.f[idx])) * m;
            }
        }
    }
}

template <int K, int MI, bool WIDE>
__global__ __launch_bounds__(FWD_THREADS) void fwd_single_kernel(ProbDev P,
                                                                 const FwdChunk* __restrict__ chunks,
                                                                 int nchunks, int mode)
{
    extern __shared__ float sh[];
    const int work = xcd_work_id(blockIdx.x, gridDim.x);
    const FwdChunk ch = chunks[work % nchunks];
    const FwdItem I{0, ch.cls, ch.a0, ch.na, ch.b0, ch.nb, (work / nchunks) * K, 0};
    fwd_body<K, MI, WIDE>(P, I, mode, sh);
}

template <int K, int MI, bool WIDE>
__global__ __launch_bounds__(FWD_THREADS) void fwd_batch_kernel(const ProbDev* __restrict__ probs,
                                                                const FwdItem* __restrict__ items,
                                                                int mode)
{
    extern __shared__ float sh[];
    // items are sorted largest first; plain block order deals them
    // round-robin over the XCDs, which balances the load
    const FwdItem I = items[blockIdx.x];
    const ProbDev P = load_prob(probs, I.prob);
    fwd_body<K, MI, WIDE>(P, I, mode, sh);
}

// A small batch's gathered items and its items by lines: bound by the latency of
// one work-group and by the launch, of which two need two.
__global__ __launch_bounds__(FWD_THREADS) void fwd_mixed_batch_kernel(
    const ProbDev* __restrict__ probs, const FwdItem* __restrict__ items, int mode)
{
    extern __shared__ float sh[];
    const FwdItem I = items[blockIdx.x];
    const ProbDev P = load_prob(probs, I.prob);
    if (I.nb == 0) {
        fwd_line_item<0>(P, I, mode, sh);
        return;
    }
    switch (I.k) {
    case 4: fwd_body<4, 1, false>(P, I, mode, sh); break;
    case 2: fwd_body<2, 1, false>(P, I, mode, sh); break;
    default: fwd_body<1, 1, false>(P, I, mode, sh);
    }
}

// --------------------------------------------------------------------------
// Primal step at one voxel-channel (update_u 2D:340-357 / 3D:706-729,
// update_p 2D:359-376 / 3D:734-757, update_extra 2D:637-638):
//   u+ = max(0, u + tau (div v - ktl / L)),  ubar = 2 u+ - u
//   p+ = p + tau (v + div2 w),               pbar = 2 p+ - p
// i indexes u[c][z][y][x] (= slice s = z + nz c), z = s % nz.
// --------------------------------------------------------------------------
template <int DIM, bool TGV, int PART = PRIMAL_UP, bool ZH = false, bool NT = false>
__device__ __forceinline__ void primal_update_r(
    float* __restrict__ u, float* __restrict__ ubar, float* __restrict__ p,
    float* __restrict__ pbar, const float* __restrict__ v, const float* __restrict__ w, int nx,
    int ny, int nz, size_t cs, float hinv, float tau, float norming, size_t i, int x, int y, int z,
    float ktl, const ProbDev* zh)
{
    constexpr bool NU = (PART & PRIMAL_U) != 0, NP = (PART & PRIMAL_P) != 0;
    float un, ub, pn[3], pb[3];
    primal_point<DIM, TGV, NU, NP, true, ZH, NT>(u, p, v, w, ktl, nx, ny, nz, cs, hinv, tau, norming, i, x, y,
                                   z, un, ub, pn, pb, zh);
    // streamed once per iteration (NT: with the non-temporal hint)
    if constexpr (NU) {
        st_stream<NT>(un, &u[i]);
        st_stream<NT>(ub, &ubar[i]);
    }
    if constexpr (TGV && NP) {
#pragma unroll
        for (int k = 0; k < DIM; ++k) {
            st_stream<NT>(pn[k], &p[i + k * cs]);
            st_stream<NT>(pb[k], &pbar[i + k * cs]);
        }
    }
}

template <int DIM, bool TGV, int PART = PRIMAL_UP, bool ZH = false, bool NT = false>
__device__ __forceinline__ void primal_update(const ProbDev& P, size_t i, int x, int y, int z,
                                              float ktl)
{
    const size_t cs = (size_t)P.nx * P.ny * P.nz * P.nch;  // component stride
    primal_update_r<DIM, TGV, PART, ZH, NT>(P.u, P.ubar, P.p, P.pbar, P.v, P.w, P.nx, P.ny, P.nz,
                                            cs, P.hinv, P.tau, P.norming, i, x, y, z, ktl, &P);
}

// Primal step of one voxel-channel per thread with K^T lam read from memory
// (the unfused form: high occupancy for the memory-bound update).
template <int DIM, bool TGV, int PART = PRIMAL_UP, bool ZH = false, bool NT = false>
__device__ __forceinline__ void primal_body(const ProbDev& P, const DualItem& I)
{
    const int x = I.x0 + (int)(threadIdx.x & (DUAL_BX - 1));
    const int y = I.y0 + (int)(threadIdx.x / DUAL_BX);
    const int s = I.z;  // slice z + nz * c
    if (x >= P.nx || y >= P.ny) return;
    const size_t i = (size_t)s * P.nx * P.ny + (size_t)y * P.nx + x;
    const float ktl = (PART & PRIMAL_U) ? ld_stream<NT>(&P.ktl[i]) : 0.f;
    primal_update<DIM, TGV, PART, ZH, NT>(P, i, x, y, s % P.nz, ktl);
}

// PART selects the u half (needs K^T lam), the p half (needs only v and w,
// so it can run beside the projections) or both.
template <int DIM, bool TGV, int PART, bool ZH, bool NT>
__global__ __launch_bounds__(DUAL_BX* DUAL_BY) void primal_single_kernel(ProbDev P, int tiles_x,
                                                                         int tiles_y)
{
    const int b = stencil_block<PRIMAL_GROUP>();
    const int tx = b % tiles_x, rest = b / tiles_x;
    const DualItem I{0, tx * DUAL_BX, (rest % tiles_y) * DUAL_BY, rest / tiles_y};
    primal_body<DIM, TGV, PART, ZH, NT>(P, I);
}

// The u half with all channels of a voxel in one thread (a quarter of the
// work-groups of the per-channel form for 4 channels, each thread with as
// many independent load streams): 0.779 against 0.786 ms per two-stream
// iteration on 256x256x64x4 on one box, 0.791 against 0.798 ms on another,
// same bits.  The p half stays per channel (0.810 ms in this form).
template <int DIM, bool TGV, bool NT>
__global__ __launch_bounds__(DUAL_BX* DUAL_BY) void primal_u_voxel_kernel(ProbDev P, int tiles_x,
                                                                          int tiles_y)
{
    const int b = stencil_block<PRIMAL_GROUP>();
    const int tx = b % tiles_x, rest = b / tiles_x;
    const int x = tx * DUAL_BX + (int)(threadIdx.x & (DUAL_BX - 1));
    const int y = (rest % tiles_y) * DUAL_BY + (int)(threadIdx.x / DUAL_BX);
    const int z = rest / tiles_y;
    if (x >= P.nx || y >= P.ny) return;
    const size_t plane = (size_t)P.nx * P.ny;
    for (int c = 0; c < P.nch; ++c) {
        const size_t i = (size_t)(z + P.nz * c) * plane + (size_t)y * P.nx + x;
        const float ktl = ld_stream<NT>(&P.ktl[i]);
        primal_update<DIM, TGV, PRIMAL_U, false, NT>(P, i, x, y, z, ktl);
    }
}

template <int DIM, bool TGV, int PART>
__global__ __launch_bounds__(DUAL_BX* DUAL_BY) void primal_batch_kernel(
    const ProbDev* __restrict__ probs, const DualItem* __restrict__ items)
{
    const DualItem I = items[blockIdx.x];
    const ProbDev P = load_prob(probs, I.prob);
    primal_body<DIM, TGV, PART>(P, I);
}

// --------------------------------------------------------------------------
// Backprojection of one tile: 64 x tile_y pixels of K slices s0...  Per
// chunk of angles it stages, for each angle, only the sinogram segment the
// tile projects onto (bins outside [0, nd) staged as zeros, which reproduces
// the reference's edge guards), then every thread interpolates for its
// tile_y/4 pixels, tile_y <= 4 * MAXR (the accumulators a lane holds: 8 rows
// take 126 VGPRs, 4 rows 70).  PRIMAL fuses the primal step into the epilogue.
// --------------------------------------------------------------------------
template <int K, bool PRIMAL, int DIM, bool TGV, int MAXR = ADJ_MAXR>
__device__ __forceinline__ void adj_body(const ProbDev& P, const AdjItem& I, float* sh)
{
    const int nx = P.nx, ny = P.ny, nd = P.nd, na = P.na;
    const int nslices = P.nz * P.nch;
    const int tile_y = P.adj_tile_y, segw = P.adj_segw, achunk = P.adj_achunk;
    float* seg = sh;                                  // achunk * segw * K
    const int hs = achunk * segw * 4;                 // K = 8: the second plane
    float4* par = reinterpret_cast<float4*>(sh + (size_t)achunk * segw * K);
    int* lo_s = reinterpret_cast<int*>(par + achunk);

    const int x0 = I.x0, y0 = I.y0, s0 = I.s0;
    const int tid = threadIdx.x;
    const int lane = tid & 63, wv = tid >> 6;
    const int R = tile_y >> 2;
    const float xf = (float)(x0 + lane);
    const float* __restrict__ sino = P.lam;

    float acc[MAXR][K];
#pragma unroll
    for (int r = 0; r < MAXR; ++r)
#pragma unroll
        for (int k = 0; k < K; ++k) acc[r][k] = 0.f;

    const size_t sino_slice = (size_t)na * nd;
    const int sg_a0 = tid / segw, sg_b0 = tid - sg_a0 * segw;
    const int sg_da = ADJ_THREADS / segw, sg_db = ADJ_THREADS - sg_da * segw;
    for (int a0 = 0; a0 < na; a0 += achunk) {
        const int A = min(achunk, na - a0);
        __syncthreads();
        if (tid < A) {
            const float4 o = P.ofs[a0 + tid];
            const float tmin = o.z + (float)x0 * o.x + (float)y0 * o.y +
                               fminf(0.f, (float)(ADJ_TX - 1) * o.x) +
                               fminf(0.f, (float)(tile_y - 1) * o.y);
            const int lo = (int)floorf(tmin) - 1;
            par[tid] = make_float4(o.x, o.y, o.z - (float)lo, 0.f);
            lo_s[tid] = lo;
        }
        __syncthreads();
        // element e = tid + j * ADJ_THREADS as (angle, bin) = (e / segw, e % segw),
        // stepped rather than divided
        for (int al = sg_a0, b = sg_b0; al < A;) {
            const int gb = lo_s[al] + b;
            float v[K];
#pragma unroll
            for (int k = 0; k < K; ++k) {
                const int s = s0 + k;
                v[k] = (gb >= 0 && gb < nd && s < nslices)
                           ? sino[(size_t)s * sino_slice + (size_t)(a0 + al) * nd + gb]
                           : 0.f;
            }
            lds_store<K>(seg, al * segw + b, v, hs);
            b += sg_db;
            al += sg_da;
            if (b >= segw) {
                b -= segw;
                ++al;
            }
        }
        __syncthreads();
        for (int al = 0; al < A; ++al) {
            const float4 pa = par[al];
            const float tb = fmaf(xf, pa.x, pa.z);
            const int base = al * segw;
#pragma unroll
            for (int r = 0; r < MAXR; ++r) {
                if (r >= R) break;
                // t >= 1 over the whole tile (the segment starts at
                // floor(min t) - 1), so truncation is the floor
                const float t = fmaf((float)(y0 + wv + 4 * r), pa.y, tb);
                const float p = __builtin_amdgcn_fractf(t);
                const float q = 1.f - p;
                const int i0 = base + (int)t;
                const Pack<K> v0 = lds_load<K>(seg, i0, hs);
                const Pack<K> v1 = lds_load<K>(seg, i0 + 1, hs);
#pragma unroll
                for (int k = 0; k < K; ++k)
                    acc[r][k] = fmaf(p, v1.v[k], fmaf(q, v0.v[k], acc[r][k]));
            }
        }
    }

    const int x = x0 + lane;
    if (x >= nx) return;
    const size_t plane = (size_t)nx * ny;
#pragma unroll
    for (int r = 0; r < MAXR; ++r) {
        if (r >= R) break;
        const int y = y0 + wv + 4 * r;
        if (y >= ny) continue;
#pragma unroll
        for (int k = 0; k < K; ++k) {
            const int s = s0 + k;
            if (s >= nslices) continue;
            const size_t i = (size_t)s * plane + (size_t)y * nx + x;
            if constexpr (PRIMAL)
                primal_update<DIM, TGV>(P, i, x, y, s % P.nz, acc[r][k]);
            else
                P.ktl[i] = acc[r][k];
        }
    }
}

// Backprojection of 64 x 4 pixels of K slices, bins read from memory: the
// positions, weights and order of the tile the pixels belong to (y0 a multiple
// of 4, tile_y as well), so the same bits.  For stacks that leave most CUs
// without a tile: four to eight times the waves, no staging between barriers,
// and 8 angles' reads in flight.  Bound by the latency of these reads; 183 x
// 183, 90 angles 32 us by tiles, 9.8 so; 317 x 317 x 3, 71 angles 43 and 16.
// UDIM: the u half of the primal step of 2 or 3 dimensions follows for the
// pixel (0: none).
template <int K, int UDIM, bool TGV>
__device__ __forceinline__ void adj_direct_body(const ProbDev& P, const AdjItem& I)
{
    __shared__ float4 par[ADJ_THREADS];
    const int nx = P.nx, ny = P.ny, nd = P.nd, na = P.na;
    const int last = P.nz * P.nch - 1, tile_y = P.adj_tile_y;
    const int tid = threadIdx.x, lane = tid & 63, wv = tid >> 6;
    const int x = I.x0 + lane, y = I.y0 + wv, ty0 = I.y0 / tile_y * tile_y;
    const float xf = (float)x, yf = (float)y;
    const size_t slice = (size_t)na * nd;
    const float* __restrict__ sino[K];
#pragma unroll
    for (int k = 0; k < K; ++k) sino[k] = P.lam + (size_t)min(I.s0 + k, last) * slice;
    float acc[K];
#pragma unroll
    for (int k = 0; k < K; ++k) acc[k] = 0.f;
    for (int a0 = 0; a0 < na; a0 += ADJ_THREADS) {
        const int A = min(ADJ_THREADS, na - a0);
        __syncthreads();
        if (tid < A) {
            const float4 o = P.ofs[a0 + tid];
            const float tmin = o.z + (float)I.x0 * o.x + (float)ty0 * o.y +
                               fminf(0.f, (float)(ADJ_TX - 1) * o.x) +
                               fminf(0.f, (float)(tile_y - 1) * o.y);
            const int lo = (int)floorf(tmin) - 1;
            par[tid] = make_float4(o.x, o.y, o.z - (float)lo, __int_as_float(lo));
        }
        __syncthreads();
#pragma unroll 8
        for (int al = 0; al < A; ++al) {
            const float4 pa = par[al];
            const float t = fmaf(yf, pa.y, fmaf(xf, pa.x, pa.z));
            const float p = __builtin_amdgcn_fractf(t);
            const float q = 1.f - p;
            const int i = __float_as_int(pa.w) + (int)t;
            const bool in0 = (unsigned)i < (unsigned)nd, in1 = (unsigned)(i + 1) < (unsigned)nd;
            const unsigned row = (unsigned)((a0 + al) * nd);
            const unsigned e0 = row + (in0 ? i : 0), e1 = row + (in1 ? i + 1 : 0);
#pragma unroll
            for (int k = 0; k < K; ++k) {
                const float g0 = sino[k][e0], g1 = sino[k][e1];
                acc[k] = fmaf(p, in1 ? g1 : 0.f, fmaf(q, in0 ? g0 : 0.f, acc[k]));
            }
        }
    }
    if (x >= nx || y >= ny) return;
    const size_t plane = (size_t)nx * ny;
#pragma unroll
    for (int k = 0; k < K; ++k) {
        const int s = I.s0 + k;
        if (s > last) continue;
        const size_t i = (size_t)s * plane + (size_t)y * nx + x;
        P.ktl[i] = acc[k];
        if constexpr (UDIM > 0) primal_update<UDIM, TGV, PRIMAL_U>(P, i, x, y, s % P.nz, acc[k]);
    }
}

template <int K, int UDIM = 0, bool TGV = false>
__global__ __launch_bounds__(ADJ_THREADS) void adj_direct_kernel(ProbDev P, int tiles_x,
                                                                 int ntiles)
{
    const int work = xcd_work_id(blockIdx.x, gridDim.x), tile = work % ntiles;
    adj_direct_body<K, UDIM, TGV>(P, AdjItem{0, tile % tiles_x * ADJ_TX, tile / tiles_x * 4,
                                              (work / ntiles) * K});
}

template <int K, bool PRIMAL, int DIM, bool TGV, int MAXR>
__global__ __launch_bounds__(ADJ_THREADS) void adj_single_kernel(ProbDev P, int tiles_x,
                                                                 int ntiles)
{
    extern __shared__ float sh[];
    const int work = xcd_work_id(blockIdx.x, gridDim.x);
    const int tile = work % ntiles;
    const AdjItem I{0, (tile % tiles_x) * ADJ_TX, (tile / tiles_x) * P.adj_tile_y,
                    (work / ntiles) * K};
    adj_body<K, PRIMAL, DIM, TGV, MAXR>(P, I, sh);
}

template <int K, bool PRIMAL, int DIM, bool TGV>
__global__ __launch_bounds__(ADJ_THREADS) void adj_batch_kernel(const ProbDev* __restrict__ probs,
                                                                const AdjItem* __restrict__ items)
{
    extern __shared__ float sh[];
    const AdjItem I = items[xcd_work_id(blockIdx.x, gridDim.x)];
    const ProbDev P = load_prob(probs, I.prob);
    adj_body<K, PRIMAL, DIM, TGV>(P, I, sh);
}

}  // namespace

// --------------------------------------------------------------------------
// sizes
// --------------------------------------------------------------------------
int fwd_table_choice(const Geometry& g, long long groups, double wg_per_cu)
{
    const double target = wg_per_cu * 256;  // work-groups per CU on 256 CUs
    int best = 0;
    double best_d = 1e30;
    for (int t = 0; t < 4; ++t) {
        const double wg = (double)groups * (g.tab_off[t + 1] - g.tab_off[t]);
        const double d = std::fabs(std::log(std::max(wg, 1.0) / target));
        if (d < best_d - 1e-9) {
            best_d = d;
            best = t;
        }
    }
    return best;
}

int fwd_pitch_of(int nx, int ny)
{
    int p = std::max(nx, ny) + FWD_PADL + 4;
    if ((p & 1) == 0) ++p;  // odd pitch: conflict-free transposed stores
    return p;
}

int fwd_band_auto(int pitch, int K, int lds_kb)
{
    // lines per band within lds_kb of LDS per work-group (36 KB: four per CU)
    int b = (int)((size_t)lds_kb * 1024 / ((size_t)pitch * K * sizeof(float)));
    return std::max(4, std::min(32, b & ~3));
}

int adj_segw_of(int tile_y, float bin_span)
{
    const double diag = std::sqrt((double)(ADJ_TX - 1) * (ADJ_TX - 1) +
                                  (double)(tile_y - 1) * (tile_y - 1));
    // capped past what LDS can hold
    int w = (int)std::ceil(std::min(diag * bin_span, 1e6)) + 6;
    return (w + 3) & ~3;
}

static int adj_lds_budget()
{
    static int kb = -1;
    if (kb < 0) {
        const char* e = getenv("GRAPTOR_ADJ_LDS_KB");
        kb = e ? std::max(4, std::min(150, atoi(e))) : 36;
    }
    return kb;
}

int adj_achunk_of(int na, int segw, int K)
{
    const size_t per_angle = (size_t)segw * K * sizeof(float) + sizeof(float4) + sizeof(int);
    int a = (int)std::min<size_t>((size_t)na, (adj_lds_budget() * 1024) / per_angle);
    return std::max(a, 1);
}

size_t fwd_lds_bytes(const ProbDev& P, int K)
{
    return (size_t)P.fwd_band * P.fwd_pitch * K * sizeof(float);
}

size_t adj_lds_bytes(const ProbDev& P, int K)
{
    return (size_t)P.adj_achunk * ((size_t)P.adj_segw * K * sizeof(float) + sizeof(float4) +
                                   sizeof(int));
}

// three slices take a group of four with one padded slot: one pass instead of
// a pair and a single
int slice_group(int nslices) { return nslices >= 3 ? 4 : (nslices == 2 ? 2 : 1); }

// --------------------------------------------------------------------------
// single-problem launchers
// --------------------------------------------------------------------------
template <int K, int MI, bool WIDE = false>
static void fwd_single_launch(const ProbDev& P, const FwdChunk* chunks, int nchunks, int groups,
                              size_t lds, int mode, hipStream_t st)
{
    hipLaunchKernelGGL((fwd_single_kernel<K, MI, WIDE>), dim3((unsigned)(groups * nchunks)),
                       dim3(FWD_THREADS), lds, st, P, chunks, nchunks, mode);
}

template <int K>
static int fwd_single_k(const ProbDev& Pin, const Geometry& g, int nslices, int mode,
                        hipStream_t st)
{
    ProbDev P = Pin;
    const int groups = (nslices + K - 1) / K;
    // chunk table: items per thread (8, 4, 2, 1) whose grid is closest to
    // three work-groups per CU, or 1.5 beside the dual step, where fewer,
    // larger work-groups leave it more of the CUs (measured: 0.827 against
    // 0.856 ms per two-stream iteration on 256x256x64x4, although the
    // forward projection alone is slower); GRAPTOR_FWD_MI = 8, 4, 2 or 1
    // forces the table
    int t = fwd_table_choice(g, groups, (mode & FWD_BESIDE) ? 1.5 : 3.0);
    static const int forced = [] {
        const char* e = getenv("GRAPTOR_FWD_MI");
        const int v = e ? atoi(e) : 0;
        return v == 8 ? 0 : v == 4 ? 1 : v == 2 ? 2 : v == 1 ? 3 : -1;
    }();
    if (forced >= 0) t = forced;
    if (g.wide_bins) t = FWD_WIDE_TABLE;
    const int nchunks = g.tab_off[t + 1] - g.tab_off[t];
    const FwdChunk* chunks = g.chunks_dev + g.tab_off[t];
    P.fwd_pitch = fwd_pitch_of(P.nx, P.ny);
    if (P.fwd_band <= 0) P.fwd_band = fwd_band_auto(P.fwd_pitch, K);
    if ((mode & FWD_BESIDE) && (mode & FWD_AUTOBAND)) {
        // beside the dual step, bands as tall as an even spread of the grid
        // over the 256 CUs allows: the LDS of a work-group then caps the
        // work-groups a CU takes, leaving every CU room for the dual step
        // (256^2 images: 512 work-groups, 2 per CU, 16-line bands: 0.786
        // against 0.804 ms per iteration with 8; 512^2: grids of thousands
        // keep 4 per CU and 4 lines, 18.6 against 19.2 ms with 8)
        const long long per_cu =
            std::min(4LL, std::max(1LL, ((long long)groups * nchunks + 255) / 256));
        P.fwd_band = fwd_band_auto(P.fwd_pitch, K, (int)(160 / per_cu) - 1);
    }
    const size_t lds = fwd_lds_bytes(P, K);
    if (lds > LDS_LIMIT) {
        set_error("radon: band %d does not fit LDS (%zu bytes)", P.fwd_band, lds);
        return GR_ERR_INVALID;
    }
    const long long blocks = (long long)groups * nchunks;
    if (blocks <= 0 || blocks > 0x7fffffff) {
        set_error("radon: invalid grid (%lld blocks)", blocks);
        return GR_ERR_INVALID;
    }
    if (g.wide_bins)
        fwd_single_launch<K, (8 >> FWD_WIDE_TABLE), true>(P, chunks, nchunks, groups, lds, mode, st);
    else switch (t) {
    case 0: fwd_single_launch<K, 8>(P, chunks, nchunks, groups, lds, mode, st); break;
    case 1: fwd_single_launch<K, 4>(P, chunks, nchunks, groups, lds, mode, st); break;
    case 2: fwd_single_launch<K, 2>(P, chunks, nchunks, groups, lds, mode, st); break;
    default: fwd_single_launch<K, 1>(P, chunks, nchunks, groups, lds, mode, st); break;
    }
    GR_LAUNCH_CHECK("fwd_single_kernel");
    return GR_OK;
}

// Where a call projects by lines: it needs the shear tables, angles of at most
// 16 waves, and P.ktl to hold the transposed slices (with the primal step
// fused into the backprojection it stays as it is).
//
// Alone, gather / by lines in us for N x N x S, 60 angles: N = 64: S 4 15 / 9,
// 64 16 / 15, 128 17 / 23; 128: 1 20 / 11, 32 30 / 21, 64 33 / 32, 128 42 / 57;
// 200: 4 63 / 16, 64 79 / 65, 128 101 / 107; 256: 4 90 / 19, 128 154 / 128,
// 512 471 / 465; 512: 4 341 / 48, 64 683 / 245, 256 1069 / 1028; 180 angles:
// N = 96: 4 21 / 14, 32 25 / 33; 200: 32 94 / 82, 64 148 / 146; 512: 128 1609 /
// 1207: angles x groups of slices against pixels.
//
// In an iteration the gather shares the GPU with the dual step, for whose
// work-groups it leaves room.  Time of an iteration by gather over that by
// lines (TGV, 4 channels, 60 angles): N = 96: S 4 1.2, 64 0.91; 128: 32 1.26,
// 128 1.02, 256 0.91; 200: 32 1.42, 80 1.04; 256: 8 2.2, 32 1.55, 64 1.00, 128
// 0.85; 384: 32 1.35; 512: 16 1.9, 64 1.05; one slice: N = 48 0.94, 96 1.05,
// 183 1.6, 512 4.
bool fwd_by_lines(const ProbDev& P, const Geometry& g, bool alone)
{
    const long long S = (long long)P.nz * P.nch, px = (long long)P.nx * P.ny;
    const long long groups = (long long)P.na * ((S + 3) / 4);
    if (g.shear_waves == 0 || 64 * g.shear_waves > FWD_LINE_ITEMS) return false;
    if (alone) return 24 * groups <= px && S * px <= (1ll << 25);
    return !P.fuse_primal && S <= 64 && groups <= 960 && 17 * groups <= px;
}

// LDS bytes of a work-group of that many waves (one or two runs of lines)
static size_t fwd_line_lds(int K, int waves)
{
    return (size_t)3 * K * waves * 64 * sizeof(float);
}

template <int K>
static int fwd_line_k(const ProbDev& P, const Geometry& g, int nslices, int mode, hipStream_t st)
{
    const int groups = (nslices + K - 1) / K, J = g.shear_waves;
    const int ns = J <= 8 ? 2 : 1;
    const int tx = (P.nx + 31) / 32, ty = (P.ny + 31) / 32;
    const long long tiles = (long long)tx * ty * nslices, blocks = (long long)groups * P.na;
    if (tiles > 0x7fffffff || blocks > 0x7fffffff) {
        set_error("radon: invalid grid (%lld blocks)", std::max(tiles, blocks));
        return GR_ERR_INVALID;
    }
    hipLaunchKernelGGL(transpose_kernel, dim3((unsigned)tiles), dim3(256), 0, st, P, tx, ty);
    hipLaunchKernelGGL((fwd_line_kernel<K>), dim3((unsigned)blocks), dim3(64 * J * ns),
                       fwd_line_lds(K, J), st, P, J, ns, mode);
    GR_LAUNCH_CHECK("fwd_line_kernel");
    return GR_OK;
}

int launch_fwd(const ProbDev& P, const Geometry& g, int nslices, int mode, hipStream_t st)
{
    if (nslices <= 0) return GR_OK;
    if ((mode & FWD_SCRATCH) &&
        ((mode & FWD_LINES) || fwd_by_lines(P, g, mode & FWD_ALONE))) {
        // fewer slices per work-group where angles x groups would not give
        // every CU one: 317 x 317 x 3, 71 angles, 10 iterations 1000 / 932 /
        // 898 us with 4 / 2 / 1 (71, 142 and 213 work-groups); 199 x 199 x 42,
        // 45 angles, 5 iterations 483 / 521 / 605 us (495 work-groups and up)
        int K = slice_group(nslices);
        while (K > 1 && (long long)((nslices + K - 1) / K) * P.na < 256) K /= 2;
        switch (K) {
        case 4: return fwd_line_k<4>(P, g, nslices, mode, st);
        case 2: return fwd_line_k<2>(P, g, nslices, mode, st);
        default: return fwd_line_k<1>(P, g, nslices, mode, st);
        }
    }
    switch (slice_group(nslices)) {
    case 4: return fwd_single_k<4>(P, g, nslices, mode, st);
    case 2: return fwd_single_k<2>(P, g, nslices, mode, st);
    default: return fwd_single_k<1>(P, g, nslices, mode, st);
    }
}

template <int K, bool PRIMAL, int DIM, bool TGV>
static void adj_single_launch(const ProbDev& P, int blocks, int tiles_x, int ntiles, size_t lds,
                              hipStream_t st)
{
    // the backprojection alone takes accumulators for the rows of its tile
    // (tiles of <= 16 rows: 7 instead of 4 waves per SIMD); the fused primal
    // epilogue keeps the 8-row form
    if constexpr (!PRIMAL) {
        if (P.adj_tile_y <= 16) {
            hipLaunchKernelGGL((adj_single_kernel<K, PRIMAL, DIM, TGV, 4>),
                               dim3((unsigned)blocks), dim3(ADJ_THREADS), lds, st, P, tiles_x,
                               ntiles);
            return;
        }
    }
    hipLaunchKernelGGL((adj_single_kernel<K, PRIMAL, DIM, TGV, ADJ_MAXR>), dim3((unsigned)blocks),
                       dim3(ADJ_THREADS), lds, st, P, tiles_x, ntiles);
}

template <int K>
static int adj_single_k(const ProbDev& Pin, int nslices, bool primal, hipStream_t st)
{
    ProbDev P = Pin;
    if (P.adj_tile_y < 4 || P.adj_tile_y > 4 * ADJ_MAXR || (P.adj_tile_y & 3)) {
        set_error("radon_ad: tile_y %d must be a multiple of 4 in [4, %d]", P.adj_tile_y,
                  4 * ADJ_MAXR);
        return GR_ERR_INVALID;
    }
    P.adj_segw = adj_segw_of(P.adj_tile_y, P.bin_span);
    P.adj_achunk = adj_achunk_of(P.na, P.adj_segw, K);
    const size_t lds = adj_lds_bytes(P, K);
    if (lds > LDS_LIMIT) {
        set_error("radon_ad: bins of 1/%.0f pixel are too narrow for the fused primal step",
                  P.bin_span);
        return GR_ERR_INVALID;
    }
    const int tiles_x = (P.nx + ADJ_TX - 1) / ADJ_TX;
    const int tiles_y = (P.ny + P.adj_tile_y - 1) / P.adj_tile_y;
    const int ntiles = tiles_x * tiles_y;
    const int groups = (nslices + K - 1) / K;
    const long long blocks = (long long)groups * ntiles;
    if (blocks <= 0 || blocks > 0x7fffffff) {
        set_error("radon_ad: invalid grid (%lld blocks)", blocks);
        return GR_ERR_INVALID;
    }
    const int b = (int)blocks;
    if (!primal) {
        adj_single_launch<K, false, 2, false>(P, b, tiles_x, ntiles, lds, st);
    } else if constexpr (K <= 4) {  // the fused primal epilogue takes up to 4 slices
        if (P.dim == 2) {
            if (P.tgv) adj_single_launch<K, true, 2, true>(P, b, tiles_x, ntiles, lds, st);
            else adj_single_launch<K, true, 2, false>(P, b, tiles_x, ntiles, lds, st);
        } else {
            if (P.tgv) adj_single_launch<K, true, 3, true>(P, b, tiles_x, ntiles, lds, st);
            else adj_single_launch<K, true, 3, false>(P, b, tiles_x, ntiles, lds, st);
        }
    }
    GR_LAUNCH_CHECK("adj_single_kernel");
    return GR_OK;
}

template <int K>
static int adj_direct_k(const ProbDev& P, int nslices, bool u_half, hipStream_t st)
{
    const int tiles_x = (P.nx + ADJ_TX - 1) / ADJ_TX, ntiles = tiles_x * ((P.ny + 3) / 4);
    const dim3 grd((unsigned)((nslices + K - 1) / K * ntiles)), blk(ADJ_THREADS);
#define GR_AD(...) \
    hipLaunchKernelGGL((adj_direct_kernel<__VA_ARGS__>), grd, blk, 0, st, P, tiles_x, ntiles)
    if constexpr (K == 1) {
        if (u_half && P.dim == 2) { if (P.tgv) GR_AD(1, 2, true); else GR_AD(1, 2, false); }
        else if (u_half) { if (P.tgv) GR_AD(1, 3, true); else GR_AD(1, 3, false); }
        else GR_AD(1);
    } else {
        GR_AD(K);
    }
#undef GR_AD
    GR_LAUNCH_CHECK("adj_direct_kernel");
    return GR_OK;
}

// Where the tiles would not give every CU a work-group, a small stack is
// read directly, in at most 6144 waves and with as few slices per wave as
// that allows.  One call, 60 angles, us with 1 / 2 / 4 slices a wave
// against tiles: 64 x 64 x 1 12.5 to 20, x 64 12.6 / 12.2 / 12.4 to 32;
// 183 x 183 x 3 12 to 22, x 16 21 / 19 / 19 to 32, x 64 (288 work-groups)
// 64 / 49 / 43 to 37; 256 x 256 x 24 (192) 46 / 36 / 32 to 33, x 32 (256)
// 58 / 45 / 39 to 33; 512 x 512 x 1 12 to 33, x 4 31 / 25 / 24 to 35.
// Whole iterations: 183 x 183 x 16 71 to 78, 512 x 512 x 4 94 to 109, but
// 64 x 64 x 256 (256 work-groups) 89 to 86, 256 x 256 x 24 (384) 116 to 108.
// Bins so narrow that not one angle's shadow of a tile fits LDS are read
// directly at every size.
// Returns the slices per wave, 0: by tiles.
static int adj_direct_slices(const ProbDev& P, int nslices, bool wide)
{
    if (P.adj_tile_y < 4 || P.adj_tile_y % 4 != 0) return 0;
    const long long cols = (P.nx + ADJ_TX - 1) / ADJ_TX, rows = cols * P.ny;
    const long long tiles = cols * ((P.ny + P.adj_tile_y - 1) / P.adj_tile_y);
    const int K = wide ? 8 : slice_group(nslices);
    const size_t shadow = (size_t)adj_segw_of(P.adj_tile_y, P.bin_span) * K * sizeof(float);
    if (shadow + sizeof(float4) + sizeof(int) > LDS_LIMIT) return slice_group(nslices);
    if (tiles * ((nslices + K - 1) / K) >= 256) return 0;
    for (int d = 1; d <= 4; d *= 2)
        if (rows * ((nslices + d - 1) / d) <= 6144) return d;
    return 0;
}

// With one slice per wave: iterations of 64 x 64 x 1 48 to 41 us, 183 x 183 x 4
// 55 to 48, 256 x 256 x 4 61 to 51, 512 x 512 x 1 79 to 76 (a launch and a gap
// less).  With more, the reads of an angle are no longer issued ahead (41
// registers instead of 89): 512 x 512 x 4 94 to 127 us.
bool adj_takes_u(const ProbDev& P, int nslices)
{
    return nslices > 0 && adj_direct_slices(P, nslices, false) == 1;
}

int launch_adj_u(const ProbDev& P, int nslices, hipStream_t st)
{
    return adj_direct_k<1>(P, nslices, true, st);
}

int launch_adj(const ProbDev& P, int nslices, bool primal, hipStream_t st, bool beside)
{
    if (nslices <= 0) return GR_OK;
    // eight slices per work-group: each interpolation weight serves twice the
    // multiply-adds (256^2 x 256 slices, 60 angles, 16-row tiles: 0.111
    // against 0.131 ms alone, same bits).  Not with 32-row tiles (8 rows x 8
    // slices of accumulators per lane: 2.92 against 2.47 ms on 512^2 x 1024
    // slices, 90 angles), nor beside the dual step (0.7874 against 0.7860 ms
    // per two-stream iteration).
    const bool wide = nslices >= 8 && !primal && !beside && P.adj_tile_y <= 16;
    const int direct = primal ? 0 : adj_direct_slices(P, nslices, wide);
    if (direct == 4) return adj_direct_k<4>(P, nslices, false, st);
    if (direct == 2) return adj_direct_k<2>(P, nslices, false, st);
    if (direct == 1) return adj_direct_k<1>(P, nslices, false, st);
    if (wide) return adj_single_k<8>(P, nslices, primal, st);
    switch (slice_group(nslices)) {
    case 4: return adj_single_k<4>(P, nslices, primal, st);
    case 2: return adj_single_k<2>(P, nslices, primal, st);
    default: return adj_single_k<1>(P, nslices, primal, st);
    }
}

template <int DIM, bool TGV, bool ZH, bool NT>
static void primal_single_part_nt(const ProbDev& P, int part, dim3 grd, dim3 blk, int tiles_x,
                                  int tiles_y, hipStream_t st)
{
    if (part == PRIMAL_U)
        hipLaunchKernelGGL((primal_single_kernel<DIM, TGV, PRIMAL_U, ZH, NT>), grd, blk, 0, st,
                           P, tiles_x, tiles_y);
    else if (part == PRIMAL_P)
        hipLaunchKernelGGL((primal_single_kernel<DIM, TGV, PRIMAL_P, ZH, NT>), grd, blk, 0, st,
                           P, tiles_x, tiles_y);
    else
        hipLaunchKernelGGL((primal_single_kernel<DIM, TGV, PRIMAL_UP, ZH, NT>), grd, blk, 0, st,
                           P, tiles_x, tiles_y);
}

template <int DIM, bool TGV, bool ZH>
static void primal_single_part_zh(const ProbDev& P, int part, dim3 grd, dim3 blk, int tiles_x,
                                  int tiles_y, hipStream_t st)
{
    if (stream_hints(P))
        primal_single_part_nt<DIM, TGV, ZH, true>(P, part, grd, blk, tiles_x, tiles_y, st);
    else
        primal_single_part_nt<DIM, TGV, ZH, false>(P, part, grd, blk, tiles_x, tiles_y, st);
}

template <int DIM, bool TGV>
static void primal_u_voxel_launch(const ProbDev& P, dim3 grd, dim3 blk, int tiles_x, int tiles_y,
                                  hipStream_t st)
{
    if (stream_hints(P))
        hipLaunchKernelGGL((primal_u_voxel_kernel<DIM, TGV, true>), grd, blk, 0, st, P, tiles_x,
                           tiles_y);
    else
        hipLaunchKernelGGL((primal_u_voxel_kernel<DIM, TGV, false>), grd, blk, 0, st, P,
                           tiles_x, tiles_y);
}

// a z-slab with halo planes takes the kernels that read them
template <int DIM, bool TGV>
static void primal_single_part(const ProbDev& P, int part, dim3 grd, dim3 blk, int tiles_x,
                               int tiles_y, hipStream_t st)
{
    if (DIM == 3 && (P.halo_ubar_hi || P.halo_v_lo))
        primal_single_part_zh<DIM, TGV, DIM == 3>(P, part, grd, blk, tiles_x, tiles_y, st);
    else
        primal_single_part_zh<DIM, TGV, false>(P, part, grd, blk, tiles_x, tiles_y, st);
}

int launch_primal(const ProbDev& P, hipStream_t st) { return launch_primal_part(P, PRIMAL_UP, st); }

int launch_primal_part(const ProbDev& P, int part, hipStream_t st)
{
    if (part != PRIMAL_U && part != PRIMAL_P && part != PRIMAL_UP) {
        set_error("primal step: invalid part %d", part);
        return GR_ERR_INVALID;
    }
    if (part == PRIMAL_P && !P.tgv) return GR_OK;  // TV: no p
    const int tiles_x = (P.nx + DUAL_BX - 1) / DUAL_BX;
    const int tiles_y = (P.ny + DUAL_BY - 1) / DUAL_BY;
    const long long blocks = (long long)tiles_x * tiles_y * P.nz * P.nch;
    if (blocks > 0x7fffffff) {
        set_error("primal step: grid too large");
        return GR_ERR_INVALID;
    }
    dim3 grd((unsigned)blocks), blk(DUAL_BX * DUAL_BY);
    const long long voxel_blocks = (long long)tiles_x * tiles_y * P.nz;
    if (part == PRIMAL_U && P.nch > 1 && voxel_blocks >= 4096 && !P.halo_ubar_hi &&
        !P.halo_v_lo) {
        // enough work-groups with one per voxel tile: the per-voxel u half
        const dim3 gv((unsigned)voxel_blocks);
        if (P.dim == 2) {
            if (P.tgv) primal_u_voxel_launch<2, true>(P, gv, blk, tiles_x, tiles_y, st);
            else primal_u_voxel_launch<2, false>(P, gv, blk, tiles_x, tiles_y, st);
        } else {
            if (P.tgv) primal_u_voxel_launch<3, true>(P, gv, blk, tiles_x, tiles_y, st);
            else primal_u_voxel_launch<3, false>(P, gv, blk, tiles_x, tiles_y, st);
        }
        GR_LAUNCH_CHECK("primal_u_voxel_kernel");
        return GR_OK;
    }
    if (P.dim == 2) {
        if (P.tgv) primal_single_part<2, true>(P, part, grd, blk, tiles_x, tiles_y, st);
        else primal_single_part<2, false>(P, part, grd, blk, tiles_x, tiles_y, st);
    } else {
        if (P.tgv) primal_single_part<3, true>(P, part, grd, blk, tiles_x, tiles_y, st);
        else primal_single_part<3, false>(P, part, grd, blk, tiles_x, tiles_y, st);
    }
    GR_LAUNCH_CHECK("primal_single_kernel");
    return GR_OK;
}

template <int DIM, bool TGV>
static void primal_batch_part(const ProbDev* probs, const DualItem* items, dim3 grd, dim3 blk,
                              int part, hipStream_t st)
{
    if (part == PRIMAL_U)
        hipLaunchKernelGGL((primal_batch_kernel<DIM, TGV, PRIMAL_U>), grd, blk, 0, st, probs,
                           items);
    else if (part == PRIMAL_P)
        hipLaunchKernelGGL((primal_batch_kernel<DIM, TGV, PRIMAL_P>), grd, blk, 0, st, probs,
                           items);
    else
        hipLaunchKernelGGL((primal_batch_kernel<DIM, TGV, PRIMAL_UP>), grd, blk, 0, st, probs,
                           items);
}

int launch_primal_batch(const ProbDev* probs, const DualItem* items, int nitems, int dim,
                        bool tgv, int part, hipStream_t st)
{
    if (part != PRIMAL_U && part != PRIMAL_P && part != PRIMAL_UP) {
        set_error("primal step: invalid part %d", part);
        return GR_ERR_INVALID;
    }
    if (nitems <= 0 || (part == PRIMAL_P && !tgv)) return GR_OK;  // TV: no p
    dim3 grd((unsigned)nitems), blk(DUAL_BX * DUAL_BY);
    if (dim == 2) {
        if (tgv) primal_batch_part<2, true>(probs, items, grd, blk, part, st);
        else primal_batch_part<2, false>(probs, items, grd, blk, part, st);
    } else {
        if (tgv) primal_batch_part<3, true>(probs, items, grd, blk, part, st);
        else primal_batch_part<3, false>(probs, items, grd, blk, part, st);
    }
    GR_LAUNCH_CHECK("primal_batch_kernel");
    return GR_OK;
}

// --------------------------------------------------------------------------
// batch launchers
// --------------------------------------------------------------------------
int launch_fwd_batch(const ProbDev* probs, const FwdItem* items, int nitems, int K, int mi,
                     bool wide, size_t lds, int mode, hipStream_t st)
{
    if (nitems <= 0) return GR_OK;
    dim3 grd((unsigned)nitems), blk(FWD_THREADS);
#define GR_FB(KK, MM) \
    hipLaunchKernelGGL((fwd_batch_kernel<KK, MM, false>), grd, blk, lds, st, probs, items, mode)
#define GR_FB_K(KK)                                  \
    if (wide)                                        \
        hipLaunchKernelGGL((fwd_batch_kernel<KK, (8 >> FWD_WIDE_TABLE), true>), grd, blk, lds, st, \
                           probs, items, mode);      \
    else switch (mi) {                               \
    case 8: GR_FB(KK, 8); break;                     \
    case 4: GR_FB(KK, 4); break;                     \
    case 2: GR_FB(KK, 2); break;                     \
    default: GR_FB(KK, 1); break;                    \
    }
    if (K == 4) { GR_FB_K(4) } else if (K == 2) { GR_FB_K(2) } else { GR_FB_K(1) }
#undef GR_FB_K
#undef GR_FB
    GR_LAUNCH_CHECK("fwd_batch_kernel");
    return GR_OK;
}

int launch_line_tables(const Geometry& g, const int* first)
{
    hipLaunchKernelGGL(line_tables_kernel, dim3((unsigned)g.na), dim3(256), 0, nullptr, g.fwd_dev,
                       g.line0_dev, first, g.nd, g.shear_stride, g.shear_dev, g.lines_dev,
                       g.bins_dev);
    GR_LAUNCH_CHECK("line_tables_kernel");
    GR_HIP(hipStreamSynchronize(nullptr));  // for users on any stream
    return GR_OK;
}

int launch_fwd_mixed_batch(const ProbDev* probs, const FwdItem* items, int nitems, int K,
                           size_t lds, int mode, hipStream_t st)
{
    if (nitems <= 0) return GR_OK;
    hipLaunchKernelGGL(fwd_mixed_batch_kernel, dim3((unsigned)nitems), dim3(FWD_THREADS),
                       std::max(lds, fwd_line_lds(K, FWD_THREADS / 64)), st, probs, items, mode);
    GR_LAUNCH_CHECK("fwd_mixed_batch_kernel");
    return GR_OK;
}

int launch_transpose_batch(const ProbDev* probs, const DualItem* items, int nitems,
                           hipStream_t st)
{
    if (nitems <= 0) return GR_OK;
    hipLaunchKernelGGL(transpose_batch_kernel, dim3((unsigned)nitems), dim3(256), 0, st, probs,
                       items);
    GR_LAUNCH_CHECK("transpose_batch_kernel");
    return GR_OK;
}

int launch_fwd_line_batch(const ProbDev* probs, const FwdItem* items, int nitems, int K,
                          bool one_k, int waves, int mode, hipStream_t st)
{
    if (nitems <= 0) return GR_OK;
    const dim3 grd((unsigned)nitems), blk(64 * waves);
    const size_t lds = fwd_line_lds(K, waves);
#define GR_FL(KK) \
    hipLaunchKernelGGL(fwd_line_batch_kernel<KK>, grd, blk, lds, st, probs, items, mode)
    if (!one_k) GR_FL(0);
    else if (K == 4) GR_FL(4);
    else if (K == 2) GR_FL(2);
    else GR_FL(1);
#undef GR_FL
    GR_LAUNCH_CHECK("fwd_line_batch_kernel");
    return GR_OK;
}

int launch_adj_batch(const ProbDev* probs, const AdjItem* items, int nitems, int K, int dim,
                     bool tgv, bool primal, size_t lds, hipStream_t st)
{
    if (nitems <= 0) return GR_OK;
    dim3 grd((unsigned)nitems), blk(ADJ_THREADS);
#define GR_AB(KK, DD, TT) \
    hipLaunchKernelGGL((adj_batch_kernel<KK, true, DD, TT>), grd, blk, lds, st, probs, items)
#define GR_AB_K(KK)                                          \
    if (!primal) hipLaunchKernelGGL((adj_batch_kernel<KK, false, 2, false>), grd, blk, lds, st, probs, items); \
    else if (dim == 2) { if (tgv) GR_AB(KK, 2, true); else GR_AB(KK, 2, false); } \
    else { if (tgv) GR_AB(KK, 3, true); else GR_AB(KK, 3, false); }
    if (K == 4) { GR_AB_K(4) } else if (K == 2) { GR_AB_K(2) } else { GR_AB_K(1) }
#undef GR_AB_K
#undef GR_AB
    GR_LAUNCH_CHECK("adj_batch_kernel");
    return GR_OK;
}

}  // namespace gr
