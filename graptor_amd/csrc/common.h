// Shared declarations of the graptor_amd HIP library (gfx950 / CDNA4).
#pragma once
#include <hip/hip_runtime.h>
#include <stddef.h>
#include <stdint.h>

#include <vector>

#include "../../include/graptor_amd.h"

namespace gr {

// Status plumbing: every extern "C" entry point returns an int status and
// records a message retrievable through gr_last_error().
void set_error(const char* fmt, ...);
int hip_status(hipError_t e, const char* where);

#define GR_HIP(call)                                                        \
    do {                                                                    \
        hipError_t e_ = (call);                                             \
        if (e_ != hipSuccess) return ::gr::hip_status(e_, #call);           \
    } while (0)

#define GR_LAUNCH_CHECK(where)                                              \
    do {                                                                    \
        hipError_t e_ = hipGetLastError();                                  \
        if (e_ != hipSuccess) return ::gr::hip_status(e_, where);           \
    } while (0)

// Per-angle constants of the gather forward projector.  For an angle whose
// rays run closer to the x axis (|sin| >= |cos|) the kernel steps along x and
// picks candidate rows; otherwise it steps along y and picks candidate
// columns.  t(x, y) = x*cos + y*sin + off is the detector coordinate.
struct FwdAngle {
    float mstep;  // coefficient of the stepping coordinate in t
    float mcand;  // coefficient of the candidate coordinate in t
    float off;    // offset term of t
    float invc;   // 1 / mcand
    float hc;     // 1 / |mcand|: half-width of the hat support in candidates
    int cls;      // 0: step x / candidates y, 1: step y / candidates x
    int id;       // angle index in the caller's table
    int pad;
};

// One work chunk of the forward projector: angles [a0, a0+na) of one class
// (indices into the class-sorted FwdAngle array) times bins [b0, b0+nb).
struct FwdChunk {
    int cls, a0, na, b0, nb, pad0, pad1, pad2;
};

// Tables of the sheared forward projection.  An item follows the line
// candidate = j + s(l) through the image, s(l) = rint(-l mstep / mcand), along
// which the detector coordinate is j mcand + off + d(l), |d| <= |mcand| / 2.
struct Shear {
    float d;
    int s;
};
struct FwdLine {
    int j;
    float rel;  // j mcand + off - m, m the nearest bin
};
// Items that reach a bin: `first`, relative to the angle's first item, and in
// `code` three bits per item: 0 past the last, 1 / 2 / 3 for m = bin + 1 / bin
// / bin - 1.
constexpr int FWD_BIN_ITEMS = 6;
struct FwdBin {
    int first, code;
};
// Everything a kernel needs to know about one reconstruction problem (or one
// standalone projector call): sizes, derived scalars, geometry tables and
// device state.  Passed by value for single problems and through a device
// table for batches.
struct ProbDev {
    int dim, nx, ny, nz, nch, nd, na;
    int coupling, tgv, disc;
    float hinv, sigma, tau, sigma_p, norming, ainv0, ainv1;
    int fwd_band, fwd_pitch, adj_tile_y, adj_segw, adj_achunk, fuse_primal;
    const float4* ofs;     // na x (cos, sin, off, 1/cos)
    const FwdAngle* fwd;   // na, sorted by class
    // sheared projection: na x shear_stride (lines), items, per angle its
    // first item, na x nd bins
    const Shear* shear;
    const FwdLine* lines;
    const int* line0;
    const FwdBin* bins;
    int shear_stride;
    float bin_span;        // most bins that a step of one pixel crosses, at least 1
    // state; for standalone projector calls: ubar = image in, ku = sinogram
    // out (forward), lam = sinogram in, ktl = image out (backprojection)
    float *u, *ubar, *p, *pbar, *v, *w, *lam, *ktl, *ku;
    const float *f, *mfac;
    // z halo of a slab (3D; NULL: boundary plane), planes [c][y][x]:
    // ubar above, pbar below [k][c], v_z below, (w_xz, w_yz, w_zz) above [j][c]
    const float *halo_ubar_hi, *halo_pbar_lo, *halo_v_lo, *halo_w_hi;
};

// Buffers of the fused primal + next-dual step: the previous state is read
// from *_in, the next written to *_out (u, p, v, w alternate between the
// caller's arrays and a second set).
struct FusedBufs {
    const float *u_in, *p_in, *v_in, *w_in;
    float *u_out, *p_out, *v_out, *w_out;
};

struct FwdItem { int prob, cls, a0, na, b0, nb, s0, k; };
struct AdjItem { int prob, x0, y0, s0; };
// Stencil items: a 64 x 4 tile of plane z (dual step) or of slice
// z + nz * channel (primal step).  prob < 0 among dual items: a 32 x 32 tile of
// slice z of problem ~prob, transposed for the projection by lines.
struct DualItem { int prob, x0, y0, z; };

// Chunk table (FWD_THREADS x 8 >> t items) of geometries with wide bins, the only
// one whose gather is built for them.
constexpr int FWD_WIDE_TABLE = 2;

constexpr int SHEAR_BLOCK = 8;       // lines per table read
constexpr double FWD_SHEAR_MIN = 0.7;
constexpr int FWD_LINE_ITEMS = 1024;  // items of an angle: 16 waves
constexpr long long FWD_LINE_PIXELS = 6400;  // smaller slices are never projected by lines

// Device-side geometry (owned by gr_geometry).
struct Geometry {
    int nx, ny, nd, na;
    // device tables, one allocation owned by ofs_dev
    float* ofs_dev;          // na x float4 (cos, sin, off, 1/cos) as given
    FwdAngle* fwd_dev;       // na, sorted by class
    FwdChunk* chunks_dev;    // four chunk tables back to back
    int tab_off[5];          // table t = chunks [tab_off[t], tab_off[t+1]),
                             // built for 8, 4, 2, 1 items per thread
    std::vector<FwdChunk> chunks_host;
    // sheared projection: waves of items of the angle with the most, or 0 and no
    // tables where it does not apply (every |mcand| in [FWD_SHEAR_MIN, 1], i.e.
    // unit detector bins; see item_table)
    int shear_waves;
    Shear* shear_dev = nullptr;  // na x shear_stride
    FwdLine* lines_dev = nullptr;
    int* line0_dev = nullptr;    // na + 1
    FwdBin* bins_dev = nullptr;  // na x nd
    int shear_stride;
    int fwd_band;            // lines per LDS band (0: automatic)
    int adj_tile_y;          // rows per backprojection tile
    float bin_span;          // most bins that a step of one pixel crosses, at least 1
    int wide_bins;           // some |mcand| below 2/3: hats over more than 3 candidates
    int fuse_primal;         // 1: primal step in the backprojection epilogue
};

// Modes of the forward projector epilogue.
// FWD_PROX applies each problem's own discrepancy (batches).
// FWD_BESIDE: the launch shares the GPU with the dual step of the same
// iteration (two-stream schedule): fewer, larger work-groups.
// FWD_AUTOBAND: the geometry's band height is automatic, so a launch beside
// the dual step may size it for its grid.
// FWD_SCRATCH: P.ktl (as large as the image) may be overwritten: inside an
// iteration, where the backprojection fills it afterwards, or because the
// caller says so.  FWD_ALONE: no dual step beside the launch.  FWD_LINES: by
// lines, whatever fwd_by_lines says of this stack.
enum {
    FWD_WRITE = 1, FWD_KL = 2, FWD_L2 = 4, FWD_PROX = 8, FWD_BESIDE = 16, FWD_AUTOBAND = 32,
    FWD_SCRATCH = 64, FWD_ALONE = 128, FWD_LINES = 256
};

// Map hardware block order (dealt round-robin over the 8 XCDs) to a work
// order in which consecutive work ids run on the same XCD and share its L2.
__device__ __forceinline__ int xcd_work_id(int bid, int nb)
{
    const int xcd = bid & 7, local = bid >> 3;
    const int per = nb >> 3, rem = nb & 7;
    return (xcd < rem) ? xcd * (per + 1) + local
                       : rem * (per + 1) + (xcd - rem) * per + local;
}

// A batch problem's descriptor.  The pointers of a descriptor read from memory
// are generic to the compiler, which would access them by flat instructions
// (slower, and counted with LDS: a wait for one is a wait for all); they are
// global.  The cast goes through an integer, or it is folded away.  10 batch
// iterations of 64 mixed slices: 10.68 ms before, 10.49 ms with it.
template <class T>
__device__ __forceinline__ T* as_global(T* p)
{
    return (T*)(__attribute__((address_space(1))) T*)(uintptr_t)p;
}
__device__ __forceinline__ ProbDev load_prob(const ProbDev* __restrict__ probs, int i)
{
    ProbDev P = probs[i];
    P.ofs = as_global(P.ofs); P.fwd = as_global(P.fwd);
    P.shear = as_global(P.shear); P.lines = as_global(P.lines);
    P.line0 = as_global(P.line0); P.bins = as_global(P.bins);
    P.u = as_global(P.u); P.ubar = as_global(P.ubar); P.p = as_global(P.p);
    P.pbar = as_global(P.pbar); P.v = as_global(P.v); P.w = as_global(P.w);
    P.lam = as_global(P.lam); P.ktl = as_global(P.ktl); P.ku = as_global(P.ku);
    P.f = as_global(P.f); P.mfac = as_global(P.mfac);
    P.halo_ubar_hi = as_global(P.halo_ubar_hi); P.halo_pbar_lo = as_global(P.halo_pbar_lo);
    P.halo_v_lo = as_global(P.halo_v_lo); P.halo_w_hi = as_global(P.halo_w_hi);
    return P;
}

// Loads / stores of arrays a stencil kernel streams once, with the
// non-temporal hint when NT: single problems whose state outgrows the
// Infinity Cache (their arrays would otherwise displace the lines of the
// neighbour reads; stream_hints decides), not problems or batches of small
// problems whose arrays stay in that cache from one phase to the next (the
// hint there: 1.135 against 1.109 ms per batch iteration).
template <bool NT>
__device__ __forceinline__ float ld_stream(const float* p)
{
    if constexpr (NT) return __builtin_nontemporal_load(p);
    else return *p;
}
template <bool NT>
__device__ __forceinline__ void st_stream(float v, float* p)
{
    if constexpr (NT) __builtin_nontemporal_store(v, p);
    else *p = v;
}

constexpr int FWD_THREADS = 256;
constexpr int FWD_PADL = 4;          // zero candidates left of position 0
constexpr int ADJ_THREADS = 256;
constexpr int ADJ_TX = 64;           // backprojection tile width (one wave)
constexpr int ADJ_MAXR = 8;          // rows per thread (tile_y <= 32)
// stencil tile (threads per work-group = DUAL_BX * DUAL_BY); the macros
// allow other shapes to be built for measurement
#ifndef GR_DUAL_BX
#define GR_DUAL_BX 64
#endif
#ifndef GR_DUAL_BY
#define GR_DUAL_BY 4
#endif
constexpr int DUAL_BX = GR_DUAL_BX, DUAL_BY = GR_DUAL_BY;
// the stencils take x +- 1 neighbours from the adjacent lanes of a wave
// (wave-wide shifts with memory loads at lanes 0 and 63): a tile row must be
// exactly one wave
static_assert(DUAL_BX == 64, "stencil tiles are one 64-lane wave wide");

#ifndef GR_DUAL_GROUP
#define GR_DUAL_GROUP 8
#endif
#ifndef GR_PRIMAL_GROUP
#define GR_PRIMAL_GROUP 4
#endif
constexpr int DUAL_GROUP = GR_DUAL_GROUP, PRIMAL_GROUP = GR_PRIMAL_GROUP;
// Work id of a single-problem stencil work-group.  Hardware dispatch deals
// work-groups round-robin over the 8 XCDs; here runs of G consecutive tiles
// (neighbours in x, then y) are kept on one XCD so that the cache lines their
// neighbour reads share are fetched into one L2, while the 8 XCDs still work
// on adjacent runs (dense, concurrently active addresses).  Grids that are
// not a multiple of 8 runs keep hardware order.
template <int G>
__device__ __forceinline__ int stencil_block()
{
    const int b = blockIdx.x;
    if (G <= 1 || gridDim.x % (8 * G) != 0) return b;
    const int xcd = b & 7, local = b >> 3;
    return ((local / G) * 8 + xcd) * G + local % G;
}

// P.ktl = slice s of P.ubar transposed, one 32 x 32 tile, by 256 threads
// through TRANSPOSE_FLOATS floats of LDS.
constexpr int TRANSPOSE_FLOATS = 32 * 33;
__device__ __forceinline__ void transpose_tile(float* tile, const ProbDev& P, int s, int x0,
                                               int y0)
{
    const int nx = P.nx, ny = P.ny, tx = threadIdx.x & 31, ty = threadIdx.x >> 5;
    const float* __restrict__ src = P.ubar + (size_t)s * nx * ny;
    float* __restrict__ dst = P.ktl + (size_t)s * nx * ny;
#pragma unroll
    for (int r = 0; r < 32; r += 8) {
        const int x = x0 + tx, y = y0 + ty + r;
        if (x < nx && y < ny) tile[(ty + r) * 33 + tx] = src[(size_t)y * nx + x];
    }
    __syncthreads();
#pragma unroll
    for (int r = 0; r < 32; r += 8) {
        const int x = x0 + ty + r, y = y0 + tx;
        if (x < nx && y < ny) dst[(size_t)x * ny + y] = tile[tx * 33 + ty + r];
    }
}

inline void set_shear(ProbDev& P, const Geometry& g)
{
    P.shear = g.shear_dev; P.lines = g.lines_dev; P.line0 = g.line0_dev; P.bins = g.bins_dev;
    P.shear_stride = g.shear_stride;
}

// Kernel-side sizes derived from a problem and its tuning.
int fwd_pitch_of(int nx, int ny);
int fwd_table_choice(const Geometry& g, long long groups, double wg_per_cu = 3.0);
int fwd_band_auto(int pitch, int K, int lds_kb = 36);
int adj_segw_of(int tile_y, float bin_span);
int adj_achunk_of(int na, int segw, int K);
size_t fwd_lds_bytes(const ProbDev& P, int K);
size_t adj_lds_bytes(const ProbDev& P, int K);
constexpr size_t LDS_LIMIT = 160 * 1024;  // of a work-group
int slice_group(int nslices);  // K = 4 (3 or more slices), 2 or 1 slices sharing geometry

// ---- launchers (single problem: descriptor by value) ---------------------
int launch_fwd(const ProbDev& P, const Geometry& g, int nslices, int mode, hipStream_t st);
// adjoint only (primal == false: writes K^T lam into P.ktl) or fused with
// the primal step of the iteration (primal == true); beside: the launch
// shares the GPU with the dual step (two-stream schedule)
int launch_adj(const ProbDev& P, int nslices, bool primal, hipStream_t st, bool beside = false);
// Backprojection and u half of the primal step in one launch, where the bins of
// a small stack are read directly (adj_takes_u); the dual step has to be over.
bool adj_takes_u(const ProbDev& P, int nslices);
int launch_adj_u(const ProbDev& P, int nslices, hipStream_t st);
// Whether the single-problem stencil kernels stream with the non-temporal
// hint: the stencil state (u, ubar, p, pbar, v, w, K^T lam) above
// STREAM_HINT_MB; GRAPTOR_STREAM_HINTS = 0 or 1 forces the choice.  Per
// two-stream iteration, 4 channels, hints off / on: 3D 256x256x8 (144 MB)
// 0.191 / 0.207 ms, x16 (288 MB) 0.289 / 0.291, x24 (432 MB) 0.410 / 0.389,
// x64 (1152 MB) 0.779 / 0.741; 2D 1024^2 (192 MB) 1.677 / 1.698, 2048^2
// (768 MB) 13.57 / 13.41.
constexpr double STREAM_HINT_MB = 320;
bool stream_hints(const ProbDev& P);
int launch_dual(const ProbDev& P, hipStream_t st);
int launch_fused_pd(const ProbDev& P, const FusedBufs& B, hipStream_t st);
int launch_primal(const ProbDev& P, hipStream_t st);
// the u half (PRIMAL_U), the p half (PRIMAL_P) or both (PRIMAL_UP)
enum { PRIMAL_U = 1, PRIMAL_P = 2, PRIMAL_UP = 3 };
int launch_primal_part(const ProbDev& P, int part, hipStream_t st);

// ---- launchers (batches: descriptor table + item table) -------------------
int launch_fwd_batch(const ProbDev* probs_dev, const FwdItem* items, int nitems, int K,
                     int mi, bool wide, size_t lds, int mode, hipStream_t st);
// The sheared forward projection of batch problems: items {prob, J, first
// angle, angles, 0, 0, s0, slices} of at most K slices, J = waves of items of
// one angle and angles * J <= waves; the slices are transposed before, by
// launch_transpose_batch (items: 32 x 32 tiles x0, y0 of slice z) or the dual
// step.  With FWD_LINE_WAVES waves the forward phase of 64 mixed slices (96^2
// to 384^2) takes 0.45 ms; with 9, 10 and 16: 0.58, 0.56, 0.54 (a multiple of 4
// loads the SIMDs evenly, and 16 leave room for one work-group less); one
// launch per J 0.48.  Small plans have work-groups of one angle: 28 slices of
// 89^2 to 130^2 117 us an iteration, 130 with 12 waves.  one_k: every item has
// K slices.
constexpr int FWD_LINE_WAVES = 12;
int launch_fwd_line_batch(const ProbDev* probs_dev, const FwdItem* items, int nitems, int K,
                          bool one_k, int waves, int mode, hipStream_t st);
// Fills the tables of the sheared projection (line0 is there; first: each angle's
// first item) and waits.
int launch_line_tables(const Geometry& g, const int* first);
// Gathered items (FWD_THREADS chunks of one item per thread, unit bins) and items
// by lines (nb = 0, FWD_THREADS / 64 waves) of at most K slices, in one launch;
// lds: bytes that the former need.
int launch_fwd_mixed_batch(const ProbDev* probs_dev, const FwdItem* items, int nitems, int K,
                           size_t lds, int mode, hipStream_t st);
int launch_transpose_batch(const ProbDev* probs_dev, const DualItem* items, int nitems,
                           hipStream_t st);
// Whether an iteration of this problem (alone: a projection outside one)
// projects forward by lines.
bool fwd_by_lines(const ProbDev& P, const Geometry& g, bool alone = false);
int launch_adj_batch(const ProbDev* probs_dev, const AdjItem* items, int nitems, int K,
                     int dim, bool tgv, bool primal, size_t lds, hipStream_t st);
int launch_primal_batch(const ProbDev* probs_dev, const DualItem* items, int nitems, int dim,
                        bool tgv, int part, hipStream_t st);
int launch_dual_batch(const ProbDev* probs_dev, const DualItem* items, int nitems, int dim,
                      int coupling, bool tgv, int maxc, bool tiles, hipStream_t st);

// ---- auxiliary (aux.hip) ---------------------------------------------------
int launch_normest(const Geometry& g, const double* x0_host, int iters, int mode,
                   double tol, double* out, hipStream_t st);
int launch_feasible(const Geometry& g, float* f, int nslices, hipStream_t st);
int launch_energy(const ProbDev& P, double a0, double a1, double* out_reg, hipStream_t st);
int launch_energy_noalloc(const ProbDev& P, const double* mu, double a0, double a1,
                          size_t per_ch, double* out_data, double* out_reg, hipStream_t st);
int launch_data_energy(const float* ku, const float* f, const double* mu, int nch,
                       size_t per_ch, int disc, double* out, hipStream_t st);

}  // namespace gr
