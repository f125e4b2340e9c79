// Which rows and pixels a wave of the weight-gradient kernel visits (cnn.hip).
// Plain C++, so that a host compiler can replay the walk of every wave.
#pragma once
#include <algorithm>

#ifdef __HIPCC__
#define GR_HD __host__ __device__ __forceinline__
#else
#define GR_HD inline
#endif

namespace gr {

// Work of one wave: rows r0 .. r0 + nrows - 1 of the SEG pixels from x0 of an
// image.  Waves are launched in fours: those past the last unit have no rows.
struct WgradUnit {
    int img, x0, r0, nrows;
};

template <int SEG>
GR_HD WgradUnit wgrad_unit(int unit, int n, int H, int W, int rows)
{
    const int segs = (W + SEG - 1) / SEG, row_chunks = (H + rows - 1) / rows;
    const int img = unit / (segs * row_chunks), us = unit - img * segs * row_chunks;
    const int r0 = us % row_chunks * rows, left = H - r0;
    return {img, us / row_chunks * SEG, r0, img < n ? (rows < left ? rows : left) : 0};
}

// Step t of the walk, wgrad_first <= t < nrows, meets row r0 + t of dy; the rows
// of x that the taps reach (`halo` above and below) are read ahead of it, from
// two steps earlier on.  A wave without rows takes no step: its image may lie
// beyond the tensor.
GR_HD int wgrad_first(int nrows, int halo) { return nrows > 0 ? -2 * halo : 0; }

// The row of x or dy that is loaded for step t, and whether it is there.
GR_HD int wgrad_row(int r0, int t, bool is_x, int halo) { return r0 + t + (is_x ? halo : 0); }

GR_HD bool wgrad_row_ok(int row, int t, int nrows, int H, bool is_x)
{
    return row >= 0 && row < H && t < nrows && (is_x || t >= 0);
}

// Rows per wave: long walks read x once and add fewer partial sums, but every
// CU should have work.  One work-group per CU, one and a half where that leaves
// long walks.  Training steps of n images of 256 x 256 with 256 / 384 / 512
// work-groups: n = 2 1162 / 1255 / 1292 us, n = 8 2003 / 1983 / 2095, n = 16
// 3215 / 3141 / 3215; with 128, n = 16 3451.
inline int wgrad_rows(long long columns, int H, long long tiles)
{
    long long rows = columns * H * tiles / (4 * 256);
    if (rows >= 12) rows = rows * 2 / 3;
    return (int)std::max<long long>(1, std::min<long long>(H, rows));
}

}  // namespace gr
