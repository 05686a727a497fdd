// Index arithmetic of the 3D march (rsg_fd3d.h), kept free of HIP so that the
// CPU tests compile it alone.
#pragma once

#ifdef __HIPCC__
#define RSG_HD __host__ __device__ __forceinline__
#else
#define RSG_HD inline
#endif

namespace rsg {

// Raw buffers over the tile's part of an array: every lane either has an
// offset inside its tile's window of the grid, or kOut, which no descriptor
// covers: loads return 0 and stores are dropped, so lanes outside the grid
// need no branches.  A live descriptor covers every offset below kOut.
constexpr unsigned kOut = 0xFFFFFF00u;

// Byte offset of row r, column c counted from the base of a tile's buffer, rows
// nx cells apart.  Unsigned: 32-bit offsets reach 4 GiB.
RSG_HD unsigned tile_off(int r, int nx, int c) { return ((unsigned)r * (unsigned)nx + (unsigned)c) * 4u; }

// First row of the window of a tile whose first row is y0, halo hy: rows above
// the grid hold no cells and are not counted, so that offsets of a window span
// at most the plane.
RSG_HD int window_row0(int y0, int hy) { return y0 > hy ? y0 - hy : 0; }

// Do the offsets of every tile's windows stay below kOut?  ty: rows of a tile.
// The largest is that of the last cell of the last of the window's rows inside
// the grid, counted from `order` columns before the row in the leftmost tile.
inline bool tiles_fit(int nx, int ny, int ty, int order) {
    const long long rows = ny < ty + 2 * order ? ny : ty + 2 * order;
    return (rows * nx + order) * 4 <= (long long)kOut;
}

}  // namespace rsg
