// Launch layout and index arithmetic of the 3D march (rsg_fd3d.h), kept free
// of HIP so that the CPU tests compile it alone.
#pragma once
#include <algorithm>

#ifdef __HIPCC__
#define RSG_HD __host__ __device__ __forceinline__
#else
#define RSG_HD inline
#endif

namespace rsg {

constexpr int R3 = 2, B3 = 256;  // rows a thread, threads a block

// Tile order.  ncx x ncy columns of TX x TY cells; the z planes in three
// zones (strips or shortened stencils at the low face, neither, the high
// face), zone i of planes z[i] .. z[i+1]-1 in n[i] chunks of zc planes; ncomp
// components (blocks that update different arrays of one tile from partly the
// same inputs), the first `first` (0 or 1) of them before all others.  With
// xgroups blocks are dealt round-robin to the 8 XCDs (XCD k runs blocks k,
// k+8, ...).  xgroups 1: XCD k marches its own contiguous group of columns
// cg[k] .. cg[k+1]-1 through the chunks, components fastest (those after the
// first), then columns: the blocks an XCD holds at once are neighbours at the
// same depth, so shared inputs, halos and the lines that tile rows share are
// fetched into that XCD's L2 once.  xgroups 2, for few columns: XCD k marches
// an eighth of all chunks, those of one depth after those of the one before.
struct Tiles3 {
    int tx, xgroups, ncx, ncy, zc, ncomp, first;
    int z[4], n[3];
    int cg[9];
};

struct Pos3 {
    int x0, y0, zb, ze, comp, zone;
};

// Component of block r of n blocks a component; r: its block.
RSG_HD bool comp_of(const Tiles3 &t, int n, int &r, int &comp) {
    const int m = t.ncomp - t.first;
    comp = 0;
    if (r >= t.first * n) {
        r -= t.first * n;
        comp = t.first + r % m;
        r /= m;
    }
    return r < n;
}

// Tile, chunk and component of block r; false for surplus blocks.
template <int TX>
RSG_HD bool tile3_at(const Tiles3 &t, int r, Pos3 &p) {
    int col, ck;
    const int nck = t.n[0] + t.n[1] + t.n[2];
    if (!t.xgroups) {
        if (!comp_of(t, t.ncx * t.ncy * nck, r, p.comp)) return false;
        ck = r / (t.ncx * t.ncy);
        col = r - ck * (t.ncx * t.ncy);
    } else if (t.xgroups == 2) {
        const int k = r % 8, ncol = t.ncx * t.ncy, i0 = (int)((long)ncol * nck * k / 8);
        r /= 8;
        if (!comp_of(t, (int)((long)ncol * nck * (k + 1) / 8) - i0, r, p.comp)) return false;
        ck = (i0 + r) / ncol;
        col = i0 + r - ck * ncol;
    } else {
        const int k = r % 8, ncol = t.cg[k + 1] - t.cg[k];
        r /= 8;
        if (ncol <= 0 || !comp_of(t, ncol * nck, r, p.comp)) return false;
        ck = r / ncol;
        col = t.cg[k] + (r - ck * ncol);
    }
    const int cy = col / t.ncx;
    p.x0 = (col - cy * t.ncx) * TX;
    p.y0 = cy * (R3 * B3 / TX);
    int zone = 0;
    if (ck >= t.n[0]) {
        ck -= t.n[0];
        zone = 1;
        if (ck >= t.n[1]) {
            ck -= t.n[1];
            zone = 2;
        }
    }
    p.zb = t.z[zone] + ck * t.zc;
    p.ze = p.zb + t.zc < t.z[zone + 1] ? p.zb + t.zc : t.z[zone + 1];
    p.zone = zone;
    return p.zb < p.ze;
}

// Does the tile hold cells of x or y strips, or whose x or y stencils the
// array's ends shorten, or cells outside the grid?
RSG_HD bool tile_pxy(int tx, int nx, int ny, int lpml, int order, const Pos3 &p) {
    const int m = lpml > order ? lpml : order;
    return p.x0 < m || p.x0 + tx > nx - m || p.y0 < m || p.y0 + R3 * B3 / tx > ny - m;
}

// A launch holds less than 2^32 threads along x; past that the runtime drops
// blocks without an error (20,000,000 of 256 threads asked for, 3,222,784 run).
constexpr long kMaxBlocks = 0xFFFFFFFFL / B3;

// Blocks of a launch of ncomp components, and the tile order.  zc, xcd: the
// knobs zc3d (0: chosen here) and xcd3d.
inline unsigned layout_tiles3(Tiles3 &t, int nx, int ny, int nz, int lpml, int order, int ncomp, int first, int zc,
                              int xcd) {
    // Rows of 64 touch fewer partly used cache lines (440^3, order 4: 778 + 474
    // us a step against 873 + 514 with 32), unless they waste much more of a
    // narrow grid's last tile (160 x 150 x 140: 36 + 33 us against 33 + 29).
    const long w64 = (nx + 63L) / 64 * 64, w32 = (nx + 31L) / 32 * 32;
    t.tx = 10 * w64 <= 11 * w32 ? 64 : 32;
    const int ty = R3 * B3 / t.tx;
    t.ncx = (nx + t.tx - 1) / t.tx;
    t.ncy = (ny + ty - 1) / ty;
    t.ncomp = ncomp;
    t.first = first;
    // the low zone ends before the high strip, so that a chunk has one face
    const int m = std::max(lpml, order), lo = std::min(m, nz - lpml), hi = std::max(lo, nz - m);
    t.z[0] = 0;
    t.z[1] = lo;
    t.z[2] = hi;
    t.z[3] = nz;
    const long ncol = (long)t.ncx * t.ncy;
    auto split = [&](int planes) {
        t.zc = planes;
        for (int i = 0; i < 3; i++) t.n[i] = (t.z[i + 1] - t.z[i] + planes - 1) / planes;
        return t.n[0] + t.n[1] + t.n[2];
    };
    // Short chunks give many blocks, long ones amortise the queue's filling:
    // 8 planes where that gives enough blocks, else 4.  One component: four
    // rounds (320 x 300 x 280: 229 + 154 us a step with 8, 230 + 161 with 4;
    // 200 x 190 x 180, 2400 blocks: 69 + 50 with 8, 62 + 50 with 4).  The
    // elastic components' blocks do less each and start cheaper on lines their
    // neighbours read: two rounds (140 x 130 x 120: 50 + 60 us with 8, 53 + 64
    // with 4; 88 x 65 x 267, velocity, 1575 blocks: 50, 43).  Where all their
    // blocks run at once a step lasts as long as one block, and chunks of 1 or 2
    // planes end sooner: three or four blocks a compute unit (order 4: 24^3 12 +
    // 13 us with 4 planes, 6.2 + 6.6 with 1; 64^3 13.7 + 13.9 with 4, 11.1 + 11.8
    // with 2, 13.6 + 15.7 with 1).
    if (zc <= 0) {
        zc = ncol * ncomp * split(8) >= (ncomp > 1 ? 2048 : 4096) ? 8 : 4;
        for (int c = 2; c >= 1 && ncomp > 1; c--)
            if (ncol * ncomp * split(c) <= (c == 2 ? 1024 : 768)) zc = c;
    }
    long most = 0;  // columns of the largest group
    for (int x = 0; x <= 8; x++) {
        t.cg[x] = (int)(ncol * x / 8);
        if (x) most = std::max(most, (long)t.cg[x] - t.cg[x - 1]);
    }
    // Few columns split unevenly: where the largest group is more than an
    // eighth above the mean, the chunks are split by depth (us a velocity + a
    // stress step by columns, by depth; elastic, order 4: 20 x 20 x 400, 2 columns,
    // 6 of 8 XCDs idle: 34 + 41, 15 + 16; 60 x 40 x 1000: 71 + 86, 44 + 63; 120 x
    // 110 x 100, 28 columns: 35 + 41, 33 + 37; 90 x 64 x 64: 15.6 + 19.1, 16.1 +
    // 15.6; acoustic: 120 x 110 x 100 order 4 18.6 + 17.3, 16.6 + 16.0, order 8,
    // where three blocks a compute unit are resident, 31.2 + 25.1, 22.9 + 23.0).
    t.xgroups = !xcd ? 0 : (64 * most <= 9 * ncol ? 1 : 2);
    // Longer chunks where these give more blocks than a launch holds (thin or
    // very large grids, a small zc3d)
    for (zc = std::min(zc, nz);; zc = std::min(2 * zc, nz)) {
        const long nck = split(zc);
        const long blocks = (t.xgroups == 2 ? (ncol * nck + 7) / 8 * 8 : (t.xgroups ? 8 * most : ncol) * nck) * ncomp;
        if (blocks <= kMaxBlocks || zc == nz) return (unsigned)blocks;
    }
}

// Raw buffers over the tile's part of an array: every lane either has an
// offset inside its tile's window of the grid, or kOut, which no descriptor
// covers: loads return 0 and stores are dropped, so lanes outside the grid
// need no branches.  A live descriptor covers every offset below kOut.
constexpr unsigned kOut = 0xFFFFFF00u;

// Byte offset of row r, column c counted from the base of a tile's buffer, rows
// nx cells apart.  Unsigned: 32-bit offsets reach 4 GiB.
RSG_HD unsigned tile_off(int r, int nx, int c) { return ((unsigned)r * (unsigned)nx + (unsigned)c) * 4u; }

// First row that the offsets of the window of a tile whose first row is y0, halo
// hy, count from.  clip: not the rows above the grid, which hold no cells, so that
// the offsets span at most the plane.  The acoustic planes (under 2^29 cells, at
// least 2 hy + 2 rows) fit without: ny + hy rows are at most one and a half planes.
RSG_HD int window_row0(int y0, int hy, bool clip) { return clip && y0 < hy ? 0 : y0 - hy; }

// Do the offsets of every tile's clipped windows stay below kOut?  ty: rows of a tile.
// The largest is that of the last cell of the last of the window's rows inside
// the grid, counted from `order` columns before the row in the leftmost tile.
inline bool tiles_fit(int nx, int ny, int ty, int order) {
    const long long rows = ny < ty + 2 * order ? ny : ty + 2 * order;
    return (rows * nx + order) * 4 <= (long long)kOut;
}

}  // namespace rsg
