// Device side of the 3D half steps (acoustic fd3d.hip, elastic
// fd3d_elastic.hip): the z march both share, and the host code that lays out
// their launches.
//
// A block owns a column tile of TX x TY = 512 cells in (x, y), 64 x 8 or
// 32 x 16, and marches through a chunk of z planes; a thread owns two rows of
// one column.  The x and y taps of a plane come from LDS (the plane's window
// with its halo, double buffered: one barrier a plane), the z taps from a
// register queue of 2*ORDER values per cell.
//
// Everything a plane needs is loaded a plane ahead, PML memory variables
// included, the queue's new values two.  For that to hide the latency no load
// may be waited for early, and the compiler waits early wherever a value still
// in flight is moved (so the queue takes its two new values at the top of the
// next round, two planes after their loads) or wherever a branch makes the
// number of loads in flight unknown.  So the march has no branches around
// loads: tiles with strips or shortened stencils in x or y (PXY) and chunks
// with them in z (PZ) are instantiations of their own, and loads past the end
// of a chunk use an empty descriptor.  Two planes ahead (a second set of
// registers) costs order 8 its fourth wave a SIMD, which hides more.
//
// What bounds it: HBM on large acoustic grids (440^3, order 4: velocity 4.25 GB a
// launch at 5.5 TB/s, stress 2.43 GB at 5.0; each array once would be 1/1.18 and
// 1/1.09 of that), the march's latency, a memory latency a plane, on small ones.
// Three or four blocks read each field's window and queue in the elastic steps,
// from the caches for the most part: a third more than each array once reaches
// HBM, at 4.4 TB/s (240^3, order 8).  Against the kernels before (acoustic: 64 x 8
// tiles that loaded the memory variables where they were used; elastic: a thread
// a cell, all taps through L1 and L2), us a velocity + a stress step:
//   acoustic, order 4:  320 x 300 x 280  315 + 251 -> 229 + 151, 440^3  901 + 674 ->
//                       765 + 465, 160 x 150 x 140  66 + 57 -> 30 + 28,
//                       120 x 110 x 100  41 + 36 -> 16.6 + 16.0
//   acoustic, order 8:  320 x 300 x 280  518 + 444 -> 251 + 183
//   elastic, order 4:   200 x 190 x 180  285 + 318 -> 144 + 189,
//                       140 x 130 x 120  80 + 85 -> 51 + 61,
//                       70 x 60 x 50  17.0 + 16.9 -> 13.3 + 14.0
//   elastic, order 8:   200 x 190 x 180  414 + 449 -> 175 + 220,
//                       240^3  672 + 729 -> 287 + 372
// Of 60 random elastic grids of 100 thousand to 1.2 million cells, strips of 8 to
// 20, all are faster here from order 4 on; at orders 1 to 3 single ones under 400
// thousand are up to a fifth slower than a thread a cell was (rows that fill 64
// lanes: 56^3, order 2, 7.2 + 7.6 us, 9.3 + 9.5 here), the mean is 1.0 to 1.2 faster.
#pragma once
#include <algorithm>
#include <type_traits>

#include "rsg_common.h"
#include "rsg_tiles3.h"

namespace rsg {

// Lambdas of the march: one left out of line would put the arrays it captures,
// the queue among them, in scratch memory.
#define RSG_INLINE __attribute__((always_inline))

// Four waves a SIMD, 128 VGPRs (three for the acoustic velocity step from order 7
// on, fd3d.hip).  Three with two planes ahead, 168 VGPRs, take 222 us for the
// acoustic stress step on 320 x 300 x 280 at order 8 where four take 185; five
// spill.
#define RSG3_BOUNDS __launch_bounds__(B3) __attribute__((amdgpu_waves_per_eu(4, 8)))

// The tile's part of an array; a descriptor that is not live covers nothing.
__device__ __forceinline__ Buf tile_buf(const float *f, long off, bool live = true) {
    return mkbuf(f + off, live ? kOut : 0u);
}

// A uniform value the optimiser may not see through (v is uniform;
// readfirstlane says so where the compiler lost sight of it): for plane
// offsets, where it would otherwise keep one running address per array, load
// and store instead of two scalar adds where one is used.
__device__ __forceinline__ long opaque(long v) {
    int lo = __builtin_amdgcn_readfirstlane((int)v), hi = __builtin_amdgcn_readfirstlane((int)(v >> 32));
    asm volatile("" : "+s"(lo), "+s"(hi));
    return ((long)hi << 32) | (unsigned)lo;
}
// One derivative term: the field, its two strips (low, high face), and
// whether it is the forward (1) or backward (0) difference.
struct Term3 {
    const float *f;
    float *lo, *hi;
    int fw;
};

// Tile, chunk and component of this block; false for surplus blocks.
template <int TX>
__device__ __forceinline__ bool tile3_of(const Tiles3 &t, Pos3 &p) {
    return tile3_at<TX>(t, blockIdx.x, p);
}

// Grid, step and stencil description every 3D kernel takes.
struct G3 {
    int nx, ny, nz, lpml, fs, order;
    float dt, inv[3];
    const float *tab;
    float c[3][8];   // the stencil's coefficients over the step, per axis
    float cz[9][8];  // z: of every order (0 past it), for the planes at the ends
    Tiles3 t;
};

template <int TX>
__device__ __forceinline__ bool tile_pxy(const G3 &g, const Pos3 &p) {
    return tile_pxy(TX, g.nx, g.ny, g.lpml, g.order, p);
}

// z-derivative from a queue q[j] = f(z + off + j): both the forward
// (off = 1-H) and the backward (off = -H) staggered forms reduce to
// sum_io c_io (q[H+io] - q[H-1-io]).  The queue holds two more values than a
// plane takes: odd planes of a chunk (S = 1) read it one further, and it
// shifts once every two planes.
template <int H, int S>
__device__ __forceinline__ float dq(const float (&q)[2 * H + 2], const float *c) {
    float acc = c[0] * (q[S + H] - q[S + H - 1]);
#pragma unroll
    for (int io = 1; io < H; io++) acc += c[io] * (q[S + H + io] - q[S + H - 1 - io]);
    return acc;
}
// The same where the array's end may shorten the stencil to order k (uniform):
// the taps past it are masked out, whatever they hold (selects would take more
// registers than order 8 has).
template <int H, int S>
__device__ __forceinline__ float dq_edge(const float (&q)[2 * H + 2], const float *c, int k) {
    float acc = c[0] * __int_as_float(__float_as_int(q[S + H] - q[S + H - 1]) & (k > 0 ? -1 : 0));
#pragma unroll
    for (int io = 1; io < H; io++)
        acc += c[io] * __int_as_float(__float_as_int(q[S + H + io] - q[S + H - 1 - io]) & (k > io ? -1 : 0));
    return acc;
}
template <int N>
__device__ __forceinline__ void shift2(float (&q)[R3][N], const float (&qn)[2][R3]) {
#pragma unroll
    for (int r = 0; r < R3; r++) {
#pragma unroll
        for (int j = 0; j < N - 2; j++) q[r][j] = q[r][j + 2];
        q[r][N - 2] = qn[0][r];
        q[r][N - 1] = qn[1][r];
    }
}

// The forward difference of a cell whose stencil the array's end shortens to
// order k, coefficients from a table in LDS (a global load here would wait
// for every load in flight).
__device__ __forceinline__ float dfw_edge(const float *s, int st, int k, float invd, const float *ce) {
    const float *c = ce + cind(k);
    float acc = 0.f;
#pragma unroll 1
    for (int io = 0; io < k; io++) acc += c[io] * (s[(io + 1) * st] - s[-io * st]);
    return acc * invd;
}

// Window of one plane, TY + 2*HY rows of TX + 2*HX: each thread's element
// list (offsets from the window's base, kOut outside the grid) is fixed for
// the whole march; fetch loads into registers, store writes them to LDS.
// The base is the corner of the window's rows inside the grid, or, with halos
// on both axes (acoustic velocity, planes under 2^29 cells), the window's own:
// there the clipped base costs order 8 a register it has not (440^3 816 -> 823
// us, 502 x 122 x 52 42.2 -> 43.5).
template <int TX, int HX, int HY>
struct Win3 {
    static constexpr int LD = TX + 2 * HX, N = LD * (R3 * B3 / TX + 2 * HY), K = (N + B3 - 1) / B3;
    static constexpr bool CLIP = HY && !HX;
    unsigned off[K];
    long corner;  // from the tile's first cell to the base
    __device__ __forceinline__ void init(int nx, int ny, int x0, int y0) {
        const int row0 = CLIP ? window_row0(y0, HY, true) : y0 - HY;
        corner = (long)(row0 - y0) * nx - HX;
#pragma unroll
        for (int k = 0; k < K; k++) {
            const int i = (int)threadIdx.x + k * B3, r = i / LD, c = i - r * LD;
            const int y = y0 - HY + r, x = x0 - HX + c;
            off[k] = (i < N && x >= 0 && x < nx && y >= 0 && y < ny) ? tile_off(CLIP ? y - row0 : r, nx, c) : kOut;
        }
    }
    // f at plane offset `at` (of the tile's first cell)
    __device__ __forceinline__ void fetch(float (&v)[K], const float *f, long at, int nx, bool live) const {
        const Buf b = tile_buf(f, CLIP ? at + corner : at - (long)HY * nx - HX, live);
#pragma unroll
        for (int k = 0; k < K; k++) v[k] = b.ld(off[k], 0);
    }
    __device__ __forceinline__ void store(const float (&v)[K], float *lds) const {
#pragma unroll
        for (int k = 0; k < K; k++)
            if (N % B3 == 0 || (int)threadIdx.x + k * B3 < N) lds[threadIdx.x + k * B3] = v[k];
    }
};

// A lane's cell against the strips of the x or y axis: its memory variable on
// the chunk's first plane (a lane outside the strips points at some cell of
// theirs, so that its load needs no branch) and its profile values.
struct Face3 {
    float *psi;
    float A, B, C;
    bool in;
    // i: the cell on the axis (any, where not ok); off(j): index of strip cell j
    template <class F>
    __device__ __forceinline__ void init(int i, int n, int L, bool ok, float *lo, float *hi, F &&off, const float *tab,
                                         int stag) {
        const bool h = i >= n - L;
        in = ok && (i < L || h);
        const int j = !in ? 0 : (h ? i - (n - L) : i), s = (h ? T_RBB : 0) + stag * T_STAG;
        psi = (h ? hi : lo) + off(j);
        A = tab[(s + T_A) * L + j];
        B = tab[(s + T_B) * L + j];
        C = tab[(s + T_C) * L + j];
    }
};

// A thread's cells: column x, rows y .. y+R3-1, and their offsets in the
// tile's part of a plane (kOut outside the grid).
template <int TX>
struct Lane3 {
    int tx, ty, x, y;
    unsigned oc[R3];
    bool ok[R3];
    long t0;  // the tile's first cell in a plane
    __device__ __forceinline__ Lane3(const G3 &g, const Pos3 &p) {
        tx = threadIdx.x % TX;
        ty = threadIdx.x / TX;
        x = p.x0 + tx;
        y = p.y0 + ty * R3;
#pragma unroll
        for (int r = 0; r < R3; r++) {
            ok[r] = x < g.nx && y + r < g.ny;
            oc[r] = ok[r] ? tile_off(ty * R3 + r, g.nx, tx) : kOut;
        }
        t0 = (long)p.y0 * g.nx + p.x0;
    }
    __device__ __forceinline__ long at(const G3 &g, int z) const { return opaque(z * ((long)g.nx * g.ny) + t0); }
    __device__ __forceinline__ void ld(const float *f, long o, float (&v)[R3], bool live = true) const {
        const Buf b = tile_buf(f, o, live);
#pragma unroll
        for (int r = 0; r < R3; r++) v[r] = b.ld(oc[r], 0);
    }
    __device__ __forceinline__ void st(float *f, long o, const float (&v)[R3], bool live = true) const {
        const Buf b = tile_buf(f, o, live);
#pragma unroll
        for (int r = 0; r < R3; r++) b.st(v[r], oc[r], 0);
    }
    // the queue before its first shift: f of the own cells at planes z .. (0
    // outside the grid) in q[2 ..] and qn
    template <int N>
    __device__ __forceinline__ void fill(const float *f, int z, const G3 &g, float (&q)[R3][N], float (&qn)[2][R3]) const {
#pragma unroll
        for (int j = 0; j < N; j++) {
            float v[R3];
            ld(f, at(g, z + j), v, z + j >= 0 && z + j < g.nz);
#pragma unroll
            for (int r = 0; r < R3; r++) (j < N - 2 ? q[r][j + 2] : qn[j - (N - 2)][r]) = v[r];
        }
#pragma unroll
        for (int r = 0; r < R3; r++) q[r][0] = q[r][1] = 0.f;
    }
};

// The x and y strips of a PXY tile.
template <int TX>
struct Sides3 {
    Face3 x, y[R3];
    bool inx[R3];
    bool px, py, ex, ey;  // does the tile (uniform) hold cells of x / y strips, of shortened x / y stencils?
    int xr;               // rows apart in an x strip (0: the second row is outside the grid)
    long xstep, ystep;    // planes apart
    int kx, ky[R3];       // stencil orders
    __device__ __forceinline__ void init(const G3 &g, const Pos3 &p, const Lane3<TX> &ln, const Term3 &tx, const Term3 &ty) {
        constexpr int TY = R3 * B3 / TX;
        const int nx = g.nx, ny = g.ny, L = g.lpml, H = g.order;
        px = p.x0 < L || p.x0 + TX > nx - L;
        py = p.y0 < L || p.y0 + TY > ny - L;
        ex = p.x0 < H || p.x0 + TX > nx - H;
        ey = p.y0 < H || p.y0 + TY > ny - H;
        xstep = (long)ny * L;
        ystep = (long)L * nx;
        const int xc = min(ln.x, nx - 1), yc = min(ln.y, ny - 1);
        xr = ln.ok[1] ? L : 0;
        if (tx.f)
            x.init(xc, nx, L, ln.ok[0], tx.lo, tx.hi, [&](int j) RSG_INLINE { return p.zb * xstep + (long)yc * L + j; }, g.tab, tx.fw);
        kx = tx.fw ? kfw(ln.x, nx, H) : kbw(ln.x, nx, H);
#pragma unroll
        for (int r = 0; r < R3; r++) {
            inx[r] = tx.f && x.in && ln.ok[r];
            if (ty.f)
                y[r].init(min(ln.y + r, ny - 1), ny, L, ln.ok[r], ty.lo, ty.hi,
                          [&](int j) RSG_INLINE { return p.zb * ystep + (long)j * nx + xc; }, g.tab, ty.fw);
            ky[r] = ty.fw ? kfw(ln.y + r, ny, H) : kbw(ln.y + r, ny, H);
        }
        xstep = opaque(xstep);
        ystep = opaque(ystep);
    }
    // memory variables `at` values on from the strips' current plane
    __device__ __forceinline__ void load_x(float (&v)[R3], long at) const {
#pragma unroll
        for (int r = 0; r < R3; r++) v[r] = x.psi[at + r * xr];
    }
    __device__ __forceinline__ void load_y(float (&v)[R3], long at) const {
#pragma unroll
        for (int r = 0; r < R3; r++) v[r] = y[r].psi[at];
    }
    __device__ __forceinline__ void store_x(const float (&v)[R3], long at) const {
#pragma unroll
        for (int r = 0; r < R3; r++)
            if (inx[r]) x.psi[at + r * xr] = v[r];
    }
    __device__ __forceinline__ void store_y(const float (&v)[R3], long at) const {
#pragma unroll
        for (int r = 0; r < R3; r++)
            if (y[r].in) y[r].psi[at] = v[r];
    }
};

// The z strip of a PZ chunk (one face): the memory variables of its planes'
// own cells and their profile values.  A plane between the strips (of a grid
// whose strips are thinner than the stencil) loads and stores nothing.
struct ZStrip {
    float *psi;
    const float *tab;
    int L, z0;  // strip plane of z: z - z0
    __device__ __forceinline__ void init(const G3 &g, const Pos3 &p, const Term3 &t) {
        const bool h = p.zone == 2;
        L = g.lpml;
        z0 = h ? g.nz - L : 0;
        psi = h ? t.hi : t.lo;
        tab = g.tab + ((h ? T_RBB : 0) + t.fw * T_STAG) * L;
    }
    __device__ __forceinline__ bool in(int z) const { return z >= z0 && z < z0 + L; }
};
struct ZVals {
    float A, B, C, v[R3];
};
template <int TX>
__device__ __forceinline__ void zload(ZVals &v, const ZStrip &s, const G3 &g, int z, const Lane3<TX> &ln, bool live) {
    const bool in = s.in(z) && live;
    const int j = in ? z - s.z0 : 0;
    v.A = s.tab[T_A * s.L + j];
    v.B = s.tab[T_B * s.L + j];
    v.C = s.tab[T_C * s.L + j];
    ln.ld(s.psi, j * ((long)g.nx * g.ny) + ln.t0, v.v, in);
}
template <int TX>
__device__ __forceinline__ void zstore(const ZVals &v, const ZStrip &s, const G3 &g, int z, const Lane3<TX> &ln) {
    const bool in = s.in(z);
    ln.st(s.psi, (in ? z - s.z0 : 0) * ((long)g.nx * g.ny) + ln.t0, v.v, in);
}

// psi = B psi + A d; F -= m (psi + C d) for a cell in the strip.
__device__ __forceinline__ void strip3(float &F, float m, float d, bool in, float C, float psi) {
    F = in ? F - m * (psi + C * d) : F;
}

// Two planes a round: top(z) before each pair, then body(S, z) for the even
// (S = 0) and the odd (S = 1) plane of the chunk.
template <class T, class B>
__device__ __forceinline__ void march3(int zb, int ze, T &&top, B &&body) {
    constexpr std::integral_constant<int, 0> S0;
    constexpr std::integral_constant<int, 1> S1;
#pragma unroll 1
    for (int z = zb;;) {
        top(z);
        body(S0, z);
        if (z + 1 >= ze) break;
        body(S1, z + 1);
        z += 2;
        if (z >= ze) break;
    }
}

// ---------------------------------------------------------------------------
// F_i += dt M_i (Dx fx + Dy fy + Dz fz), each term with its CFS-PML memory
// variable: the acoustic stress step, an elastic velocity component, the
// elastic normal stresses (NOUT 3: moduli L + 2 mu of the component's own
// axis, L of the others; UNIT: F_i += dt of its own term) and, with one term
// left out, an elastic shear stress.
// ---------------------------------------------------------------------------

struct Comp3 {
    Term3 t[3];         // x, y, z
    float *F[3];        // NOUT of them
    const float *M[2];  // the modulus (NOUT 1), or L, L + 2 mu
};

template <int TX, int ORDER, bool HX, bool HY, bool HZ, int NOUT, bool UNIT, bool FULL = true>
struct Div3 {
    static constexpr int H = ORDER, NM = UNIT ? 0 : (NOUT == 3 ? 2 : 1);
    using WX = Win3<TX, H, 0>;
    using WY = Win3<TX, 0, H>;
    // floats of LDS: two buffers of both windows, and the edge coefficients
    static constexpr int LX = HX ? WX::N : 0, LY = HY ? WY::N : 0, LDS = 2 * (LX + LY) + 36;

    template <bool PXY, bool PZ>
    static __device__ __forceinline__ void march(const G3 &g, const Comp3 &c, const Pos3 &p, float *lds) {
        const int fx = c.t[0].fw, fy = c.t[1].fw, fz = c.t[2].fw, nx = g.nx, ze = p.ze;
        const Lane3<TX> ln(g, p);
        float *const ce = lds + 2 * (LX + LY);
        WX wx;
        WY wy;
        if (HX) wx.init(nx, g.ny, p.x0, p.y0);
        if (HY) wy.init(nx, g.ny, p.x0, p.y0);
        Sides3<TX> sd;
        ZStrip zs;
        if (PXY) {
            sd.init(g, p, ln, c.t[0], c.t[1]);
            if (threadIdx.x < 36) ce[threadIdx.x] = kCoefC[threadIdx.x];
        }
        if (PZ && HZ) zs.init(g, p, c.t[2]);
        const float *const f[3] = {c.t[0].f, c.t[1].f, c.t[2].f};
        float *Fp[NOUT];
        const float *Mp[NM ? NM : 1];
#pragma unroll
        for (int i = 0; i < NOUT; i++) Fp[i] = c.F[i];
#pragma unroll
        for (int i = 0; i < NM; i++) Mp[i] = c.M[i];
        const long nxy = opaque((long)nx * g.ny);
        long o = ln.at(g, p.zb);      // the current plane's part of the tile
        long xo = 0, yo = 0;          // and of its strips
        // the next plane's values, once the current plane's are used
        float F[NOUT][R3], M[NM ? NM : 1][R3], sx[R3], sy[R3], q[R3][2 * H + 2], qn[2][R3], wvx[WX::K], wvy[WY::K];
        ZVals zv;
        // plane z, k planes after the current one
        auto window = [&](int z, int k) RSG_INLINE {
            const bool live = z < ze;
            const long at = opaque(o + k * nxy);
            if (HX) wx.fetch(wvx, f[0], at, nx, live);
            if (HY) wy.fetch(wvy, f[1], at, nx, live);
        };
        auto own = [&](int z, int k) RSG_INLINE {
            const bool live = z < ze;
            const long at = opaque(o + k * nxy);
#pragma unroll
            for (int i = 0; i < NOUT; i++) ln.ld(Fp[i], at, F[i], live);
#pragma unroll
            for (int i = 0; i < NM; i++) ln.ld(Mp[i], at, M[i], live);
            if (PXY && HX) sd.load_x(sx, xo + (live ? k * sd.xstep : 0));
            if (PXY && HY) sd.load_y(sy, yo + (live ? k * sd.ystep : 0));
            if (PZ && HZ) zload(zv, zs, g, z, ln, live);
        };
        if (HZ) ln.fill(f[2], p.zb + fz - H, g, q, qn);
        window(p.zb, 0);
        own(p.zb, 0);
        const int qz = fz + H;  // the queue's next plane, from two planes on
        auto top = [&](int z) RSG_INLINE {
            o = opaque(o);
            if (HZ) {
                shift2(q, qn);
                ln.ld(f[2], o + (qz + 2) * nxy, qn[0], z + 2 < ze && z + 2 + qz < g.nz);
                ln.ld(f[2], o + (qz + 3) * nxy, qn[1], z + 3 < ze && z + 3 + qz < g.nz);
            }
        };
        auto body = [&](auto S, int z) RSG_INLINE {
            constexpr int sb = decltype(S)::value;
            float *const bx = lds + sb * (LX + LY), *const by = bx + LX;
            if (HX) wx.store(wvx, bx);
            if (HY) wy.store(wvy, by);
            __syncthreads();
            window(z + 1, 1);
            const int kz = PZ ? (fz ? kfw(z, g.nz, H) : kbw(z, g.nz, H)) : H;
            const float *const cz = g.cz[kz];
            const bool zin = PZ && HZ && zs.in(z);
#pragma unroll
            for (int r = 0; r < R3; r++) {
                const int yl = ln.ty * R3 + r;
                auto m = [&](int a, int i) RSG_INLINE { return UNIT ? g.dt : g.dt * M[NOUT == 3 && i == a ? NM - 1 : 0][r]; };
                auto plain = [&](int a, float d) RSG_INLINE {
#pragma unroll
                    for (int i = 0; i < NOUT; i++)
                        if (!(NOUT == 3 && UNIT && i != a)) F[i][r] += m(a, i) * d;
                };
                auto strip = [&](int a, float d, bool in, float C, float psi) RSG_INLINE {
#pragma unroll
                    for (int i = 0; i < NOUT; i++)
                        if (!(NOUT == 3 && UNIT && i != a)) strip3(F[i][r], m(a, i), d, in, C, psi);
                };
                auto term_x = [&]() RSG_INLINE {
                    if (!HX) return;
                    // the backward difference is the forward one a cell before
                    const float *w = bx + yl * WX::LD + ln.tx + H - 1 + fx;
                    float d = dfw<ORDER>(w, 1, g.c[0]);
                    if (PXY && sd.ex)
                        if (sd.kx != H) d = dfw_edge(w, 1, sd.kx, g.inv[0], ce);
                    plain(0, d);
                    if (PXY && sd.px) {
                        sx[r] = fmaf(sd.x.A, d, sd.x.B * sx[r]);
                        strip(0, d, sd.inx[r], sd.x.C, sx[r]);
                    }
                };
                auto term_y = [&]() RSG_INLINE {
                    if (!HY) return;
                    const float *w = by + (yl + H - 1 + fy) * WY::LD + ln.tx;
                    float d = dfw<ORDER>(w, WY::LD, g.c[1]);
                    if (PXY && sd.ey)
                        if (sd.ky[r] != H) d = dfw_edge(w, WY::LD, sd.ky[r], g.inv[1], ce);
                    plain(1, d);
                    if (PXY && sd.py) {
                        sy[r] = fmaf(sd.y[r].A, d, sd.y[r].B * sy[r]);
                        strip(1, d, sd.y[r].in, sd.y[r].C, sy[r]);
                    }
                };
                auto term_z = [&]() RSG_INLINE {
                    if (!HZ) return;
                    const float d = PZ ? dq_edge<H, sb>(q[r], cz, kz) : dq<H, sb>(q[r], g.c[2]);
                    plain(2, d);
                    if (PZ && zin) {
                        zv.v[r] = fmaf(zv.A, d, zv.B * zv.v[r]);
                        strip(2, d, true, zv.C, zv.v[r]);
                    }
                };
                // the reference's order: x, y, z, but z, y for Syz and y, x for Sxy
                if (HX && HZ) {
                    term_x();
                    term_y();
                    term_z();
                } else {
                    term_z();
                    term_y();
                    term_x();
                }
                // free surface: the plane lpml lies in no z strip, so zeroing
                // after the strips is the reference's zeroing before them
                if (NOUT == 3 && g.fs && z == g.lpml) F[NOUT - 1][r] = 0.f;
            }
#pragma unroll
            for (int i = 0; i < NOUT; i++) ln.st(Fp[i], o, F[i]);
            if (PZ && HZ) zstore(zv, zs, g, z, ln);
            if (PXY && HX && sd.px) sd.store_x(sx, xo);
            if (PXY && HY && sd.py) sd.store_y(sy, yo);
            own(z + 1, 1);
            o += nxy;
            if (PXY) {
                xo += sd.xstep;
                yo += sd.ystep;
            }
        };
        march3(p.zb, ze, top, body);
    }

    static __device__ __forceinline__ void run(const G3 &g, const Comp3 &c, const Pos3 &p, float *lds) {
        const bool pxy = tile_pxy<TX>(g, p), pz = p.zone != 1;
        if (FULL && pxy && !pz)
            march<true, false>(g, c, p, lds);
        else if (FULL && HZ && pz && !pxy)
            march<false, true>(g, c, p, lds);
        else if (pxy || pz)
            march<true, true>(g, c, p, lds);
        else
            march<false, false>(g, c, p, lds);
    }
};

// ---------------------------------------------------------------------------
// Acoustic velocity: V_a += dt R_a D+_a P, each with its memory variable.  One
// field in, three out: P's window carries both halos.
// ---------------------------------------------------------------------------

struct Grad3Args {
    Term3 t[3];  // f: P, fw: 1
    float *V[3];
    const float *R[3];
};

template <int TX, int ORDER>
struct Grad3 {
    static constexpr int H = ORDER;
    using W = Win3<TX, H, H>;
    static constexpr int LDS = 2 * W::N + 36;

    template <bool PXY, bool PZ>
    static __device__ __forceinline__ void march(const G3 &g, const Grad3Args &c, const Pos3 &p, float *lds) {
        const int nx = g.nx, ze = p.ze;
        const Lane3<TX> ln(g, p);
        float *const ce = lds + 2 * W::N;
        W w;
        w.init(nx, g.ny, p.x0, p.y0);
        Sides3<TX> sd;
        ZStrip zs;
        if (PXY) {
            sd.init(g, p, ln, c.t[0], c.t[1]);
            if (threadIdx.x < 36) ce[threadIdx.x] = kCoefC[threadIdx.x];
        }
        if (PZ) zs.init(g, p, c.t[2]);
        const float *const P = c.t[0].f;
        float *const Vp[3] = {c.V[0], c.V[1], c.V[2]};
        const float *const Rp[3] = {c.R[0], c.R[1], c.R[2]};
        const long nxy = opaque((long)nx * g.ny);
        long o = ln.at(g, p.zb), xo = 0, yo = 0;
        float V[3][R3], R[3][R3], sx[R3], sy[R3], wv[W::K], q[R3][2 * H + 2], qn[2][R3];
        ZVals zv;
        auto window = [&](int z, int k) RSG_INLINE {
            w.fetch(wv, P, opaque(o + k * nxy), nx, z < ze);
        };
        auto own = [&](int z, int k) RSG_INLINE {
            const bool live = z < ze;
            const long at = opaque(o + k * nxy);
#pragma unroll
            for (int a = 0; a < 3; a++) {
                ln.ld(Vp[a], at, V[a], live);
                ln.ld(Rp[a], at, R[a], live);
            }
            if (PXY) {
                sd.load_x(sx, xo + (live ? k * sd.xstep : 0));
                sd.load_y(sy, yo + (live ? k * sd.ystep : 0));
            }
            if (PZ) zload(zv, zs, g, z, ln, live);
        };
        ln.fill(P, p.zb + 1 - H, g, q, qn);
        window(p.zb, 0);
        own(p.zb, 0);
        auto top = [&](int z) RSG_INLINE {
            o = opaque(o);
            shift2(q, qn);
            ln.ld(P, o + (H + 3) * nxy, qn[0], z + 2 < ze && z + 3 + H < g.nz);
            ln.ld(P, o + (H + 4) * nxy, qn[1], z + 3 < ze && z + 4 + H < g.nz);
        };
        auto body = [&](auto S, int z) RSG_INLINE {
            constexpr int sb = decltype(S)::value;
            float *const b = lds + sb * W::N;
            w.store(wv, b);
            __syncthreads();
            window(z + 1, 1);
            const int kz = PZ ? kfw(z, g.nz, H) : H;
            const float *const cz = g.cz[kz];
            const bool zin = PZ && zs.in(z);
#pragma unroll
            for (int r = 0; r < R3; r++) {
                const float *t = b + (ln.ty * R3 + r + H) * W::LD + ln.tx + H;
                float m = g.dt * R[0][r], d = dfw<ORDER>(t, 1, g.c[0]);
                if (PXY && sd.ex)
                    if (sd.kx != H) d = dfw_edge(t, 1, sd.kx, g.inv[0], ce);
                V[0][r] += m * d;
                if (PXY && sd.px) {
                    sx[r] = fmaf(sd.x.A, d, sd.x.B * sx[r]);
                    strip3(V[0][r], m, d, sd.inx[r], sd.x.C, sx[r]);
                }
                m = g.dt * R[1][r];
                d = dfw<ORDER>(t, W::LD, g.c[1]);
                if (PXY && sd.ey)
                    if (sd.ky[r] != H) d = dfw_edge(t, W::LD, sd.ky[r], g.inv[1], ce);
                V[1][r] += m * d;
                if (PXY && sd.py) {
                    sy[r] = fmaf(sd.y[r].A, d, sd.y[r].B * sy[r]);
                    strip3(V[1][r], m, d, sd.y[r].in, sd.y[r].C, sy[r]);
                }
                m = g.dt * R[2][r];
                d = PZ ? dq_edge<H, sb>(q[r], cz, kz) : dq<H, sb>(q[r], g.c[2]);
                V[2][r] += m * d;
                if (PZ && zin) {
                    zv.v[r] = fmaf(zv.A, d, zv.B * zv.v[r]);
                    strip3(V[2][r], m, d, true, zv.C, zv.v[r]);
                }
            }
#pragma unroll
            for (int a = 0; a < 3; a++) ln.st(Vp[a], o, V[a]);
            if (PZ) zstore(zv, zs, g, z, ln);
            if (PXY && sd.px) sd.store_x(sx, xo);
            if (PXY && sd.py) sd.store_y(sy, yo);
            own(z + 1, 1);
            o += nxy;
            if (PXY) {
                xo += sd.xstep;
                yo += sd.ystep;
            }
        };
        march3(p.zb, ze, top, body);
    }

    static __device__ __forceinline__ void run(const G3 &g, const Grad3Args &c, const Pos3 &p, float *lds) {
        if (tile_pxy<TX>(g, p)) {
            if (p.zone != 1)
                march<true, true>(g, c, p, lds);
            else
                march<true, false>(g, c, p, lds);
        } else {
            if (p.zone != 1)
                march<false, true>(g, c, p, lds);
            else
                march<false, false>(g, c, p, lds);
        }
    }
};

// ---------------------------------------------------------------------------
// Host side
// ---------------------------------------------------------------------------

static G3 make_g3(const rsg_grid *g, const float *tab, int order) {
    G3 k{};
    k.nx = g->nx;
    k.ny = g->ny;
    k.nz = g->nz;
    k.lpml = g->lpml;
    k.fs = g->fs;
    k.order = order;
    k.dt = g->dt;
    const float d[3] = {g->dx, g->dy, g->dz};
    for (int a = 0; a < 3; a++) {
        k.inv[a] = 1.0f / d[a];
        const Coefs cf = scaled_coefs(d[a]);
        for (int i = 0; i < order; i++) k.c[a][i] = cf.c[cind(order) + i];
        if (a == 2)
            for (int o = 1; o <= order; o++)
                for (int i = 0; i < o; i++) k.cz[o][i] = cf.c[cind(o) + i];
    }
    k.tab = tab;
    return k;
}

// Launch grid of ncomp components, and the tile order.
static unsigned layout3(G3 &k, int ncomp, int first = 0) {
    return layout_tiles3(k.t, k.nx, k.ny, k.nz, k.lpml, k.order, ncomp, first, tuning().zc3d, tuning().xcd3d);
}

#define RSG3_ORDER_CASES(LAUNCH, X, ORDER) \
    switch (ORDER) {                        \
    case 1: LAUNCH(X, 1); break;            \
    case 2: LAUNCH(X, 2); break;            \
    case 3: LAUNCH(X, 3); break;            \
    case 4: LAUNCH(X, 4); break;            \
    case 5: LAUNCH(X, 5); break;            \
    case 6: LAUNCH(X, 6); break;            \
    case 7: LAUNCH(X, 7); break;            \
    default: LAUNCH(X, 8); break;           \
    }
#define RSG3_DISPATCH(K, LAUNCH)                    \
    if ((K).t.tx == 64) {                           \
        RSG3_ORDER_CASES(LAUNCH, 64, (K).order)     \
    } else {                                        \
        RSG3_ORDER_CASES(LAUNCH, 32, (K).order)     \
    }

}  // namespace rsg
