// 3D acoustic staggered-grid half steps for gfx950 (WavesAcoustic3D,
// waves.cpp:710-996): fused velocity and stress updates with the CFS-PML
// memory variables of all six faces, on the z march of rsg_fd3d.h.
#include "rsg_fd3d.h"

namespace rsg {

// The queue, three fields and three moduli are a few registers too many for
// four waves a SIMD from order 7 on (four spill 20 and 60 bytes a lane).  us at
// order 8, three waves against four with their spills: 120 x 110 x 100 22.9, 25.0,
// 140 x 130 x 120 36.3, 38.2, 160 x 150 x 140 46.0, 41.8, 200 x 190 x 180 76.8, 70.0,
// 320 x 300 x 280 251, 250, 440^3 822, 822.
template <int TX, int ORDER>
__global__ __launch_bounds__(B3) __attribute__((amdgpu_waves_per_eu((ORDER) >= 7 ? 3 : 4, 8))) void a3d_velocity_kernel(const G3 g, const Grad3Args a) {
    using K = Grad3<TX, ORDER>;
    __shared__ float lds[K::LDS];
    Pos3 p;
    if (tile3_of<TX>(g.t, p)) K::run(g, a, p, lds);
}

template <int TX, int ORDER>
__global__ RSG3_BOUNDS void a3d_stress_kernel(const G3 g, const Comp3 c) {
    using K = Div3<TX, ORDER, true, true, true, 1, false>;
    __shared__ float lds[K::LDS];
    Pos3 p;
    if (tile3_of<TX>(g.t, p)) K::run(g, c, p, lds);
}

static int check_grid3d(const rsg_grid *g, const rsg_state *s) {
    if (!g || !s) return fail(RSG_EINVAL, "null grid/state");
    if (g->order < 1 || g->order > 8) return fail(RSG_EINVAL, "order must be 1..8");
    if (g->lpml < 1 || g->nx <= 2 * g->lpml || g->ny <= 2 * g->lpml || g->nz <= 2 * g->lpml)
        return fail(RSG_EINVAL, "grid must exceed 2*lpml on every axis");
    if (g->nx < 2 * g->order + 2 || g->ny < 2 * g->order + 2 || g->nz < 2 * g->order + 2)
        return fail(RSG_EINVAL, "grid too small for the stencil order");
    if ((long long)g->nx * g->ny * 4 >= (1LL << 31))
        return fail(RSG_EINVAL, "3D plane larger than 2^29 cells (32-bit in-plane offsets)");
    if (!s->tab || !s->P || !s->Vx || !s->Vy || !s->Vz) return fail(RSG_EINVAL, "a3d: null array");
    return RSG_OK;
}

}  // namespace rsg

using namespace rsg;

extern "C" int rsg_a3d_forward_velocity(const rsg_grid *g, const rsg_state *s, void *stream) {
    if (int rc = check_grid3d(g, s)) return rc;
    if (!s->Rx || !s->Ry || !s->Rz) return fail(RSG_EINVAL, "a3d: null model");
    G3 k = make_g3(g, s->tab, g->order);
    const unsigned blocks = layout3(k, 1);
    const Grad3Args a{{{s->P, s->psi[RSG_A3D_P_LEFT], s->psi[RSG_A3D_P_RIGHT], 1},
                       {s->P, s->psi[RSG_A3D_P_FRONT], s->psi[RSG_A3D_P_BACK], 1},
                       {s->P, s->psi[RSG_A3D_P_TOP], s->psi[RSG_A3D_P_BOTTOM], 1}},
                      {s->Vx, s->Vy, s->Vz},
                      {s->Rx, s->Ry, s->Rz}};
#define L_(X, O) a3d_velocity_kernel<X, O><<<blocks, B3, 0, (hipStream_t)stream>>>(k, a)
    RSG3_DISPATCH(k, L_)
#undef L_
    RSG_LAUNCH_CHECK("a3d_velocity_kernel");
    return RSG_OK;
}

extern "C" int rsg_a3d_forward_stress(const rsg_grid *g, const rsg_state *s, void *stream) {
    if (int rc = check_grid3d(g, s)) return rc;
    if (!s->L) return fail(RSG_EINVAL, "a3d: null model");
    G3 k = make_g3(g, s->tab, g->order);
    k.fs = 0;  // the acoustic free surface is in the model (L is zero there)
    const unsigned blocks = layout3(k, 1);
    const Comp3 c{{{s->Vx, s->psi[RSG_A3D_VXX_LEFT], s->psi[RSG_A3D_VXX_RIGHT], 0},
                   {s->Vy, s->psi[RSG_A3D_VYY_FRONT], s->psi[RSG_A3D_VYY_BACK], 0},
                   {s->Vz, s->psi[RSG_A3D_VZZ_TOP], s->psi[RSG_A3D_VZZ_BOTTOM], 0}},
                  {s->P, nullptr, nullptr},
                  {s->L, nullptr}};
#define L_(X, O) a3d_stress_kernel<X, O><<<blocks, B3, 0, (hipStream_t)stream>>>(k, c)
    RSG3_DISPATCH(k, L_)
#undef L_
    RSG_LAUNCH_CHECK("a3d_stress_kernel");
    return RSG_OK;
}
