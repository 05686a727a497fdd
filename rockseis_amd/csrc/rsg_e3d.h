// The elastic 3D half steps on the z march: component descriptions and the
// stress kernels.  The forward and the adjoint-state stress kernels are
// compiled from this header in two files, so that they build in parallel.
#pragma once
#include "rsg_fd3d.h"

namespace rsg {

int e3d_stress_forward(const rsg_grid *g, const rsg_state_e3d *s, hipStream_t st);
int e3d_stress_backward(const rsg_grid *g, const rsg_state_e3d *s, hipStream_t st);

// The components of a half step.
struct Comps3 {
    Comp3 c[4];
};

inline Term3 term(const float *f, const rsg_state_e3d *s, int slot, int fw) {
    return Term3{f, s->psi[slot], s->psi[slot + 1], fw};
}
// The elastic steps take planes of any size (the acoustic ones up to 2^29
// cells, whose offsets always fit): those whose windows reach past 32-bit
// offsets, a row's cells times the window's rows (8 + 2 order, or ny) from 2^30
// on, are left to no kernel.  Rows that long are tiled 64 cells by 8 rows.
inline int check_tiles3(const rsg_grid *g) {
    if (!tiles_fit(g->nx, g->ny, R3 * B3 / 64, std::min(std::max(g->order, 1), 8)))
        return fail(RSG_EINVAL, "e3d: rows too long for 32-bit offsets (nx min(ny, 8 + 2 order) >= 2^30)");
    return RSG_OK;
}
inline G3 make_g3e(const rsg_grid *g, const rsg_state_e3d *s) {
    return make_g3(g, s->tab, std::min(std::max(g->order, 1), 8));
}

// forwardstepStress (waves.cpp:2861-3258), or with BW backwardstepStress
// (waves.cpp:3715-4103): the same terms and strips with unit moduli.
// Component 0: Sxx, Syy, Szz; 1: Sxz; 2: Syz; 3: Sxy.  All blocks of component
// 0 run before the others: side by side on one compute unit their marches and
// the shears' push each other out of the instruction cache (200 x 190 x 180,
// order 8: 279 us mixed, 215 in this order, 252 as four launches; 70 x 60 x 50,
// order 4: 21, 16, 44).  The three shears side by side cost nothing and share
// their inputs.  Two marches a component (FULL off) keep the kernel's eight
// in registers; twelve put the queue in scratch memory.
template <int TX, int ORDER, bool BW>
__global__ RSG3_BOUNDS void e3d_stress_kernel(const G3 g, const Comps3 a) {
    using KN = Div3<TX, ORDER, true, true, true, 3, BW, false>;
    using KXZ = Div3<TX, ORDER, true, false, true, 1, BW, false>;
    using KYZ = Div3<TX, ORDER, false, true, true, 1, BW, false>;
    using KXY = Div3<TX, ORDER, true, true, false, 1, BW, false>;
    __shared__ float lds[KN::LDS];  // both windows: no component needs more
    Pos3 p;
    if (!tile3_of<TX>(g.t, p)) return;
    if (p.comp == 0)
        KN::run(g, a.c[0], p, lds);
    else if (p.comp == 1)
        KXZ::run(g, a.c[1], p, lds);
    else if (p.comp == 2)
        KYZ::run(g, a.c[2], p, lds);
    else
        KXY::run(g, a.c[3], p, lds);
}

template <bool BW>
int launch_stress(const rsg_grid *g, const rsg_state_e3d *s, hipStream_t st) {
    G3 k = make_g3e(g, s);
    const Comps3 a{{{{term(s->Vx, s, RSG_E3D_VXX_LEFT, 0), term(s->Vy, s, RSG_E3D_VYY_FRONT, 0), term(s->Vz, s, RSG_E3D_VZZ_TOP, 0)},
                     {s->Sxx, s->Syy, s->Szz},
                     {s->L, s->L2M}},
                    {{term(s->Vz, s, RSG_E3D_VZX_LEFT, 1), Term3{}, term(s->Vx, s, RSG_E3D_VXZ_TOP, 1)},
                     {s->Sxz, nullptr, nullptr},
                     {s->Mxz, nullptr}},
                    {{Term3{}, term(s->Vz, s, RSG_E3D_VZY_FRONT, 1), term(s->Vy, s, RSG_E3D_VYZ_TOP, 1)},
                     {s->Syz, nullptr, nullptr},
                     {s->Myz, nullptr}},
                    {{term(s->Vy, s, RSG_E3D_VYX_LEFT, 1), term(s->Vx, s, RSG_E3D_VXY_FRONT, 1), Term3{}},
                     {s->Sxy, nullptr, nullptr},
                     {s->Mxy, nullptr}}}};
    const unsigned blocks = layout3(k, 4, 1);
#define L_(X, O) e3d_stress_kernel<X, O, BW><<<blocks, B3, 0, st>>>(k, a)
    RSG3_DISPATCH(k, L_)
#undef L_
    RSG_LAUNCH_CHECK("e3d_stress_kernel");
    return RSG_OK;
}

}  // namespace rsg
