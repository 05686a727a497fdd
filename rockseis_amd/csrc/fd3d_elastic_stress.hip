// WavesElastic3D::forwardstepStress (waves.cpp:2861-3258).
#include "rsg_e3d.h"

int rsg::e3d_stress_forward(const rsg_grid *g, const rsg_state_e3d *s, hipStream_t st) { return launch_stress<false>(g, s, st); }
