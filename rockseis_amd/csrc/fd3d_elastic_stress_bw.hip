// WavesElastic3D::backwardstepStress (waves.cpp:3715-4103).
#include "rsg_e3d.h"

int rsg::e3d_stress_backward(const rsg_grid *g, const rsg_state_e3d *s, hipStream_t st) { return launch_stress<true>(g, s, st); }
