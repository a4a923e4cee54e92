// Per-pair work of the expansion and of its adjoint, one wavefront per centre
// (or a few for small batches), for spline radial functions and l_max <= 9.
#pragma once

#include <hip/hip_runtime.h>

#include "radial.hh"
#include "soap_kernels.hh"

namespace rgpu {

// whether the kernels below apply to these hypers
bool pair_kernels_apply(const RadialDev& rad);

// Pair phase of the adjoint: from dL/dc [n][S][(L+1)^2][N] (T) of each
// centre, the pair and centre forces of dL/dr (pv.pair_force,
// pv.centre_force; launch_force_gather sums them per atom) and the per-centre
// virials centre_virial[n_centres][6] (sum over the centre's pairs of r_ji (x)
// dL/dr_j, Voigt xx,yy,zz,yz,xz,xy, not divided by the volume).  dc has
// kPairSlack readable values past its last row.
constexpr int kPairSlack = 32;
template <class T>
void launch_pair_forces(const RadialDev& rad, int S, const PairView& pv, const T* dc, double* centre_virial,
                        hipStream_t stream);

// Expansion c[n][S][N][(L+1)^2] and key masks, as launch_expansion
template <class T>
void launch_expansion_wave(const RadialDev& rad, int S, const PairView& pv, T* c, unsigned long long* keymask,
                           hipStream_t stream);

}  // namespace rgpu
