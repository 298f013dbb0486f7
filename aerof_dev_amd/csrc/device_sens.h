// device_sens.h -- templated pieces of the residual shared by its derivative
// passes (adjoint.hip: reverse mode, tangent.hip: forward mode).  With
// T = Dual face_flux carries one directional derivative.
#pragma once
#include <hip/hip_runtime.h>

#include "context.h"
#include "device_dual.h"

namespace aerofx {

// The vertices (c, d) opposite to a tet's edge (a, b), in the order that makes
// the tet's part of the median dual face, from a to b,
// (c - d) x (a + b - c - d) / 24 (ElemTet edge and face tables,
// ElemTetCore.C:19-21)
constexpr int kOpp[6][2] = {{3, 2}, {1, 3}, {2, 1}, {3, 0}, {0, 2}, {1, 0}};

// LSQ weights W(dx; L) (computeLocalWeightsLeastSquares, SubDomain.C:137-159)
// in the gradient pass's operation order; linear in dx: W = M^-1 dx with the
// moments M.
__device__ __forceinline__ void lsq_weights(const double L[6], double dx0, double dx1, double dx2, double w[3]) {
  const double or11 = L[0], or22 = L[1], or33 = L[2], r12or11 = L[3], r23or22 = L[4], psi = L[5];
  const double alpha1 = dx0 * or11 * or11;
  const double alpha2 = (dx1 - r12or11 * dx0) * or22 * or22;
  const double alpha3 = (dx2 - r23or22 * dx1 + psi * dx0) * or33 * or33;
  w[0] = alpha1 - r12or11 * alpha2 + psi * alpha3;
  w[1] = alpha2 - r23or22 * alpha3;
  w[2] = alpha3;
}

// boundary flux of one face node; nv = (1/3) face normal
template <class T>
__device__ __forceinline__ void face_flux(const FluxConsts &fc, int code, const T nv[3], const T V[5], T fl[5]) {
  if (is_wall_code(code)) {
    wallflux(nv, 0.0, V, fl);
  } else {
    const double *ub = (code == AEROFX_BC_INLET || code == -AEROFX_BC_INLET) ? fc.ub_in : fc.ub_out;
    boundflux5(fc.gas, nv, 0.0, V, ub, fl);
  }
}

}  // namespace aerofx
