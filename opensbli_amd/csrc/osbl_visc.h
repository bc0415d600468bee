// osbl_visc.h -- the viscous residual of a point from its transformed
// derivatives, shared by the per-point and the tiled kernels.
#pragma once

#include "osbl_device.h"

namespace osbl {

// The viscous residual from the transformed derivatives at a point (D_j u_m,
// D_a D_b u_m, D_jj T, D_j T, D_j mu).
template <int ND>
__device__ __forceinline__ void viscous_assemble(double mu, const double um_[3], const double (&DU)[ND][ND],
                                                 const double (&DD)[ND][ND][ND], const double (&D2T)[ND],
                                                 const double (&DT)[ND], const double (&DMU)[ND], const Phys& ph,
                                                 bool suth, double vr[ND + 2]) {
  double divu = 0.0;
#pragma unroll
  for (int k = 0; k < ND; ++k) divu += DU[k][k];
  double energy = 0.0;
#pragma unroll
  for (int j = 0; j < ND; ++j) {
    if (suth) energy += ph.cq * (mu * D2T[j] + DMU[j] * DT[j]);
    else energy += ph.cq * D2T[j];
  }
#pragma unroll
  for (int m = 0; m < ND; ++m) {
    const double um = um_[m];
    double visc = 0.0;
#pragma unroll
    for (int j = 0; j < ND; ++j) {
      double tt = DD[m][j][j] + DD[j][m][j];
      if (j == m) {
        double sk = 0.0;
#pragma unroll
        for (int k = 0; k < ND; ++k) sk += DD[k][m][k];
        tt -= (2.0 / 3.0) * sk;
      }
      const double sr = DU[m][j] + DU[j][m] - (j == m ? (2.0 / 3.0) * divu : 0.0);
      double dtau, tau;
      if (suth) {
        dtau = ph.inv_re * mu * tt + ph.inv_re * DMU[j] * sr;
        tau = ph.inv_re * mu * sr;
      } else {
        dtau = ph.inv_re * tt;
        tau = ph.inv_re * sr;
      }
      visc += dtau;
      energy += DU[m][j] * tau + um * dtau;
    }
    vr[1 + m] += visc;
  }
  vr[ND + 1] += energy;
}

}  // namespace osbl
