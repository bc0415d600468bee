// osbl_line.h -- one RK stage of the 1-D Euler equations (characteristic
// WENO/TENO flux, zeroth-order extrapolation ends) on part of a line, by one
// wave: shared by the ensembles (osbl_batch.hip) and the 1-D blocks.
//
// The lanes of a wave take 64 consecutive interfaces, whose 69 points are
// staged in LDS with their constituent relations; a cell's flux difference is
// its lane's flux minus that of the lane below.  Zeroth-order extrapolation
// (extrapolation.py:29-58) gives the boundary point and its halos the value
// of the first point inside, so a point is read at its index clamped to
// [1, n-2] and no boundary pass runs between the stages.
#pragma once

#include "osbl_device.h"

namespace osbl {

constexpr int LINE_PTS = 64 + 5;  // points staged per 64 interfaces
constexpr int LINE_CELLS = 63;    // cells one such chunk completes
constexpr int LINE_NF = 9;        // doubles per staged point: q, u, p, a, sqrt(rho), sqrt(rho) H; odd, no bank conflicts

__device__ __forceinline__ void line_wave_sync() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// Cells [s0, s1) of a line of n points.  ld(x, q) reads the state at the
// (clamped) point x, rk_in(x, qo) the RK register of cell x ahead of the flux,
// put(x, qn, qo) stores the new state and register.  MODE as k_update.
template <int CONV, int AVG, int MODE, class Ld, class RkIn, class Put>
__device__ __forceinline__ void line_segment(double (*S)[LINE_NF], int lane, int n, int s0, int s1, double dt,
                                             double inv_dx, const Phys& ph, double cA, double cB, bool first,
                                             Ld&& ld, RkIn&& rk_in, Put&& put) {
  constexpr bool ROE = AVG == OSBL_AVG_ROE;
  if (s0 >= s1) return;
  auto point = [&](int x, double (&q)[3]) { ld(max(1, min(x, n - 2)), q); };
  auto stage = [&](int slot, const double (&q)[3], bool on) {
    Pt<1> p;
#pragma unroll
    for (int m = 0; m < 3; ++m) p.q[m] = q[m];
    finish_pt<1>(p, ph);
    double sq = 0.0, h = 0.0;
    if constexpr (ROE) roe_factors<1>(p, sq, h);
    if (on) {
#pragma unroll
      for (int m = 0; m < 3; ++m) S[slot][m] = p.q[m];
      S[slot][3] = p.u[0];
      S[slot][4] = p.p;
      S[slot][5] = p.a;
      S[slot][6] = sq;
      S[slot][7] = h;
    }
  };
  // slot s holds point base - 2 + s, lane l the interface base + l + 1/2
  int base = s0 - 1;
  double nq[3], prev[3] = {0.0, 0.0, 0.0};
  {
    double q5[3];
    point(base - 2 + lane, q5);
    point(base + 3 + lane, nq);
    stage(lane, q5, lane < 5);
  }
  for (;;) {
    const int I = base + lane;
    const bool own = I >= s0 && I < s1, more = base + 64 < s1;
    stage(5 + lane, nq, true);
    line_wave_sync();
    // the next points and the cell's RK register, in flight during the flux
    double qo[3] = {0.0, 0.0, 0.0};
    if (own && !(MODE == 0 ? first : cA == 0.0)) rk_in(I, qo);
    if (more) point(base + 67 + lane, nq);
    double fh[3];
    {
      const LdsPoints<1, LINE_NF> w{S[lane]};
      RoeF rf{};
      if constexpr (ROE) rf = RoeF{S[lane + 2][6], S[lane + 2][7], S[lane + 3][6], S[lane + 3][7]};
      char_flux_w<1, 0, CONV, AVG, true>(w, ph, fh, ph.teno_ct, rf);
    }
    double qn[3];
#pragma unroll
    for (int m = 0; m < 3; ++m) {
      const double up = __shfl_up(fh[m], 1);
      const double r = ((lane == 0 ? prev[m] : up) - fh[m]) * inv_dx;
      const double q = S[lane + 2][m];
      if constexpr (MODE == 0) {
        const double o = first ? q : qo[m];
        qn[m] = __fma_rn(dt * cA, r, o);
        qo[m] = __fma_rn(dt * cB, r, o);
      } else {
        qo[m] = __fma_rn(dt, r, __dmul_rn(cA, qo[m]));
        qn[m] = __fma_rn(cB, qo[m], q);
      }
    }
    if (own) put(I, qn, qo);
    if (!more) return;
#pragma unroll
    for (int m = 0; m < 3; ++m) prev[m] = __shfl(fh[m], 63);
    line_wave_sync();
    if (lane < 5) {
#pragma unroll
      for (int e = 0; e < 8; ++e) S[lane][e] = S[64 + lane][e];
    }
    line_wave_sync();  // the next points go into slots 64..68
    base += 64;
  }
}

}  // namespace osbl
