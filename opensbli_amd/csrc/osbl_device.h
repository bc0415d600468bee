// osbl_device.h -- device-side building blocks of the OpenSBLI RHS on gfx950:
// grid indexing, constituent relations, Roe averaging, the Euler
// eigensystems, WENO5-JS/Z and TENO5/6 reconstructions.
//
// All arithmetic is FP64.  Formulas follow the reference's symbolic
// definitions; where an expression is rearranged to save divisions the
// rearrangement is algebraically exact and noted at the function.
#pragma once

#include <hip/hip_runtime.h>

#include <type_traits>
#include <utility>

#include "../../include/opensbli_amd.h"

namespace osbl {

// ---------------------------------------------------------------------------
// Storage: one array per field, x fastest.  The interior x range starts at a
// 128-byte boundary (offset OX doubles into each row), y and z carry `h`
// halo points.  Absent dimensions have n = 1 and no halo.
// ---------------------------------------------------------------------------
constexpr int OX = 16;

struct Grid {
  int nd;
  int n[3];
  int h[3];
  int pitch;  // doubles per row
  int rows;   // rows per plane
  int planes;
  int plane;  // doubles per plane
  long long fs;  // doubles per field (padded)
  int periodic_x;  // x faces periodic
  __host__ __device__ __forceinline__ int idx(int i, int j, int k) const {
    return (i + OX) + pitch * ((j + h[1]) + rows * (k + h[2]));
  }
  __host__ __device__ __forceinline__ int stride(int d) const { return d == 0 ? 1 : (d == 1 ? pitch : plane); }
};

// Segment length of a sliding-window sweep: `seg` cells per thread, halved
// (down to `lo`) while the launch would have fewer than 2^17 threads, so small
// blocks (2-D, 1-D lines) still give the GPU a few thousand waves.
__host__ __forceinline__ int fit_segment(long long lines, int n, int seg, int lo) {
  while (seg > lo && lines * ((n + seg - 1) / seg) < (1LL << 17)) seg /= 2;
  return seg;
}

// Workgroups are dispatched to the 8 XCDs round-robin by linear id.  The
// tile of a workgroup: linear ids are renumbered so that each XCD gets one
// contiguous range of tiles (x fastest, then y, then z) and tiles sharing
// halo rows sit behind one L2.  A bijection when the tile count is a
// multiple of 8, the identity otherwise.
__device__ __forceinline__ void xcd_tile(int& bx, int& by, int& bz) {
  const int nx = gridDim.x, ny = gridDim.y, total = nx * ny * gridDim.z;
  const int lin = blockIdx.x + nx * (blockIdx.y + ny * blockIdx.z);
  const int logical = (total % 8 == 0) ? (lin % 8) * (total / 8) + lin / 8 : lin;
  bx = logical % nx;
  by = (logical / nx) % ny;
  bz = logical / (nx * ny);
}

struct Phys {
  double gama, gm1, Minf, Re, Pr, dt, eps, teno_ct;
  double inv_delta[3];
  double inv_re, cq;  // 1/Re and 1/((gama-1) Minf^2 Pr Re)
  double suth;        // SuthT/RefT of the Sutherland law
  double teno_a1, teno_a2, sensor_eps;  // adaptive TENO cut-off and Ducros sensor constants
  double igm1;        // 1/(gama-1)
  double force[3];    // c_j of the constant body force (zero without one)
  int has_force;
  int nt;             // non-temporal hint on the residual and RK registers
};

// 10^n for an integer n by repeated products (exact for |n| <= 22)
__host__ __device__ __forceinline__ double pow10i(int n) {
  double r = 1.0;
  const int m = n < 0 ? -n : n;
  for (int i = 0; i < m; ++i) r *= 10.0;
  return n < 0 ? 1.0 / r : r;
}

// adaptive TENO cut-off from the sensor at an interface's left point
// (teno.py:430-443): C_T = 1/10^floor(a1 - a2 (1 - (1-theta)^4 (1 + 4 theta))),
// each operation rounded separately so that floor() sees the same value as a
// build without contraction
__device__ __forceinline__ double adaptive_ct(double m, const Phys& ph) {
#pragma clang fp contract(off)
  const double t = 1.0 - m;
  const double t2 = t * t;
  const double t4 = t2 * t2;
  const double q = t4 * (1.0 + 4.0 * m);
  const double beta = ph.teno_a1 - ph.teno_a2 * (1.0 - q);
  return 1.0 / pow10i((int)floor(beta));
}

// Near-boundary stencils and metric of a block with non-periodic faces
// (bc_core.py:15-16, opensblifunctions.py:523-534, metric.py:72-212).
struct Bnd {
  int mod[3][2];        // 0: central stencil; 1 + OSBL_BS_* where the face's BC replaces it
  const double* dm[3];  // D_dd of a direction stretched along itself (n[d] values), or nullptr
  const double* sd[3];  // SD_ddd = CD(D_dd, xi_d)
  const double* cw;     // closure rows (6 weights each): Carpenter first derivative rows 0-3 at 0,
                        // ReducedAccess first derivative rows 0-1 at 24, second derivative rows 0-1 at 36
};
constexpr int CW_CARP = 0, CW_RA = 24, CW_D2 = 36, CW_SIZE = 48;

// ---------------------------------------------------------------------------
// compile-time loop
// ---------------------------------------------------------------------------
template <int B, int E, class F>
__device__ __forceinline__ void sfor(F&& f) {
  if constexpr (B < E) {
    f(std::integral_constant<int, B>{});
    sfor<B + 1, E>(f);
  }
}

// ---------------------------------------------------------------------------
// Point state: conservative variables and the constituent relations
// u_i = rhou_i/rho, p = (gama-1)(rhoE - rho/2 u.u), a = (gama p/rho)^0.5
// (taylor_green_vortex.py:29-31, Sod_shock_tube.py:26-28).
// ---------------------------------------------------------------------------
template <int ND>
struct Pt {
  double q[ND + 2];
  double u[ND];
  double p, a;
};

// Loads and stores of the arrays a stage kernel touches once per cell (the
// residual and the RK registers).  On blocks whose fields exceed the
// last-level cache (Phys::nt) they carry the non-temporal hint, so that they
// stream through L2 without evicting the Q planes the stencils of
// neighbouring tiles and rows still re-read from it; on smaller blocks the
// whole working set stays cached between kernels and plain accesses keep it
// there.
__device__ __forceinline__ double ld_once(const double* p, int nt) {
  return nt ? __builtin_nontemporal_load(p) : *p;
}
__device__ __forceinline__ void st_once(double v, double* p, int nt) {
  if (nt) __builtin_nontemporal_store(v, p);
  else *p = v;
}

// Quotients and roots of positive normal operands far from the overflow range,
// from the hardware estimates (measured: v_rcp_f64 within 2^-24.4, v_rsq_f64
// within 2^-24.2), in about half the instructions of the IEEE sequences, which
// must also handle scaling and special operands.
//
// a/b and sqrt(x): one Newton-Raphson step, the result then corrected once by
// its residual (Markstein's method; for the root the residual times the
// estimate itself is enough): 0.50 ulp.  1/b: the first two terms of the series
// in the estimate's error e (2^-24, so e^3 is below rounding) in one step,
// 1/(1-e) = 1 + e + e^2, also 0.50 ulp.
__device__ __forceinline__ double quot_pos(double a, double b) {
  double r = __builtin_amdgcn_rcp(b);
  r = __fma_rn(__fma_rn(-b, r, 1.0), r, r);
  const double q = a * r;
  return __fma_rn(__fma_rn(-b, q, a), r, q);
}
__device__ __forceinline__ double recip_pos(double b) {
  const double r = __builtin_amdgcn_rcp(b);
  const double e = __fma_rn(-b, r, 1.0);
  return __fma_rn(r, __fma_rn(e, e, e), r);
}
__device__ __forceinline__ double sqrt_pos(double x) {
  const double r = __builtin_amdgcn_rsq(x);
  const double h = 0.5 * r, y = x * r;
  const double z = __fma_rn(y, __fma_rn(-h, y, 0.5), y);
  return __fma_rn(h, __fma_rn(-z, z, x), z);
}
// max(m, |x|) in one instruction (fmax first quiets its operands)
__device__ __forceinline__ double max_abs(double m, double x) {
  double r;
  asm("v_max_f64 %0, %1, |%2|" : "=v"(r) : "v"(m), "v"(x));
  return r;
}

// Every kernel and every place in one takes a point's values from here, so they
// are the same bits in a sweep's prologue and in its loop, and a direction along
// which the state is uniform keeps exactly zero flux differences.  (The
// compiler may contract the operations; it does so alike wherever they are
// inlined.)
template <int ND>
__device__ __forceinline__ void finish_pt(Pt<ND>& s, const Phys& ph) {
  const double ir = recip_pos(s.q[0]);
  double ke = 0.0;
#pragma unroll
  for (int m = 0; m < ND; ++m) {
    s.u[m] = __dmul_rn(s.q[1 + m], ir);
    ke = __dadd_rn(ke, __dmul_rn(s.u[m], s.u[m]));
  }
  s.p = __dmul_rn(ph.gm1, __dsub_rn(s.q[ND + 1], __dmul_rn(__dmul_rn(0.5, s.q[0]), ke)));
  s.a = sqrt_pos(__dmul_rn(__dmul_rn(ph.gama, s.p), ir));
}

// raw conservative variables of one point
template <int ND>
__device__ __forceinline__ void fetch_q(double (&q)[ND + 2], const double* __restrict__ Q, long long fs, int off) {
#pragma unroll
  for (int m = 0; m < ND + 2; ++m) q[m] = Q[m * fs + off];
}

template <int ND>
__device__ __forceinline__ void load_pt(Pt<ND>& s, const double* __restrict__ Q, long long fs, int off,
                                         const Phys& ph) {
  fetch_q<ND>(s.q, Q, fs, off);
  finish_pt<ND>(s, ph);
}

// ---------------------------------------------------------------------------
// Interface state between points i and i+1 (the averaged symbols of the
// eigensystem).  Roe: averaging.py:70-114.  Simple: averaging.py:38-59.
// ---------------------------------------------------------------------------
template <int ND, class T = double>
struct AvgT {
  T rho, a, u[ND];
  T ia, ir;           // 1/a, 1/rho (inv_AVG_a, inv_AVG_rho, shock_capturing.py:319-331)
  T phi;              // (gama-1)|u|^2/2
  T alpha, bta;       // rho/(a sqrt2), 1/(rho a sqrt2)
  T Hh;               // a^2/(gama-1) + |u|^2/2  (1-D eigensystem)
};
template <int ND>
using Avg = AvgT<ND, double>;

// the derived symbols of an averaged state (rho, a, u)
template <int ND, class T>
__device__ __forceinline__ void finish_avg(AvgT<ND, T>& v, const Phys& ph) {
  T uu = v.u[0] * v.u[0];
#pragma unroll
  for (int m = 1; m < ND; ++m) uu = uu + v.u[m] * v.u[m];
  if constexpr (std::is_same_v<T, double>) {
    // 1/a and 1/rho from one division
    const double t = recip_pos(v.a * v.rho);
    v.ia = v.rho * t;
    v.ir = v.a * t;
  } else {
    // dual numbers (the adjoint's tangents): two plain reciprocals are cheaper
    v.ia = 1.0 / v.a;
    v.ir = 1.0 / v.rho;
  }
  v.phi = ph.gm1 * 0.5 * uu;
  constexpr double RS2 = 0.70710678118654752440;  // 1/sqrt(2.0)
  v.alpha = v.rho * v.ia * RS2;
  v.bta = v.ir * v.ia * RS2;
  v.Hh = v.a * v.a * ph.igm1 + 0.5 * uu;
}

// the per-point factors of the Roe average: sqrt(rho) and
// sqrt(rho) H = (rhoE + p)/sqrt(rho).  Sweeps that visit every point once
// compute them once per point and pass them in (RoeF); the result is the same.
struct RoeF {
  double sL, hL, sR, hR;
};
template <int ND>
__device__ __forceinline__ void roe_factors(const Pt<ND>& P, double& sq, double& h) {
  sq = sqrt_pos(P.q[0]);
  h = (P.q[ND + 1] + P.p) * quot_pos(sq, P.q[0]);
}

template <int ND>
__device__ __forceinline__ void roe_state(Avg<ND>& v, const Pt<ND>& L, const Pt<ND>& R, const RoeF& f,
                                          const Phys& ph) {
  const double inv = recip_pos(f.sR + f.sL);
  v.rho = f.sL * f.sR;  // sqrt(rho_L rho_R)
  double ke = 0.0;
#pragma unroll
  for (int m = 0; m < ND; ++m) {
    v.u[m] = (f.sL * L.u[m] + f.sR * R.u[m]) * inv;
    ke += v.u[m] * v.u[m];
  }
  const double hh = (f.hL + f.hR) * inv;
  v.a = sqrt_pos(ph.gm1 * (hh - 0.5 * ke));
}

template <int ND, int AVG>
__device__ __forceinline__ void interface_state(Avg<ND>& v, const Pt<ND>& L, const Pt<ND>& R, const Phys& ph) {
  if constexpr (AVG == OSBL_AVG_ROE) {
    RoeF f;
    roe_factors<ND>(L, f.sL, f.hL);
    roe_factors<ND>(R, f.sR, f.hR);
    roe_state<ND>(v, L, R, f, ph);
  } else {
    v.rho = 0.5 * (L.q[0] + R.q[0]);
#pragma unroll
    for (int m = 0; m < ND; ++m) v.u[m] = 0.5 * (L.u[m] + R.u[m]);
    v.a = 0.5 * (L.a + R.a);
  }
  finish_avg<ND>(v, ph);
}

// ---------------------------------------------------------------------------
// Left/right eigenvectors of the Euler flux Jacobian for a Cartesian
// direction D (unit normal k = e_D), euler_eigensystem.py:57-135.  Field
// order follows the reference: 3-D (U,U,U,U+a,U-a), 2-D (U,U,U+a,U-a),
// 1-D (u-a,u,u+a).  In 3-D the rows k != D are the two shear waves whose
// non-zero entries sit at component c = 3-D-k with sign eps(D,k,c); this is
// the reference's k_t algebra with k_t = e_D substituted.
// ---------------------------------------------------------------------------
__host__ __device__ constexpr int lc3(int D, int k) { return 3 - D - k; }
__host__ __device__ constexpr int eps3(int a, int b, int c) {
  return (a == 0 && b == 1 && c == 2) || (a == 1 && b == 2 && c == 0) || (a == 2 && b == 0 && c == 1) ? 1 : -1;
}

// bit m set when L[k][m] is structurally non-zero
template <int ND, int D, int K>
__host__ __device__ constexpr unsigned lmask() {
  if constexpr (ND == 3) {
    if constexpr (K < 3 && K != D) return 1u | (1u << (1 + lc3(D, K)));
    else return 0x1Fu;
  } else if constexpr (ND == 2) {
    if constexpr (K == 1) return 1u | (1u << (1 + (1 - D)));
    else return 0xFu;
  } else {
    return 0x7u;
  }
}
template <int ND, int D, int K>
__host__ __device__ constexpr unsigned rmask() {
  if constexpr (ND == 3) {
    if constexpr (K < 3 && K != D) return (1u << (1 + lc3(D, K))) | (1u << 4);
    else return 0x1Fu;
  } else if constexpr (ND == 2) {
    if constexpr (K == 1) return (1u << (1 + (1 - D))) | (1u << 3);
    else return 0xFu;
  } else {
    return 0x7u;
  }
}

// row K of the left eigenvector matrix (T: double, or a dual number type for
// the derivatives with respect to the averaged state)
template <int ND, int D, int K, class T = double>
__device__ __forceinline__ void lrow(const AvgT<ND, T>& v, const Phys& ph, T l[ND + 2]) {
  const double gm1 = ph.gm1;
  if constexpr (ND == 3) {
    const T ia2 = v.ia * v.ia;
    if constexpr (K == D) {
      l[0] = 1.0 - v.phi * ia2;
      l[1] = gm1 * v.u[0] * ia2;
      l[2] = gm1 * v.u[1] * ia2;
      l[3] = gm1 * v.u[2] * ia2;
      l[4] = -gm1 * ia2;
    } else if constexpr (K < 3) {
      constexpr int c = lc3(D, K);
      constexpr double s = (double)eps3(D, K, c);
      l[0] = -s * v.u[c] * v.ir;
      l[1 + c] = s * v.ir;
    } else {
      constexpr double sg = (K == 3) ? 1.0 : -1.0;
      const T th = v.u[D];
      l[0] = v.bta * (v.phi - sg * th * v.a);
#pragma unroll
      for (int m = 0; m < 3; ++m) {
        if (m == D) l[1 + m] = -v.bta * (gm1 * v.u[m] - sg * v.a);
        else l[1 + m] = -v.bta * (gm1 * v.u[m]);
      }
      l[4] = v.bta * gm1;
    }
  } else if constexpr (ND == 2) {
    const T ia2 = v.ia * v.ia;
    if constexpr (K == 0) {
      l[0] = 1.0 - v.phi * ia2;
      l[1] = gm1 * v.u[0] * ia2;
      l[2] = gm1 * v.u[1] * ia2;
      l[3] = -gm1 * ia2;
    } else if constexpr (K == 1) {
      constexpr int c = 1 - D;
      constexpr double s = (D == 0) ? -1.0 : 1.0;
      l[0] = -s * v.u[c] * v.ir;
      l[1 + c] = s * v.ir;
    } else {
      constexpr double sg = (K == 2) ? 1.0 : -1.0;
      const T th = v.u[D];
      l[0] = v.bta * (v.phi - sg * v.a * th);
#pragma unroll
      for (int m = 0; m < 2; ++m) {
        if (m == D) l[1 + m] = -v.bta * (gm1 * v.u[m] - sg * v.a);
        else l[1 + m] = -v.bta * (gm1 * v.u[m]);
      }
      l[3] = v.bta * gm1;
    }
  } else {
    const T u = v.u[0], a = v.a, Hh = v.Hh;
    const T den = 2.0 * Hh - u * u;
    const T iden = 1.0 / den;
    if constexpr (K == 0) {
      l[0] = u * (2.0 * Hh + a * u - u * u) * v.ia * 0.5 * iden;
      l[1] = (-Hh - a * u + 0.5 * u * u) * v.ia * iden;
      l[2] = iden;
    } else if constexpr (K == 1) {
      l[0] = 2.0 * (Hh - u * u) * iden;
      l[1] = 2.0 * u * iden;
      l[2] = -2.0 * iden;
    } else {
      l[0] = u * (-2.0 * Hh + a * u + u * u) * v.ia * 0.5 * iden;
      l[1] = (Hh - a * u - 0.5 * u * u) * v.ia * iden;
      l[2] = iden;
    }
  }
}

// column K of the right eigenvector matrix
template <int ND, int D, int K, class T = double>
__device__ __forceinline__ void rcol(const AvgT<ND, T>& v, const Phys& ph, T r[ND + 2]) {
  const double igm1 = ph.igm1;
  if constexpr (ND == 3) {
    if constexpr (K == D) {
      r[0] = 1.0;
      r[1] = v.u[0];
      r[2] = v.u[1];
      r[3] = v.u[2];
      r[4] = v.phi * igm1;
    } else if constexpr (K < 3) {
      constexpr int c = lc3(D, K);
      constexpr double s = (double)eps3(D, K, c);
      r[1 + c] = s * v.rho;
      r[4] = s * v.rho * v.u[c];
    } else {
      constexpr double sg = (K == 3) ? 1.0 : -1.0;
      r[0] = v.alpha;
#pragma unroll
      for (int m = 0; m < 3; ++m) {
        if (m == D) r[1 + m] = v.alpha * (v.u[m] + sg * v.a);
        else r[1 + m] = v.alpha * v.u[m];
      }
      r[4] = v.alpha * ((v.phi + v.a * v.a) * igm1 + sg * v.u[D] * v.a);
    }
  } else if constexpr (ND == 2) {
    if constexpr (K == 0) {
      r[0] = 1.0;
      r[1] = v.u[0];
      r[2] = v.u[1];
      r[3] = v.phi * igm1;
    } else if constexpr (K == 1) {
      constexpr int c = 1 - D;
      constexpr double s = (D == 0) ? -1.0 : 1.0;
      r[1 + c] = s * v.rho;
      r[3] = s * v.rho * v.u[c];
    } else {
      constexpr double sg = (K == 2) ? 1.0 : -1.0;
      r[0] = v.alpha;
#pragma unroll
      for (int m = 0; m < 2; ++m) {
        if (m == D) r[1 + m] = v.alpha * (v.u[m] + sg * v.a);
        else r[1 + m] = v.alpha * v.u[m];
      }
      r[3] = v.alpha * ((v.phi + v.a * v.a) * igm1 + sg * v.a * v.u[D]);
    }
  } else {
    const T u = v.u[0], a = v.a, Hh = v.Hh;
    if constexpr (K == 0) {
      r[0] = 1.0; r[1] = u - a; r[2] = Hh - u * a;
    } else if constexpr (K == 1) {
      r[0] = 1.0; r[1] = u; r[2] = 0.5 * u * u;
    } else {
      r[0] = 1.0; r[1] = u + a; r[2] = Hh + u * a;
    }
  }
}

// WENO5-JS (weno.py:341-369, eps = 1e-6) of values f[-2..2], also returning the
// shock sensor of its non-linear weights (weno.py:415-431, normalised, sensor_theta = 4):
// rj = sum_r |omega_r/d_r - 1|^4 / (|1/min d - 1|^4 + 2) = (...)/6563.
__device__ __forceinline__ double weno5js_sensor(double fm2, double fm1, double f0, double f1, double f2, double& rj) {
  const double t0 = f0 - 2.0 * f1 + f2, s0 = 3.0 * f0 - 4.0 * f1 + f2;
  const double t1 = fm1 - 2.0 * f0 + f1, s1 = fm1 - f1;
  const double t2 = fm2 - 2.0 * fm1 + f0, s2 = fm2 - 4.0 * fm1 + 3.0 * f0;
  constexpr double C13 = 13.0 / 12.0;
  const double e0 = 1.0e-6 + (C13 * t0 * t0 + 0.25 * s0 * s0);
  const double e1 = 1.0e-6 + (C13 * t1 * t1 + 0.25 * s1 * s1);
  const double e2 = 1.0e-6 + (C13 * t2 * t2 + 0.25 * s2 * s2);
  const double q0 = e0 * e0, q1 = e1 * e1, q2 = e2 * e2;
  const double A0 = 0.3 * (q1 * q2), A1 = 0.6 * (q0 * q2), A2 = 0.1 * (q0 * q1);
  const double ia = 1.0 / (A0 + A1 + A2);
  const double w0 = A0 * ia, w1 = A1 * ia, w2 = A2 * ia;
  const double z0 = w0 / 0.3 - 1.0, z1 = w1 / 0.6 - 1.0, z2 = w2 / 0.1 - 1.0;
  const double y0 = z0 * z0, y1 = z1 * z1, y2 = z2 * z2;
  rj = (y0 * y0 + y1 * y1 + y2 * y2) / 6563.0;
  constexpr double S6 = 1.0 / 6.0;
  const double r0 = (2.0 * f0 + 5.0 * f1 - f2) * S6;
  const double r1 = (-fm1 + 5.0 * f0 + 2.0 * f1) * S6;
  const double r2 = (2.0 * fm2 - 7.0 * fm1 + 11.0 * f0) * S6;
  return w0 * r0 + w1 * r1 + w2 * r2;
}

// Flux of the WENO non-linear filter for one characteristic field
// (shock_capturing.py:82-96, 401-416, 438-443; WENO_filter.py:324-326): the
// WENO-JS reconstructions of f+ and f- summed, minus the sixth-order central
// flux (1, -8, 37, 37, -8, 1)/60 of the characteristic fluxes on points
// -2..3, times rj = max(sensor(f+ side), sensor(f- side)).
__device__ __forceinline__ double weno_filter_flux(const double fp[6], const double fm[6], const double cf[6]) {
  double rr, rl;
  const double rec = weno5js_sensor(fp[0], fp[1], fp[2], fp[3], fp[4], rr) +
                     weno5js_sensor(fm[5], fm[4], fm[3], fm[2], fm[1], rl);
  const double central = (cf[0] - 8.0 * cf[1] + 37.0 * cf[2] + 37.0 * cf[3] - 8.0 * cf[4] + cf[5]) / 60.0;
  return fmax(rr, rl) * (rec - central);
}

// scheme tag of the WENO filter's characteristic sweeps (not a convective scheme)
constexpr int CONV_WFILTER = 16;

__device__ __forceinline__ double pow6(double x) {
  const double x2 = x * x;
  return x2 * x2 * x2;
}

// ---------------------------------------------------------------------------
// The six stencil points of an interface, as char_flux reads them: from a
// sliding register window (RegWindow), or from the LDS slots of a staged
// chunk (LdsWindow, fields q, u, p, a in rows of `stride` doubles).  With the
// LDS window every characteristic field re-reads the points it needs instead
// of holding all six in registers across the fields.
// ---------------------------------------------------------------------------
template <int ND>
struct RegWindow {
  static constexpr bool STREAM = false;
  const Pt<ND>* w;
  __device__ __forceinline__ double q(int p, int m) const { return w[p].q[m]; }
  __device__ __forceinline__ double u(int p, int m) const { return w[p].u[m]; }
  __device__ __forceinline__ double pr(int p) const { return w[p].p; }
  __device__ __forceinline__ double a(int p) const { return w[p].a; }
  __device__ __forceinline__ void point(int p, Pt<ND>& out) const { out = w[p]; }
};

template <int ND>
struct LdsWindow {
  static constexpr bool STREAM = true;
  const double* s;  // field 0 of point 0
  int stride;       // doubles between fields
  __device__ __forceinline__ double f(int p, int e) const { return s[e * stride + p]; }
  __device__ __forceinline__ double q(int p, int m) const { return f(p, m); }
  __device__ __forceinline__ double u(int p, int m) const { return f(p, ND + 2 + m); }
  __device__ __forceinline__ double pr(int p) const { return f(p, 2 * ND + 2); }
  __device__ __forceinline__ double a(int p) const { return f(p, 2 * ND + 3); }
  __device__ __forceinline__ void point(int p, Pt<ND>& out) const {
#pragma unroll
    for (int m = 0; m < ND + 2; ++m) out.q[m] = q(p, m);
#pragma unroll
    for (int m = 0; m < ND; ++m) out.u[m] = u(p, m);
    out.p = pr(p);
    out.a = a(p);
  }
};

// The same from LDS with the fields of a point next to each other, STRIDE
// doubles from point to point: with an odd stride the lanes of a wave, on
// consecutive points, hit different banks, and one address with constant
// offsets reaches every value of the six points.
template <int ND, int STRIDE>
struct LdsPoints {
  static constexpr bool STREAM = true;
  const double* s;  // field 0 of point 0
  __device__ __forceinline__ double f(int p, int e) const { return s[p * STRIDE + e]; }
  __device__ __forceinline__ double q(int p, int m) const { return f(p, m); }
  __device__ __forceinline__ double u(int p, int m) const { return f(p, ND + 2 + m); }
  __device__ __forceinline__ double pr(int p) const { return f(p, 2 * ND + 2); }
  __device__ __forceinline__ double a(int p) const { return f(p, 2 * ND + 3); }
  __device__ __forceinline__ void point(int p, Pt<ND>& out) const {
#pragma unroll
    for (int m = 0; m < ND + 2; ++m) out.q[m] = q(p, m);
#pragma unroll
    for (int m = 0; m < ND; ++m) out.u[m] = u(p, m);
    out.p = pr(p);
    out.a = a(p);
  }
};

// ---------------------------------------------------------------------------
// Reconstructions in difference form.  A reconstruction at i+1/2 is the value
// at the upwind point plus a combination of the differences of neighbouring
// points, so it is evaluated from the differences A = f[-1]-f[-2],
// B = f[0]-f[-1], C = f[1]-f[0], Dd = f[2]-f[1] (and E = f[3]-f[2], TENO6) of
// the stencil alone: the candidates are f[0] + c_r/6 with
//   c_0 = 4C - Dd, c_1 = B + 2C, c_2 = 5B - 2A,
// and *_gap return sum(omega_r c_r) as num/den.  The left reconstruction
// (weno.py side -1, of f- on the mirrored points) is the right one of the
// mirrored differences with the sign turned -- except for TENO6, whose
// right-side fourth indicator has the unsquared 781/720 term
// (teno.py:166-167), hence the QUIRK flag.
// ---------------------------------------------------------------------------

// WENO5-Z (weno.py:283-338, eps = 1e-14, p = 2) and WENO5-JS
// (weno.py:341-369, eps = 1e-6).  The indicators are taken 12/13 times:
// t^2 + 3/13 s^2, with eps 12/13 times to match.  The weights
// d_r (1 + tau^2/e_r^2) (Z) and d_r/e_r^2 (JS) are multiplied by
// 10 e_0^2 e_1^2 e_2^2, which leaves omega_r unchanged and needs no division.
template <bool Z>
__device__ __forceinline__ void weno5_gap(double A, double B, double C, double Dd, double eps, double& num,
                                          double& den) {
  constexpr double K = 3.0 / 13.0;
  const double t0 = Dd - C, t1 = C - B, t2 = B - A;
  const double s0 = __fma_rn(-2.0, C, t0), s1 = B + C, s2 = __fma_rn(2.0, B, t2);
  const double e0 = __fma_rn(t0, t0, __fma_rn(K * s0, s0, eps));
  const double e1 = __fma_rn(t1, t1, __fma_rn(K * s1, s1, eps));
  const double e2 = __fma_rn(t2, t2, __fma_rn(K * s2, s2, eps));
  const double q0 = e0 * e0, q1 = e1 * e1, q2 = e2 * e2;
  double a0 = q1 * q2, a1 = q0 * q2, a2 = q0 * q1;
  if constexpr (Z) {
    const double tau = e0 - e2;
    const double tt = tau * tau, q = a2 * q2;
    a0 = __fma_rn(tt, a0, q);
    a1 = __fma_rn(tt, a1, q);
    a2 = __fma_rn(tt, a2, q);
  }
  a0 *= 3.0;
  a1 *= 6.0;
  num = a0 * __fma_rn(4.0, C, -Dd) + a1 * __fma_rn(2.0, C, B) + a2 * __fma_rn(5.0, B, -2.0 * A);
  den = a0 + a1 + a2;
}

// TENO5 / TENO6 (teno.py:57-234, 407-465): alpha_r = (1 + tau/e_r)^6,
// e_r = eps + beta_r; delta_r = 0 where alpha_r < C_T sum(alpha), and
// omega_r = d_r delta_r / sum(d delta).  The quotients tau/e_r share a
// division by the product of two e_r (one by the product of all took as many
// instructions, but leaves the range of a double for differences beyond 1e37
// or eps below 1e-75; these products hold to 1e75 and 1e-150).
template <bool SIX, bool QUIRK>
__device__ __forceinline__ void teno_gap(double A, double B, double C, double Dd, double E, double eps, double ct,
                                         double& num, double& den) {
  constexpr double C13 = 13.0 / 12.0;
  const double t0 = C - B, s0 = B + C;
  const double t1 = Dd - C, s1 = __fma_rn(-2.0, C, t1);
  const double t2 = B - A, s2 = __fma_rn(2.0, B, t2);
  const double b0 = C13 * t0 * t0 + 0.25 * s0 * s0;
  const double b1 = C13 * t1 * t1 + 0.25 * s1 * s1;
  const double b2 = C13 * t2 * t2 + 0.25 * s2 * s2;
  const double e0 = eps + b0, e1 = eps + b1, e2 = eps + b2;
  const double c0 = __fma_rn(2.0, C, B), c1 = __fma_rn(4.0, C, -Dd), c2 = __fma_rn(5.0, B, -2.0 * A);
  if constexpr (SIX) {
    const double p3 = 11.0 * C - 7.0 * Dd + 2.0 * E;
    const double r3 = 3.0 * Dd - 2.0 * C - E;
    const double q3 = C - 2.0 * Dd + E;
    double b3 = (1.0 / 36.0) * p3 * p3 + C13 * r3 * r3;
    // f+- are half the differences that come in: the unsquared term counts double
    if constexpr (QUIRK) b3 += 2.0 * (781.0 / 720.0) * q3;
    else b3 += (781.0 / 720.0) * q3 * q3;
    const double c3 = 4.5 * C - 2.0 * Dd + 0.5 * E;
    const double tau = fabs(b3 - (b0 + b2 - 4.0 * b1) * (1.0 / 6.0));
    const double e3 = eps + b3;
    const double x01 = quot_pos(tau, e0 * e1), x23 = quot_pos(tau, e2 * e3);
    const double a0 = pow6(__fma_rn(e1, x01, 1.0)), a1 = pow6(__fma_rn(e0, x01, 1.0));
    const double a2 = pow6(__fma_rn(e3, x23, 1.0)), a3 = pow6(__fma_rn(e2, x23, 1.0));
    const double cut = ct * (a0 + a1 + a2 + a3);
    const double w0 = a0 < cut ? 0.0 : 231.0 / 500.0, w1 = a1 < cut ? 0.0 : 3.0 / 10.0;
    const double w2 = a2 < cut ? 0.0 : 27.0 / 500.0, w3 = a3 < cut ? 0.0 : 23.0 / 125.0;
    num = w0 * c0 + w1 * c1 + w2 * c2 + w3 * c3;
    den = w0 + w1 + w2 + w3;
  } else {
    const double tau = fabs(b0 - b2);
    const double x01 = quot_pos(tau, e0 * e1);
    const double a0 = pow6(__fma_rn(e1, x01, 1.0)), a1 = pow6(__fma_rn(e0, x01, 1.0));
    const double a2 = pow6(1.0 + quot_pos(tau, e2));
    const double cut = ct * (a0 + a1 + a2);
    const double w0 = a0 < cut ? 0.0 : 11.0 / 20.0, w1 = a1 < cut ? 0.0 : 4.0 / 10.0, w2 = a2 < cut ? 0.0 : 1.0 / 20.0;
    num = w0 * c0 + w1 * c1 + w2 * c2;
    den = w0 + w1 + w2;
  }
}

// Twice the reconstructed value of one characteristic field less the sum of
// its flux at the interface's two points: the right reconstruction of
// f+ = (cf + lam cs)/2 and the left one of f- = (cf - lam cs)/2
// (shock_capturing.py:257-265) from the differences dcs, dcf of cs and cf
// between the six points; the halves are left out (eps counts four times).
template <int CONV>
__device__ __forceinline__ double recon_gap(const double dcs[5], const double dcf[5], double lam, double eps,
                                            double ct) {
  double p[5], m[5];
#pragma unroll
  for (int g = 0; g < 5; ++g) {
    p[g] = __fma_rn(lam, dcs[g], dcf[g]);
    m[g] = __fma_rn(-lam, dcs[g], dcf[g]);
  }
  if constexpr (CONV == CONV_WFILTER) {
    // the filter flux, which vanishes on equal values, of the variables less their first
    double fp[6], fm[6], cf[6];
    fp[0] = fm[0] = cf[0] = 0.0;
#pragma unroll
    for (int g = 0; g < 5; ++g) {
      fp[g + 1] = fp[g] + 0.5 * p[g];
      fm[g + 1] = fm[g] + 0.5 * m[g];
      cf[g + 1] = cf[g] + dcf[g];
    }
    return 2.0 * weno_filter_flux(fp, fm, cf);
  } else {
    double n1, d1, n2, d2;
    if constexpr (CONV == OSBL_CONV_WENO_Z || CONV == OSBL_CONV_WENO_JS) {
      constexpr bool Z = CONV == OSBL_CONV_WENO_Z;
      weno5_gap<Z>(p[0], p[1], p[2], p[3], eps, n1, d1);
      weno5_gap<Z>(m[4], m[3], m[2], m[1], eps, n2, d2);
    } else {
      constexpr bool SIX = CONV == OSBL_CONV_TENO6;
      teno_gap<SIX, true>(p[0], p[1], p[2], p[3], p[4], eps, ct, n1, d1);
      teno_gap<SIX, false>(m[4], m[3], m[2], m[1], m[0], eps, ct, n2, d2);
    }
    return __fma_rn(1.0 / 6.0, quot_pos(n1, d1) - quot_pos(n2, d2), -lam * dcs[2]);
  }
}

// ---------------------------------------------------------------------------
// LLF characteristic flux at the interface between window points 2 and 3
// (shock_capturing.py:357-448), as the mean of the two points' fluxes plus
// R times the rest of the reconstructions: R L = 1, so the values that the
// reconstructions start from (f+ at point 2, f- at point 3) add up to that
// mean and -lam (cs_3 - cs_2)/2, and only differences between points have to
// be projected.  They are projected in the frame that moves with the
// averaged velocity v.u, where the eigenvectors lose most entries: with
// m' = m - v.u rho and E' = E - v.u.m + rho v.u^2/2,
//   entropy   rho - (gama-1)/a^2 E'
//   acoustic  s (E' +- a/(gama-1) m'_D), s = (gama-1)/(sqrt2 rho a)
//             (1-D: (gama-1)/(2 a^2))
//   shear     +-m'_c/rho
// and the flux in that frame is (m_D, u_D m'_c, u_D m'_D + p,
// u_D E' + p (u_D - v.u_D)).
//
// The sweeps are bound by FP64 issue (and the clock that its power allows):
// against projecting every point on the full rows of L this takes the y
// sweep of WENO5-Z, Roe, 3-D, from ~1300 to ~980 VALU instructions per cell;
// 256^3: y 0.785 -> 0.57 ms, z with the RK update 0.83 -> 0.67, x 0.89 -> 0.62
// (with its pipelined walk); the step 8.9 -> 7.3 ms, TENO6 12.8 -> 10.8.
// ---------------------------------------------------------------------------
template <int ND, int D, int CONV, class W>
__device__ __forceinline__ void char_fields(const W& w, const Avg<ND>& v, const Phys& ph, double ct,
                                            double fh[ND + 2]) {
  constexpr int NV = ND + 2, E = NV - 1;
  // WENO's indicators are taken 12/13 times
  constexpr bool WENO = CONV == OSBL_CONV_WENO_Z || CONV == OSBL_CONV_WENO_JS;
  const double eps = 4.0 * (WENO ? 12.0 / 13.0 * (CONV == OSBL_CONV_WENO_Z ? 1.0e-14 : 1.0e-6) : ph.eps);
  // the points are re-read per use from a streamed window, and a field's
  // reconstruction is finished before the next one starts, so that little of
  // either stays in registers across the fields
  auto reload = [] {
    if constexpr (W::STREAM) asm volatile("" ::: "memory");
    __builtin_amdgcn_sched_barrier(0);
  };
  auto finish = [&](double& x) {
    asm volatile("" : "+v"(x));
    reload();
  };
  double l0 = 0.0, lp = 0.0, lm = 0.0;
#pragma unroll
  for (int p = 0; p < 6; ++p) {
    const double ud = w.u(p, D), a = w.a(p);
    l0 = max_abs(l0, ud);
    lp = max_abs(lp, ud + a);
    lm = max_abs(lm, ud - a);
  }
  double hu = 0.0;  // v.u^2/2
#pragma unroll
  for (int m = 0; m < ND; ++m) hu = __fma_rn(0.5 * v.u[m], v.u[m], hu);
#pragma unroll
  for (int m = 0; m < NV; ++m) fh[m] = 0.0;
  reload();
  sfor<0, ND>([&](auto cc) {
    constexpr int c = decltype(cc)::value;
    if constexpr (c != D) {
      constexpr double sg = ND == 3 ? (double)eps3(D, 3 - D - c, c) : (D == 0 ? -1.0 : 1.0);
      const double lc = sg * v.ir, lr = -lc * v.u[c];
      double dcs[5], dcf[5], ps = 0.0, pf = 0.0;
#pragma unroll
      for (int p = 0; p < 6; ++p) {
        const double cs = __fma_rn(lr, w.q(p, 0), lc * w.q(p, 1 + c));
        const double cf = w.u(p, D) * cs;
        if (p > 0) {
          dcs[p - 1] = cs - ps;
          dcf[p - 1] = cf - pf;
        }
        ps = cs;
        pf = cf;
      }
      double h = 0.5 * sg * v.rho * recon_gap<CONV>(dcs, dcf, l0, eps, ct);
      finish(h);
      fh[1 + c] += h;
      fh[E] = __fma_rn(v.u[c], h, fh[E]);
    }
  });
  // differences of s E', m'_D and of their fluxes
  const double ia2 = v.ia * v.ia;
  const double s = ND == 1 ? 0.5 * ph.gm1 * ia2 : v.bta * ph.gm1;
  const double kap = ND == 1 ? 0.5 * v.ia : v.bta * v.a;  // s a/(gama-1)
  double dE[5], gE[5], dm[5], gm[5];
  {
    double pE = 0.0, pg = 0.0, pm = 0.0, pn = 0.0;
#pragma unroll
    for (int p = 0; p < 6; ++p) {
      const double r = w.q(p, 0), ud = w.u(p, D), pr = w.pr(p);
      const double mD = __fma_rn(-v.u[D], r, w.q(p, 1 + D));
      double En = __fma_rn(hu, r, w.q(p, E));
#pragma unroll
      for (int m = 0; m < ND; ++m) En = __fma_rn(-v.u[m], w.q(p, 1 + m), En);
      const double fD = __fma_rn(ud, mD, pr);
      const double fE = __fma_rn(pr, ud - v.u[D], ud * En);
      if (p > 0) {
        dE[p - 1] = s * (En - pE);
        gE[p - 1] = s * (fE - pg);
        dm[p - 1] = mD - pm;
        gm[p - 1] = fD - pn;
      }
      pE = En;
      pg = fE;
      pm = mD;
      pn = fD;
      if constexpr (W::STREAM) {
        if (p & 1) {
          asm volatile("" : "+v"(pE), "+v"(pg), "+v"(pm), "+v"(pn));
          reload();
        }
      }
    }
  }
  reload();
  double w0, wp, wm;
  double cs[5], cf[5];
  {
    // -(gama-1)/a^2 / s
    const double ce = ND == 1 ? -2.0 : -1.41421356237309504880 * v.rho * v.ia;
#pragma unroll
    for (int g = 0; g < 5; ++g) {
      cs[g] = __fma_rn(ce, dE[g], w.q(g + 1, 0) - w.q(g, 0));
      cf[g] = __fma_rn(ce, gE[g], w.q(g + 1, 1 + D) - w.q(g, 1 + D));
    }
    w0 = 0.5 * recon_gap<CONV>(cs, cf, l0, eps, ct);
  }
  finish(w0);
  // R's first entries: alpha (1-D: 1)
  const double ha = ND == 1 ? 0.5 : 0.5 * v.alpha;
#pragma unroll
  for (int g = 0; g < 5; ++g) {
    cs[g] = __fma_rn(kap, dm[g], dE[g]);
    cf[g] = __fma_rn(kap, gm[g], gE[g]);
  }
  wp = ha * recon_gap<CONV>(cs, cf, lp, eps, ct);
  finish(wp);
#pragma unroll
  for (int g = 0; g < 5; ++g) {
    cs[g] = __fma_rn(-kap, dm[g], dE[g]);
    cf[g] = __fma_rn(-kap, gm[g], gE[g]);
  }
  wm = ha * recon_gap<CONV>(cs, cf, lm, eps, ct);
  finish(wm);
  const double S = wp + wm, G = w0 + S, M = v.a * (wp - wm);
  fh[0] += G;
#pragma unroll
  for (int m = 0; m < ND; ++m) fh[1 + m] = __fma_rn(v.u[m], G, fh[1 + m]);
  fh[1 + D] += M;
  fh[E] = __fma_rn(hu, G, fh[E]);
  fh[E] = __fma_rn(v.a * v.a * ph.igm1, S, fh[E]);
  fh[E] = __fma_rn(v.u[D], M, fh[E]);
  if constexpr (CONV != CONV_WFILTER) {
    const double u2 = 0.5 * w.u(2, D), u3 = 0.5 * w.u(3, D), p2 = w.pr(2), p3 = w.pr(3);
    fh[0] += 0.5 * (w.q(2, 1 + D) + w.q(3, 1 + D));
#pragma unroll
    for (int m = 0; m < ND; ++m) {
      const double f = __fma_rn(u2, w.q(2, 1 + m), u3 * w.q(3, 1 + m));
      fh[1 + m] += m == D ? __fma_rn(0.5, p2 + p3, f) : f;
    }
    fh[E] += __fma_rn(u2, w.q(2, E) + p2, u3 * (w.q(3, E) + p3));
  }
}

template <int ND, int D, int CONV, int AVG, bool CACHED = false, class W>
__device__ __forceinline__ void char_flux_w(const W& w, const Phys& ph, double fh[ND + 2], double ct,
                                            const RoeF& rf = RoeF{}) {
  Avg<ND> v;
  {
    Pt<ND> L, R;
    w.point(2, L);
    w.point(3, R);
    if constexpr (CACHED && AVG == OSBL_AVG_ROE) {
      roe_state<ND>(v, L, R, rf, ph);
      finish_avg<ND>(v, ph);
    } else {
      interface_state<ND, AVG>(v, L, R, ph);
    }
  }
  char_fields<ND, D, CONV>(w, v, ph, ct, fh);
}

template <int ND, int D, int CONV, int AVG, bool CACHED = false>
__device__ __forceinline__ void char_flux(const Pt<ND> (&w)[6], const Phys& ph, double fh[ND + 2], double ct,
                                          const RoeF& rf = RoeF{}) {
  char_flux_w<ND, D, CONV, AVG, CACHED>(RegWindow<ND>{w}, ph, fh, ct, rf);
}

}  // namespace osbl
