// osbl_curvilinear.hip -- the shock-capturing right-hand side on a general
// curvilinear grid: the Euler equations in strong conservation form
//   d(Q)/dt = -(1/detJ) sum_j d(detJ F_j)/d xi_j,
//   F_j = (rho U_j, rhou_i U_j + p D_ji, (p + rhoE) U_j),  U_j = D_jm u_m
// (apps/euler_wave_curvilinear/euler_wave.py:17-47), with the metric
// D = d xi/d x and detJ = det(d x/d xi) of MetricsEquation (metric.py:72-147).
//
// The LLF characteristic reconstruction (shock_capturing.py:357-448) runs
// about the metric direction k = (D_d0, .., D_d(nd-1)) of each interface:
// k is the simple average of the two neighbours' metric (averaging.py:49-57,
// 104-113), L and R are the Euler eigenvectors about the unit normal k/|k|
// (euler_eigensystem.py:18-40, 88-135), and the local wave speeds use every
// stencil point's own metric, |U|, |U +- a|k|| (shock_capturing.py:512-536).
// The characteristic fluxes are L (detJ F_d) and the characteristic state L Q.
//
// Layout: the padded fields of the block (Grid); the metric holds nd*nd + 1
// padded fields, D_ab at a*nd + b and detJ last.  One kernel per direction
// forms detJ F_d of a tile's points in LDS, the interface fluxes from them and
// their differences; the last direction divides by detJ and applies the RK
// update.  Curvilinear blocks are periodic: points are read at their images.
#include "osbl_kernels.h"

namespace osbl {

namespace {

// A point's fields in LDS: q, G = detJ F_d, U, a|k|, the metric k (not scaled
// by detJ), and of the average 1/sqrt(rho), sqrt(rho) H (Roe) or 1/rho, a
template <int ND>
struct CurvPt {
  static constexpr int NV = ND + 2, Q = 0, G = NV, U = 2 * NV, AK = U + 1, K = U + 2, IS = K + ND, H = IS + 1,
                       NF = H + 1, STRIDE = NF | 1;  // odd stride: lanes on consecutive points hit different banks
};

// LLF characteristic flux about the metric normal at the interface between
// points 2 and 3 of six, ST doubles apart: the mean of the two G plus R times
// the rest of the reconstructions, from differences between points alone
// (R L = 1), projected in the frame of the averaged velocity u.  There
// m' = m - u rho, E' = E - u.m + rho u^2/2 of both q and G, and with kt the
// unit normal the rows of L are
//   2-D: rho - (gama-1)/a^2 E' =: e;  (kt x m')/rho (shear)
//   3-D: kt_f e - (kt x m')_f/rho, f = 0, 1, 2
//   (+-a kt.m' + (gama-1) E')/(sqrt2 rho a)
// (euler_eigensystem.py:18-40, 88-135).
template <int ND, int CONV, int AVG, int ST>
__device__ __forceinline__ void curv_flux(const double* __restrict__ s, const Phys& ph, double (&fh)[ND + 2]) {
  using P = CurvPt<ND>;
  constexpr int NV = ND + 2, E = NV - 1;
  constexpr bool WENO = CONV == OSBL_CONV_WENO_Z || CONV == OSBL_CONV_WENO_JS;
  const double eps = 4.0 * (WENO ? 12.0 / 13.0 * (CONV == OSBL_CONV_WENO_Z ? 1.0e-14 : 1.0e-6) : ph.eps);
  const double ct = ph.teno_ct;
  auto at = [&](int p, int e) { return s[p * ST + e]; };
  auto finish = [](double& x) {  // a field's reconstruction is finished before the next one starts
    asm volatile("" : "+v"(x));
    __builtin_amdgcn_sched_barrier(0);
  };
  Avg<ND> v;
  {
    const double iL = at(2, P::IS), iR = at(3, P::IS);
    if constexpr (AVG == OSBL_AVG_ROE) {
      const double sL = at(2, 0) * iL, sR = at(3, 0) * iR, inv = recip_pos(sL + sR);
      v.rho = sL * sR;
      double ke = 0.0;
#pragma unroll
      for (int m = 0; m < ND; ++m) {
        v.u[m] = (at(2, 1 + m) * iL + at(3, 1 + m) * iR) * inv;
        ke += v.u[m] * v.u[m];
      }
      v.a = sqrt_pos(ph.gm1 * ((at(2, P::H) + at(3, P::H)) * inv - 0.5 * ke));
    } else {
      v.rho = 0.5 * (at(2, 0) + at(3, 0));
#pragma unroll
      for (int m = 0; m < ND; ++m) v.u[m] = 0.5 * (at(2, 1 + m) * iL + at(3, 1 + m) * iR);
      v.a = 0.5 * (at(2, P::H) + at(3, P::H));
    }
    finish_avg<ND>(v, ph);
  }
  double kt[ND], kk = 0.0;
#pragma unroll
  for (int m = 0; m < ND; ++m) {
    kt[m] = at(2, P::K + m) + at(3, P::K + m);
    kk = __fma_rn(kt[m], kt[m], kk);
  }
  const double ik = recip_pos(sqrt_pos(kk));
#pragma unroll
  for (int m = 0; m < ND; ++m) kt[m] *= ik;
  double l0 = 0.0, lp = 0.0, lm = 0.0, hu = 0.0;
#pragma unroll
  for (int m = 0; m < ND; ++m) hu = __fma_rn(0.5 * v.u[m], v.u[m], hu);
  // differences of q and G in the moving frame
  double dq[NV][5], dg[NV][5];
  {
    double pq[NV], pg[NV];
#pragma unroll
    for (int p = 0; p < 6; ++p) {
      const double U = at(p, P::U), ak = at(p, P::AK);
      l0 = max_abs(l0, U);
      lp = max_abs(lp, U + ak);
      lm = max_abs(lm, U - ak);
      auto moved = [&](int base, double (&o)[NV]) {
        o[0] = at(p, base);
        o[E] = __fma_rn(hu, o[0], at(p, base + E));
#pragma unroll
        for (int m = 0; m < ND; ++m) {
          const double mm = at(p, base + 1 + m);
          o[1 + m] = __fma_rn(-v.u[m], o[0], mm);
          o[E] = __fma_rn(-v.u[m], mm, o[E]);
        }
      };
      double nq[NV], ng[NV];
      moved(P::Q, nq);
      moved(P::G, ng);
#pragma unroll
      for (int m = 0; m < NV; ++m) {
        if (p > 0) {
          dq[m][p - 1] = nq[m] - pq[m];
          dg[m][p - 1] = ng[m] - pg[m];
        }
        pq[m] = nq[m];
        pg[m] = ng[m];
      }
    }
  }
  __builtin_amdgcn_sched_barrier(0);
  double cs[5], cf[5];
  double w0 = 0.0, mo[ND];  // R's sums in the moving frame: of the entropy columns, momentum
  const double ce = -ph.gm1 * v.ia * v.ia;
  if constexpr (ND == 2) {
    const double t0 = kt[1] * v.ir, t1 = -kt[0] * v.ir;
#pragma unroll
    for (int g = 0; g < 5; ++g) {
      cs[g] = __fma_rn(t0, dq[1][g], t1 * dq[2][g]);
      cf[g] = __fma_rn(t0, dg[1][g], t1 * dg[2][g]);
    }
    double ws = 0.5 * v.rho * recon_gap<CONV>(cs, cf, l0, eps, ct);
    finish(ws);
    mo[0] = kt[1] * ws;
    mo[1] = -kt[0] * ws;
#pragma unroll
    for (int g = 0; g < 5; ++g) {
      cs[g] = __fma_rn(ce, dq[E][g], dq[0][g]);
      cf[g] = __fma_rn(ce, dg[E][g], dg[0][g]);
    }
    w0 = 0.5 * recon_gap<CONV>(cs, cf, l0, eps, ct);
    finish(w0);
  } else {
    double w[3];
    sfor<0, 3>([&](auto fc) {
      constexpr int f = decltype(fc)::value, c1 = (f + 1) % 3, c2 = (f + 2) % 3;
      const double t1 = kt[c2] * v.ir, t2 = -kt[c1] * v.ir, e0 = kt[f], e1 = kt[f] * ce;
#pragma unroll
      for (int g = 0; g < 5; ++g) {
        cs[g] = __fma_rn(t1, dq[1 + c1][g], __fma_rn(t2, dq[1 + c2][g], __fma_rn(e1, dq[E][g], e0 * dq[0][g])));
        cf[g] = __fma_rn(t1, dg[1 + c1][g], __fma_rn(t2, dg[1 + c2][g], __fma_rn(e1, dg[E][g], e0 * dg[0][g])));
      }
      w[f] = 0.5 * recon_gap<CONV>(cs, cf, l0, eps, ct);
      finish(w[f]);
    });
    w0 = kt[0] * w[0] + kt[1] * w[1] + kt[2] * w[2];
#pragma unroll
    for (int c = 0; c < 3; ++c) {
      const int c1 = (c + 1) % 3, c2 = (c + 2) % 3;
      mo[c] = v.rho * (kt[c1] * w[c2] - kt[c2] * w[c1]);
    }
  }
  const double sE = v.bta * ph.gm1, sn = v.bta * v.a, ha = 0.5 * v.alpha;
  double wa[2];
#pragma unroll
  for (int k = 0; k < 2; ++k) {
    double n[ND];
#pragma unroll
    for (int m = 0; m < ND; ++m) n[m] = (k == 0 ? sn : -sn) * kt[m];
#pragma unroll
    for (int g = 0; g < 5; ++g) {
      cs[g] = sE * dq[E][g];
      cf[g] = sE * dg[E][g];
#pragma unroll
      for (int m = 0; m < ND; ++m) {
        cs[g] = __fma_rn(n[m], dq[1 + m][g], cs[g]);
        cf[g] = __fma_rn(n[m], dg[1 + m][g], cf[g]);
      }
    }
    wa[k] = ha * recon_gap<CONV>(cs, cf, k == 0 ? lp : lm, eps, ct);
    finish(wa[k]);
  }
  const double S = wa[0] + wa[1], r0 = w0 + S, M = v.a * (wa[0] - wa[1]);
  double en = __fma_rn(hu, r0, v.a * v.a * ph.igm1 * S);
#pragma unroll
  for (int m = 0; m < ND; ++m) {
    mo[m] = __fma_rn(kt[m], M, mo[m]);
    en = __fma_rn(v.u[m], mo[m], en);
    fh[1 + m] = __fma_rn(v.u[m], r0, mo[m]) + 0.5 * (at(2, P::G + 1 + m) + at(3, P::G + 1 + m));
  }
  fh[0] = r0 + 0.5 * (at(2, P::G) + at(3, P::G));
  fh[E] = en + 0.5 * (at(2, P::G + E) + at(3, P::G + E));
}

// ---------------------------------------------------------------------------
// Direction D of a stage.  A workgroup takes TI - 1 cells along D of TL lines:
// 31 x 8 for the x direction, 15 x 16 (16 along x, whole cache lines) for the
// others.  Its (TI + 5) TL points are staged in LDS with G, U and a|k|; thread
// (i, l) evaluates the flux below cell i of line l and finishes cell i - 1.
// The first direction assigns R, the others add; the last one divides by detJ
// and leaves R (mode 2) or applies the RK update (mode as k_update).
//
// What bounds it is FP64 issue.  A stage of WENO5-Z, Roe at 1024^2 under the
// profiler: 53 + 62 us, against 214 of a point, a flux (all six points
// projected on the full rows of L) and a difference kernel per direction, the
// update and the halo exchange.  3-D keeps 50 differences in 172 to 200
// registers: two waves per SIMD (96^3: 70 + 63 + 75 us), as three spill (79 +
// 79 + 94; TENO6 116 + 115 + 131 against 89 + 80 + 89).
// Tiles of 63 x 4 along x gained 5 % at 1024^2 and 1 % at 96^3 and waste more on
// other extents; 31 x 8 along y and z, half cache lines, took 72 and 91 us there.
// ---------------------------------------------------------------------------
template <int ND, int D, int CONV, int AVG>
__global__ void __launch_bounds__(256, ND == 3 ? 2 : 3) k_curv_sweep(const double* __restrict__ Q, const double* __restrict__ M,
                                                       double* __restrict__ R, double* __restrict__ Qo,
                                                       double* __restrict__ Qn, Grid g, Phys ph, int mode, double cA,
                                                       double cB, int first) {
  using P = CurvPt<ND>;
  constexpr int NV = ND + 2, TI = D == 0 ? 32 : 16, TL = 256 / TI, NP = (TI + 5) * TL;
  constexpr bool LAST = D == ND - 1;
  constexpr int AL = D == 0 ? 1 : 0, AO = D == 2 ? 1 : 2;  // axis of the lines, and the one of single planes
  static_assert(NP <= 512);
  __shared__ double S[NP * P::STRIDE];
  const int t = threadIdx.x;
  // neighbours in LDS: points along x
  const int i = D == 0 ? t % TI : t / TL, l = D == 0 ? t / TI : t % TL;
  const int i0 = (D == 0 ? blockIdx.x : blockIdx.y) * (TI - 1), l0 = (D == 0 ? blockIdx.y : blockIdx.x) * TL;
  const int o = blockIdx.z;
  auto index = [&](int ci, int cl) {
    int c[3];
    c[D] = ci < 0 ? ci + g.n[D] : (ci >= g.n[D] ? ci - g.n[D] : ci);
    c[AL] = min(cl, g.n[AL] - 1);
    c[AO] = o;
    return g.idx(c[0], c[1], c[2]);
  };
  double nq[2][NV], nm[2][ND + 1];
#pragma unroll
  for (int k = 0; k < 2; ++k) {
    const int p = min(t + 256 * k, NP - 1);
    const int pi = D == 0 ? p % (TI + 5) : p / TL, pl = D == 0 ? p / (TI + 5) : p % TL;
    const int y = index(min(i0 - 3 + pi, g.n[D] + 2), l0 + pl);
    fetch_q<ND>(nq[k], Q, g.fs, y);
#pragma unroll
    for (int m = 0; m < ND; ++m) nm[k][m] = M[(D * ND + m) * g.fs + y];
    nm[k][ND] = M[ND * ND * g.fs + y];
  }
  const int ci = i0 + i - 1, cl = l0 + l;
  const bool own = i > 0 && ci < g.n[D] && cl < g.n[AL];
  const int x = index(max(ci, 0), cl);
#pragma unroll
  for (int k = 0; k < 2; ++k) {
    const int p = t + 256 * k;
    Pt<ND> s;
#pragma unroll
    for (int m = 0; m < NV; ++m) s.q[m] = nq[k][m];
    finish_pt<ND>(s, ph);
    double U = 0.0, kk = 0.0;
#pragma unroll
    for (int m = 0; m < ND; ++m) {
      U = __fma_rn(nm[k][m], s.u[m], U);
      kk = __fma_rn(nm[k][m], nm[k][m], kk);
    }
    const double w = nm[k][ND] * U, jp = nm[k][ND] * s.p;
    if (p < NP) {
      double* o_ = S + p * P::STRIDE;
#pragma unroll
      for (int m = 0; m < NV; ++m) o_[P::Q + m] = s.q[m];
      o_[P::G] = w * s.q[0];
#pragma unroll
      for (int m = 0; m < ND; ++m) {
        o_[P::G + 1 + m] = __fma_rn(w, s.q[1 + m], jp * nm[k][m]);
        o_[P::K + m] = nm[k][m];
      }
      o_[P::G + NV - 1] = w * (s.q[NV - 1] + s.p);
      o_[P::U] = U;
      o_[P::AK] = s.a * sqrt_pos(kk);
      if constexpr (AVG == OSBL_AVG_ROE) {
        const double is = recip_pos(sqrt_pos(s.q[0]));
        o_[P::IS] = is;
        o_[P::H] = (s.q[NV - 1] + s.p) * is;
      } else {
        o_[P::IS] = recip_pos(s.q[0]);
        o_[P::H] = s.a;
      }
    }
  }
  __syncthreads();
  double f[NV];
  constexpr int ST = (D == 0 ? 1 : TL) * P::STRIDE;
  curv_flux<ND, CONV, AVG, ST>(S + (D == 0 ? l * (TI + 5) + i : i * TL + l) * P::STRIDE, ph, f);
  double q[NV];
  if constexpr (LAST) {
    const double* c = S + (D == 0 ? l * (TI + 5) + i + 2 : (i + 2) * TL + l) * P::STRIDE;  // cell i - 1
#pragma unroll
    for (int m = 0; m < NV; ++m) q[m] = c[m];
  }
  // (loaded here, not ahead of the fluxes: 22 registers less there, no spills)
  double fl[NV], r[NV], qo[NV], ij = 1.0;
  auto load = [&] {
    if constexpr (D > 0) {
      if (!own) return;
#pragma unroll
      for (int m = 0; m < NV; ++m) r[m] = R[m * g.fs + x];
      if constexpr (LAST) {
        ij = M[ND * ND * g.fs + x];
        if (mode == 0 ? !first : (mode == 1 && cA != 0.0)) {
#pragma unroll
          for (int m = 0; m < NV; ++m) qo[m] = Qo[m * g.fs + x];
        }
      }
    }
  };
  if constexpr (D == 0) {
#pragma unroll
    for (int m = 0; m < NV; ++m) fl[m] = __shfl_up(f[m], 1);
  } else {
    __syncthreads();
    load();
#pragma unroll
    for (int m = 0; m < NV; ++m) S[m * 256 + t] = f[m];
    __syncthreads();
#pragma unroll
    for (int m = 0; m < NV; ++m) fl[m] = S[m * 256 + max(t - TL, 0)];
  }
  if (!own) return;
  if constexpr (LAST) ij = 1.0 / ij;
#pragma unroll
  for (int m = 0; m < NV; ++m) {
    const double df = fl[m] - f[m];
    r[m] = D == 0 ? df * ph.inv_delta[D] : __fma_rn(df, ph.inv_delta[D], r[m]);
    if constexpr (LAST) r[m] *= ij;
    if (!LAST || mode == 2) {
      R[m * g.fs + x] = r[m];
    } else if (mode == 0) {
      const double o_ = first ? q[m] : qo[m];
      Qn[m * g.fs + x] = __fma_rn(ph.dt * cA, r[m], o_);
      Qo[m * g.fs + x] = __fma_rn(ph.dt * cB, r[m], o_);
    } else {
      const double tmp = cA != 0.0 ? __fma_rn(ph.dt, r[m], cA * qo[m]) : ph.dt * r[m];
      Qo[m * g.fs + x] = tmp;
      Qn[m * g.fs + x] = __fma_rn(cB, tmp, q[m]);
    }
  }
}

// J_ab = CD(x_a, xi_b) from the coordinates X (nd arrays over the interior
// extended by 2 points on every side, x fastest, extents e), detJ = det J and
// D = adj(J)/detJ over the interior
template <int ND>
__global__ void __launch_bounds__(256) k_curv_metric(const double* __restrict__ X, double* __restrict__ M, Grid g,
                                                     Phys ph, int e0, int e1, int e2) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= g.n[0]) return;
  const int j = blockIdx.y, k = blockIdx.z;
  const long long per = (long long)e0 * e1 * e2;
  const long long base = (i + 2) + (long long)e0 * ((j + (ND > 1 ? 2 : 0)) + (long long)e1 * (k + (ND > 2 ? 2 : 0)));
  const long long sx[3] = {1, e0, (long long)e0 * e1};
  double J[3][3] = {{0.0, 0.0, 0.0}, {0.0, 0.0, 0.0}, {0.0, 0.0, 0.0}};
#pragma unroll
  for (int a = 0; a < ND; ++a)
#pragma unroll
    for (int b = 0; b < ND; ++b) {
      const double* f = X + a * per + base;
      const long long s = sx[b];
      J[a][b] = ph.inv_delta[b] *
                ((1.0 / 12.0) * f[-2 * s] + (-2.0 / 3.0) * f[-s] + (2.0 / 3.0) * f[s] + (-1.0 / 12.0) * f[2 * s]);
    }
  double adj[3][3], det;
  if constexpr (ND == 2) {
    det = J[0][0] * J[1][1] - J[0][1] * J[1][0];
    adj[0][0] = J[1][1];
    adj[0][1] = -J[0][1];
    adj[1][0] = -J[1][0];
    adj[1][1] = J[0][0];
  } else {
#pragma unroll
    for (int a = 0; a < 3; ++a)
#pragma unroll
      for (int b = 0; b < 3; ++b) {
        const int r0 = (b + 1) % 3, r1 = (b + 2) % 3, c0 = (a + 1) % 3, c1 = (a + 2) % 3;
        adj[a][b] = J[r0][c0] * J[r1][c1] - J[r0][c1] * J[r1][c0];  // cofactor C_ba
      }
    det = J[0][0] * adj[0][0] + J[0][1] * adj[1][0] + J[0][2] * adj[2][0];
  }
  const int x = g.idx(i, j, k);
  const long long fs = g.fs;
  M[(ND * ND) * fs + x] = det;
#pragma unroll
  for (int a = 0; a < ND; ++a)
#pragma unroll
    for (int b = 0; b < ND; ++b) M[(a * ND + b) * fs + x] = adj[a][b] / det;
}

template <int ND, int CONV, int AVG>
void launch_sweeps(const double* Q, const double* M, double* R, double* Qo, double* Qn, const Grid& g, const Phys& ph,
                   int d, int mode, double cA, double cB, int first, hipStream_t s) {
  auto go = [&](auto dc) {
    constexpr int D = decltype(dc)::value, TI = D == 0 ? 32 : 16, TL = 256 / TI, AL = D == 0 ? 1 : 0;
    const unsigned ti = (g.n[D] + TI - 2) / (TI - 1), tl = (g.n[AL] + TL - 1) / TL;
    const dim3 grid(D == 0 ? ti : tl, D == 0 ? tl : ti, g.n[D == 2 ? 1 : 2]);
    k_curv_sweep<ND, D, CONV, AVG><<<grid, 256, 0, s>>>(Q, M, R, Qo, Qn, g, ph, mode, cA, cB, first);
  };
  if (d == 0) go(std::integral_constant<int, 0>{});
  else if (d == 1) go(std::integral_constant<int, 1>{});
  else if constexpr (ND == 3) go(std::integral_constant<int, 2>{});
}

}  // namespace

// direction d of a curvilinear stage; the last one ends it (k_curv_sweep).  Q
// needs no halos; M is the metric.
void launch_curv_sweep(int nd, int d, int conv, int avg, int mode, const double* Q, const double* M, double* R,
                       double* Qo, double* Qn, const Grid& g, const Phys& ph, double cA, double cB, int first,
                       hipStream_t s) {
  auto with_avg = [&](auto nc, auto cc) {
    constexpr int ND = decltype(nc)::value, C = decltype(cc)::value;
    if (avg == OSBL_AVG_ROE) launch_sweeps<ND, C, OSBL_AVG_ROE>(Q, M, R, Qo, Qn, g, ph, d, mode, cA, cB, first, s);
    else launch_sweeps<ND, C, OSBL_AVG_SIMPLE>(Q, M, R, Qo, Qn, g, ph, d, mode, cA, cB, first, s);
  };
  auto with_conv = [&](auto nc) {
    switch (conv) {
      case OSBL_CONV_WENO_JS: with_avg(nc, std::integral_constant<int, OSBL_CONV_WENO_JS>{}); break;
      case OSBL_CONV_WENO_Z: with_avg(nc, std::integral_constant<int, OSBL_CONV_WENO_Z>{}); break;
      case OSBL_CONV_TENO5: with_avg(nc, std::integral_constant<int, OSBL_CONV_TENO5>{}); break;
      default: with_avg(nc, std::integral_constant<int, OSBL_CONV_TENO6>{}); break;
    }
  };
  if (nd == 3) with_conv(std::integral_constant<int, 3>{});
  else with_conv(std::integral_constant<int, 2>{});
}

// metric over the interior from the coordinates X (extents e[3]: n[d] + 4 on
// the block's directions, 1 elsewhere), then its periodic halos
void launch_curv_metric(int nd, const double* X, double* M, const Grid& g, const Phys& ph, const int e[3],
                        hipStream_t s) {
  dim3 grid((g.n[0] + 255) / 256, g.n[1], g.n[2]);
  if (nd == 3) k_curv_metric<3><<<grid, 256, 0, s>>>(X, M, g, ph, e[0], e[1], e[2]);
  else k_curv_metric<2><<<grid, 256, 0, s>>>(X, M, g, ph, e[0], e[1], e[2]);
  launch_halo_periodic(M, nd * nd + 1, g, s);
}

}  // namespace osbl
