// osbl_adjoint.hip -- discrete adjoint of the central (skew-symmetric) Euler
// RHS and of the 3-register RK3 step, on periodic blocks.
//
// Forward residual (parsing.py:75-111, scheme.py:187-252), per direction j:
//   R_m -= 1/2 [D_j(q_m u_j) + u_j D_j q_m + q_m D_j u_j]
//   R_{1+j} -= D_j p,   R_E -= D_j(p u_j)
// with u_j = q_{1+j}/rho, p = (gama-1)(q_E - rho |u|^2/2).  The central D_j
// has antisymmetric weights, so on a periodic grid D_j^T = -D_j and the
// vector-Jacobian product lambda = (dR/dQ)^T mu is again a stencil:
//   g_q[m] += 1/2 u_j D_j mu_m + 1/2 D_j(mu_m u_j) - 1/2 mu_m D_j u_j
//   g_u[j] += 1/2 sum_m q_m D_j mu_m - 1/2 sum_m mu_m D_j q_m
//             + 1/2 D_j(sum_m mu_m q_m) + p D_j mu_E
//   g_p    += D_j mu_{1+j} + u_j D_j mu_E
// followed by the chain rule through u_j and p.
#include "osbl_kernels.h"

namespace osbl {

template <int ND>
__global__ void __launch_bounds__(128) k_rhs_vjp(const double* __restrict__ Q, const double* __restrict__ P,
                                                 const double* __restrict__ M, double* __restrict__ out, Grid g,
                                                 Phys ph) {
  constexpr int NV = ND + 2, E = NV - 1;
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= g.n[0]) return;
  const int j0 = blockIdx.y, k0 = blockIdx.z;
  const int x = g.idx(i, j0, k0);
  const int st[3] = {1, g.pitch, g.plane};
  const long long fs = g.fs;
  double q[NV], mu[NV], u[ND];
#pragma unroll
  for (int m = 0; m < NV; ++m) {
    q[m] = Q[m * fs + x];
    mu[m] = M[m * fs + x];
  }
#pragma unroll
  for (int d = 0; d < ND; ++d) u[d] = P[d * fs + x];
  const double p = P[ND * fs + x];
  double gq[NV], gu[ND], gp = 0.0;
#pragma unroll
  for (int m = 0; m < NV; ++m) gq[m] = 0.0;
#pragma unroll
  for (int j = 0; j < ND; ++j) {
    const int sj = st[j];
    const double inv = ph.inv_delta[j];
    const int offs[4] = {x - 2 * sj, x - sj, x + sj, x + 2 * sj};
    constexpr double W1A = 1.0 / 12.0, W1B = 2.0 / 3.0;
    const double wts[4] = {W1A, -W1B, W1B, -W1A};
    double dmu[NV], dmuu[NV], dq[NV], dmuq = 0.0, duj = 0.0;
#pragma unroll
    for (int m = 0; m < NV; ++m) { dmu[m] = 0.0; dmuu[m] = 0.0; dq[m] = 0.0; }
#pragma unroll
    for (int s = 0; s < 4; ++s) {
      const int y = offs[s];
      const double w = wts[s];
      const double uj = P[j * fs + y];
      double sq = 0.0;
#pragma unroll
      for (int m = 0; m < NV; ++m) {
        const double my = M[m * fs + y], qy = Q[m * fs + y];
        dmu[m] += w * my;
        dmuu[m] += w * (my * uj);
        dq[m] += w * qy;
        sq += my * qy;
      }
      dmuq += w * sq;
      duj += w * uj;
    }
#pragma unroll
    for (int m = 0; m < NV; ++m) { dmu[m] *= inv; dmuu[m] *= inv; dq[m] *= inv; }
    dmuq *= inv;
    duj *= inv;
    double gu_j = 0.5 * dmuq + p * dmu[E];
#pragma unroll
    for (int m = 0; m < NV; ++m) {
      gq[m] += 0.5 * u[j] * dmu[m] + 0.5 * dmuu[m] - 0.5 * mu[m] * duj;
      gu_j += 0.5 * q[m] * dmu[m] - 0.5 * mu[m] * dq[m];
    }
    gu[j] = gu_j;
    gp += dmu[1 + j] + u[j] * dmu[E];
  }
  const double rho = q[0], ir = 1.0 / rho;
  double uu = 0.0;
#pragma unroll
  for (int d = 0; d < ND; ++d) uu += u[d] * u[d];
  const long long cells = (long long)g.n[0] * g.n[1] * g.n[2];
  const long long c = (long long)i + (long long)g.n[0] * (j0 + (long long)g.n[1] * k0);
  double l0 = gq[0] + gp * ph.gm1 * 0.5 * uu;
#pragma unroll
  for (int d = 0; d < ND; ++d) {
    l0 -= gu[d] * u[d] * ir;
    out[(1 + d) * cells + c] += gq[1 + d] + gu[d] * ir - gp * ph.gm1 * u[d];
  }
  out[c] += l0;
  out[E * cells + c] += gq[E] + gp * ph.gm1;
}

// out = a*x + b*y (packed arrays of n doubles); y may be null
__global__ void __launch_bounds__(256) k_lincomb(double* __restrict__ out, double a, const double* __restrict__ xv,
                                                  double b, const double* __restrict__ yv, long long n) {
  const long long t = (long long)blockIdx.x * blockDim.x + threadIdx.x;
  if (t >= n) return;
  double v = a * xv[t];
  if (yv) v += b * yv[t];
  out[t] = v;
}

// ---------------------------------------------------------------------------
// One reverse RK stage in one launch, on packed interior arrays with periodic
// wrap (no halo copies): the adjoint weights are mu = alpha*A + beta*B,
// formed on the fly at every stencil point, V = (dR/dQ at Qs)^T mu, and
//   out1 = c*(A + B) + V      (c = 0 or 1)
//   out2 = A + B              (when out2 is given)
// ---------------------------------------------------------------------------
template <int ND>
__global__ void __launch_bounds__(128) k_adj_stage(const double* __restrict__ Qs, const double* __restrict__ A,
                                                   const double* __restrict__ B, double alpha, double beta,
                                                   double c, double* __restrict__ out1, double* __restrict__ out2,
                                                   int n0, int n1, int n2, Phys ph) {
  constexpr int NV = ND + 2, E = NV - 1;
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n0) return;
  const int j0 = blockIdx.y, k0 = blockIdx.z;
  const long long cells = (long long)n0 * n1 * n2;
  const int nn[3] = {n0, n1, n2};
  const int co[3] = {i, j0, k0};
  const long long sd[3] = {1, n0, (long long)n0 * n1};
  const long long x = i + (long long)n0 * (j0 + (long long)n1 * k0);
  auto muv = [&](int m, long long y) {
    double v = alpha * A[m * cells + y];
    if (B) v += beta * B[m * cells + y];
    return v;
  };
  auto prim = [&](long long y, double* u, double& p, double* q) {
#pragma unroll
    for (int m = 0; m < NV; ++m) q[m] = Qs[m * cells + y];
    const double ir = 1.0 / q[0];
    double ke = 0.0;
#pragma unroll
    for (int d = 0; d < ND; ++d) {
      u[d] = q[1 + d] * ir;
      ke += u[d] * u[d];
    }
    p = ph.gm1 * (q[E] - 0.5 * q[0] * ke);
  };
  double q[NV], u[ND], p, mu[NV];
  prim(x, u, p, q);
#pragma unroll
  for (int m = 0; m < NV; ++m) mu[m] = muv(m, x);
  double gq[NV], gu[ND], gp = 0.0;
#pragma unroll
  for (int m = 0; m < NV; ++m) gq[m] = 0.0;
#pragma unroll
  for (int j = 0; j < ND; ++j) {
    const double inv = ph.inv_delta[j];
    constexpr double W1A = 1.0 / 12.0, W1B = 2.0 / 3.0;
    const int offs[4] = {-2, -1, 1, 2};
    const double wts[4] = {W1A, -W1B, W1B, -W1A};
    double dmu[NV], dmuu[NV], dq[NV], dmuq = 0.0, duj = 0.0;
#pragma unroll
    for (int m = 0; m < NV; ++m) { dmu[m] = 0.0; dmuu[m] = 0.0; dq[m] = 0.0; }
#pragma unroll
    for (int s = 0; s < 4; ++s) {
      int cj = co[j] + offs[s];
      cj = cj < 0 ? cj + nn[j] : (cj >= nn[j] ? cj - nn[j] : cj);
      const long long y = x + (long long)(cj - co[j]) * sd[j];
      const double w = wts[s];
      double qy[NV], uy[ND], py;
      prim(y, uy, py, qy);
      const double uj = uy[j];
      double sq = 0.0;
#pragma unroll
      for (int m = 0; m < NV; ++m) {
        const double my = muv(m, y);
        dmu[m] += w * my;
        dmuu[m] += w * (my * uj);
        dq[m] += w * qy[m];
        sq += my * qy[m];
      }
      dmuq += w * sq;
      duj += w * uj;
    }
#pragma unroll
    for (int m = 0; m < NV; ++m) { dmu[m] *= inv; dmuu[m] *= inv; dq[m] *= inv; }
    dmuq *= inv;
    duj *= inv;
    double gu_j = 0.5 * dmuq + p * dmu[E];
#pragma unroll
    for (int m = 0; m < NV; ++m) {
      gq[m] += 0.5 * u[j] * dmu[m] + 0.5 * dmuu[m] - 0.5 * mu[m] * duj;
      gu_j += 0.5 * q[m] * dmu[m] - 0.5 * mu[m] * dq[m];
    }
    gu[j] = gu_j;
    gp += dmu[1 + j] + u[j] * dmu[E];
  }
  const double ir = 1.0 / q[0];
  double uu = 0.0;
#pragma unroll
  for (int d = 0; d < ND; ++d) uu += u[d] * u[d];
  double v[NV];
  v[0] = gq[0] + gp * ph.gm1 * 0.5 * uu;
#pragma unroll
  for (int d = 0; d < ND; ++d) {
    v[0] -= gu[d] * u[d] * ir;
    v[1 + d] = gq[1 + d] + gu[d] * ir - gp * ph.gm1 * u[d];
  }
  v[E] = gq[E] + gp * ph.gm1;
#pragma unroll
  for (int m = 0; m < NV; ++m) {
    const double ab = A[m * cells + x] + (B ? B[m * cells + x] : 0.0);
    out1[m * cells + x] = c * ab + v[m];
    if (out2) out2[m * cells + x] = ab;
  }
}

// ---------------------------------------------------------------------------
// The same on 2-D blocks in one tiled kernel, with the viscous terms' VJP (the
// formulas of osbl_adjoint_visc.hip): a workgroup takes 16 x 16 cells and
// stages rho, u, rhoE and mu = alpha A + beta B of the points around them in
// LDS (two layers; four with viscous terms), forms w and 2 mu_E tau on the
// cells and two layers, and finishes every cell.
//   EULER: out1 = c (A + B) + V and out2 as k_adj_stage, V with the viscous
//   part when VISC; otherwise out1 += the viscous part alone.
//
// What bounds it is one tile's latency at three workgroups a CU, and the points
// staged more than once (2.25 per cell).  512^2, central, viscous, under the
// profiler: stage 23.5, padded copies 8.0, w and tau 11.5, viscous part 12.2 us
// -> 34 us in one launch.
// ---------------------------------------------------------------------------
constexpr int A2C = 16;

template <bool EULER, bool VISC>
__global__ void __launch_bounds__(256, VISC ? 3 : 4) k_adj_tile2d(const double* __restrict__ Qs,
                                                                  const double* __restrict__ A,
                                                                  const double* __restrict__ B, double alpha,
                                                                  double beta, double c, double* __restrict__ out1,
                                                                  double* __restrict__ out2, int n0, int n1, Phys ph) {
  constexpr int NV = 4, E = 3;
  constexpr int H = VISC ? 4 : 2, PX = A2C + 2 * H, NP = PX * PX;  // staged points
  constexpr int MX = A2C + 4, NM = VISC ? MX * MX : 1;             // points of w and tau
  constexpr int U = 0, MU = 1;                                     // fields of S: MU + m is mu_m, m > 0
  constexpr int TX = A2C + 4;                                      // rho, rhoE, mu_0: the cells and two layers
  // odd strides: no bank conflicts along x.  49 KB with viscous terms: three
  // workgroups a CU (two, with eight fields at every point, took as long)
  __shared__ double S[NP][5];       // u, mu_1, mu_2, mu_E
  __shared__ double T[TX * TX][3];  // rho, rhoE, mu_0
  __shared__ double W[NM][5];       // w, 2 mu_E tau_00, _01, _11
  const int t = threadIdx.x, i = t % A2C, j = t / A2C;
  const int x0 = blockIdx.x * A2C, y0 = blockIdx.y * A2C;
  const long long cells = (long long)n0 * n1;
  // a tile's points beyond the block's reach (n + H - 1) feed no cell
  auto image = [](int a, int n) {
    a = min(a, n + H - 1);
    return a < 0 ? a + n : (a >= n ? a - n : a);
  };
#pragma unroll
  for (int k = 0; k < (NP + 255) / 256; ++k) {
    const int p = t + 256 * k;
    if (p < NP) {
      const long long y = image(x0 - H + p % PX, n0) + (long long)n0 * image(y0 - H + p / PX, n1);
      double q[NV], mu[NV];
#pragma unroll
      for (int m = 0; m < NV; ++m) {
        q[m] = Qs[m * cells + y];
        mu[m] = alpha * A[m * cells + y];
        if (B) mu[m] = __fma_rn(beta, B[m * cells + y], mu[m]);
      }
      const double ir = recip_pos(q[0]);
      S[p][U] = q[1] * ir;
      S[p][U + 1] = q[2] * ir;
#pragma unroll
      for (int m = 1; m < NV; ++m) S[p][MU + m] = mu[m];
      const int tx = p % PX - (H - 2), ty = p / PX - (H - 2);
      if (tx >= 0 && ty >= 0 && tx < TX && ty < TX) {
        T[ty * TX + tx][0] = q[0];
        T[ty * TX + tx][1] = q[E];
        T[ty * TX + tx][2] = mu[0];
      }
    }
  }
  __syncthreads();
  constexpr double WA = 1.0 / 12.0, WB = 2.0 / 3.0;
  // first, second and mixed derivative (without 1/Delta) at o of f(point), rows st and PR apart
  auto d1 = [&](int o, int st, auto&& f) {
    return WA * (f(o - 2 * st) - f(o + 2 * st)) + WB * (f(o + st) - f(o - st));
  };
  auto d2 = [&](int o, int st, auto&& f) {
    return (-1.0 / 12.0) * (f(o - 2 * st) + f(o + 2 * st)) + (4.0 / 3.0) * (f(o - st) + f(o + st)) - 2.5 * f(o);
  };
  auto dmix = [&](int o, int row, auto&& f) { return d1(o, row, [&](int z) { return d1(z, 1, f); }); };
  // the loads of a part stay in it, so that few registers hold points
  auto part = [](double& v) {
    asm volatile("" : "+v"(v) : : "memory");
    __builtin_amdgcn_sched_barrier(0);
  };
  const double id0 = ph.inv_delta[0], id1 = ph.inv_delta[1];
  if constexpr (VISC) {
#pragma unroll
    for (int k = 0; k < (NM + 255) / 256; ++k) {
      const int p = t + 256 * k;
      if (p < NM) {
        const int o = (p / MX + 2) * PX + p % MX + 2;
        auto u0 = [&](int z) { return S[z][U]; };
        auto u1 = [&](int z) { return S[z][U + 1]; };
        const double d00 = id0 * d1(o, 1, u0), d01 = id1 * d1(o, PX, u0);
        const double d10 = id0 * d1(o, 1, u1), d11 = id1 * d1(o, PX, u1);
        const double muE = S[o][MU + E], f = 2.0 * muE * ph.inv_re, div = (2.0 / 3.0) * (d00 + d11);
        W[p][0] = __fma_rn(muE, S[o][U], S[o][MU + 1]);
        W[p][1] = __fma_rn(muE, S[o][U + 1], S[o][MU + 2]);
        W[p][2] = f * (2.0 * d00 - div);
        W[p][3] = f * (d01 + d10);
        W[p][4] = f * (2.0 * d11 - div);
      }
    }
    __syncthreads();
  }
  const int cx = x0 + i, cy = y0 + j;
  if (cx >= n0 || cy >= n1) return;
  const long long x = cx + (long long)n0 * cy;
  const int o = (j + H) * PX + i + H, to = (j + 2) * TX + i + 2;
  const double rho = T[to][0], ir = recip_pos(rho);
  const double u[2] = {S[o][U], S[o][U + 1]};
  const double uu = u[0] * u[0] + u[1] * u[1];
  const double p = ph.gm1 * (T[to][1] - 0.5 * rho * uu);
  double gq[NV] = {0.0, 0.0, 0.0, 0.0}, gu[2] = {0.0, 0.0}, gp = 0.0;
  if constexpr (EULER) {
    double q[NV], mu[NV];
    q[0] = rho;
    q[1] = rho * u[0];
    q[2] = rho * u[1];
    q[E] = T[to][1];
    mu[0] = T[to][2];
#pragma unroll
    for (int m = 1; m < NV; ++m) mu[m] = S[o][MU + m];
#pragma unroll
    for (int d = 0; d < 2; ++d) {
      const int st = d == 0 ? 1 : PX;
      double dmu[NV] = {0.0, 0.0, 0.0, 0.0}, dmuu[NV] = {0.0, 0.0, 0.0, 0.0};
      double duj = 0.0, dmuq = 0.0, mdq = 0.0;  // D u_j, D(mu.q), mu.D q
#pragma unroll
      for (int k = 0; k < 4; ++k) {
        const int off[4] = {-2, -1, 1, 2};
        const double w4[4] = {WA, -WB, WB, -WA};
        const double* y = S[o + off[k] * st];
        const double* z = T[to + off[k] * (d == 0 ? 1 : TX)];
        const double w = w4[k], wu = w * y[U + d], r = z[0];
        const double qy[NV] = {r, r * y[U], r * y[U + 1], z[1]};
        double sq = 0.0, sm = 0.0;
#pragma unroll
        for (int m = 0; m < NV; ++m) {
          const double my = m == 0 ? z[2] : y[MU + m];
          dmu[m] = __fma_rn(w, my, dmu[m]);
          dmuu[m] = __fma_rn(wu, my, dmuu[m]);
          sq = __fma_rn(my, qy[m], sq);
          sm = __fma_rn(mu[m], qy[m], sm);
        }
        dmuq = __fma_rn(w, sq, dmuq);
        mdq = __fma_rn(w, sm, mdq);
        duj += wu;
      }
      const double inv = ph.inv_delta[d];
      double qdm = 0.0;
#pragma unroll
      for (int m = 0; m < NV; ++m) {
        gq[m] = __fma_rn(0.5 * inv, u[d] * dmu[m] + dmuu[m] - mu[m] * duj, gq[m]);
        qdm = __fma_rn(q[m], dmu[m], qdm);
        asm volatile("" : "+v"(gq[m]));
      }
      gu[d] = inv * (0.5 * (dmuq - mdq + qdm) + p * dmu[E]);
      gp = __fma_rn(inv, __fma_rn(u[d], dmu[E], dmu[1 + d]), gp);
      asm volatile("" : "+v"(gu[d]));
      part(gp);
    }
  }
  double gT = 0.0;
  if constexpr (VISC) {
    const int mo = (j + 2) * MX + i + 2;
    const double muE = S[o][MU + E], id[2] = {id0, id1};
#pragma unroll
    for (int k = 0; k < 2; ++k) {
      // (sum_j M_jj w_k + 1/3 sum_m M_mk w_m) / Re - sum_b D_b(2 mu_E tau_kb), and mu_E times the same of u
      auto wk = [&](int z) { return W[z][k]; };
      auto wo = [&](int z) { return W[z][1 - k]; };
      auto uk = [&](int z) { return S[z][U + k]; };
      auto uo = [&](int z) { return S[z][U + 1 - k]; };
      double c0 = id0 * id0, c1 = id1 * id1;
      (k == 0 ? c0 : c1) *= 4.0 / 3.0;
      const double cm = (1.0 / 3.0) * id0 * id1;
      double vw = c0 * d2(mo, 1, wk) + c1 * d2(mo, MX, wk) + cm * dmix(mo, MX, wo);
      part(vw);
      double vu = c0 * d2(o, 1, uk) + c1 * d2(o, PX, uk) + cm * dmix(o, PX, uo);
      part(vu);
      double s = ph.inv_re * __fma_rn(muE, vu, vw);
      s -= id[0] * d1(mo, 1, [&](int z) { return W[z][2 + k]; });
      s -= id[1] * d1(mo, MX, [&](int z) { return W[z][3 + k]; });
      gu[k] += s;
      part(gu[k]);
    }
    auto me = [&](int z) { return S[z][MU + E]; };
    gT = ph.cq * (id0 * id0 * d2(o, 1, me) + id1 * id1 * d2(o, PX, me));
  }
  // chain rule through u = rhou / rho, p and T = gama Minf^2 p / rho
  double v[NV];
  v[0] = gq[0];
  if constexpr (VISC) {
    const double gM = ph.gama * ph.Minf * ph.Minf * ir;
    gp = __fma_rn(gT, gM, gp);
    v[0] -= gT * (p * gM) * ir;
  }
  v[0] += gp * ph.gm1 * 0.5 * uu;
#pragma unroll
  for (int d = 0; d < 2; ++d) {
    v[0] -= gu[d] * u[d] * ir;
    v[1 + d] = gq[1 + d] + gu[d] * ir - gp * ph.gm1 * u[d];
  }
  v[E] = gq[E] + gp * ph.gm1;
#pragma unroll
  for (int m = 0; m < NV; ++m) {
    if constexpr (EULER) {
      const double ab = A[m * cells + x] + (B ? B[m * cells + x] : 0.0);
      out1[m * cells + x] = c * ab + v[m];
      if (out2) out2[m * cells + x] = ab;
    } else {
      out1[m * cells + x] += v[m];
    }
  }
}

void launch_adj_tile2d(bool euler, bool visc, const double* Qs, const double* A, const double* B, double alpha,
                       double beta, double c, double* out1, double* out2, const Grid& g, const Phys& ph,
                       hipStream_t s) {
  const dim3 grid((g.n[0] + A2C - 1) / A2C, (g.n[1] + A2C - 1) / A2C);
  auto go = [&](auto ee, auto vv) {
    k_adj_tile2d<decltype(ee)::value, decltype(vv)::value>
        <<<grid, 256, 0, s>>>(Qs, A, B, alpha, beta, c, out1, out2, g.n[0], g.n[1], ph);
  };
  if (!euler) go(std::false_type{}, std::true_type{});
  else if (visc) go(std::true_type{}, std::true_type{});
  else go(std::true_type{}, std::false_type{});
}

void launch_adj_stage(int nd, const double* Qs, const double* A, const double* B, double alpha, double beta, double c,
                      double* out1, double* out2, const Grid& g, const Phys& ph, hipStream_t s) {
  dim3 grid((g.n[0] + 127) / 128, g.n[1], g.n[2]);
  if (nd == 3) k_adj_stage<3><<<grid, 128, 0, s>>>(Qs, A, B, alpha, beta, c, out1, out2, g.n[0], g.n[1], g.n[2], ph);
  else k_adj_stage<1><<<grid, 128, 0, s>>>(Qs, A, B, alpha, beta, c, out1, out2, g.n[0], g.n[1], g.n[2], ph);
}

// pack every variable of a bundle into contiguous interior blocks in one launch
__global__ void __launch_bounds__(256) k_pack_all(const double* __restrict__ F, double* __restrict__ out, Grid g, int nv) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= g.n[0]) return;
  const int j = blockIdx.y, k = blockIdx.z;
  const long long cells = (long long)g.n[0] * g.n[1] * g.n[2];
  const long long c = (long long)i + (long long)g.n[0] * (j + (long long)g.n[1] * k);
  const int x = g.idx(i, j, k);
  for (int m = 0; m < nv; ++m) out[m * cells + c] = F[m * g.fs + x];
}

void launch_pack_all(const double* F, double* out, const Grid& g, int nv, hipStream_t s) {
  dim3 grid((g.n[0] + 255) / 256, g.n[1], g.n[2]);
  k_pack_all<<<grid, 256, 0, s>>>(F, out, g, nv);
}

void launch_rhs_vjp(int nd, const double* Q, const double* P, const double* M, double* out, const Grid& g,
                    const Phys& ph, hipStream_t s) {
  dim3 grid((g.n[0] + 127) / 128, g.n[1], g.n[2]);
  if (nd == 3) k_rhs_vjp<3><<<grid, 128, 0, s>>>(Q, P, M, out, g, ph);
  else if (nd == 2) k_rhs_vjp<2><<<grid, 128, 0, s>>>(Q, P, M, out, g, ph);
  else k_rhs_vjp<1><<<grid, 128, 0, s>>>(Q, P, M, out, g, ph);
}

void launch_lincomb(double* out, double a, const double* x, double b, const double* y, long long n, hipStream_t s) {
  k_lincomb<<<(unsigned)((n + 255) / 256), 256, 0, s>>>(out, a, x, b, y, n);
}

}  // namespace osbl
