// osbl_tile2d.hip -- one stage of a 2-D block in one kernel.  Characteristic
// schemes: both sweeps, the viscous terms with closures, metric and mu(T), the
// body force, the adaptive TENO's sensor, and the RK update.  Central schemes
// (uniform grid, no closures): convective and viscous terms and the RK update.
#include "osbl_kernels.h"
#include "osbl_visc.h"

namespace osbl {

namespace {

constexpr int T2C = 15, T2P = T2C + 6;  // cells and staged points per side

}  // namespace

// ---------------------------------------------------------------------------
// A workgroup takes 15 x 15 cells.  The 21 x 21 points around them are staged
// in LDS with their constituent relations, once for both directions; thread
// (i, j) evaluates the flux left of cell i in row j (x) and below cell j in
// column i - 1 (y), 16 interfaces per 15 cells, and finishes cell (i - 1, j):
// its left flux comes from the lane below, its upper one through LDS.  The
// same points serve the sensor (evaluated at the left points of the
// interfaces, 16 x 16) and the viscous terms; the residual stays in registers.
// The last tile of a direction is moved back so that it ends with the block
// (its cells that another tile owns are left alone): the one-sided closure
// rows reach at most six points inward and so stay inside the tile.
//
// What bounds it is FP64 issue at three waves per SIMD; small blocks are bound
// by the launch and one tile's latency.  400^2 Euler stage: 16 us in three
// launches -> 11 us; 500x250 with sensor, Sutherland viscosity, closures and
// metric: five launches -> one.
//
// mode as k_update (2: residual into R).  wrap: periodic in both directions,
// points are read at their periodic images and the halos need not be filled.
// SENSOR: theta is formed here and left in TH (interior).  PK, when given,
// takes the packed stage input (the adjoint's; a pass of 5.5 us at 512^2).
// ---------------------------------------------------------------------------
template <int CONV, int AVG, bool VISC, bool SENSOR>
__global__ void __launch_bounds__(256, 3) k_char_tile2d(const double* __restrict__ Q, double* __restrict__ R,
                                                        double* __restrict__ Qo, double* __restrict__ Qn, Grid g,
                                                        Phys ph, Bnd b, double cA, double cB, int first, int mode,
                                                        double* __restrict__ TH, int suth, int wrap,
                                                        double* __restrict__ PK) {
  constexpr int ND = 2, NV = 4;
  constexpr bool ROE = AVG == OSBL_AVG_ROE;
  constexpr int NF = NV + ND + 2 + ((ROE || VISC) ? 2 : 0);  // q, u, p, a (, sqrt(rho), sqrt(rho) H; then T, mu)
  constexpr int NS = NF | 1;                                 // odd stride: no bank conflicts along x
  __shared__ double S[T2P * T2P][NS];
  __shared__ double Fy[NV][256];
  __shared__ double W[VISC || SENSOR ? CW_SIZE : 1];
  const int t = threadIdx.x, i = t & 15, j = t >> 4;
  const int bx = blockIdx.x * T2C, by = blockIdx.y * T2C;  // first own cell
  const int x0 = min(bx, max(g.n[0] - T2C, 0)), y0 = min(by, max(g.n[1] - T2C, 0));
  auto image = [&](int a, int n) { return !wrap ? a : (a < 0 ? a + n : (a >= n ? a - n : a)); };
  // point (px, py) of the tile is (x0 - 3 + px, y0 - 3 + py); those beyond
  // the block's reach (n + 2) feed no cell
  double nq[2][NV];
#pragma unroll
  for (int k = 0; k < 2; ++k) {
    const int p = min(t + 256 * k, T2P * T2P - 1);
    const int gx = min(x0 - 3 + p % T2P, g.n[0] + 2), gy = min(y0 - 3 + p / T2P, g.n[1] + 2);
    fetch_q<ND>(nq[k], Q, g.fs, g.idx(image(gx, g.n[0]), image(gy, g.n[1]), 0));
  }
  if constexpr (VISC || SENSOR)
    if (t < CW_SIZE) W[t] = b.cw[t];
  const int cx = x0 + i - 1, cy = y0 + j;
  const int x = g.idx(cx, cy, 0);
  const bool own = i > 0 && j < T2C && cx >= bx && cy >= by && cx < g.n[0] && cy < g.n[1];
  double qo[NV] = {0.0, 0.0, 0.0, 0.0};
  if (own && (mode == 0 ? !first : (mode == 1 && cA != 0.0))) {
#pragma unroll
    for (int m = 0; m < NV; ++m) qo[m] = Qo[m * g.fs + x];
  }
#pragma unroll
  for (int k = 0; k < 2; ++k) {
    const int p = t + 256 * k;
    Pt<ND> s;
#pragma unroll
    for (int m = 0; m < NV; ++m) s.q[m] = nq[k][m];
    finish_pt<ND>(s, ph);
    double sq = 0.0, h = 0.0;
    if constexpr (ROE) roe_factors<ND>(s, sq, h);
    if (p < T2P * T2P) {
#pragma unroll
      for (int m = 0; m < NV; ++m) S[p][m] = s.q[m];
      S[p][4] = s.u[0];
      S[p][5] = s.u[1];
      S[p][6] = s.p;
      S[p][7] = s.a;
      if constexpr (ROE) {
        S[p][8] = sq;
        S[p][9] = h;
      }
    }
  }
  __syncthreads();

  // derivative of order ORDER in the computational coordinate (without
  // 1/Delta) of f(point) along d, at tile point p with grid index c: dxi of
  // the per-point kernels with the closure rows in LDS
  auto deriv = [&](auto order, int d, int c, int p, auto&& f) {
    constexpr int ORDER = decltype(order)::value;
    const int st = d == 0 ? 1 : T2P, N = g.n[d], lo = b.mod[d][0], hi = b.mod[d][1], r = N - 1 - c;
    const int nlo = ORDER == 2 ? 2 : (lo == 1 ? 4 : 2), nhi = ORDER == 2 ? 2 : (hi == 1 ? 4 : 2);
    const bool at_lo = lo && c >= 0 && c < nlo, at_hi = !at_lo && hi && r >= 0 && r < nhi;
    if (at_lo || at_hi) {
      const int bs = at_lo ? lo : hi, k0 = at_lo ? c : r, s = at_lo ? st : -st;
      const double* w = W + (ORDER == 2 ? CW_D2 : (bs == 1 ? CW_CARP : CW_RA)) + 6 * k0;
      const int np = ORDER == 1 && bs == 1 ? 6 : 5;
      double acc = 0.0;
      for (int k = 0; k < np; ++k) acc += w[k] * f(p + (k - k0) * s);
      return at_hi && ORDER == 1 ? -acc : acc;
    }
    if constexpr (ORDER == 1) return (1.0 / 12.0) * (f(p - 2 * st) - f(p + 2 * st)) + (2.0 / 3.0) * (f(p + st) - f(p - st));
    else return (-1.0 / 12.0) * (f(p - 2 * st) + f(p + 2 * st)) + (4.0 / 3.0) * (f(p - st) + f(p + st)) - 2.5 * f(p);
  };
  using One = std::integral_constant<int, 1>;
  using Sec = std::integral_constant<int, 2>;

  if constexpr (SENSOR) {
    // the modified Ducros sensor (k_sensor) at point (x0 - 1 + i, y0 - 1 + j),
    // where an own interface has its left point
    const int px = x0 - 1 + i, py = y0 - 1 + j, p = (j + 2) * T2P + i + 2;
    double th = 0.0;
    if (px >= bx - 1 && py >= by - 1 && px < g.n[0] + 1 && py < g.n[1] + 1) {
      auto metric = [&](int d, int c) {
        if (!b.dm[d]) return 1.0;
        const int N = g.n[d];
        if (c < 0) c = -c;
        if (c > N - 1) c = 2 * (N - 1) - c;
        return b.dm[d][c];
      };
      double du[2][2];
#pragma unroll
      for (int m = 0; m < 2; ++m) {
        auto u = [&](int q) { return S[q][4 + m]; };
        du[m][0] = metric(0, px) * (ph.inv_delta[0] * deriv(One{}, 0, px, p, u));
        du[m][1] = metric(1, py) * (ph.inv_delta[1] * deriv(One{}, 1, py, p, u));
      }
      const double div = du[0][0] + du[1][1], w = du[1][0] - du[0][1];
      const double filt = 0.5 * (1.0 - tanh(2.5 * (1.0 + 100.0 * div)));
      th = filt * (div * div) / (div * div + w * w + ph.sensor_eps);
      if (px >= bx && py >= by && px < min(x0 + T2C, g.n[0]) && py < min(y0 + T2C, g.n[1])) TH[g.idx(px, py, 0)] = th;
    }
    Fy[0][t] = th;
    __syncthreads();
  }
  auto flux = [&](auto dc, int p0, int th, double (&fh)[NV]) {
    constexpr int D = decltype(dc)::value, ST = D == 0 ? NS : T2P * NS, PS = D == 0 ? 1 : T2P;
    [[maybe_unused]] RoeF rf{};
    if constexpr (ROE) rf = RoeF{S[p0 + 2 * PS][8], S[p0 + 2 * PS][9], S[p0 + 3 * PS][8], S[p0 + 3 * PS][9]};
    double ct = ph.teno_ct;
    if constexpr (SENSOR) ct = adaptive_ct(Fy[0][th], ph);
    char_flux_w<ND, D, CONV, AVG, true>(LdsPoints<ND, ST>{S[p0]}, ph, fh, ct, rf);
  };
  double r[NV], f[NV];
  const int jr = min(j, T2C - 1), ic = max(i, 1);
  flux(std::integral_constant<int, 0>{}, (jr + 3) * T2P + i, (jr + 1) * 16 + i, f);
  const double g0 = b.dm[0] && own ? ph.inv_delta[0] * b.dm[0][cx] : ph.inv_delta[0];
#pragma unroll
  for (int m = 0; m < NV; ++m) r[m] = (__shfl_up(f[m], 1) - f[m]) * g0;
  flux(std::integral_constant<int, 1>{}, j * T2P + ic + 2, j * 16 + ic, f);
  __syncthreads();  // the sensor's values and the Roe factors have been read
#pragma unroll
  for (int m = 0; m < NV; ++m) Fy[m][t] = f[m];
  if constexpr (VISC) {
    // T and mu(T) of the staged points take the Roe factors' place
#pragma unroll
    for (int k = 0; k < 2; ++k) {
      const int p = t + 256 * k;
      if (p < T2P * T2P) {
        const double T = S[p][6] * ph.gama * ph.Minf * ph.Minf * recip_pos(S[p][0]);
        S[p][8] = T;
        S[p][9] = suth ? T * sqrt_pos(T) * quot_pos(1.0 + ph.suth, T + ph.suth) : 1.0;
      }
    }
  }
  __syncthreads();
  if (!own) return;
  const double g1 = b.dm[1] ? ph.inv_delta[1] * b.dm[1][cy] : ph.inv_delta[1];
  const int pc = (j + 3) * T2P + i + 2;
#pragma unroll
  for (int m = 0; m < NV; ++m) r[m] = __fma_rn(f[m] - Fy[m][t + 16], g1, r[m]);
  if constexpr (VISC) {
    const int ci[2] = {cx, cy};
    const bool metric = b.dm[0] || b.dm[1];
    double DU[2][2], DD[2][2][2], D2T[2], DT[2], DMU[2];
#pragma unroll
    for (int d = 0; d < 2; ++d) {
      const double id = ph.inv_delta[d];
      const double G = b.dm[d] ? b.dm[d][ci[d]] : 1.0, H = b.sd[d] ? b.sd[d][ci[d]] : 0.0;
      auto both = [&](int fld, double& first_, double& second_) {
        auto v = [&](int q) { return S[q][fld]; };
        const double d1 = id * deriv(One{}, d, ci[d], pc, v), d2 = id * id * deriv(Sec{}, d, ci[d], pc, v);
        first_ = G * d1;
        second_ = G * G * d2 + G * H * d1;
      };
#pragma unroll
      for (int m = 0; m < 2; ++m) both(4 + m, DU[m][d], DD[m][d][d]);
      both(8, DT[d], D2T[d]);
      DMU[d] = suth ? G * (id * deriv(One{}, d, ci[d], pc, [&](int q) { return S[q][9]; })) : 0.0;
    }
#pragma unroll
    for (int m = 0; m < 2; ++m) {  // D_1(D_0 u_m)
      auto inner = [&](int q) {
        return ph.inv_delta[0] * deriv(One{}, 0, cx, q, [&](int z) { return S[z][4 + m]; });
      };
      double v = ph.inv_delta[1] * deriv(One{}, 1, cy, pc, inner);
      if (metric) v *= (b.dm[0] ? b.dm[0][cx] : 1.0) * (b.dm[1] ? b.dm[1][cy] : 1.0);
      DD[m][0][1] = DD[m][1][0] = v;
    }
    const double um[3] = {S[pc][4], S[pc][5], 0.0};
    viscous_assemble<2>(S[pc][9], um, DU, DD, D2T, DT, DMU, ph, suth != 0, r);
  }
  if constexpr (CONV != CONV_WFILTER) {  // the filter's R holds flux differences alone
    if (ph.has_force) {
      r[1] -= ph.force[0];
      r[2] -= ph.force[1];
      r[3] -= ph.force[0] * S[pc][4] + ph.force[1] * S[pc][5];
    }
  }
  if (PK) {
#pragma unroll
    for (int m = 0; m < NV; ++m) PK[((long long)m * g.n[1] + cy) * g.n[0] + cx] = S[pc][m];
  }
#pragma unroll
  for (int m = 0; m < NV; ++m) {
    if (mode == 2) {
      R[m * g.fs + x] = r[m];
    } else if (mode == 0) {
      const double o = first ? S[pc][m] : qo[m];
      Qn[m * g.fs + x] = __fma_rn(ph.dt * cA, r[m], o);
      Qo[m * g.fs + x] = __fma_rn(ph.dt * cB, r[m], o);
    } else {
      const double tmp = __fma_rn(ph.dt, r[m], cA * qo[m]);
      Qo[m * g.fs + x] = tmp;
      Qn[m * g.fs + x] = __fma_rn(cB, tmp, S[pc][m]);
    }
  }
}

// ---------------------------------------------------------------------------
// Central schemes.  A workgroup takes 32 x 8 cells (a wave: two rows of 32, so
// stores are whole cache lines) and stages the 36 x 12 points around them in
// LDS with their constituent relations; mode and wrap as above.  The terms are
// those of central_convective and viscous_terms, the skew-symmetric form
// summed point by point: sum_y w (q_m(y) (u_j(y) + u_j(x)) + q_m(x) u_j(y)).
//
// What bounds it is one tile's latency on small blocks, memory on large ones.
// 512^2, skew, viscous, under the profiler: halo pass 4.6 + constituent
// relations 7.0 + update 14.5 us -> 11.5 us in one launch.
// ---------------------------------------------------------------------------
constexpr int C2X = 32, C2Y = 8, C2PX = C2X + 4, C2PY = C2Y + 4, C2P = C2PX * C2PY;

template <int CONV, bool VISC>
__global__ void __launch_bounds__(256, 4) k_central2d(const double* __restrict__ Q, double* __restrict__ R,
                                                      double* __restrict__ Qo, double* __restrict__ Qn, Grid g,
                                                      Phys ph, double cA, double cB, int first, int mode, int wrap,
                                                      double* __restrict__ PK) {
  constexpr int ND = 2, NV = 4, E = 3;
  __shared__ double S[C2P][9];  // q, u, p, T; odd stride: no bank conflicts along x
  const int t = threadIdx.x, i = t % C2X, j = t / C2X;
  const int x0 = blockIdx.x * C2X, y0 = blockIdx.y * C2Y;
  auto image = [&](int a, int n) { return !wrap ? a : (a < 0 ? a + n : (a >= n ? a - n : a)); };
  double nq[2][NV];
#pragma unroll
  for (int k = 0; k < 2; ++k) {
    const int p = min(t + 256 * k, C2P - 1);
    const int gx = min(x0 - 2 + p % C2PX, g.n[0] + 1), gy = min(y0 - 2 + p / C2PX, g.n[1] + 1);
    fetch_q<ND>(nq[k], Q, g.fs, g.idx(image(gx, g.n[0]), image(gy, g.n[1]), 0));
  }
  const int cx = x0 + i, cy = y0 + j;
  const bool own = cx < g.n[0] && cy < g.n[1];
  const int x = g.idx(cx, cy, 0);
  double qo[NV] = {0.0, 0.0, 0.0, 0.0};
  if (own && (mode == 0 ? !first : (mode == 1 && cA != 0.0))) {
#pragma unroll
    for (int m = 0; m < NV; ++m) qo[m] = Qo[m * g.fs + x];
  }
#pragma unroll
  for (int k = 0; k < 2; ++k) {
    const int p = t + 256 * k;
    const double ir = recip_pos(nq[k][0]);
    const double u0 = nq[k][1] * ir, u1 = nq[k][2] * ir;
    const double pr = ph.gm1 * (nq[k][E] - 0.5 * (nq[k][1] * u0 + nq[k][2] * u1));
    if (p < C2P) {
#pragma unroll
      for (int m = 0; m < NV; ++m) S[p][m] = nq[k][m];
      S[p][4] = u0;
      S[p][5] = u1;
      S[p][6] = pr;
      S[p][7] = pr * ph.gama * ph.Minf * ph.Minf * ir;
    }
  }
  __syncthreads();
  if (!own) return;
  const int pc = (j + 2) * C2PX + i + 2;
  constexpr double WA = 1.0 / 12.0, WB = 2.0 / 3.0;
  // the loads of a part stay in it, so that few registers hold points
  auto part = [] {
    asm volatile("" ::: "memory");
    __builtin_amdgcn_sched_barrier(0);
  };
  double q[NV], r[NV] = {0.0, 0.0, 0.0, 0.0};
#pragma unroll
  for (int m = 0; m < NV; ++m) q[m] = S[pc][m];
#pragma unroll
  for (int d = 0; d < 2; ++d) {
    const int st = d == 0 ? 1 : C2PX;
    const double uc = S[pc][4 + d], id = ph.inv_delta[d];
    double a[NV] = {0.0, 0.0, 0.0, 0.0}, su = 0.0, sp = 0.0, spu = 0.0;
#pragma unroll
    for (int k = 0; k < 4; ++k) {
      const int off[4] = {-2, -1, 1, 2};
      const double w4[4] = {WA, -WB, WB, -WA};
      const double* y = S[pc + off[k] * st];
      const double w = w4[k], u = y[4 + d], p = y[6];
      if constexpr (CONV == OSBL_CONV_CENTRAL_SKEW) {
        const double wu = w * (u + uc);
#pragma unroll
        for (int m = 0; m < NV; ++m) a[m] = __fma_rn(wu, y[m], a[m]);
        su = __fma_rn(w, u, su);
        spu = __fma_rn(w * u, p, spu);
      } else {
        const double wu = w * u;
        a[0] = __fma_rn(w, y[1 + d], a[0]);
#pragma unroll
        for (int m = 1; m < E; ++m) a[m] = __fma_rn(wu, y[m], a[m]);
        a[E] = __fma_rn(wu, y[E] + p, a[E]);
      }
      sp = __fma_rn(w, p, sp);
    }
#pragma unroll
    for (int m = 0; m < NV; ++m) {
      double s = CONV == OSBL_CONV_CENTRAL_SKEW ? 0.5 * __fma_rn(q[m], su, a[m]) : a[m];
      if (m == 1 + d) s += sp;
      if (m == E) s += spu;
      r[m] = __fma_rn(-id, s, r[m]);
      asm volatile("" : "+v"(r[m]));
    }
    part();
  }
  if constexpr (VISC) {
    auto d1 = [&](int st, auto&& f) {
      return WA * (f(pc - 2 * st) - f(pc + 2 * st)) + WB * (f(pc + st) - f(pc - st));
    };
    auto d2 = [&](int st, auto&& f) {
      return (-1.0 / 12.0) * (f(pc - 2 * st) + f(pc + 2 * st)) + (4.0 / 3.0) * (f(pc - st) + f(pc + st)) - 2.5 * f(pc);
    };
    double DU[2][2], DD[2][2][2], D2T[2];
    const double none[2] = {0.0, 0.0};
#pragma unroll
    for (int m = 0; m < 2; ++m) {
      auto v = [&](int z) { return S[z][4 + m]; };
#pragma unroll
      for (int d = 0; d < 2; ++d) {
        const int st = d == 0 ? 1 : C2PX;
        const double id = ph.inv_delta[d];
        DU[m][d] = id * d1(st, v);
        DD[m][d][d] = id * id * d2(st, v);
        asm volatile("" : "+v"(DU[m][d]), "+v"(DD[m][d][d]));
      }
      // D_1(D_0 u_m)
      auto inner = [&](int z) {
        return WA * (S[z - 2][4 + m] - S[z + 2][4 + m]) + WB * (S[z + 1][4 + m] - S[z - 1][4 + m]);
      };
      double mix = ph.inv_delta[0] * ph.inv_delta[1] * d1(C2PX, inner);
      asm volatile("" : "+v"(mix));
      DD[m][0][1] = DD[m][1][0] = mix;
      part();
    }
#pragma unroll
    for (int d = 0; d < 2; ++d)
      D2T[d] = ph.inv_delta[d] * ph.inv_delta[d] * d2(d == 0 ? 1 : C2PX, [&](int z) { return S[z][7]; });
    const double um[3] = {S[pc][4], S[pc][5], 0.0};
    viscous_assemble<2>(1.0, um, DU, DD, D2T, none, none, ph, false, r);
  }
  if (PK) {
#pragma unroll
    for (int m = 0; m < NV; ++m) PK[((long long)m * g.n[1] + cy) * g.n[0] + cx] = q[m];
  }
#pragma unroll
  for (int m = 0; m < NV; ++m) {
    if (mode == 2) {
      R[m * g.fs + x] = r[m];
    } else if (mode == 0) {
      const double o = first ? q[m] : qo[m];
      Qn[m * g.fs + x] = __fma_rn(ph.dt * cA, r[m], o);
      Qo[m * g.fs + x] = __fma_rn(ph.dt * cB, r[m], o);
    } else {
      const double tmp = __fma_rn(ph.dt, r[m], cA * qo[m]);
      Qo[m * g.fs + x] = tmp;
      Qn[m * g.fs + x] = __fma_rn(cB, tmp, q[m]);
    }
  }
}

void launch_central2d(int conv, bool visc, int mode, const double* Q, double* R, double* Qo, double* Qn, const Grid& g,
                      const Phys& ph, double cA, double cB, int first, int wrap, double* PK, hipStream_t s) {
  const dim3 grid((g.n[0] + C2X - 1) / C2X, (g.n[1] + C2Y - 1) / C2Y);
  auto go = [&](auto cc, auto vv) {
    k_central2d<decltype(cc)::value, decltype(vv)::value>
        <<<grid, 256, 0, s>>>(Q, R, Qo, Qn, g, ph, cA, cB, first, mode, wrap, PK);
  };
  auto with_visc = [&](auto cc) {
    if (visc) go(cc, std::true_type{});
    else go(cc, std::false_type{});
  };
  if (conv == OSBL_CONV_CENTRAL_SKEW) with_visc(std::integral_constant<int, OSBL_CONV_CENTRAL_SKEW>{});
  else with_visc(std::integral_constant<int, OSBL_CONV_CENTRAL_CONS>{});
}

void launch_char_tile2d(int conv, int avg, int mode, bool visc, const double* Q, double* R, double* Qo, double* Qn,
                        const Grid& g, const Phys& ph, const Bnd& b, double cA, double cB, int first, double* theta,
                        int suth, int wrap, double* PK, hipStream_t s) {
  const dim3 grid((g.n[0] + T2C - 1) / T2C, (g.n[1] + T2C - 1) / T2C);
  auto go = [&](auto cc, auto aa, auto vv, auto ss) {
    k_char_tile2d<decltype(cc)::value, decltype(aa)::value, decltype(vv)::value, decltype(ss)::value>
        <<<grid, 256, 0, s>>>(Q, R, Qo, Qn, g, ph, b, cA, cB, first, mode, theta, suth, wrap, PK);
  };
  if (conv == CONV_WFILTER) {  // SimpleAverage (WENO_filter.py:324)
    go(std::integral_constant<int, CONV_WFILTER>{}, std::integral_constant<int, OSBL_AVG_SIMPLE>{}, std::false_type{},
       std::false_type{});
    return;
  }
  auto with_avg = [&](auto cc) {
    constexpr bool TENO = decltype(cc)::value == OSBL_CONV_TENO5 || decltype(cc)::value == OSBL_CONV_TENO6;
    auto rest = [&](auto aa) {
      auto sensor = [&](auto vv) {
        if constexpr (TENO) {
          if (theta) {
            go(cc, aa, vv, std::true_type{});
            return;
          }
        }
        go(cc, aa, vv, std::false_type{});
      };
      if (visc) sensor(std::true_type{});
      else sensor(std::false_type{});
    };
    if (avg == OSBL_AVG_ROE) rest(std::integral_constant<int, OSBL_AVG_ROE>{});
    else rest(std::integral_constant<int, OSBL_AVG_SIMPLE>{});
  };
  switch (conv) {
    case OSBL_CONV_WENO_JS: with_avg(std::integral_constant<int, OSBL_CONV_WENO_JS>{}); break;
    case OSBL_CONV_WENO_Z: with_avg(std::integral_constant<int, OSBL_CONV_WENO_Z>{}); break;
    case OSBL_CONV_TENO5: with_avg(std::integral_constant<int, OSBL_CONV_TENO5>{}); break;
    default: with_avg(std::integral_constant<int, OSBL_CONV_TENO6>{}); break;
  }
}

}  // namespace osbl
