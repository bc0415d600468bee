// osbl_kernels.hip -- gfx950 kernels of one RK stage of the OpenSBLI RHS:
//   * the periodic halo pass and the constituent relations of what still reads them,
//   * one characteristic LLF sweep per direction of 1-D and 3-D blocks
//     (WENO5-JS/Z, TENO5/6), their viscous terms and RK update,
//   * the central (skew or conservative) stage of 3-D blocks in one kernel, of
//     1-D blocks as a fused update.
// (2-D blocks: osbl_tile2d.hip; 1-D lines with extrapolation ends: osbl_line.h.)
#include "osbl_kernels.h"

namespace osbl {

// ---------------------------------------------------------------------------
// Periodic boundary (periodic.py:42-56): every halo point of the shell takes
// the value of its periodic image, corners and edges included, in one pass.
// The shell is enumerated as z-slabs (full x,y extent), then y-slabs of the
// interior z range, then x-slabs of the interior y,z range.
// ---------------------------------------------------------------------------
__global__ void __launch_bounds__(256) k_halo_periodic(double* __restrict__ Q, int nv, Grid g, long long total) {
  long long t = (long long)blockIdx.x * blockDim.x + threadIdx.x;
  if (t >= total) return;
  const int hx = g.h[0], hy = g.h[1], hz = g.h[2];
  const int PX = g.n[0] + 2 * hx, PY = g.n[1] + 2 * hy;
  const long long nzs = 2LL * hz * PY * PX;
  const long long nys = 2LL * hy * g.n[2] * PX;
  int i, j, k;
  if (t < nzs) {
    const int ii = (int)(t % PX);
    const long long r = t / PX;
    const int jj = (int)(r % PY);
    const int kk = (int)(r / PY);
    i = ii - hx;
    j = jj - hy;
    k = kk < hz ? kk - hz : g.n[2] + (kk - hz);
  } else if (t < nzs + nys) {
    const long long u = t - nzs;
    const int ii = (int)(u % PX);
    const long long r = u / PX;
    const int jj = (int)(r % (2 * hy));
    k = (int)(r / (2 * hy));
    i = ii - hx;
    j = jj < hy ? jj - hy : g.n[1] + (jj - hy);
  } else {
    const long long u = t - nzs - nys;
    const int ii = (int)(u % (2 * hx));
    const long long r = u / (2 * hx);
    j = (int)(r % g.n[1]);
    k = (int)(r / g.n[1]);
    i = ii < hx ? ii - hx : g.n[0] + (ii - hx);
  }
  auto wrap = [](int a, int n) { return a < 0 ? a + n : (a >= n ? a - n : a); };
  const int dst = g.idx(i, j, k);
  const int src = g.idx(wrap(i, g.n[0]), wrap(j, g.n[1]), wrap(k, g.n[2]));
  for (int m = 0; m < nv; ++m) Q[m * g.fs + dst] = Q[m * g.fs + src];
}

// ---------------------------------------------------------------------------
// Constituent relations over the padded domain: u_m, p, T
// (taylor_green_vortex.py:29-31).  Read by the central and viscous stencils.
// ---------------------------------------------------------------------------
template <int ND>
__global__ void __launch_bounds__(256) k_prims(const double* __restrict__ Q, double* __restrict__ P, Grid g, Phys ph) {
  const int PX = g.n[0] + 2 * g.h[0];
  const int PY = g.n[1] + 2 * g.h[1];
  const int PZ = g.n[2] + 2 * g.h[2];
  const int i = blockIdx.x * blockDim.x + threadIdx.x - g.h[0];
  const int j = blockIdx.y - g.h[1];
  const int k = blockIdx.z - g.h[2];
  if (i >= g.n[0] + g.h[0]) return;
  (void)PX; (void)PY; (void)PZ;
  const int x = g.idx(i, j, k);
  const double rho = Q[x];
  const double ir = recip_pos(rho);
  double ke = 0.0;
#pragma unroll
  for (int m = 0; m < ND; ++m) {
    const double u = Q[(1 + m) * g.fs + x] * ir;
    P[m * g.fs + x] = u;
    ke += u * u;
  }
  const double p = ph.gm1 * (Q[(ND + 1) * g.fs + x] - 0.5 * rho * ke);
  P[ND * g.fs + x] = p;
  P[(ND + 1) * g.fs + x] = p * ph.gama * ph.Minf * ph.Minf * ir;
}

// ---------------------------------------------------------------------------
// Characteristic sweep along direction D.  Each thread owns a segment of
// `seg` cells of one grid line and slides a 6-point window along it: every
// point's constituent relations are evaluated once, every interface flux
// once, and the residual of a cell is the difference of its two interface
// fluxes (shock_capturing.py:21-34).  Threads of a wave are adjacent in x,
// except for D = 0, where they are adjacent lines.
//
// RKM >= 0: the sweep is the stage's last contribution to the residual, so a
// cell's complete residual R + (this direction's difference) goes straight
// into the RK update (RKM = 0: 3-register stage, 1: low-storage stage, as in
// k_update) and R is not written back.
// ---------------------------------------------------------------------------
struct RkArgs {
  double* Qo;
  double* Qn;
  double cA, cB;
  int first;
};

template <int ND, int D, int CONV, int AVG, bool ACC, int RKM = -1>
__global__ void __launch_bounds__(256) k_char_sweep(const double* __restrict__ Q, double* __restrict__ R, Grid g,
                                                     Phys ph, int seg, long long total,
                                                     const double* __restrict__ met,
                                                     const double* __restrict__ theta, RkArgs rk) {
  constexpr int NV = ND + 2;
  const long long t = (long long)blockIdx.x * blockDim.x + threadIdx.x;
  if (t >= total) return;
  int c[3];
  int s;
  if constexpr (D == 0) {
    c[1] = (int)(t % g.n[1]);
    const long long r = t / g.n[1];
    c[2] = (int)(r % g.n[2]);
    s = (int)(r / g.n[2]);
  } else {
    constexpr int O = (D == 1) ? 2 : 1;
    c[0] = (int)(t % g.n[0]);
    const long long r = t / g.n[0];
    c[O] = (int)(r % g.n[O]);
    s = (int)(r / g.n[O]);
  }
  const int c0 = s * seg;
  const int c1 = min(c0 + seg, g.n[D]);
  c[D] = c0 - 3;
  const int st = g.stride(D);
  int off = g.idx(c[0], c[1], c[2]);
  const double inv = ph.inv_delta[D];

  Pt<ND> w[6];
#pragma unroll
  for (int p = 0; p < 5; ++p) load_pt<ND>(w[p], Q, g.fs, off + p * st, ph);
  // the next point's raw values are fetched one iteration ahead
  double nxt[NV];
  fetch_q<ND>(nxt, Q, g.fs, off + 5 * st);
  double fprev[NV];
  // Roe factors of the interface's two points, carried along the window
  [[maybe_unused]] RoeF rf{};
  if constexpr (AVG == OSBL_AVG_ROE) roe_factors<ND>(w[2], rf.sL, rf.hL);
  for (int f = c0 - 1; f < c1; ++f) {
#pragma unroll
    for (int m = 0; m < NV; ++m) w[5].q[m] = nxt[m];
    finish_pt<ND>(w[5], ph);
    if (f + 1 < c1) fetch_q<ND>(nxt, Q, g.fs, off + 6 * st);
    double fh[NV];
    // the residual (and RK register) of this iteration's cell are fetched
    // before the flux, so that the loads overlap its arithmetic instead of
    // stalling the update after it -- except for TENO6, whose sweep would
    // then need more registers than two waves per SIMD leave it
    constexpr bool EARLY = CONV != OSBL_CONV_TENO6;
    [[maybe_unused]] double rin[NV], qoin[NV];
    if constexpr ((RKM >= 0 || ACC) && EARLY) {
      if (f >= c0) {
        const int x = off + 2 * st;
#pragma unroll
        for (int m = 0; m < NV; ++m) {
          rin[m] = ld_once(&R[m * g.fs + x], ph.nt);
          if constexpr (RKM >= 0) qoin[m] = (RKM == 0 && rk.first) ? 0.0 : ld_once(&rk.Qo[m * g.fs + x], ph.nt);
        }
      }
    }
    // interface between window points 2 and 3: its left point is at off + 2 st
    const double ct = theta ? adaptive_ct(theta[off + 2 * st], ph) : ph.teno_ct;
    if constexpr (AVG == OSBL_AVG_ROE) roe_factors<ND>(w[3], rf.sR, rf.hR);
    char_flux<ND, D, CONV, AVG, true>(w, ph, fh, ct, rf);
    if constexpr (AVG == OSBL_AVG_ROE) {
      rf.sL = rf.sR;
      rf.hL = rf.hR;
    }
    if (f >= c0) {
      const int x = off + 2 * st;
      // a stretched direction scales the flux difference by D_dd (opensblifunctions.py:607-616)
      const double gi = met ? met[f] * inv : inv;
#pragma unroll
      for (int m = 0; m < NV; ++m) {
        const double v = (fprev[m] - fh[m]) * gi;
        if constexpr (RKM == 0) {
          const double r = (EARLY ? rin[m] : R[m * g.fs + x]) + v;
          const double qo = rk.first ? w[2].q[m] : (EARLY ? qoin[m] : rk.Qo[m * g.fs + x]);
          st_once(qo + ph.dt * rk.cA * r, &rk.Qn[m * g.fs + x], ph.nt);
          st_once(qo + ph.dt * rk.cB * r, &rk.Qo[m * g.fs + x], ph.nt);
        } else if constexpr (RKM == 1) {
          const double r = (EARLY ? rin[m] : R[m * g.fs + x]) + v;
          const double tmp = (rk.cA == 0.0 ? 0.0 : rk.cA * (EARLY ? qoin[m] : rk.Qo[m * g.fs + x])) + ph.dt * r;
          st_once(tmp, &rk.Qo[m * g.fs + x], ph.nt);
          st_once(w[2].q[m] + rk.cB * tmp, &rk.Qn[m * g.fs + x], ph.nt);
        } else if constexpr (ACC) {
          st_once((EARLY ? rin[m] : R[m * g.fs + x]) + v, &R[m * g.fs + x], ph.nt);
        } else {
          st_once(v, &R[m * g.fs + x], ph.nt);
        }
      }
    }
#pragma unroll
    for (int m = 0; m < NV; ++m) fprev[m] = fh[m];
#pragma unroll
    for (int p = 0; p < 5; ++p) w[p] = w[p + 1];
    off += st;
  }
}

// ---------------------------------------------------------------------------
// Characteristic sweep along x with the lanes of a wave along x.  A wave owns
// `cells` consecutive cells of one (y, z) row and walks them in chunks of 64
// interfaces: the 69 points around a chunk are staged in LDS with their
// constituent relations, lane l evaluates the flux at interface base + l + 1/2
// from LDS, and the residual of cell base + l is its difference with lane
// l-1's flux (a shuffle; lane 0 takes the previous chunk's last flux).  Stores
// are coalesced 512-byte rows.  On a periodic row of one wave the flux left of
// cell 0 is the row's last interface flux, so cell 0 is finished after the
// walk; otherwise the walk starts with the flux left of the first cell.
//
// Slot s of a chunk holds point base - 2 + s; slots 0..4 are slots 64..68 of
// the chunk before, so each chunk stages one new point per lane, whose raw
// values are fetched while the previous chunk evaluates its fluxes.
// ---------------------------------------------------------------------------
constexpr int XW = 4;             // waves per block
constexpr int XP = 64 + 5;        // points staged per chunk

// Cells per wave: the whole row, or the 63 that one chunk completes, whichever
// leaves the busiest of the 1024 SIMDs fewer chunks (a row costs a chunk per 64
// interfaces, one less where the periodic flux is shared; 63 cells per wave
// cost more of them but spread them out); the whole row once the rows alone
// give every SIMD the three waves its registers hold.  Measured (us, WENO5-Z,
// whole row and 63 cells): 512x8x8 29 and 9, 400x20x20 29 and 16, 1000x30x30 59
// and 47, 128x50x50 periodic 23 and 28, 256x55x55 periodic 39 and 48, 96^3 54
// and 57.  Two to eight chunks per wave lay between or above the two.
static int sweep_xl_cells(const Grid& g) {
  const long long rows = (long long)g.n[1] * g.n[2];
  const int n = g.n[0];
  if (rows >= 3072 || n <= 63) return n;
  const long long whole = (rows + 1023) / 1024 * ((n + (g.periodic_x ? 0 : 1) + 63) / 64);
  const long long single = (rows * ((n + 62) / 63) + 1023) / 1024;
  return whole < single ? n : 63;
}

// (at least three waves per SIMD)
template <int ND, int CONV, int AVG>
__global__ void __launch_bounds__(64 * XW, 3) k_char_sweep_xl(const double* __restrict__ Q, double* __restrict__ R,
                                                          Grid g, Phys ph, int nwaves, int cells, int periodic,
                                                          const double* __restrict__ met,
                                                          const double* __restrict__ theta) {
  constexpr int NV = ND + 2;
  constexpr bool ROE = AVG == OSBL_AVG_ROE;
  constexpr int NF = NV + ND + 2 + (ROE ? 2 : 0);  // q, u, p, a (, sqrt(rho), sqrt(rho) H)
  constexpr int NS = NF | 1;                       // odd stride: no bank conflicts
  __shared__ double sh[XW][XP][NS];
  __shared__ double edge[XW][2][NV];
  const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
  const int id = __builtin_amdgcn_readfirstlane(blockIdx.x * XW + wv);
  if (id >= nwaves) return;  // whole waves only: no block-wide barrier below
  double (*S)[NS] = sh[wv];
  const int N = g.n[0];
  const int nseg = (N + cells - 1) / cells;
  const int row = id / nseg, s0 = (id % nseg) * cells, s1 = min(s0 + cells, N);
  const int line = g.idx(0, row % g.n[1], row / g.n[1]);
  const double inv = ph.inv_delta[0];
  const bool wrap = periodic && nseg == 1;
  const int xmax = N + g.h[0] - 1;  // last stored point of the row
  auto clampx = [&](int x) { return max(-g.h[0], min(x, xmax)); };
  auto stage_q = [&](int slot, const double (&q)[NV]) {
    Pt<ND> p;
#pragma unroll
    for (int m = 0; m < NV; ++m) p.q[m] = q[m];
    finish_pt<ND>(p, ph);
#pragma unroll
    for (int m = 0; m < NV; ++m) S[slot][m] = p.q[m];
#pragma unroll
    for (int m = 0; m < ND; ++m) S[slot][NV + m] = p.u[m];
    S[slot][NV + ND] = p.p;
    S[slot][NV + ND + 1] = p.a;
    if constexpr (ROE) roe_factors<ND>(p, S[slot][NV + ND + 2], S[slot][NV + ND + 3]);
  };
  auto wave_sync = [&] {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
  };
  auto emit = [&](int x, const double* r) {
    const double gi = met ? -met[x] * inv : -inv;
#pragma unroll
    for (int m = 0; m < NV; ++m) {
      st_once(r[m] * gi, &R[m * g.fs + line + x], ph.nt);
    }
  };
  int base = wrap ? s0 : s0 - 1;
  double nq[NV];
  if (lane < 5) {
    double q0[NV];
    fetch_q<ND>(q0, Q, g.fs, line + clampx(base - 2 + lane));
    stage_q(lane, q0);
  }
  fetch_q<ND>(nq, Q, g.fs, line + clampx(base + 3 + lane));
  for (bool start = true; base < s1; base += 64, start = false) {
    stage_q(5 + lane, nq);
    wave_sync();
    // the next chunk's point, in flight while this chunk's fluxes are evaluated
    fetch_q<ND>(nq, Q, g.fs, line + clampx(base + 67 + lane));
    const int I = base + lane;
    double fh[NV];
    {
      const LdsPoints<ND, NS> w{S[lane]};
      [[maybe_unused]] RoeF rf{};
      if constexpr (ROE) {
        rf.sL = S[lane + 2][NV + ND + 2];
        rf.hL = S[lane + 2][NV + ND + 3];
        rf.sR = S[lane + 3][NV + ND + 2];
        rf.hR = S[lane + 3][NV + ND + 3];
      }
      const double ct = theta ? adaptive_ct(theta[line + min(I, xmax)], ph) : ph.teno_ct;
      char_flux_w<ND, 0, CONV, AVG, true>(w, ph, fh, ct, rf);
    }
    double r[NV];
#pragma unroll
    for (int m = 0; m < NV; ++m) {
      const double up = __shfl_up(fh[m], 1);
      r[m] = fh[m] - (lane == 0 ? edge[wv][0][m] : up);
    }
    // the first flux and the chunk's last one wait in LDS (registers are what bounds the kernel)
    const int last = min(63, s1 - 1 - base);
    if (lane == 0 && start) {
#pragma unroll
      for (int m = 0; m < NV; ++m) edge[wv][1][m] = fh[m];
    }
    wave_sync();
    if (lane == last) {
#pragma unroll
      for (int m = 0; m < NV; ++m) edge[wv][0][m] = fh[m];
    }
    if (I >= s0 && I < s1 && !(wrap && I == 0)) emit(I, r);
    // slots 64..68 become slots 0..4 of the next chunk
    wave_sync();
    if (lane < 5) {
#pragma unroll
      for (int e = 0; e < NF; ++e) S[lane][e] = S[64 + lane][e];
    }
    wave_sync();
  }
  if (wrap && lane == 0) {
    // the row's last interface flux is the flux left of cell 0
    double r[NV];
#pragma unroll
    for (int m = 0; m < NV; ++m) r[m] = edge[wv][1][m] - edge[wv][0][m];
    emit(0, r);
  }
}

// ---------------------------------------------------------------------------
// Central fourth-order stencils (scheme.py:81-85): D1 weights
// [1/12, -2/3, 0, 2/3, -1/12], D2 weights [-1/12, 4/3, -5/2, 4/3, -1/12].
// ---------------------------------------------------------------------------
__device__ __forceinline__ double d1(const double* __restrict__ f, int x, int st) {
  return (1.0 / 12.0) * (f[x - 2 * st] - f[x + 2 * st]) + (2.0 / 3.0) * (f[x + st] - f[x - st]);
}
__device__ __forceinline__ double d2(const double* __restrict__ f, int x, int st) {
  return (-1.0 / 12.0) * (f[x - 2 * st] + f[x + 2 * st]) + (4.0 / 3.0) * (f[x - st] + f[x + st]) - 2.5 * f[x];
}

// Viscous terms of the constant-viscosity stress tensor and heat flux
// (taylor_green_vortex.py:14-19), expanded by the product rule as the
// reference's Der.differentiate does (parsing.py:141-186): second derivatives
// with the D2 stencil, mixed derivatives as D_b(D_a u) with a < b
// (opensblifunctions.py:341-353, scheme.py:360-387).  P holds u_0..u_{ND-1}, p, T.
template <int ND>
__device__ __forceinline__ void viscous_terms(const double* __restrict__ P, long long fs, int x, const int st[3],
                                              const Phys& ph, double vr[ND + 2]) {
  const double* U[3] = {P, P + fs, P + 2 * fs};
  const double* T = P + (ND + 1) * fs;
  double du[ND][ND], dd[ND][ND][ND];  // du[m][j] = D_j u_m; dd[m][a][b] = D_a D_b u_m (symmetric use)
#pragma unroll
  for (int m = 0; m < ND; ++m)
#pragma unroll
    for (int j = 0; j < ND; ++j) {
      du[m][j] = ph.inv_delta[j] * d1(U[m], x, st[j]);
      dd[m][j][j] = ph.inv_delta[j] * ph.inv_delta[j] * d2(U[m], x, st[j]);
    }
  // mixed derivatives needed: u_a and u_b for every pair a < b
#pragma unroll
  for (int a = 0; a < ND; ++a)
#pragma unroll
    for (int b = a + 1; b < ND; ++b)
#pragma unroll
      for (int q = 0; q < 2; ++q) {
        const int m = q == 0 ? a : b;
        const double* f = U[m];
        const int sa = st[a], sb = st[b];
        const double im2 = ph.inv_delta[a] * d1(f, x - 2 * sb, sa);
        const double im1 = ph.inv_delta[a] * d1(f, x - sb, sa);
        const double ip1 = ph.inv_delta[a] * d1(f, x + sb, sa);
        const double ip2 = ph.inv_delta[a] * d1(f, x + 2 * sb, sa);
        const double v = ph.inv_delta[b] * ((1.0 / 12.0) * (im2 - ip2) + (2.0 / 3.0) * (ip1 - im1));
        dd[m][a][b] = v;
        dd[m][b][a] = v;
      }
  double divu = 0.0;
#pragma unroll
  for (int k = 0; k < ND; ++k) divu += du[k][k];
  double energy = 0.0;
#pragma unroll
  for (int j = 0; j < ND; ++j) energy += ph.cq * ph.inv_delta[j] * ph.inv_delta[j] * d2(T, x, st[j]);
#pragma unroll
  for (int m = 0; m < ND; ++m) {
    const double um = U[m][x];
    double sk = 0.0;
#pragma unroll
    for (int k = 0; k < ND; ++k) sk += dd[k][m][k];
    double visc = 0.0;
#pragma unroll
    for (int j = 0; j < ND; ++j) {
      double tt = dd[m][j][j] + dd[j][m][j];
      if (j == m) tt -= (2.0 / 3.0) * sk;
      const double dtau = ph.inv_re * tt;
      const double tau = ph.inv_re * (du[m][j] + du[j][m] - (j == m ? (2.0 / 3.0) * divu : 0.0));
      visc += dtau;
      energy += du[m][j] * tau + um * dtau;
    }
    vr[1 + m] += visc;
  }
  vr[ND + 1] += energy;
}

// Central convective terms.  Skew/Blaisdell form (parsing.py:75-111,
// scheme.py:187-252) or the conservative flux form (parsing.py:189-216).
template <int ND, int CONV>
__device__ __forceinline__ void central_convective(const double* __restrict__ Q, const double* __restrict__ P,
                                                   long long fs, int x, const int st[3], const Phys& ph,
                                                   double r[ND + 2]) {
  constexpr int NV = ND + 2;
  const double* U[3] = {P, P + fs, P + 2 * fs};
  const double* Pp = P + ND * fs;
#pragma unroll
  for (int m = 0; m < NV; ++m) r[m] = 0.0;
#pragma unroll
  for (int j = 0; j < ND; ++j) {
    const int sj = st[j];
    const double inv = ph.inv_delta[j];
    constexpr double W1A = 1.0 / 12.0, W1B = 2.0 / 3.0;
    // points -2, -1, +1, +2 with weights  W1A, -W1B, W1B, -W1A
    const int offs[4] = {x - 2 * sj, x - sj, x + sj, x + 2 * sj};
    const double wts[4] = {W1A, -W1B, W1B, -W1A};
    if constexpr (CONV == OSBL_CONV_CENTRAL_SKEW) {
      double d_ru[NV], d_q[NV], d_uj = 0.0, d_p = 0.0, d_puj = 0.0;
#pragma unroll
      for (int m = 0; m < NV; ++m) { d_ru[m] = 0.0; d_q[m] = 0.0; }
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        const int y = offs[q];
        const double w = wts[q];
        const double uj = U[j][y];
        const double pp = Pp[y];
#pragma unroll
        for (int m = 0; m < NV; ++m) {
          const double qm = Q[m * fs + y];
          d_ru[m] += w * (qm * uj);
          d_q[m] += w * qm;
        }
        d_uj += w * uj;
        d_p += w * pp;
        d_puj += w * (pp * uj);
      }
      const double uj = U[j][x];
      const double duj = inv * d_uj;
#pragma unroll
      for (int m = 0; m < NV; ++m) {
        const double qm = Q[m * fs + x];
        double t = -0.5 * (inv * d_ru[m] + uj * (inv * d_q[m]) + qm * duj);
        if (m == 1 + j) t -= inv * d_p;
        if (m == NV - 1) t -= inv * d_puj;
        r[m] += t;
      }
    } else {
      double dF[NV];
#pragma unroll
      for (int m = 0; m < NV; ++m) dF[m] = 0.0;
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        const int y = offs[q];
        const double w = wts[q];
        const double uj = U[j][y];
        const double pp = Pp[y];
        dF[0] += w * Q[(1 + j) * fs + y];
#pragma unroll
        for (int m = 0; m < ND; ++m) dF[1 + m] += w * (Q[(1 + m) * fs + y] * uj + (m == j ? pp : 0.0));
        dF[NV - 1] += w * ((pp + Q[(NV - 1) * fs + y]) * uj);
      }
#pragma unroll
      for (int m = 0; m < NV; ++m) r[m] -= inv * dF[m];
    }
  }
}

// ---------------------------------------------------------------------------
// Residual assembly + RK update for one interior cell.
//   MODE 0: 3-register RK3 stage (rk_sbli.py:117-124): Qn = Qo + dt*cA*R,
//           Qo += dt*cB*R; at the first stage Qo is read from Q (the save of
//           rk_sbli.py:126-133 fused into the stage).
//   MODE 1: low-storage stage (rk_LS.py:155-166): Qo = cA*Qo + dt*R,
//           Qn = Q + cB*Qo (Qo not read when cA == 0).
//   MODE 2: residual only (written to R).
// For characteristic schemes the convective residual is already in R.
// ---------------------------------------------------------------------------
template <int ND, int CONV, bool VISC, int MODE>
__global__ void __launch_bounds__(256) k_update(const double* __restrict__ Q, const double* __restrict__ P,
                                                double* __restrict__ R, double* __restrict__ Qo,
                                                double* __restrict__ Qn, Grid g, Phys ph, double cA, double cB,
                                                int first) {
  constexpr int NV = ND + 2;
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= g.n[0]) return;
  const int j = blockIdx.y, k = blockIdx.z;
  const int x = g.idx(i, j, k);
  const int st[3] = {1, g.pitch, g.plane};
  double r[NV];
  if constexpr (CONV == OSBL_CONV_CENTRAL_SKEW || CONV == OSBL_CONV_CENTRAL_CONS) {
    central_convective<ND, CONV>(Q, P, g.fs, x, st, ph, r);
  } else {
#pragma unroll
    for (int m = 0; m < NV; ++m) r[m] = R[m * g.fs + x];
  }
  if constexpr (VISC) viscous_terms<ND>(P, g.fs, x, st, ph, r);
  if constexpr (MODE == 2) {
#pragma unroll
    for (int m = 0; m < NV; ++m) R[m * g.fs + x] = r[m];
  } else if constexpr (MODE == 0) {
#pragma unroll
    for (int m = 0; m < NV; ++m) {
      const double qo = first ? Q[m * g.fs + x] : Qo[m * g.fs + x];
      Qn[m * g.fs + x] = qo + ph.dt * cA * r[m];
      Qo[m * g.fs + x] = qo + ph.dt * cB * r[m];
    }
  } else {
#pragma unroll
    for (int m = 0; m < NV; ++m) {
      const double tmp = (cA == 0.0 ? 0.0 : cA * Qo[m * g.fs + x]) + ph.dt * r[m];
      Qo[m * g.fs + x] = tmp;
      Qn[m * g.fs + x] = Q[m * g.fs + x] + cB * tmp;
    }
  }
}

// ---------------------------------------------------------------------------
// 3-D viscous terms + RK update for the characteristic schemes, tiled 2.5-D.
// A VTX x VTY block of (x, y) columns marches along z.  Each z plane of the
// constituent relations u_0..u_2, T (computed here from Q, with a 2-point
// x/y halo) is staged in one of four rotating LDS slots; the x/y stencils
// read LDS, the z stencils read a per-thread register queue of the five
// planes z-2..z+2 holding u, T and the inner derivatives D_x u_0, D_x u_2,
// D_y u_1, D_y u_2 of the mixed terms D_z(D_x u), D_z(D_y u).  The formulas
// are those of viscous_terms (scheme.py:299-387).
//
// Software pipeline: while plane z is evaluated, the raw Q of plane z+3 and
// the cell's residual / RK registers are already in flight (loaded at the
// top of the iteration into registers); plane z+3 then goes into the slot
// plane z-1 vacated, and one barrier per plane separates those writes from
// the next plane's reads.
// ---------------------------------------------------------------------------
constexpr int VTX = 64, VTY = 8, VPX = VTX + 4, VPY = VTY + 4, VPL = VPX * VPY;
constexpr int VNT = VTX * VTY;                 // threads per block
constexpr int VPP = (VPL + VNT - 1) / VNT;     // staged points per thread and plane

__global__ void __launch_bounds__(VNT, 2) k_visc_update3d(const double* __restrict__ Q, double* __restrict__ R, Grid g,
                                                       Phys ph, int sz) {
  __shared__ double sp[4][4][VPL];
  const int tx = threadIdx.x, ty = threadIdx.y;
  const int tid = ty * VTX + tx;
  int bx, by, bz;
  xcd_tile(bx, by, bz);
  const int x0 = bx * VTX, y0 = by * VTY;
  const int z0 = bz * sz;
  const int z1 = min(z0 + sz, g.n[2]);
  const int x = x0 + tx, y = y0 + ty;
  const bool inside = x < g.n[0] && y < g.n[1];
  const double ix = ph.inv_delta[0], iy = ph.inv_delta[1], iz = ph.inv_delta[2];

  // this thread's staged points: slot index and in-plane offset (plane z = 0)
  int sidx[VPP], soff[VPP];
  bool sval[VPP];
#pragma unroll
  for (int k = 0; k < VPP; ++k) {
    const int p = tid + k * VNT;
    const int xx = p % VPX, yy = p / VPX;
    const int gx = x0 - 2 + xx, gy = y0 - 2 + yy;
    sidx[k] = p;
    sval[k] = p < VPL && gx < g.n[0] + g.h[0] && gy < g.n[1] + g.h[1];
    soff[k] = sval[k] ? g.idx(gx, gy, 0) : 0;
  }
  double pq[VPP][5];  // raw Q of the plane in flight
  auto fetch = [&](int zp) {
    const int zo = zp * g.plane;
#pragma unroll
    for (int k = 0; k < VPP; ++k)
      if (sval[k]) {
#pragma unroll
        for (int m = 0; m < 5; ++m) pq[k][m] = Q[m * g.fs + soff[k] + zo];
      }
  };
  auto store = [&](int slot) {
#pragma unroll
    for (int k = 0; k < VPP; ++k)
      if (sval[k]) {
        const double rho = pq[k][0];
        const double ir = recip_pos(rho);
        const double u0 = pq[k][1] * ir, u1 = pq[k][2] * ir, u2 = pq[k][3] * ir;
        const double pr = ph.gm1 * (pq[k][4] - 0.5 * rho * (u0 * u0 + u1 * u1 + u2 * u2));
        const int p = sidx[k];
        sp[slot][0][p] = u0;
        sp[slot][1][p] = u1;
        sp[slot][2][p] = u2;
        sp[slot][3][p] = pr * ph.gama * ph.Minf * ph.Minf * ir;
      }
  };
  const int c = (ty + 2) * VPX + tx + 2;  // this thread's point in a slot
  auto dx1 = [&](const double* f, int o) {
    return (1.0 / 12.0) * (f[o - 2] - f[o + 2]) + (2.0 / 3.0) * (f[o + 1] - f[o - 1]);
  };
  auto dy1 = [&](const double* f, int o) {
    return (1.0 / 12.0) * (f[o - 2 * VPX] - f[o + 2 * VPX]) + (2.0 / 3.0) * (f[o + VPX] - f[o - VPX]);
  };
  auto dx2 = [&](const double* f, int o) {
    return (-1.0 / 12.0) * (f[o - 2] + f[o + 2]) + (4.0 / 3.0) * (f[o - 1] + f[o + 1]) - 2.5 * f[o];
  };
  auto dy2 = [&](const double* f, int o) {
    return (-1.0 / 12.0) * (f[o - 2 * VPX] + f[o + 2 * VPX]) + (4.0 / 3.0) * (f[o - VPX] + f[o + VPX]) - 2.5 * f[o];
  };
  // column quantities of a plane: u0,u1,u2,T, Dx u0, Dx u2, Dy u1, Dy u2
  auto column = [&](int slot, double* cq) {
    const double* u0 = sp[slot][0];
    const double* u1 = sp[slot][1];
    const double* u2 = sp[slot][2];
    cq[0] = u0[c];
    cq[1] = u1[c];
    cq[2] = u2[c];
    cq[3] = sp[slot][3][c];
    cq[4] = ix * dx1(u0, c);
    cq[5] = ix * dx1(u2, c);
    cq[6] = iy * dy1(u1, c);
    cq[7] = iy * dy1(u2, c);
  };
  auto slot_of = [](int zp) { return (zp + 8) & 3; };

  double zq[5][8];
  // prologue: planes z0-2 .. z0+1 into the four slots, their columns into
  // queue entries 0..3, then plane z0+2 into the slot of plane z0-2
  for (int k = 0; k < 4; ++k) {
    fetch(z0 - 2 + k);
    store(slot_of(z0 - 2 + k));
  }
  __syncthreads();
#pragma unroll
  for (int k = 0; k < 4; ++k) column(slot_of(z0 - 2 + k), zq[k]);
  fetch(z0 + 2);
  __syncthreads();
  store(slot_of(z0 + 2));
  __syncthreads();
  column(slot_of(z0 + 2), zq[4]);

  for (int z = z0; z < z1; ++z) {
    const bool more = z + 1 < z1;  // plane z+3 feeds the next plane's queue entry
    if (more) fetch(z + 3);
    const int o = g.idx(x, y, z);
    // the cell's residual, in flight during the arithmetic
    double rin[5];
    if (inside) {
#pragma unroll
      for (int m = 0; m < 5; ++m) rin[m] = ld_once(&R[m * g.fs + o], ph.nt);
      const int sl = slot_of(z);
      const double* U[3] = {sp[sl][0], sp[sl][1], sp[sl][2]};
      const double* T = sp[sl][3];
      double du[3][3], dd[3][3][3];
      // x and y first / second derivatives from LDS
#pragma unroll
      for (int m = 0; m < 3; ++m) {
        du[m][0] = ix * dx1(U[m], c);
        du[m][1] = iy * dy1(U[m], c);
        dd[m][0][0] = ix * ix * dx2(U[m], c);
        dd[m][1][1] = iy * iy * dy2(U[m], c);
      }
      // z derivatives from the queue (planes z-2..z+2 at indices 0..4)
#pragma unroll
      for (int m = 0; m < 3; ++m) {
        du[m][2] = iz * ((1.0 / 12.0) * (zq[0][m] - zq[4][m]) + (2.0 / 3.0) * (zq[3][m] - zq[1][m]));
        dd[m][2][2] =
            iz * iz * ((-1.0 / 12.0) * (zq[0][m] + zq[4][m]) + (4.0 / 3.0) * (zq[1][m] + zq[3][m]) - 2.5 * zq[2][m]);
      }
      // mixed D_y(D_x u_m), m = 0, 1, from LDS
#pragma unroll
      for (int m = 0; m < 2; ++m) {
        const double* f = U[m];
        const double a2 = ix * dx1(f, c - 2 * VPX), a1 = ix * dx1(f, c - VPX);
        const double b1 = ix * dx1(f, c + VPX), b2 = ix * dx1(f, c + 2 * VPX);
        const double v = iy * ((1.0 / 12.0) * (a2 - b2) + (2.0 / 3.0) * (b1 - a1));
        dd[m][0][1] = v;
        dd[m][1][0] = v;
      }
      // mixed D_z(D_x u_m), m = 0 (queue 4), 2 (queue 5); D_z(D_y u_m), m = 1 (6), 2 (7)
      auto dzq = [&](int e) {
        return iz * ((1.0 / 12.0) * (zq[0][e] - zq[4][e]) + (2.0 / 3.0) * (zq[3][e] - zq[1][e]));
      };
      dd[0][0][2] = dd[0][2][0] = dzq(4);
      dd[2][0][2] = dd[2][2][0] = dzq(5);
      dd[1][1][2] = dd[1][2][1] = dzq(6);
      dd[2][1][2] = dd[2][2][1] = dzq(7);
      const double divu = du[0][0] + du[1][1] + du[2][2];
      double r[5];
#pragma unroll
      for (int m = 0; m < 5; ++m) r[m] = 0.0;
      double energy = ph.cq * (ix * ix * dx2(T, c) + iy * iy * dy2(T, c) +
                               iz * iz * ((-1.0 / 12.0) * (zq[0][3] + zq[4][3]) +
                                          (4.0 / 3.0) * (zq[1][3] + zq[3][3]) - 2.5 * zq[2][3]));
#pragma unroll
      for (int m = 0; m < 3; ++m) {
        const double um = zq[2][m];
        double sk = 0.0;
#pragma unroll
        for (int k = 0; k < 3; ++k) sk += dd[k][m][k];
        double visc = 0.0;
#pragma unroll
        for (int j = 0; j < 3; ++j) {
          double tt = dd[m][j][j] + dd[j][m][j];
          if (j == m) tt -= (2.0 / 3.0) * sk;
          const double dtau = ph.inv_re * tt;
          const double tau = ph.inv_re * (du[m][j] + du[j][m] - (j == m ? (2.0 / 3.0) * divu : 0.0));
          visc += dtau;
          energy += du[m][j] * tau + um * dtau;
        }
        r[1 + m] = visc;
      }
      r[4] = energy;
#pragma unroll
      for (int m = 0; m < 5; ++m) st_once(rin[m] + r[m], &R[m * g.fs + o], ph.nt);
    }
    if (more) {
      // plane z+3 replaces plane z-1 (last read before the previous barrier)
      store(slot_of(z + 3));
      __syncthreads();
#pragma unroll
      for (int k = 0; k < 4; ++k)
#pragma unroll
        for (int e = 0; e < 8; ++e) zq[k][e] = zq[k + 1][e];
      column(slot_of(z + 3), zq[4]);
    }
  }
}

void launch_visc_update3d(const double* Q, double* R, const Grid& g, const Phys& ph, int sz, hipStream_t s) {
  dim3 grid((g.n[0] + VTX - 1) / VTX, (g.n[1] + VTY - 1) / VTY, (g.n[2] + sz - 1) / sz);
  k_visc_update3d<<<grid, dim3(VTX, VTY), 0, s>>>(Q, R, g, ph, sz);
}

// ---------------------------------------------------------------------------
// One stage of a 3-D central scheme in one kernel: convective terms in the
// skew-symmetric (Blaisdell) form (parsing.py:75-111, scheme.py:187-252) or
// the conservative flux form (parsing.py:189-216), constant-viscosity terms
// (scheme.py:299-387) and the RK update, with the formulas of
// central_convective and viscous_terms.
//
// A TX x TY block of (x, y) columns (64 or 32 by 8) marches along z.  When plane z+2 is in
// LDS (conservative and primitive variables with a 2-point x/y halo), each
// thread evaluates everything that needs only that plane for its column --
// the x and y terms, added up in r -- and keeps in a register queue over
// five planes what the z stencils need: Q, 1/rho and the inner derivatives
// D_x u_0 + D_y u_1, D_x u_2, D_y u_2 of the mixed terms.  Then plane z is
// complete.  With the sums folded, the viscous terms need nothing else kept:
//   rhou_m: (1/Re) (lap u_m + D_m(div u)/3)
//   rhoE:   u . the above + (1/Re) (2 sum_m (D_m u_m)^2 - 2/3 (div u)^2
//           + sum_{m<j} (D_m u_j + D_j u_m)^2) + cq lap T
// The raw Q of the next plane is in flight during the arithmetic; two LDS
// slots alternate, one barrier per plane.  On a block periodic in every
// direction (`wrap`) the staged points are read at their periodic images, so
// the halos need not be filled between stages.
//
// The stage moves Q, the register and the new state once: 160 B per cell
// against 280 for a convective kernel that leaves R to a viscous kernel.  What
// bounds it now is a block's chain per plane (LDS reads, two waves per SIMD,
// a barrier) and, at 256^3, HBM: 0.73 ms a stage, 3.7 TB/s of those 160 B;
// the two kernels and the halo pass took 1.36 ms.  Reading a point's fields
// two at a time (ds_read_b128) took it from 0.88 to 0.75, adding up the pairs'
// differences with Q and p in one sum (fewer operations and registers) to 0.73.
//   MODE 0/1: RK update; MODE 2: the residual alone, into R.
// ---------------------------------------------------------------------------
template <int CONV, bool VISC, int MODE, int TX, int TY>
__global__ void __launch_bounds__(TX * TY, 2)
    k_central3d(const double* __restrict__ Q, double* __restrict__ R, double* __restrict__ Qo,
                double* __restrict__ Qn, Grid g, Phys ph, double cA, double cB, int first, int sz, int wrap) {
  constexpr int NV = 5, PX = TX + 4, PY = TY + 4, PL = PX * PY, NT = TX * TY;
  constexpr int PP = (PL + NT - 1) / NT;     // staged points per thread and plane
  constexpr int NF = 10;                     // Q0..Q4, p, u0, u1, u2, T
  constexpr int NQ = VISC ? 9 : 6;           // queue: Q0..Q4, 1/rho (, D_x u0 + D_y u1, D_x u2, D_y u2)
  // a point's fields lie next to each other and are read two at a time: at a
  // stride of 80 bytes 16 lanes' 16-byte reads cover the 64 banks once
  __shared__ __align__(16) double sp[2][PL][NF];
  const int tx = threadIdx.x, ty = threadIdx.y, tid = ty * TX + tx;
  int bx, by, bz;
  xcd_tile(bx, by, bz);
  const int x0 = bx * TX, y0 = by * TY, z0 = bz * sz, z1 = min(z0 + sz, g.n[2]);
  const int x = x0 + tx, y = y0 + ty;
  const bool inside = x < g.n[0] && y < g.n[1];
  const double ix = ph.inv_delta[0], iy = ph.inv_delta[1], iz = ph.inv_delta[2];
  const double cT = ph.gama * ph.Minf * ph.Minf;

  auto image = [&](int i, int n) { return !wrap ? i : (i < 0 ? i + n : (i >= n ? i - n : i)); };
  int soff[PP];
  bool sval[PP];
#pragma unroll
  for (int k = 0; k < PP; ++k) {
    const int pt = tid + k * NT;
    const int gx = x0 - 2 + pt % PX, gy = y0 - 2 + pt / PX;
    sval[k] = pt < PL && gx < g.n[0] + 2 && gy < g.n[1] + 2;
    soff[k] = sval[k] ? g.idx(image(gx, g.n[0]), image(gy, g.n[1]), 0) : 0;
  }
  double pq[PP][NV];  // raw Q of the plane in flight
  auto fetch = [&](int zp) {
    const int zo = image(zp, g.n[2]) * g.plane;
#pragma unroll
    for (int k = 0; k < PP; ++k)
      if (sval[k]) {
#pragma unroll
        for (int m = 0; m < NV; ++m) pq[k][m] = Q[m * g.fs + soff[k] + zo];
      }
  };
  auto store = [&](int slot) {
#pragma unroll
    for (int k = 0; k < PP; ++k)
      if (sval[k]) {
        const int pt = tid + k * NT;
        const double rho = pq[k][0];
        const double ir = recip_pos(rho);
        const double u0 = pq[k][1] * ir, u1 = pq[k][2] * ir, u2 = pq[k][3] * ir;
        const double pr = ph.gm1 * (pq[k][4] - 0.5 * rho * (u0 * u0 + u1 * u1 + u2 * u2));
#pragma unroll
        for (int m = 0; m < NV; ++m) sp[slot][pt][m] = pq[k][m];
        sp[slot][pt][5] = pr;
        sp[slot][pt][6] = u0;
        sp[slot][pt][7] = u1;
        if constexpr (VISC) {
          sp[slot][pt][8] = u2;
          sp[slot][pt][9] = cT * pr * ir;
        }
      }
  };
  const int c = (ty + 2) * PX + tx + 2;  // this thread's column in a slot
  auto d1 = [](double fm2, double fm1, double fp1, double fp2) {
    return (1.0 / 12.0) * (fm2 - fp2) + (2.0 / 3.0) * (fp1 - fm1);
  };
  auto d2 = [](double fm2, double fm1, double f0, double fp1, double fp2) {
    return (-1.0 / 12.0) * (fm2 + fp2) + (4.0 / 3.0) * (fm1 + fp1) - 2.5 * f0;
  };
  struct alignas(16) Two {
    double a, b;
  };
  // fields 2 i and 2 i + 1 of the point o of a slot
  auto two = [](const double (*S)[NF], int o, int i) { return *reinterpret_cast<const Two*>(&S[o][2 * i]); };
  // sums over the points -2, -1, 1, 2 of a direction: q is the convective term
  // of the conservative variables over `hi` below -- skew: first difference of
  // Q (u_j + u0) + 2 p e, conservative: of Q u_j + p e, with p e = (0, p e_j,
  // p u_j); u, uu and TT first and second differences of u_0..u_2 and T.  The
  // outer and the inner pair are each taken as a difference (a sum) before
  // they are weighted: a field uniform along the direction gives exactly zero.
  struct Sums {
    double q[NV], u[3], uu[3], TT;
  };
  constexpr bool SKEW = CONV == OSBL_CONV_CENTRAL_SKEW;
  auto gather = [&](const double (*S)[NF], int j, int st, double u0) {
    Sums a{};
#pragma unroll
    for (int s = 0; s < 2; ++s) {
      // D = 1/12 (f[-2] - f[2]) + 2/3 (f[1] - f[-1]): l minus r, weighted w
      const int l = c + (s == 0 ? -2 : 1) * st, r = c + (s == 0 ? 2 : -1) * st;
      const double w = s == 0 ? 1.0 / 12.0 : 2.0 / 3.0, w2 = s == 0 ? -1.0 / 12.0 : 4.0 / 3.0;
      const Two l3 = two(S, l, 3), r3 = two(S, r, 3);
      const double ul = j == 0 ? l3.a : l3.b, ur = j == 0 ? r3.a : r3.b;
      if constexpr (VISC) {
        const Two l4 = two(S, l, 4), r4 = two(S, r, 4);
        a.u[0] = __fma_rn(w, l3.a - r3.a, a.u[0]);
        a.u[1] = __fma_rn(w, l3.b - r3.b, a.u[1]);
        a.u[2] = __fma_rn(w, l4.a - r4.a, a.u[2]);
        a.uu[0] = __fma_rn(w2, l3.a + r3.a, a.uu[0]);
        a.uu[1] = __fma_rn(w2, l3.b + r3.b, a.uu[1]);
        a.uu[2] = __fma_rn(w2, l4.a + r4.a, a.uu[2]);
        a.TT = __fma_rn(w2, l4.b + r4.b, a.TT);
      } else {
        a.u[j] = __fma_rn(w, ul - ur, a.u[j]);
      }
      __builtin_amdgcn_sched_barrier(0);  // (the pair's fields in two parts: registers)
      const Two l0 = two(S, l, 0), l1 = two(S, l, 1), l2 = two(S, l, 2);
      const Two r0 = two(S, r, 0), r1 = two(S, r, 1), r2 = two(S, r, 2);
      const double ql[NV] = {l0.a, l0.b, l1.a, l1.b, l2.a}, qr[NV] = {r0.a, r0.b, r1.a, r1.b, r2.a};
      if constexpr (SKEW) {
        const double vl = ul + u0, vr = ur + u0;
#pragma unroll
        for (int m = 0; m < NV; ++m) a.q[m] = __fma_rn(w, __fma_rn(ql[m], vl, -(qr[m] * vr)), a.q[m]);
        a.q[1 + j] = __fma_rn(2.0 * w, l2.b - r2.b, a.q[1 + j]);
        a.q[4] = __fma_rn(2.0 * w, __fma_rn(l2.b, ul, -(r2.b * ur)), a.q[4]);
      } else {
        a.q[0] = __fma_rn(w, ql[1 + j] - qr[1 + j], a.q[0]);
#pragma unroll
        for (int m = 1; m < 4; ++m) a.q[m] = __fma_rn(w, __fma_rn(ql[m], ul, -(qr[m] * ur)), a.q[m]);
        a.q[1 + j] = __fma_rn(w, l2.b - r2.b, a.q[1 + j]);
        a.q[4] = __fma_rn(w, __fma_rn(ql[4] + l2.b, ul, -((qr[4] + r2.b) * ur)), a.q[4]);
      }
      __builtin_amdgcn_sched_barrier(0);
    }
    return a;
  };
  auto add_convect = [](const Sums& a, int j, double inv, const double (&q0)[NV], double* r) {
    const double hi = SKEW ? -0.5 * inv : -inv;
    const double du = hi * a.u[j];
#pragma unroll
    for (int m = 0; m < NV; ++m) r[m] += SKEW ? hi * a.q[m] + q0[m] * du : hi * a.q[m];
  };
  // convective terms along z: values of Q_m, u_j, p at the
  // offsets -2, -1, 1, 2 through fq, fu, fp; the cell's own Q and u_j
  auto convect = [&](int j, double inv, auto&& fq, auto&& fu, auto&& fp, const double (&q0)[NV], double u0, double* r) {
    double qv[4][NV], uv[4], pv[4];
#pragma unroll
    for (int s = 0; s < 4; ++s) {
#pragma unroll
      for (int m = 0; m < NV; ++m) qv[s][m] = fq(s, m);
      uv[s] = fu(s);
      pv[s] = fp(s);
    }
    const double dp = inv * d1(pv[0], pv[1], pv[2], pv[3]);
    if constexpr (CONV == OSBL_CONV_CENTRAL_SKEW) {
      const double hi = -0.5 * inv, hu = hi * u0;
      const double du = hi * d1(uv[0], uv[1], uv[2], uv[3]);
#pragma unroll
      for (int m = 0; m < NV; ++m) {
        const double dru = d1(qv[0][m] * uv[0], qv[1][m] * uv[1], qv[2][m] * uv[2], qv[3][m] * uv[3]);
        const double dq = d1(qv[0][m], qv[1][m], qv[2][m], qv[3][m]);
        r[m] += hi * dru + hu * dq + q0[m] * du;
        if (m == 1 + j) r[m] -= dp;
      }
      r[4] -= inv * d1(pv[0] * uv[0], pv[1] * uv[1], pv[2] * uv[2], pv[3] * uv[3]);
    } else {
      r[0] -= inv * d1(qv[0][1 + j], qv[1][1 + j], qv[2][1 + j], qv[3][1 + j]);
#pragma unroll
      for (int m = 0; m < 3; ++m) {
        r[1 + m] -= inv * d1(qv[0][1 + m] * uv[0], qv[1][1 + m] * uv[1], qv[2][1 + m] * uv[2], qv[3][1 + m] * uv[3]);
        if (m == j) r[1 + m] -= dp;
      }
      r[4] -= inv * d1((qv[0][4] + pv[0]) * uv[0], (qv[1][4] + pv[1]) * uv[1], (qv[2][4] + pv[2]) * uv[2],
                       (qv[3][4] + pv[3]) * uv[3]);
    }
  };

  // (what has been added up so far is finished before the next terms' values
  // are read from LDS: the registers hold one direction's at a time)
  auto settle = [](double* r) {
#pragma unroll
    for (int m = 0; m < NV; ++m) asm volatile("" : "+v"(r[m]) : : "memory");
    __builtin_amdgcn_sched_barrier(0);
  };

  double zq[5][NQ];   // planes z-2 .. z+2 of this column
  double rr[3][NV];   // the in-plane sums of planes z, z+1, z+2
  fetch(z0 - 2);
  store(z0 & 1);
  __syncthreads();
  for (int zp = z0 - 2; zp < z1 + 2; ++zp) {
    const int z = zp - 2;  // the plane that plane zp completes
    const bool more = zp + 1 < z1 + 2;
    if (more) fetch(zp + 1);
    const int o = g.idx(x, y, z);
    [[maybe_unused]] double qa[NV];
    if (inside && z >= z0) {
#pragma unroll
      for (int m = 0; m < NV; ++m) {
        if constexpr (MODE == 0) qa[m] = first ? 0.0 : ld_once(&Qo[m * g.fs + o], ph.nt);
        if constexpr (MODE == 1) qa[m] = cA == 0.0 ? 0.0 : ld_once(&Qo[m * g.fs + o], ph.nt);
      }
    }
    const double (*S)[NF] = sp[zp & 1];
    if (inside) {
      double* e = zq[4];
      const Two f0 = two(S, c, 0), f1 = two(S, c, 1), f2 = two(S, c, 2), f3 = two(S, c, 3);
      e[0] = f0.a;
      e[1] = f0.b;
      e[2] = f1.a;
      e[3] = f1.b;
      e[4] = f2.a;
      e[5] = recip_pos(e[0]);
      if (zp >= z0 && zp < z1) {
        double* r = rr[2];
#pragma unroll
        for (int m = 0; m < NV; ++m) r[m] = 0.0;
        const double q0[NV] = {e[0], e[1], e[2], e[3], e[4]};
        const Sums ax = gather(S, 0, 1, f3.a);
        add_convect(ax, 0, ix, q0, r);
        if constexpr (VISC) {
          const double xx = ix * ix, yy = iy * iy;
          const Two f4 = two(S, c, 4);
          // second derivatives and shears, x first
          double p0 = (4.0 / 3.0) * xx * (ax.uu[0] - 2.5 * f3.a), p1 = xx * (ax.uu[1] - 2.5 * f3.b);
          double p2 = xx * (ax.uu[2] - 2.5 * f4.a), TT = xx * (ax.TT - 2.5 * f4.b);
          double ux = ix * ax.u[0], sh = ix * ax.u[1];
          e[7] = ix * ax.u[2];
          asm volatile("" : "+v"(p0), "+v"(p1), "+v"(p2), "+v"(TT), "+v"(ux), "+v"(sh), "+v"(e[7]));
          settle(r);
          const Sums ay = gather(S, 1, PX, f3.b);
          add_convect(ay, 1, iy, q0, r);
          p0 += yy * (ay.uu[0] - 2.5 * f3.a);
          p1 += (4.0 / 3.0) * yy * (ay.uu[1] - 2.5 * f3.b);
          p2 += yy * (ay.uu[2] - 2.5 * f4.a);
          TT += yy * (ay.TT - 2.5 * f4.b);
          const double vy = iy * ay.u[1];
          sh += iy * ay.u[0];
          e[6] = ux + vy;
          e[8] = iy * ay.u[2];
          r[3] += ph.inv_re * p2;
          r[4] += ph.inv_re * (f4.a * p2 + 2.0 * (ux * ux + vy * vy) + sh * sh) + ph.cq * TT;
          asm volatile("" : "+v"(p0), "+v"(p1), "+v"(e[6]), "+v"(e[8]));
          settle(r);
          // D_y(D_x u_1) and D_y(D_x u_0)
          double m0 = 0.0, m1 = 0.0;
#pragma unroll
          for (int s = 0; s < 4; ++s) {
            const int o = c + (s < 2 ? s - 2 : s - 1) * PX;
            const double w = s == 0 ? 1.0 / 12.0 : (s == 1 ? -2.0 / 3.0 : (s == 2 ? 2.0 / 3.0 : -1.0 / 12.0));
            const Two a = two(S, o - 2, 3), b = two(S, o - 1, 3), d = two(S, o + 1, 3), f = two(S, o + 2, 3);
            m0 = __fma_rn(w, d1(a.a, b.a, d.a, f.a), m0);
            m1 = __fma_rn(w, d1(a.b, b.b, d.b, f.b), m1);
          }
          const double k = (1.0 / 3.0) * ix * iy;
          p0 += k * m1;
          p1 += k * m0;
          r[1] += ph.inv_re * p0;
          r[2] += ph.inv_re * p1;
          r[4] += ph.inv_re * (f3.a * p0 + f3.b * p1);
          settle(r);
        } else {
          settle(r);
          add_convect(gather(S, 1, PX, f3.b), 1, iy, q0, r);
          settle(r);
        }
      } else if constexpr (VISC) {
        // a plane that only the z stencils read
        auto at1 = [&](int f, int st) {
          return d1(S[c - 2 * st][f], S[c - st][f], S[c + st][f], S[c + 2 * st][f]);
        };
        e[6] = ix * at1(6, 1) + iy * at1(7, PX);
        e[7] = ix * at1(8, 1);
        e[8] = iy * at1(8, PX);
      }
      if (z >= z0) {
        double r[NV];
#pragma unroll
        for (int m = 0; m < NV; ++m) r[m] = rr[0][m];
        const double* k0 = zq[2];
        const double q0[NV] = {k0[0], k0[1], k0[2], k0[3], k0[4]};
        // velocities and pressure of the column, each rounded (no product is
        // contracted into a difference): equal values have zero derivatives
        auto rounded = [](double v) {
          asm("" : "+v"(v));
          return v;
        };
        double u[5][3], p[5];
#pragma unroll
        for (int s = 0; s < 5; ++s) {
          double ke = 0.0;
#pragma unroll
          for (int m = 0; m < 3; ++m) {
            u[s][m] = rounded(zq[s][1 + m] * zq[s][5]);
            ke += u[s][m] * zq[s][1 + m];
          }
          p[s] = rounded(ph.gm1 * (zq[s][4] - 0.5 * ke));
        }
        auto pl = [](int s) { return s < 2 ? s : s + 1; };
        convect(
            2, iz, [&](int s, int m) { return zq[pl(s)][m]; }, [&](int s) { return u[pl(s)][2]; },
            [&](int s) { return p[pl(s)]; }, q0, u[2][2], r);
        settle(r);
        if constexpr (VISC) {
          double T[5], du[3], ddu[3];
#pragma unroll
          for (int s = 0; s < 5; ++s) T[s] = rounded(cT * p[s] * zq[s][5]);
          const double zz = iz * iz;
#pragma unroll
          for (int m = 0; m < 3; ++m) {
            du[m] = iz * d1(u[0][m], u[1][m], u[3][m], u[4][m]);
            ddu[m] = zz * d2(u[0][m], u[1][m], u[2][m], u[3][m], u[4][m]);
          }
          auto dz = [&](int i) { return iz * d1(zq[0][i], zq[1][i], zq[3][i], zq[4][i]); };
          const double p0 = ddu[0] + (1.0 / 3.0) * dz(7);
          const double p1 = ddu[1] + (1.0 / 3.0) * dz(8);
          const double p2 = (4.0 / 3.0) * ddu[2] + (1.0 / 3.0) * dz(6);
          const double div = k0[6] + du[2], sx = du[0] + k0[7], sy = du[1] + k0[8];
          r[1] += ph.inv_re * p0;
          r[2] += ph.inv_re * p1;
          r[3] += ph.inv_re * p2;
          r[4] += ph.inv_re * (u[2][0] * p0 + u[2][1] * p1 + u[2][2] * p2 + 2.0 * du[2] * du[2] -
                               (2.0 / 3.0) * div * div + sx * sx + sy * sy) +
                  ph.cq * zz * d2(T[0], T[1], T[2], T[3], T[4]);
        }
#pragma unroll
        for (int m = 0; m < NV; ++m) {
          if constexpr (MODE == 2) {
            st_once(r[m], &R[m * g.fs + o], ph.nt);
          } else if constexpr (MODE == 0) {
            const double qo = first ? q0[m] : qa[m];
            st_once(qo + ph.dt * cA * r[m], &Qn[m * g.fs + o], ph.nt);
            st_once(qo + ph.dt * cB * r[m], &Qo[m * g.fs + o], ph.nt);
          } else {
            const double tmp = cA * qa[m] + ph.dt * r[m];
            st_once(tmp, &Qo[m * g.fs + o], ph.nt);
            st_once(q0[m] + cB * tmp, &Qn[m * g.fs + o], ph.nt);
          }
        }
      }
#pragma unroll
      for (int k = 0; k < 4; ++k)
#pragma unroll
        for (int i = 0; i < NQ; ++i) zq[k][i] = zq[k + 1][i];
#pragma unroll
      for (int m = 0; m < NV; ++m) {
        rr[0][m] = rr[1][m];
        rr[1][m] = rr[2][m];
      }
    }
    if (more) {
      store((zp + 1) & 1);  // (last read before the previous barrier)
      __syncthreads();
    }
  }
}

// z segment of a 2.5-D tiled kernel over tx x ty columns: `start` planes,
// halved (down to 2) while the launch would have fewer than `want` blocks.
// The viscous kernels (one 512-thread block per CU, bound by their 104-130 KB
// of LDS) take 64-plane segments from 512 blocks on: each segment stages four
// planes beyond its own, and at 256^3 two rounds of 64 planes beat four of 32
// (0.684 -> 0.673 ms for a viscous + RK kernel).
static int tile_segment(const Grid& g, int tx, int ty, long long want, int start) {
  const long long tiles = (long long)((g.n[0] + tx - 1) / tx) * ((g.n[1] + ty - 1) / ty);
  int sz = start;
  while (sz > 2 && tiles * ((g.n[2] + sz - 1) / sz) < want) sz /= 2;
  return sz;
}
int visc3d_segment(const Grid& g) { return tile_segment(g, VTX, VTY, 512, 64); }

// Tile and z segment of k_central3d.  A segment stages four planes beyond its
// own, and every plane costs a block about the same time whatever the others
// do, so the launch takes rounds * (segment + overhead).  Measured (us, skew +
// viscous): 64 x 8 tiles, one block per CU (131 KB of LDS), 4.0 per plane + 10
// per segment; 32 x 8 tiles, two per CU, 4.2 and 9, or 3.05 and 8 while there
// are no more blocks than CUs.  The cheapest of all is taken: 256^3 64 x 8 x
// 128 (0.73 ms; 4 % more with 32 planes), 128^3 about 91 us (101 with 64 x 8 x 8),
// 24x30x40 and smaller blocks 32 x 8 x 1 (8^3 to 32^3 11 us; 13.5 with two
// planes, 18 with 64-wide tiles).
void central3d_tiles(const Grid& g, int* tx, int* sz) {
  double best = 1.0e300;
  for (int w = 64; w >= 32; w -= 32) {
    const long long tiles = (long long)((g.n[0] + w - 1) / w) * ((g.n[1] + 7) / 8);
    for (int p = 1; p <= 256; ++p) {
      const long long blocks = tiles * ((g.n[2] + p - 1) / p);
      double t;
      if (w == 64) t = (double)((blocks + 255) / 256) * (4.0 * p + 10.0);
      else t = blocks <= 256 ? 3.05 * p + 8.0 : (double)((blocks + 511) / 512) * (4.2 * p + 9.0);
      if (t < best) {
        best = t;
        *tx = w;
        *sz = p;
      }
      if (p >= g.n[2]) break;
    }
  }
}

void launch_central3d(int conv, bool visc, int mode, const double* Q, double* R, double* Qo, double* Qn, const Grid& g,
                      const Phys& ph, double cA, double cB, int first, int tx, int sz, int wrap, hipStream_t s) {
  const dim3 grid((g.n[0] + tx - 1) / tx, (g.n[1] + 7) / 8, (g.n[2] + sz - 1) / sz), block(tx, 8);
  auto go = [&](auto cc, auto vv, auto mm, auto xx, auto yy) {
    k_central3d<decltype(cc)::value, decltype(vv)::value, decltype(mm)::value, decltype(xx)::value, decltype(yy)::value>
        <<<grid, block, 0, s>>>(Q, R, Qo, Qn, g, ph, cA, cB, first, sz, wrap);
  };
  auto with_tile = [&](auto cc, auto vv, auto mm) {
    if (tx == 64) go(cc, vv, mm, std::integral_constant<int, 64>{}, std::integral_constant<int, 8>{});
    else go(cc, vv, mm, std::integral_constant<int, 32>{}, std::integral_constant<int, 8>{});
  };
  auto with_mode = [&](auto cc, auto vv) {
    if (mode == 0) with_tile(cc, vv, std::integral_constant<int, 0>{});
    else if (mode == 1) with_tile(cc, vv, std::integral_constant<int, 1>{});
    else with_tile(cc, vv, std::integral_constant<int, 2>{});
  };
  auto with_visc = [&](auto cc) {
    if (visc) with_mode(cc, std::true_type{});
    else with_mode(cc, std::false_type{});
  };
  if (conv == OSBL_CONV_CENTRAL_SKEW) with_visc(std::integral_constant<int, OSBL_CONV_CENTRAL_SKEW>{});
  else with_visc(std::integral_constant<int, OSBL_CONV_CENTRAL_CONS>{});
}

// interior <-> contiguous copies
__global__ void __launch_bounds__(256) k_pack(const double* __restrict__ F, double* __restrict__ out, Grid g) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= g.n[0]) return;
  const int j = blockIdx.y, k = blockIdx.z;
  out[(long long)i + (long long)g.n[0] * (j + (long long)g.n[1] * k)] = F[g.idx(i, j, k)];
}
__global__ void __launch_bounds__(256) k_unpack(const double* __restrict__ in, double* __restrict__ F, Grid g) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= g.n[0]) return;
  const int j = blockIdx.y, k = blockIdx.z;
  F[g.idx(i, j, k)] = in[(long long)i + (long long)g.n[0] * (j + (long long)g.n[1] * k)];
}

// NaN values among the interior values of fields v0 .. v1-1 (OPS's
// ops_NaNcheck): counted per wave with a ballot, a wave adds to the counter
// only when it found one, so a finite state costs no atomics
__global__ void __launch_bounds__(256) k_count_nan(const double* __restrict__ F, Grid g, int v0, int v1,
                                                  unsigned long long* __restrict__ count) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  const int j = blockIdx.y, k = blockIdx.z;
  unsigned long long found = 0;
  if (i < g.n[0]) {
    const int x = g.idx(i, j, k);
    for (int v = v0; v < v1; ++v) found += __builtin_isnan(F[v * g.fs + x]) ? 1 : 0;
  }
  unsigned long long wave = 0;
  for (int v = 0; v < v1 - v0; ++v) wave += __popcll(__ballot(found > (unsigned long long)v));
  if ((threadIdx.x & 63) == 0 && wave) atomicAdd(count, wave);
}
__global__ void k_clear_count(unsigned long long* count) { *count = 0; }

// ---------------------------------------------------------------------------
// launch helpers (instantiation tables)
// ---------------------------------------------------------------------------
template <int ND, int D, int CONV, int AVG>
static void launch_sweep_t(const double* Q, double* R, const Grid& g, const Phys& ph, int seg, const double* met,
                           const double* theta, hipStream_t s) {
  if constexpr (D == 0 && ND == 3) {
    const int cells = sweep_xl_cells(g);
    const int nwaves = g.n[1] * g.n[2] * ((g.n[0] + cells - 1) / cells);
    const unsigned blocks = (unsigned)((nwaves + XW - 1) / XW);
    k_char_sweep_xl<ND, CONV, AVG>
        <<<blocks, 64 * XW, 0, s>>>(Q, R, g, ph, nwaves, cells, g.periodic_x, met, theta);
  } else {
    long long lines = 1;
    for (int e = 0; e < 3; ++e)
      if (e != D) lines *= g.n[e];
    seg = fit_segment(lines, g.n[D], seg, 4);
    const long long nseg = (g.n[D] + seg - 1) / seg;
    const long long total = lines * nseg;
    const unsigned blocks = (unsigned)((total + 255) / 256);
    const RkArgs none{nullptr, nullptr, 0.0, 0.0, 0};
    // (y and z add to the directions before them, x on a line is the only one)
    k_char_sweep<ND, D, CONV, AVG, (D > 0)><<<blocks, 256, 0, s>>>(Q, R, g, ph, seg, total, met, theta, none);
  }
}

// the last (z) sweep of a 3-D stage fused with the RK update
template <int CONV, int AVG>
static void launch_sweep_rk_t(int mode, const double* Q, double* R, const Grid& g, const Phys& ph, int seg,
                              const double* theta, const RkArgs& rk, hipStream_t s) {
  const long long lines = (long long)g.n[0] * g.n[1];
  seg = fit_segment(lines, g.n[2], seg, 4);
  const long long nseg = (g.n[2] + seg - 1) / seg;
  const long long total = lines * nseg;
  const unsigned blocks = (unsigned)((total + 255) / 256);
  if (mode == 0)
    k_char_sweep<3, 2, CONV, AVG, true, 0><<<blocks, 256, 0, s>>>(Q, R, g, ph, seg, total, nullptr, theta, rk);
  else
    k_char_sweep<3, 2, CONV, AVG, true, 1><<<blocks, 256, 0, s>>>(Q, R, g, ph, seg, total, nullptr, theta, rk);
}

template <int CONV>
static void launch_sweep_rk_avg(int avg, int mode, const double* Q, double* R, const Grid& g, const Phys& ph, int seg,
                                const double* theta, const RkArgs& rk, hipStream_t s) {
  if (avg == OSBL_AVG_ROE) launch_sweep_rk_t<CONV, OSBL_AVG_ROE>(mode, Q, R, g, ph, seg, theta, rk, s);
  else launch_sweep_rk_t<CONV, OSBL_AVG_SIMPLE>(mode, Q, R, g, ph, seg, theta, rk, s);
}

void launch_sweep_z_rk(int conv, int avg, int mode, const double* Q, double* R, double* Qo, double* Qn, const Grid& g,
                       const Phys& ph, int seg, const double* theta, double cA, double cB, int first, hipStream_t s) {
  const RkArgs rk{Qo, Qn, cA, cB, first};
  switch (conv) {
    case OSBL_CONV_WENO_JS: launch_sweep_rk_avg<OSBL_CONV_WENO_JS>(avg, mode, Q, R, g, ph, seg, theta, rk, s); break;
    case OSBL_CONV_WENO_Z: launch_sweep_rk_avg<OSBL_CONV_WENO_Z>(avg, mode, Q, R, g, ph, seg, theta, rk, s); break;
    case OSBL_CONV_TENO5: launch_sweep_rk_avg<OSBL_CONV_TENO5>(avg, mode, Q, R, g, ph, seg, theta, rk, s); break;
    default: launch_sweep_rk_avg<OSBL_CONV_TENO6>(avg, mode, Q, R, g, ph, seg, theta, rk, s); break;
  }
}

template <int ND, int D, int CONV>
static void launch_sweep_avg(int avg, const double* Q, double* R, const Grid& g, const Phys& ph, int seg,
                             const double* met, const double* theta, hipStream_t s) {
  if (avg == OSBL_AVG_ROE) launch_sweep_t<ND, D, CONV, OSBL_AVG_ROE>(Q, R, g, ph, seg, met, theta, s);
  else launch_sweep_t<ND, D, CONV, OSBL_AVG_SIMPLE>(Q, R, g, ph, seg, met, theta, s);
}

template <int ND, int D>
static void launch_sweep_conv(int conv, int avg, const double* Q, double* R, const Grid& g, const Phys& ph, int seg,
                              const double* met, const double* theta, hipStream_t s) {
  switch (conv) {
    case OSBL_CONV_WENO_JS: launch_sweep_avg<ND, D, OSBL_CONV_WENO_JS>(avg, Q, R, g, ph, seg, met, theta, s); break;
    case OSBL_CONV_WENO_Z: launch_sweep_avg<ND, D, OSBL_CONV_WENO_Z>(avg, Q, R, g, ph, seg, met, theta, s); break;
    case OSBL_CONV_TENO5: launch_sweep_avg<ND, D, OSBL_CONV_TENO5>(avg, Q, R, g, ph, seg, met, theta, s); break;
    case CONV_WFILTER:
      // the WENO filter reconstructs with SimpleAverage (WENO_filter.py:324)
      if constexpr (ND == 3) launch_sweep_t<ND, D, CONV_WFILTER, OSBL_AVG_SIMPLE>(Q, R, g, ph, seg, met, theta, s);
      break;
    default: launch_sweep_avg<ND, D, OSBL_CONV_TENO6>(avg, Q, R, g, ph, seg, met, theta, s); break;
  }
}

void launch_sweep(int nd, int d, int conv, int avg, const double* Q, double* R, const Grid& g, const Phys& ph, int seg,
                  const double* met, const double* theta, hipStream_t s) {
  if (nd == 3) {
    if (d == 0) launch_sweep_conv<3, 0>(conv, avg, Q, R, g, ph, seg, met, theta, s);
    else if (d == 1) launch_sweep_conv<3, 1>(conv, avg, Q, R, g, ph, seg, met, theta, s);
    else launch_sweep_conv<3, 2>(conv, avg, Q, R, g, ph, seg, met, theta, s);
  } else {
    launch_sweep_conv<1, 0>(conv, avg, Q, R, g, ph, seg, met, theta, s);
  }
}

template <int ND, int CONV, bool VISC>
static void launch_update_m(int mode, const double* Q, const double* P, double* R, double* Qo, double* Qn,
                            const Grid& g, const Phys& ph, double cA, double cB, int first, hipStream_t s) {
  dim3 grid((g.n[0] + 127) / 128, g.n[1], g.n[2]);
  if (mode == 0) k_update<ND, CONV, VISC, 0><<<grid, 128, 0, s>>>(Q, P, R, Qo, Qn, g, ph, cA, cB, first);
  else if (mode == 1) k_update<ND, CONV, VISC, 1><<<grid, 128, 0, s>>>(Q, P, R, Qo, Qn, g, ph, cA, cB, first);
  else k_update<ND, CONV, VISC, 2><<<grid, 128, 0, s>>>(Q, P, R, Qo, Qn, g, ph, cA, cB, first);
}

template <int ND>
static void launch_update_nd(int conv, bool visc, int mode, const double* Q, const double* P, double* R, double* Qo,
                             double* Qn, const Grid& g, const Phys& ph, double cA, double cB, int first,
                             hipStream_t s) {
  // 1-D blocks, and 3-D Euler blocks of characteristic schemes; the others' stages
  // end in k_central2d/3d, k_char_tile2d, the viscous or general kernels
  if constexpr (ND == 1) {
    if (conv == OSBL_CONV_CENTRAL_SKEW) {
      if (visc) launch_update_m<ND, OSBL_CONV_CENTRAL_SKEW, true>(mode, Q, P, R, Qo, Qn, g, ph, cA, cB, first, s);
      else launch_update_m<ND, OSBL_CONV_CENTRAL_SKEW, false>(mode, Q, P, R, Qo, Qn, g, ph, cA, cB, first, s);
      return;
    }
    if (conv == OSBL_CONV_CENTRAL_CONS) {
      if (visc) launch_update_m<ND, OSBL_CONV_CENTRAL_CONS, true>(mode, Q, P, R, Qo, Qn, g, ph, cA, cB, first, s);
      else launch_update_m<ND, OSBL_CONV_CENTRAL_CONS, false>(mode, Q, P, R, Qo, Qn, g, ph, cA, cB, first, s);
      return;
    }
    if (visc) {
      launch_update_m<ND, OSBL_CONV_WENO_Z, true>(mode, Q, P, R, Qo, Qn, g, ph, cA, cB, first, s);
      return;
    }
  }
  launch_update_m<ND, OSBL_CONV_WENO_Z, false>(mode, Q, P, R, Qo, Qn, g, ph, cA, cB, first, s);
}
void launch_update(int nd, int conv, bool visc, int mode, const double* Q, const double* P, double* R, double* Qo,
                   double* Qn, const Grid& g, const Phys& ph, double cA, double cB, int first, hipStream_t s) {
  if (nd == 3) launch_update_nd<3>(conv, visc, mode, Q, P, R, Qo, Qn, g, ph, cA, cB, first, s);
  else launch_update_nd<1>(conv, visc, mode, Q, P, R, Qo, Qn, g, ph, cA, cB, first, s);
}

void launch_prims(int nd, const double* Q, double* P, const Grid& g, const Phys& ph, hipStream_t s) {
  const int PX = g.n[0] + 2 * g.h[0];
  dim3 grid((PX + 255) / 256, g.n[1] + 2 * g.h[1], g.n[2] + 2 * g.h[2]);
  if (nd == 3) k_prims<3><<<grid, 256, 0, s>>>(Q, P, g, ph);
  else if (nd == 2) k_prims<2><<<grid, 256, 0, s>>>(Q, P, g, ph);
  else k_prims<1><<<grid, 256, 0, s>>>(Q, P, g, ph);
}

long long halo_points(const Grid& g) {
  const long long PX = g.n[0] + 2 * g.h[0], PY = g.n[1] + 2 * g.h[1];
  return 2LL * g.h[2] * PY * PX + 2LL * g.h[1] * g.n[2] * PX + 2LL * g.h[0] * g.n[1] * (long long)g.n[2];
}

void launch_halo_periodic(double* Q, int nv, const Grid& g, hipStream_t s) {
  const long long total = halo_points(g);
  if (total == 0) return;
  k_halo_periodic<<<(unsigned)((total + 255) / 256), 256, 0, s>>>(Q, nv, g, total);
}

void launch_count_nan(const double* F, int v0, int v1, unsigned long long* count, const Grid& g, hipStream_t s) {
  k_clear_count<<<1, 1, 0, s>>>(count);
  dim3 grid((g.n[0] + 255) / 256, g.n[1], g.n[2]);
  k_count_nan<<<grid, 256, 0, s>>>(F, g, v0, v1, count);
}

void launch_pack(const double* F, double* out, const Grid& g, hipStream_t s) {
  dim3 grid((g.n[0] + 255) / 256, g.n[1], g.n[2]);
  k_pack<<<grid, 256, 0, s>>>(F, out, g);
}
void launch_unpack(const double* in, double* F, const Grid& g, hipStream_t s) {
  dim3 grid((g.n[0] + 255) / 256, g.n[1], g.n[2]);
  k_unpack<<<grid, 256, 0, s>>>(in, F, g);
}

}  // namespace osbl
