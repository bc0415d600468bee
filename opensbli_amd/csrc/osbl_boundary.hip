// osbl_boundary.hip -- boundary kernels of non-periodic faces and the
// periodic exchange of one direction.  The faces' kernels run over the boundary
// planes of both faces of a direction (2-D: of all four faces) with the other
// directions' halos included (bc_core.py:163-171); one thread owns one line
// normal to a face.
#include "osbl_kernels.h"

namespace osbl {

namespace {

// temperature from the conservative variables of a point (ns_physics.py:105-106)
template <int ND>
__device__ __forceinline__ double t_cons(const double (&q)[ND + 2], const Phys& ph) {
  double m2 = 0.0;
#pragma unroll
  for (int m = 0; m < ND; ++m) m2 += q[1 + m] * q[1 + m];
  return (q[ND + 1] - 0.5 * m2 / q[0]) * (ph.gama * ph.gm1 * ph.Minf * ph.Minf) / q[0];
}

constexpr int BC_H = 4;  // halo points a block keeps at most

}  // namespace

// What a direction's two faces need: type OSBL_BC_*, halo points filled and
// the face's values [nv][n_e2][n_e1] (Dirichlet) per side.
struct BcSides {
  int type[2], nh[2];
  const double* plane[2];
};

// The line normal to face (d, side) through the face point (ia, ib) of the
// other directions (halos included); `st` below is the storage stride pointing
// inward, Q2 the other state buffer (inlet: its rhoE halos are kept equal to
// those of Q).  A line touches its own face's points and halos only and reads
// at most four points inward, so both faces of a direction (at least 8 points
// apart) can be done at once.
template <int ND>
__device__ __forceinline__ void bc_line(double* __restrict__ Q, double* __restrict__ Q2, const Grid& g,
                                        const Phys& ph, int d, int side, int type, int nh, double twall,
                                        const double* __restrict__ plane, int ia, int ib) {
  constexpr int NV = ND + 2;
  const int e1 = d == 0 ? 1 : 0, e2 = d == 2 ? 1 : 2;
  int c[3];
  c[e1] = ia;
  c[e2] = ib;
  c[d] = side == 0 ? 0 : g.n[d] - 1;
  const int x = g.idx(c[0], c[1], c[2]);
  const int st = (side == 0 ? 1 : -1) * g.stride(d);
  const long long fs = g.fs;
  const double gm = ph.gama, M2 = ph.Minf * ph.Minf;
  // A line's points are loaded at once and its new values stored at once: one
  // memory latency instead of one per halo point (a 500x250 block's faces:
  // 16 -> 13 us under the profiler).  v[k] is point k inward, w[k] halo point k.
  double v[BC_H + 1][NV], w[BC_H + 1][NV];
  auto load = [&](int first, int last) {
#pragma unroll
    for (int k = 0; k <= BC_H; ++k)
      if (k >= first && k <= last) {
#pragma unroll
        for (int m = 0; m < NV; ++m) v[k][m] = Q[m * fs + x + k * st];
      }
  };
  auto store_point = [&] {
#pragma unroll
    for (int m = 0; m < NV; ++m) Q[m * fs + x] = v[0][m];
  };
  auto store_halos = [&](int n) {
#pragma unroll
    for (int k = 1; k <= BC_H; ++k)
      if (k <= n) {
#pragma unroll
        for (int m = 0; m < NV; ++m) Q[m * fs + x - k * st] = w[k][m];
      }
  };
  auto halos_are = [&](const double (&q)[NV]) {
#pragma unroll
    for (int k = 1; k <= BC_H; ++k)
#pragma unroll
      for (int m = 0; m < NV; ++m) w[k][m] = q[m];
  };
  switch (type) {
    case OSBL_BC_PERIODIC:  // periodic.py:42-56
#pragma unroll
      for (int k = 1; k <= BC_H; ++k)
        if (k <= g.h[d]) {
#pragma unroll
          for (int m = 0; m < NV; ++m) w[k][m] = Q[m * fs + x + (g.n[d] - k) * st];
        }
      store_halos(g.h[d]);
      break;
    case OSBL_BC_EXTRAP0:  // boundary point and halos take the first point inside (extrapolation.py:29-58)
      load(1, 1);
#pragma unroll
      for (int m = 0; m < NV; ++m) v[0][m] = v[1][m];
      halos_are(v[1]);
      store_point();
      store_halos(g.h[d]);
      break;
    case OSBL_BC_EXTRAP1:  // halo i = 2 q[i-1] - q[i-2], outward (extrapolation.py:42-54)
      load(0, 1);
#pragma unroll
      for (int m = 0; m < NV; ++m) {
        w[1][m] = 2.0 * v[0][m] - v[1][m];
        w[2][m] = 2.0 * w[1][m] - v[0][m];
        w[3][m] = 2.0 * w[2][m] - w[1][m];
        w[4][m] = 2.0 * w[3][m] - w[2][m];
      }
      store_halos(nh);
      break;
    case OSBL_BC_SYMMETRY:  // symmetry.py:24-48: mirror images, normal momentum negated; the boundary point stays
      load(1, nh);
#pragma unroll
      for (int k = 1; k <= BC_H; ++k)
#pragma unroll
        for (int m = 0; m < NV; ++m) w[k][m] = (m == 1 + d) ? -v[k][m] : v[k][m];
      store_halos(nh);
      break;
    case OSBL_BC_ZERO_GRADIENT:  // q[0] = q[1]; q[-i] = q[i] (zero_gradient_outlet.py:16-23)
      load(1, nh > 1 ? nh : 1);
#pragma unroll
      for (int m = 0; m < NV; ++m) v[0][m] = v[1][m];
#pragma unroll
      for (int k = 1; k <= BC_H; ++k)
#pragma unroll
        for (int m = 0; m < NV; ++m) w[k][m] = v[k][m];
      store_point();
      store_halos(nh);
      break;
    case OSBL_BC_ADIABATIC_WALL: {  // adiabatic_wall.py:28-69
      load(0, nh > 3 ? nh : 3);
#pragma unroll
      for (int m = 0; m < ND; ++m) v[0][1 + m] = 0.0;
      const double T1 = t_cons<ND>(v[1], ph), T2 = t_cons<ND>(v[2], ph), T3 = t_cons<ND>(v[3], ph);
      // Carpenter's one-sided dT/dn = 0 at the wall
      const double Tw = (6.0 / 11.0) * (3.0 * T1 + (1.0 / 3.0) * T3 - (3.0 / 2.0) * T2);
      const double pw = v[0][0] * Tw / (gm * M2);
      v[0][ND + 1] = pw / ph.gm1;
#pragma unroll
      for (int k = 1; k <= BC_H; ++k)
#pragma unroll
        for (int m = 0; m < NV; ++m) w[k][m] = (m == 0 || m == ND + 1) ? v[k][m] : -v[k][m];
      store_point();
      store_halos(nh);
      break;
    }
    case OSBL_BC_ISOTHERMAL_WALL: {  // isothermal_wall.py:33-88
      load(0, nh > 1 ? nh : 1);
#pragma unroll
      for (int m = 0; m < ND; ++m) v[0][1 + m] = 0.0;
      v[0][ND + 1] = v[0][0] * twall / (gm * ph.gm1 * M2);
      // wall pressure from the updated wall state (momentum is zero there)
      const double pw = ph.gm1 * (v[0][ND + 1] - 0.5 * 0.0 / v[0][0]);
      const double Ta = t_cons<ND>(v[1], ph);
#pragma unroll
      for (int k = 1; k <= BC_H; ++k) {
        double uh[ND];
        double ke = 0.0;
#pragma unroll
        for (int m = 0; m < ND; ++m) {
          uh[m] = v[k][1 + m] / v[k][0];
          ke += uh[m] * uh[m];
        }
        const double Th = (k + 1) * twall - k * Ta;
        const double rh = pw * gm * M2 / Th;
#pragma unroll
        for (int m = 0; m < ND; ++m) w[k][1 + m] = -rh * uh[m];
        w[k][ND + 1] = pw / ph.gm1 + 0.5 * rh * ke;
        w[k][0] = rh;
      }
      store_point();
      store_halos(nh);
      break;
    }
    case OSBL_BC_DIRICHLET: {  // dirichlet.py:28-41
      const int n1i = g.n[e1], n2i = g.n[e2];
      const int pa = ia < 0 ? 0 : (ia >= n1i ? n1i - 1 : ia);
      const int pb = ib < 0 ? 0 : (ib >= n2i ? n2i - 1 : ib);
#pragma unroll
      for (int m = 0; m < NV; ++m) v[0][m] = plane[((long long)m * n2i + pb) * n1i + pa];
      halos_are(v[0]);
      store_point();
      store_halos(nh);
      break;
    }
    case OSBL_BC_INLET_PEXTRAP: {  // inlet_pressure_extrapolate.py:32-66, side 0
      load(0, 0);
#pragma unroll
      for (int m = 0; m < NV; ++m) w[1][m] = Q[m * fs + x - st];
      const double rb = v[0][0];
      double ke = 0.0, un = 0.0;
#pragma unroll
      for (int m = 0; m < ND; ++m) {
        const double ub = fabs(v[0][1 + m] / rb);
        ke += ub * ub;
        if (m == d) un = ub;
      }
      const double pb = ph.gm1 * (v[0][ND + 1] - 0.5 * rb * ke);
      const double ab = sqrt(gm * pb / rb);
      if (un >= ab) {
#pragma unroll
        for (int m = 0; m < NV; ++m) Q[m * fs + x] = w[1][m];
      } else {
        const double e0 = v[0][ND + 1];
        for (int hh = 1; hh <= nh; ++hh) {
          Q[(ND + 1) * fs + x - hh * st] = e0;
          Q2[(ND + 1) * fs + x - hh * st] = e0;
        }
      }
      break;
    }
    default:
      break;
  }
}

// both faces of direction d
template <int ND>
__global__ void __launch_bounds__(256) k_bc_sides(double* __restrict__ Q, double* __restrict__ Q2, Grid g, Phys ph,
                                                  int d, BcSides f, double twall) {
  const int e1 = d == 0 ? 1 : 0, e2 = d == 2 ? 1 : 2;
  const int n1 = g.n[e1] + 2 * g.h[e1], n2 = g.n[e2] + 2 * g.h[e2];
  int t = blockIdx.x * blockDim.x + threadIdx.x;
  if (t >= 2 * n1 * n2) return;
  const int side = t >= n1 * n2;
  t -= side * n1 * n2;
  bc_line<ND>(Q, Q2, g, ph, d, side, f.type[side], f.nh[side], twall, f.plane[side], t % n1 - g.h[e1],
              t / n1 - g.h[e2]);
}

// A 2-D block's four faces in one launch, direction 0 before direction 1 where
// they meet (block.py:199-210).  A line reaches four points inward (a periodic
// one the last four of its direction), so only lines within five rows or
// columns of a corner see another face's: workgroup 0 takes those of direction
// 0, waits, and takes those of direction 1; every other wave has 64 lines of
// one face to itself.  Bound by one memory round trip a phase.  The faces of a
// 500x250 block under the profiler: 4 to 7 us each in a launch per face, 16 us
// in one workgroup (its one address unit splits the x faces' lines into 64
// cache lines a load), 13 with the lines' loads made at once, 5.3 as here.
constexpr int BC_EDGE = 5;

__host__ __device__ inline int bc_mid_blocks(const Grid& g, int d) {  // waves for the inner lines of a face of d
  const int mid = g.n[1 - d] - 2 * BC_EDGE;
  return mid > 0 ? (mid + 63) / 64 : 0;
}

__global__ void __launch_bounds__(64) k_bc_block2d(double* __restrict__ Q, double* __restrict__ Q2, Grid g, Phys ph,
                                                   BcSides f0, BcSides f1, double twall) {
  if (blockIdx.x == 0) {
#pragma unroll
    for (int d = 0; d < 2; ++d) {
      const BcSides& f = d == 0 ? f0 : f1;
      const int h = g.h[1 - d], all = g.n[1 - d] + 2 * h, nc = min(2 * (h + BC_EDGE), all);
      const int t = threadIdx.x;  // 2 nc <= 36 lines
      if (t < 2 * nc) {
        const int side = t >= nc, l = t - side * nc;
        bc_line<2>(Q, Q2, g, ph, d, side, f.type[side], f.nh[side], twall, f.plane[side],
                   (l < nc / 2 ? l : all - nc + l) - h, 0);
      }
      __syncthreads();
    }
    return;
  }
  const int b0 = bc_mid_blocks(g, 0), b1 = bc_mid_blocks(g, 1);
  int b = blockIdx.x - 1;
  auto face = [&](auto dc, const BcSides& f, int per) {
    constexpr int d = decltype(dc)::value;
    const int side = b >= per, l = BC_EDGE + (b - side * per) * 64 + threadIdx.x;
    if (l < g.n[1 - d] - BC_EDGE)
      bc_line<2>(Q, Q2, g, ph, d, side, f.type[side], f.nh[side], twall, f.plane[side], l, 0);
  };
  if (b < 2 * b0) {
    face(std::integral_constant<int, 0>{}, f0, b0);
  } else {
    b -= 2 * b0;
    face(std::integral_constant<int, 1>{}, f1, b1);
  }
}

// Periodic exchange of one direction over the full extents of the others
// (periodic.py:42-56): halo points [-h, 0) and [N, N+h) take their images.
__global__ void __launch_bounds__(256) k_periodic_dir(double* __restrict__ Q, int nv, Grid g, int d) {
  const int e1 = d == 0 ? 1 : 0, e2 = d == 2 ? 1 : 2;
  const int n1 = g.n[e1] + 2 * g.h[e1], n2 = g.n[e2] + 2 * g.h[e2];
  const int h = g.h[d], N = g.n[d];
  const long long total = (long long)n1 * n2 * 2 * h;
  const long long t = (long long)blockIdx.x * blockDim.x + threadIdx.x;
  if (t >= total) return;
  const int hh = (int)(t % (2 * h));
  const long long r = t / (2 * h);
  int c[3], s[3];
  c[e1] = s[e1] = (int)(r % n1) - g.h[e1];
  c[e2] = s[e2] = (int)(r / n1) - g.h[e2];
  c[d] = hh < h ? hh - h : N + (hh - h);
  s[d] = hh < h ? c[d] + N : c[d] - N;
  const int dst = g.idx(c[0], c[1], c[2]), src = g.idx(s[0], s[1], s[2]);
  for (int m = 0; m < nv; ++m) Q[m * g.fs + dst] = Q[m * g.fs + src];
}

// Every halo point of face (d, side) takes the plane's values (the inflow
// state an inlet face keeps in its halos).
__global__ void __launch_bounds__(256) k_fill_face_halo(double* __restrict__ Q, int nv, Grid g, int d, int side,
                                                        const double* __restrict__ plane) {
  const int e1 = d == 0 ? 1 : 0, e2 = d == 2 ? 1 : 2;
  const int n1 = g.n[e1] + 2 * g.h[e1], n2 = g.n[e2] + 2 * g.h[e2];
  const int t = blockIdx.x * blockDim.x + threadIdx.x;
  if (t >= n1 * n2) return;
  int c[3];
  const int ia = t % n1 - g.h[e1], ib = t / n1 - g.h[e2];
  c[e1] = ia;
  c[e2] = ib;
  c[d] = side == 0 ? 0 : g.n[d] - 1;
  const int x = g.idx(c[0], c[1], c[2]);
  const int st = (side == 0 ? 1 : -1) * g.stride(d);
  const int n1i = g.n[e1], n2i = g.n[e2];
  const int pa = ia < 0 ? 0 : (ia >= n1i ? n1i - 1 : ia);
  const int pb = ib < 0 ? 0 : (ib >= n2i ? n2i - 1 : ib);
  for (int v = 0; v < nv; ++v) {
    const double val = plane[((long long)v * n2i + pb) * n1i + pa];
    for (int hh = 1; hh <= g.h[d]; ++hh) Q[v * g.fs + x - hh * st] = val;
  }
}

static BcSides bc_sides(const Grid& g, int d, const int type[2], const int nh[2], double* const plane[2]) {
  BcSides f;
  for (int s = 0; s < 2; ++s) {
    f.type[s] = type[s];
    f.nh[s] = nh[s] > g.h[d] ? g.h[d] : nh[s];
    f.plane[s] = plane[s];
  }
  return f;
}

void launch_bc_sides(int nd, double* Q, double* Q2, const Grid& g, const Phys& ph, int d, const int type[2],
                     const int nh[2], double twall, double* const plane[2], hipStream_t s) {
  const int e1 = d == 0 ? 1 : 0, e2 = d == 2 ? 1 : 2;
  const int n = 2 * (g.n[e1] + 2 * g.h[e1]) * (g.n[e2] + 2 * g.h[e2]);
  const BcSides f = bc_sides(g, d, type, nh, plane);
  if (nd == 3) k_bc_sides<3><<<(n + 255) / 256, 256, 0, s>>>(Q, Q2, g, ph, d, f, twall);
  else k_bc_sides<1><<<(n + 255) / 256, 256, 0, s>>>(Q, Q2, g, ph, d, f, twall);
}

void launch_bc_block2d(double* Q, double* Q2, const Grid& g, const Phys& ph, const int (*type)[2], const int (*nh)[2],
                       double twall, double* const (*plane)[2], hipStream_t s) {
  const int blocks = 1 + 2 * (bc_mid_blocks(g, 0) + bc_mid_blocks(g, 1));
  k_bc_block2d<<<blocks, 64, 0, s>>>(Q, Q2, g, ph, bc_sides(g, 0, type[0], nh[0], plane[0]),
                                  bc_sides(g, 1, type[1], nh[1], plane[1]), twall);
}

void launch_periodic_dir(double* Q, int nv, const Grid& g, int d, hipStream_t s) {
  const int e1 = d == 0 ? 1 : 0, e2 = d == 2 ? 1 : 2;
  const long long total = (long long)(g.n[e1] + 2 * g.h[e1]) * (g.n[e2] + 2 * g.h[e2]) * 2 * g.h[d];
  k_periodic_dir<<<(unsigned)((total + 255) / 256), 256, 0, s>>>(Q, nv, g, d);
}

void launch_fill_face_halo(double* Q, int nv, const Grid& g, int d, int side, const double* plane, hipStream_t s) {
  const int e1 = d == 0 ? 1 : 0, e2 = d == 2 ? 1 : 2;
  const int n = (g.n[e1] + 2 * g.h[e1]) * (g.n[e2] + 2 * g.h[e2]);
  k_fill_face_halo<<<(n + 255) / 256, 256, 0, s>>>(Q, nv, g, d, side, plane);
}

}  // namespace osbl
