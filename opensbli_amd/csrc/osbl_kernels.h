// osbl_kernels.h -- launch interface of the gfx950 kernels (host side).
#pragma once

#include "osbl_device.h"

namespace osbl {

void launch_halo_periodic(double* Q, int nv, const Grid& g, hipStream_t s);
void launch_prims(int nd, const double* Q, double* P, const Grid& g, const Phys& ph, hipStream_t s);
// the characteristic sweep of direction d (1-D, 3-D): d = 0 assigns R, the others add to it
void launch_sweep(int nd, int d, int conv, int avg, const double* Q, double* R, const Grid& g, const Phys& ph, int seg,
                  const double* met, const double* theta, hipStream_t s);
// one stage of a 2-D characteristic block (osbl_tile2d.hip); theta: the
// adaptive TENO's sensor is formed and left there; wrap: periodic in both
// directions, halos not read.  conv CONV_WFILTER, mode 2: the WENO filter's
// flux differences into R.  PK, when given: Q's interior, packed
void launch_char_tile2d(int conv, int avg, int mode, bool visc, const double* Q, double* R, double* Qo, double* Qn,
                        const Grid& g, const Phys& ph, const Bnd& b, double cA, double cB, int first, double* theta,
                        int suth, int wrap, double* PK, hipStream_t s);
// one stage of a 2-D central scheme on a uniform grid without closures; PK as above
void launch_central2d(int conv, bool visc, int mode, const double* Q, double* R, double* Qo, double* Qn, const Grid& g,
                      const Phys& ph, double cA, double cB, int first, int wrap, double* PK, hipStream_t s);
void launch_sweep_z_rk(int conv, int avg, int mode, const double* Q, double* R, double* Qo, double* Qn, const Grid& g,
                       const Phys& ph, int seg, const double* theta, double cA, double cB, int first, hipStream_t s);
void launch_sensor(int nd, const double* Q, double* theta, const Grid& g, const Phys& ph, const Bnd& b, hipStream_t s);
void launch_update(int nd, int conv, bool visc, int mode, const double* Q, const double* P, double* R, double* Qo,
                   double* Qn, const Grid& g, const Phys& ph, double cA, double cB, int first, hipStream_t s);
void launch_visc_update3d(const double* Q, double* R, const Grid& g, const Phys& ph, int sz, hipStream_t s);
int visc3d_segment(const Grid& g);  // its z segment for a grid
// one stage of a 3-D central scheme; tiles of tx x 8 columns, sz planes
// (central3d_tiles); wrap: periodic in every direction, halos not read
void launch_central3d(int conv, bool visc, int mode, const double* Q, double* R, double* Qo, double* Qn, const Grid& g,
                      const Phys& ph, double cA, double cB, int first, int tx, int sz, int wrap, hipStream_t s);
void central3d_tiles(const Grid& g, int* tx, int* sz);
void launch_update_gen(int nd, int conv, bool visc, int mode, const double* Q, const double* P, double* R,
                       double* Qo, double* Qn, const Grid& g, const Phys& ph, const Bnd& b, double cA, double cB,
                       int first, int suth, hipStream_t s);
void launch_visc_gen3d(const double* Q, const double* P, double* R, const Grid& g, const Phys& ph, const Bnd& b,
                       int suth, int sz, hipStream_t s);
void launch_body_force3d(const double* Q, double* R, const Grid& g, const Phys& ph, hipStream_t s);
void launch_prims_slab(const double* Q, double* P, const Grid& g, const Phys& ph, int suth, hipStream_t s);
void launch_prims_mu(int nd, const double* Q, double* P, const Grid& g, const Phys& ph, hipStream_t s);
// the two faces of direction d (1-D, 3-D); the four faces of a 2-D block
void launch_bc_sides(int nd, double* Q, double* Q2, const Grid& g, const Phys& ph, int d, const int type[2],
                     const int nh[2], double twall, double* const plane[2], hipStream_t s);
void launch_bc_block2d(double* Q, double* Q2, const Grid& g, const Phys& ph, const int (*type)[2], const int (*nh)[2],
                       double twall, double* const (*plane)[2], hipStream_t s);
void launch_periodic_dir(double* Q, int nv, const Grid& g, int d, hipStream_t s);
void launch_fill_face_halo(double* Q, int nv, const Grid& g, int d, int side, const double* plane, hipStream_t s);
void launch_pack(const double* F, double* out, const Grid& g, hipStream_t s);
void launch_count_nan(const double* F, int v0, int v1, unsigned long long* count, const Grid& g, hipStream_t s);
void launch_unpack(const double* in, double* F, const Grid& g, hipStream_t s);
long long halo_points(const Grid& g);
void launch_rhs_vjp(int nd, const double* Q, const double* P, const double* M, double* out, const Grid& g,
                    const Phys& ph, hipStream_t s);
// a 2-D reverse stage of the central scheme (euler) and/or of the viscous terms
// (alone: added to out1), on packed arrays
void launch_adj_tile2d(bool euler, bool visc, const double* Qs, const double* A, const double* B, double alpha,
                       double beta, double c, double* out1, double* out2, const Grid& g, const Phys& ph,
                       hipStream_t s);
void launch_adj_stage(int nd, const double* Qs, const double* A, const double* B, double alpha, double beta, double c,
                      double* out1, double* out2, const Grid& g, const Phys& ph, hipStream_t s);
void launch_pack_all(const double* F, double* out, const Grid& g, int nv, hipStream_t s);
void launch_adj_stage_char(int nd, int avg, const double* Qs, const double* A, const double* B, double alpha,
                           double beta, double c, double* out1, double* out2, const Grid& g, const Phys& ph, bool acc,
                           hipStream_t s, double* vy = nullptr);
int visc_vjp_fields(int nd);
void launch_unpack_prims(int nd, const double* q, double* Qpad, double* P, const Grid& g, const Phys& ph,
                         hipStream_t s);
void launch_visc_vjp(int nd, const double* q, const double* A, const double* B, double alpha, double beta, double* P,
                     double* Mpad, double* W, double* out, const Grid& g, const Phys& ph, hipStream_t s);
void launch_weno_filter_apply(int nd, double* Q, const double* R, double* theta, const Grid& g, const Phys& ph,
                              bool ducros, bool mach, double control, int walls, hipStream_t s);
void launch_sfd(int nd, double* Q, double* F, const Grid& g, double c, double E, hipStream_t s);
void launch_binomial(int nd, const double* Q, double* Qn, const Grid& g, const double* w, int N, double sigma,
                     const unsigned char* mask, hipStream_t s);
void launch_lincomb(double* out, double a, const double* x, double b, const double* y, long long n, hipStream_t s);

void launch_curv_sweep(int nd, int d, int conv, int avg, int mode, const double* Q, const double* M, double* R,
                       double* Qo, double* Qn, const Grid& g, const Phys& ph, double cA, double cB, int first,
                       hipStream_t s);
void launch_curv_metric(int nd, const double* X, double* M, const Grid& g, const Phys& ph, const int e[3],
                        hipStream_t s);

// 1-D block with zeroth-order extrapolation ends: nsteps iterations of a line
// of at most LINE_RUN_MAX points in one launch (state left in Q, ends filled;
// Q2 and Qo are scratch), or one stage Q -> Qn of any line (its ends are read
// as the boundary condition gives them, and left to a later boundary pass)
constexpr int LINE_RUN_MAX = 16 * 63;
int launch_line_run(int conv, int avg, int mode, double* Q, double* Q2, double* Qo, const Grid& g, const Phys& ph,
                    const double* A, const double* B, int ns, int nsteps, hipStream_t s);
void launch_line_stage(int conv, int avg, int mode, const double* Q, double* Qo, double* Qn, const Grid& g,
                       const Phys& ph, const double* A, const double* B, int ns, int stage, hipStream_t s);

// record the thread-local message osbl_last_error() returns; returns code
int set_error(int code, const char* msg);

}  // namespace osbl
