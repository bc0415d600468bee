// line_segment (osbl_line.h) on the CPU: the 64 lanes of a wave as fibers that
// run one after the other between two wave barriers or shuffles, upwards or
// downwards.  What the lanes do between two barriers may happen in any order,
// so the results must not depend on it.
#include <algorithm>
#include <ucontext.h>
#include <vector>

#include <hip/hip_runtime.h>

#include "osbl_line.h"

using namespace osbl;

namespace {

constexpr int WAVE = 64;
ucontext_t main_ctx, lane_ctx[WAVE];
bool done[WAVE];
int cur;
double exchange[WAVE];
std::vector<char> stacks;

struct Task {
  int n, s0, s1, first, conv, mode;
  double dt, inv_dx, cA, cB;
  Phys ph;
  const double* q;
  double *qo, *qn;
  double (*S)[LINE_NF];
} task;

template <int CONV, int MODE>
void segment() {
  const Task& t = task;
  line_segment<CONV, OSBL_AVG_ROE, MODE>(
      t.S, cur, t.n, t.s0, t.s1, t.dt, t.inv_dx, t.ph, t.cA, t.cB, t.first != 0,
      [&](int x, double (&q)[3]) { for (int m = 0; m < 3; ++m) q[m] = t.q[m * t.n + x]; },
      [&](int x, double (&q)[3]) { for (int m = 0; m < 3; ++m) q[m] = t.qo[m * t.n + x]; },
      [&](int x, const double (&qn)[3], const double (&qo)[3]) {
        for (int m = 0; m < 3; ++m) {
          t.qn[m * t.n + x] = qn[m];
          t.qo[m * t.n + x] = qo[m];
        }
      });
}

void lane_main() {
  if (task.conv == OSBL_CONV_WENO_Z) task.mode == 0 ? segment<OSBL_CONV_WENO_Z, 0>() : segment<OSBL_CONV_WENO_Z, 1>();
  else task.mode == 0 ? segment<OSBL_CONV_TENO6, 0>() : segment<OSBL_CONV_TENO6, 1>();
  done[cur] = true;
}

}  // namespace

void host_wave_barrier() { swapcontext(&lane_ctx[cur], &main_ctx); }

double host_shfl(double v, int delta, int lane) {
  exchange[cur] = v;
  host_wave_barrier();
  const double r = exchange[lane >= 0 ? lane : std::max(cur - delta, 0)];
  host_wave_barrier();
  return r;
}

// cells [s0, s1) of a line by one wave, lanes upwards or downwards between barriers
extern "C" void run_segment(int conv, int mode, int n, int s0, int s1, double dt, double inv_dx, double cA, double cB,
                            int first, double gama, double eps, double ct, const double* q, double* qo, double* qn,
                            int downwards) {
  std::vector<double> S((size_t)LINE_PTS * LINE_NF, 0.0);
  Phys ph{};
  ph.gama = gama;
  ph.gm1 = gama - 1.0;
  ph.igm1 = 1.0 / ph.gm1;
  ph.eps = eps;
  ph.teno_ct = ct;
  task = Task{n, s0, s1, first, conv, mode, dt, inv_dx, cA, cB, ph, q, qo, qn,
              reinterpret_cast<double (*)[LINE_NF]>(S.data())};
  constexpr size_t STACK = 1 << 16;
  stacks.resize(STACK * WAVE);
  for (int l = 0; l < WAVE; ++l) {
    done[l] = false;
    getcontext(&lane_ctx[l]);
    lane_ctx[l].uc_stack.ss_sp = stacks.data() + STACK * l;
    lane_ctx[l].uc_stack.ss_size = STACK;
    lane_ctx[l].uc_link = &main_ctx;
    makecontext(&lane_ctx[l], lane_main, 0);
  }
  for (bool any = true; any;) {
    any = false;
    for (int k = 0; k < WAVE; ++k) {
      cur = downwards ? WAVE - 1 - k : k;
      if (done[cur]) continue;
      any = true;
      swapcontext(&main_ctx, &lane_ctx[cur]);
    }
  }
}
