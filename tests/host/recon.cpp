// The TENO weights and the short quotients and roots of osbl_device.h on the CPU.
#include <algorithm>

#include <hip/hip_runtime.h>

#include "osbl_device.h"

void host_wave_barrier() {}
double host_shfl(double v, int, int) { return v; }

using namespace osbl;

// n reconstructions of the differences d[5 i ..]: numerators and denominators
extern "C" void teno(int six, int quirk, long n, const double* d, double eps, double ct, double* num, double* den) {
  for (long i = 0; i < n; ++i) {
    const double* x = d + 5 * i;
    if (six && quirk) teno_gap<true, true>(x[0], x[1], x[2], x[3], x[4], eps, ct, num[i], den[i]);
    else if (six) teno_gap<true, false>(x[0], x[1], x[2], x[3], x[4], eps, ct, num[i], den[i]);
    else teno_gap<false, false>(x[0], x[1], x[2], x[3], x[4], eps, ct, num[i], den[i]);
  }
}
