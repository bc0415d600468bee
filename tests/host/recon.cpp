// The TENO and WENO weights and the short quotients and roots of osbl_device.h on the CPU.
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

// the same of WENO5-Z and -JS, from four differences each
extern "C" void weno(int z, long n, const double* d, double eps, double* num, double* den) {
  for (long i = 0; i < n; ++i) {
    const double* x = d + 5 * i;
    if (z) weno5_gap<true>(x[0], x[1], x[2], x[3], eps, num[i], den[i]);
    else weno5_gap<false>(x[0], x[1], x[2], x[3], eps, num[i], den[i]);
  }
}

// the largest errors of a/b, 1/b and sqrt(b) over n operands, in units in the last place
extern "C" void ulps(long n, const double* a, const double* b, double* worst) {
  auto err = [](double got, long double want) {
    int e;
    std::frexp((double)want, &e);
    return (double)(std::fabs((long double)got - want) / std::ldexp(1.0L, e - 53));
  };
  worst[0] = worst[1] = worst[2] = 0.0;
  for (long i = 0; i < n; ++i) {
    worst[0] = std::max(worst[0], err(quot_pos(a[i], b[i]), (long double)a[i] / b[i]));
    worst[1] = std::max(worst[1], err(recip_pos(b[i]), 1.0L / b[i]));
    worst[2] = std::max(worst[2], err(sqrt_pos(b[i]), std::sqrt((long double)b[i])));
  }
}
