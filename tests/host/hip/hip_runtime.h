// Host stand-in for the HIP header, so that osbl_device.h and osbl_line.h run
// on the CPU: the qualifiers vanish, the hardware estimates become quotients
// and roots off by what the hardware's may be, and the cross-lane operations
// go to the fibers of line_lanes.cpp.
#pragma once
#include <cmath>
#include <cstdint>
#include <cstring>

#define __host__
#define __device__
#define __global__
#define __forceinline__ inline
struct HostDim {
  unsigned x, y, z;
};
inline HostDim gridDim{1, 1, 1}, blockIdx{0, 0, 0};
// the one instruction written out (max_abs); empty asm statements compile as they are
#define asm(...) r = std::fmax(m, std::fabs(x))

inline double __fma_rn(double a, double b, double c) { return std::fma(a, b, c); }
inline double __dmul_rn(double a, double b) { volatile double r = a * b; return r; }
inline double __dadd_rn(double a, double b) { volatile double r = a + b; return r; }
inline double __dsub_rn(double a, double b) { volatile double r = a - b; return r; }
using std::fabs;
using std::floor;
using std::fmax;
using std::max;
using std::min;

// estimates within 2^-24.2, by a fraction of that drawn from the operand's bits
inline double host_off(double x) {
  uint64_t u;
  std::memcpy(&u, &x, 8);
  u *= 0x9E3779B97F4A7C15ull;
  return 1.0 + ((double)(u >> 40) / 8388608.0 - 1.0) * 5.0e-8;
}
#define __builtin_amdgcn_rcp(x) ((1.0 / (x)) * host_off(x))
#define __builtin_amdgcn_rsq(x) ((1.0 / std::sqrt(x)) * host_off(x))
#define __builtin_nontemporal_load(p) (*(p))
#define __builtin_nontemporal_store(v, p) (void)(*(p) = (v))
#define __builtin_amdgcn_sched_barrier(x) ((void)0)
#define __builtin_amdgcn_fence(order, scope) ((void)0)
#define __builtin_amdgcn_wave_barrier() host_wave_barrier()

void host_wave_barrier();
double host_shfl(double v, int from_delta, int from_lane);
inline double __shfl_up(double v, int d) { return host_shfl(v, d, -1); }
inline double __shfl(double v, int lane) { return host_shfl(v, 0, lane); }
