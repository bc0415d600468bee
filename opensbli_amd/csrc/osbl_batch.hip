// osbl_batch.hip -- ensembles of independent 1-D Euler problems of uneven
// size (WENO/TENO characteristic LLF fluxes, zeroth-order extrapolation ends,
// 3-register or low-storage RK), integrated on one GPU.
//
// Storage: each variable is one array holding every instance's points back
// to back, each instance with H halo points on both sides.
//
// Two executions, same arithmetic (line_segment, osbl_line.h), so the results
// are bitwise identical:
//  * persistent: one launch; workgroup b integrates instance order[b]
//    through all its steps and stages, with a workgroup barrier per stage.
//    Up to 16 waves share a line; the autotuner can set the threads by size.
//  * staged: one launch per RK stage covering every instance still running;
//    the stages of a chunk of steps are captured once into a hipGraph (two,
//    when a chunk ends on the other ping-pong buffer) and replayed for every
//    chunk, the step number coming from a device counter.
#include <algorithm>
#include <cmath>
#include <cstring>
#include <mutex>
#include <string>
#include <vector>

#include "osbl_kernels.h"
#include "osbl_line.h"

using namespace osbl;

namespace {

constexpr int BH = 4;  // halo points per side

struct Inst {
  int n;           // points
  int off;         // index of point 0 in every variable array
  int nsteps;
  int threads;     // persistent mode: threads used by this instance's workgroup
  double dt;
  double inv_dx;
};

struct Coeffs {
  double A[5], B[5];
  int ns;
};

// read / write access of line_segment to a line in global memory
struct GlobalLine {
  const double* Q;
  double* Qn;
  double* Qo;
  long long fs;
  int off;
  __device__ __forceinline__ void ld(int x, double (&q)[3]) const {
#pragma unroll
    for (int m = 0; m < 3; ++m) q[m] = Q[m * fs + off + x];
  }
  __device__ __forceinline__ void rk_in(int x, double (&q)[3]) const {
#pragma unroll
    for (int m = 0; m < 3; ++m) q[m] = Qo[m * fs + off + x];
  }
  __device__ __forceinline__ void put(int x, const double (&qn)[3], const double (&qo)[3]) const {
#pragma unroll
    for (int m = 0; m < 3; ++m) {
      Qn[m * fs + off + x] = qn[m];
      Qo[m * fs + off + x] = qo[m];
    }
  }
};

template <int CONV, int AVG, int MODE>
__device__ __forceinline__ void line_segment_global(double (*S)[LINE_NF], int lane, const Inst& in, int s0, int s1,
                                                    const Phys& ph, const Coeffs& rk, int s, const GlobalLine& g) {
  line_segment<CONV, AVG, MODE>(
      S, lane, in.n, s0, s1, in.dt, in.inv_dx, ph, rk.A[s], rk.B[s], s == 0,
      [&](int x, double (&q)[3]) { g.ld(x, q); }, [&](int x, double (&q)[3]) { g.rk_in(x, q); },
      [&](int x, const double (&qn)[3], const double (&qo)[3]) { g.put(x, qn, qo); });
}

// LDS of a workgroup of W waves: the waves' staged points, then (for lines
// that fit) two copies of the state of up to LINE_CELLS * W cells
__host__ __device__ constexpr size_t line_lds(int W, bool state) {
  return sizeof(double) * ((size_t)W * LINE_PTS * LINE_NF + (state ? (size_t)W * 6 * LINE_CELLS : 0));
}

// One line through nsteps iterations by one workgroup, a barrier per stage.
//
// A line of at most LINE_CELLS cells per wave stays on the chip: its state in
// two LDS copies that alternate between the stages, its RK register in the
// registers of the lanes that own the cells.  What bounds it is the latency
// of one wave's chunk; a longer line is split into one contiguous part per
// wave, read from and written to L2, and bound by the CU's FP64 issue.
template <int CONV, int AVG, int MODE>
__device__ __forceinline__ void line_run(const Inst& in, int W, double* sm, double* QA, double* QB, double* Qo,
                                         long long fs, const Phys& ph, const Coeffs& rk) {
  const int lane = threadIdx.x & 63, wv = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), T = blockDim.x;
  double (*S)[LINE_NF] = reinterpret_cast<double (*)[LINE_NF]>(sm + (size_t)wv * LINE_PTS * LINE_NF);
  // the final state: boundary points and halos filled
  auto leave = [&](auto&& value) {
    for (int i = (int)threadIdx.x - BH; i < in.n + BH; i += T) {
      const int x = max(1, min(i, in.n - 2));
      double v[3];
      value(x, v);
#pragma unroll
      for (int m = 0; m < 3; ++m) QA[m * fs + in.off + i] = v[m];
    }
  };
  if (in.n <= LINE_CELLS * W) {
    double* L = sm + (size_t)(T >> 6) * LINE_PTS * LINE_NF;
    const int ls = LINE_CELLS * (T >> 6);  // doubles per variable
    for (int i = threadIdx.x; i < in.n; i += T)
#pragma unroll
      for (int m = 0; m < 3; ++m) L[m * ls + i] = QA[m * fs + in.off + i];
    __syncthreads();
    const int s0 = min(wv * LINE_CELLS, in.n), s1 = min(s0 + LINE_CELLS, in.n);
    double ro[3] = {0.0, 0.0, 0.0};
    int cur = 0;
    for (int step = 0; step < in.nsteps; ++step)
      for (int s = 0; s < rk.ns; ++s) {
        const double* Lq = L + cur * 3 * ls;
        double* Ln = L + (1 - cur) * 3 * ls;
        if (wv < W)
          line_segment<CONV, AVG, MODE>(
              S, lane, in.n, s0, s1, in.dt, in.inv_dx, ph, rk.A[s], rk.B[s], s == 0,
              [&](int x, double (&q)[3]) {
#pragma unroll
                for (int m = 0; m < 3; ++m) q[m] = Lq[m * ls + x];
              },
              [&](int, double (&q)[3]) {
#pragma unroll
                for (int m = 0; m < 3; ++m) q[m] = ro[m];
              },
              [&](int x, const double (&qn)[3], const double (&qo)[3]) {
#pragma unroll
                for (int m = 0; m < 3; ++m) {
                  Ln[m * ls + x] = qn[m];
                  ro[m] = qo[m];
                }
              });
        __syncthreads();
        cur ^= 1;
      }
    const double* Lq = L + cur * 3 * ls;
    leave([&](int x, double (&v)[3]) {
#pragma unroll
      for (int m = 0; m < 3; ++m) v[m] = Lq[m * ls + x];
    });
    return;
  }
  const int len = (in.n + W - 1) / W;
  const int s0 = min(wv * len, in.n), s1 = wv < W ? min(s0 + len, in.n) : s0;
  double* Q = QA;
  double* Qn = QB;
  for (int step = 0; step < in.nsteps; ++step)
    for (int s = 0; s < rk.ns; ++s) {
      line_segment_global<CONV, AVG, MODE>(S, lane, in, s0, s1, ph, rk, s, GlobalLine{Q, Qn, Qo, fs, in.off});
      __syncthreads();
      double* t = Q;
      Q = Qn;
      Qn = t;
    }
  if (Q != QA) {
    leave([&](int x, double (&v)[3]) {
#pragma unroll
      for (int m = 0; m < 3; ++m) v[m] = Q[m * fs + in.off + x];
    });
  } else {
    // the ends only: the rest is in place
    const int t = threadIdx.x;
    if (t < 2 * (BH + 1)) {
      const int i = t <= BH ? t - BH : in.n - 1 + (t - BH - 1);
      const int x = t <= BH ? 1 : in.n - 2;
#pragma unroll
      for (int m = 0; m < 3; ++m) QA[m * fs + in.off + i] = QA[m * fs + in.off + x];
    }
  }
}

template <int CONV, int AVG, int MODE>
__global__ void __launch_bounds__(1024) k_batch_persistent(const Inst* __restrict__ insts,
                                                           const int* __restrict__ order, double* __restrict__ QA,
                                                           double* __restrict__ QB, double* __restrict__ Qo,
                                                           long long fs, Phys ph, Coeffs rk) {
  extern __shared__ double sm[];
  const Inst in = insts[order[blockIdx.x]];
  line_run<CONV, AVG, MODE>(in, in.threads >> 6, sm, QA, QB, Qo, fs, ph, rk);
}

// A single 1-D block: the whole run of a line that stays on one chip (one
// workgroup), or one stage of a longer one, LINE_CELLS cells per wave.
template <int CONV, int AVG, int MODE>
__global__ void __launch_bounds__(1024) k_line_run(Inst in, double* __restrict__ Q, double* __restrict__ Q2,
                                                   double* __restrict__ Qo, long long fs, Phys ph, Coeffs rk) {
  extern __shared__ double sm[];
  line_run<CONV, AVG, MODE>(in, blockDim.x >> 6, sm, Q, Q2, Qo, fs, ph, rk);
}
template <int CONV, int AVG, int MODE>
__global__ void __launch_bounds__(64) k_line_stage(Inst in, const double* __restrict__ Q, double* __restrict__ Qo,
                                                   double* __restrict__ Qn, long long fs, Phys ph, Coeffs rk, int s) {
  __shared__ double sm[LINE_PTS][LINE_NF];
  const int c0 = blockIdx.x * LINE_CELLS;
  line_segment_global<CONV, AVG, MODE>(sm, threadIdx.x, in, c0, min(c0 + LINE_CELLS, in.n), ph, rk, s,
                                       GlobalLine{Q, Qn, Qo, fs, in.off});
}

// zeroth-order extrapolation of both ends (extrapolation.py:29-58) by lanes 0, 1
__device__ __forceinline__ void extrap_ends(double* __restrict__ Q, long long fs, const Inst& in, int lane) {
  if (lane > 1) return;
  const int b = lane == 0 ? 0 : in.n - 1;
  const int from = lane == 0 ? 1 : in.n - 2;
  const int dir = lane == 0 ? -1 : 1;
  for (int m = 0; m < 3; ++m) {
    const double v = Q[m * fs + in.off + from];
    for (int h = 0; h <= BH; ++h) Q[m * fs + in.off + b + dir * h] = v;
  }
}

// Staged mode.  The step a launch belongs to is *step0 + rel: step0 is a
// device counter the chunk's last kernel advances, so one captured chunk of
// steps serves every chunk of the run.
//
// one wave per (instance, chunk of LINE_CELLS cells); finished instances skip
constexpr int SW = 4;  // waves per workgroup
template <int CONV, int AVG, int MODE>
__global__ void __launch_bounds__(64 * SW) k_batch_stage(const Inst* __restrict__ insts,
                                                         const int* __restrict__ seg_inst,
                                                         const int* __restrict__ seg_c0, int nseg,
                                                         const double* __restrict__ Q, double* __restrict__ Qo,
                                                         double* __restrict__ Qn, long long fs, Phys ph, Coeffs rk,
                                                         int s, const int* __restrict__ step0, int rel) {
  __shared__ double sm[SW][LINE_PTS][LINE_NF];
  const int lane = threadIdx.x & 63, wv = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int t = blockIdx.x * SW + wv;
  if (t >= nseg) return;  // whole waves only: no workgroup-wide barrier below
  const Inst in = insts[seg_inst[t]];
  const int step = *step0 + rel;
  if (step >= in.nsteps) return;
  const int c0 = seg_c0[t];
  line_segment_global<CONV, AVG, MODE>(sm[wv], lane, in, c0, min(c0 + LINE_CELLS, in.n), ph, rk, s,
                                       GlobalLine{Q, Qn, Qo, fs, in.off});
}

__global__ void __launch_bounds__(256) k_batch_bc(const Inst* __restrict__ insts, int ninst, double* __restrict__ Q,
                                                   long long fs, const int* __restrict__ step0, int rel) {
  const int t = blockIdx.x * blockDim.x + threadIdx.x;
  if (t >= 2 * ninst) return;
  const Inst in = insts[t >> 1];
  if (*step0 + rel > in.nsteps) return;
  extrap_ends(Q, fs, in, t & 1);
}

// inactive instances keep their state: copy Q -> Qn so the ping-pong stays consistent
__global__ void __launch_bounds__(256) k_batch_carry(const Inst* __restrict__ insts, const int* __restrict__ pt_inst,
                                                      const int* __restrict__ pt_i, int npts, const double* __restrict__ Q,
                                                      double* __restrict__ Qn, long long fs, const int* __restrict__ step0,
                                                      int rel) {
  const int t = blockIdx.x * blockDim.x + threadIdx.x;
  if (t >= npts) return;
  const Inst in = insts[pt_inst[t]];
  if (*step0 + rel < in.nsteps) return;
  const int x = in.off + pt_i[t];
  for (int m = 0; m < 3; ++m) Qn[m * fs + x] = Q[m * fs + x];
}

// the three variables of one line, back to back, to pinned host memory
__global__ void __launch_bounds__(256) k_batch_gather(const double* __restrict__ Q, long long fs, int n,
                                                      double* __restrict__ out) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
#pragma unroll
  for (int m = 0; m < 3; ++m) out[m * (long long)n + i] = Q[m * fs + i];
}

// the staged mode's step counter: set before a run, advanced after each chunk
__global__ void k_batch_step_set(int* __restrict__ step0, int value) {
  if (threadIdx.x == 0) step0[0] = value;
}
__global__ void k_batch_step_add(int* __restrict__ step0, int add) {
  if (threadIdx.x == 0) step0[0] += add;
}

int bfail(int code, const std::string& msg) { return osbl::set_error(code, msg.c_str()); }
#define BCHK(call)                                                                         \
  do {                                                                                     \
    hipError_t e_ = (call);                                                                \
    if (e_ != hipSuccess) return bfail(OSBL_E_HIP, std::string(#call) + ": " + hipGetErrorString(e_)); \
  } while (0)

}  // namespace

struct osbl_batch {
  osbl_config base{};
  int ninst = 0;
  long long fs = 0;
  Phys ph{};
  Coeffs rk{};
  int mode_rk = 0;
  std::vector<Inst> h_inst;
  std::vector<int> order;  // instances by decreasing work
  Inst* d_inst = nullptr;
  int* d_order = nullptr;
  double* QA = nullptr;
  double* QB = nullptr;
  double* Qo = nullptr;
  double* stage_buf = nullptr;
  double* host_buf = nullptr;  // pinned: the state of the longest line
  std::mutex host_mu;          // one line at a time goes through host_buf
  hipStream_t stream = nullptr;
  // staged mode
  int* d_seg_inst = nullptr;
  int* d_seg_c0 = nullptr;
  int nseg = 0;
  int* d_pt_inst = nullptr;
  int* d_pt_i = nullptr;
  int npts = 0;
  int graph_steps = 8;
  int* d_step0 = nullptr;
  // captured chunk of graph_steps steps, by the buffer it starts from (0: QA, 1: QB)
  hipGraphExec_t chunk[2] = {nullptr, nullptr};
  // per-size thread table: threads for n <= bucket_n[k]; empty: a wave per LINE_CELLS cells
  std::vector<int> bucket_n, bucket_t;
  double last_ms = 0.0;
};

namespace {

int pick_threads(const osbl_batch* b, int n) {
  for (size_t k = 0; k < b->bucket_n.size(); ++k)
    if (n <= b->bucket_n[k]) return b->bucket_t[k];
  return 64 * std::min(16, (n + LINE_CELLS - 1) / LINE_CELLS);
}

int upload_instances(osbl_batch* b) {
  for (auto& in : b->h_inst) in.threads = pick_threads(b, in.n);
  BCHK(hipMemcpy(b->d_inst, b->h_inst.data(), sizeof(Inst) * b->ninst, hipMemcpyHostToDevice));
  return OSBL_OK;
}

template <int CONV, int AVG>
int launch_persistent_t(osbl_batch* b) {
  int maxT = 64;
  bool state = false;
  for (auto& in : b->h_inst) {
    maxT = std::max(maxT, in.threads);
    state |= in.n <= LINE_CELLS * (in.threads >> 6);
  }
  const size_t lds = line_lds(maxT >> 6, state);
  auto go = [&](auto k) -> int {
    BCHK(hipFuncSetAttribute(reinterpret_cast<const void*>(k), hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds));
    k<<<b->ninst, maxT, lds, b->stream>>>(b->d_inst, b->d_order, b->QA, b->QB, b->Qo, b->fs, b->ph, b->rk);
    BCHK(hipGetLastError());
    return OSBL_OK;
  };
  return b->mode_rk == 0 ? go(&k_batch_persistent<CONV, AVG, 0>) : go(&k_batch_persistent<CONV, AVG, 1>);
}

template <int CONV, int AVG>
void launch_stage_t(osbl_batch* b, const double* Q, double* Qn, int s, int rel) {
  const unsigned blocks = (unsigned)((b->nseg + SW - 1) / SW);
  if (b->mode_rk == 0)
    k_batch_stage<CONV, AVG, 0><<<blocks, 64 * SW, 0, b->stream>>>(b->d_inst, b->d_seg_inst, b->d_seg_c0, b->nseg, Q,
                                                                   b->Qo, Qn, b->fs, b->ph, b->rk, s, b->d_step0, rel);
  else
    k_batch_stage<CONV, AVG, 1><<<blocks, 64 * SW, 0, b->stream>>>(b->d_inst, b->d_seg_inst, b->d_seg_c0, b->nseg, Q,
                                                                   b->Qo, Qn, b->fs, b->ph, b->rk, s, b->d_step0, rel);
}

template <class F>
void dispatch(int conv, int avg, F&& f) {
  auto go = [&](auto cc) {
    constexpr int C = decltype(cc)::value;
    if (avg == OSBL_AVG_ROE) f(std::integral_constant<int, C>{}, std::integral_constant<int, OSBL_AVG_ROE>{});
    else f(std::integral_constant<int, C>{}, std::integral_constant<int, OSBL_AVG_SIMPLE>{});
  };
  switch (conv) {
    case OSBL_CONV_WENO_JS: go(std::integral_constant<int, OSBL_CONV_WENO_JS>{}); break;
    case OSBL_CONV_WENO_Z: go(std::integral_constant<int, OSBL_CONV_WENO_Z>{}); break;
    case OSBL_CONV_TENO5: go(std::integral_constant<int, OSBL_CONV_TENO5>{}); break;
    default: go(std::integral_constant<int, OSBL_CONV_TENO6>{}); break;
  }
}

int run_persistent(osbl_batch* b) {
  int rc = OSBL_OK;
  dispatch(b->base.conv, b->base.averaging, [&](auto c, auto a) {
    rc = launch_persistent_t<decltype(c)::value, decltype(a)::value>(b);
  });
  return rc;
}

void drop_chunks(osbl_batch* b) {
  for (auto& g : b->chunk)
    if (g) {
      (void)hipGraphExecDestroy(g);
      g = nullptr;
    }
}

// capture one chunk of graph_steps steps starting from buffer `start`
int capture_chunk(osbl_batch* b, int start) {
  const unsigned cpb = (unsigned)((b->npts + 255) / 256);
  double* Q = start ? b->QB : b->QA;
  double* Qn = start ? b->QA : b->QB;
  hipGraph_t graph;
  BCHK(hipStreamBeginCapture(b->stream, hipStreamCaptureModeThreadLocal));
  for (int rel = 0; rel < b->graph_steps; ++rel) {
    for (int s = 0; s < b->rk.ns; ++s) {
      dispatch(b->base.conv, b->base.averaging, [&](auto c, auto a) {
        launch_stage_t<decltype(c)::value, decltype(a)::value>(b, Q, Qn, s, rel);
      });
      k_batch_carry<<<cpb, 256, 0, b->stream>>>(b->d_inst, b->d_pt_inst, b->d_pt_i, b->npts, Q, Qn, b->fs,
                                                b->d_step0, rel);
      std::swap(Q, Qn);
    }
  }
  k_batch_step_add<<<1, 64, 0, b->stream>>>(b->d_step0, b->graph_steps);
  BCHK(hipStreamEndCapture(b->stream, &graph));
  hipError_t e = hipGraphInstantiate(&b->chunk[start], graph, nullptr, nullptr, 0);
  (void)hipGraphDestroy(graph);
  if (e != hipSuccess) {
    b->chunk[start] = nullptr;
    return bfail(OSBL_E_HIP, std::string("hipGraphInstantiate: ") + hipGetErrorString(e));
  }
  return OSBL_OK;
}

int run_staged(osbl_batch* b) {
  int maxsteps = 0;
  for (auto& in : b->h_inst) maxsteps = std::max(maxsteps, in.nsteps);
  const unsigned bcb = (unsigned)((2 * b->ninst + 255) / 256);
  // every chunk replays the same graph (at most one per starting buffer);
  // steps past an instance's nsteps leave it unchanged, so the last chunk may
  // run beyond maxsteps
  const int swaps = (b->rk.ns * b->graph_steps) & 1;
  int cur = 0;
  k_batch_step_set<<<1, 64, 0, b->stream>>>(b->d_step0, 0);
  BCHK(hipGetLastError());
  for (int step0 = 0; step0 < maxsteps; step0 += b->graph_steps) {
    if (!b->chunk[cur])
      if (int rc = capture_chunk(b, cur)) return rc;
    BCHK(hipGraphLaunch(b->chunk[cur], b->stream));
    cur ^= swaps;
  }
  if (cur) BCHK(hipMemcpyAsync(b->QA, b->QB, sizeof(double) * 3 * b->fs, hipMemcpyDeviceToDevice, b->stream));
  k_batch_step_set<<<1, 64, 0, b->stream>>>(b->d_step0, 0);
  k_batch_bc<<<bcb, 256, 0, b->stream>>>(b->d_inst, b->ninst, b->QA, b->fs, b->d_step0, 0);
  BCHK(hipGetLastError());
  return OSBL_OK;
}

}  // namespace

namespace osbl {

int launch_line_run(int conv, int avg, int mode, double* Q, double* Q2, double* Qo, const Grid& g, const Phys& ph,
                    const double* A, const double* B, int ns, int nsteps, hipStream_t st) {
  const int W = (g.n[0] + LINE_CELLS - 1) / LINE_CELLS;
  const Inst in{g.n[0], g.idx(0, 0, 0), nsteps, 64 * W, ph.dt, ph.inv_delta[0]};
  Coeffs rk{};
  rk.ns = ns;
  for (int i = 0; i < ns; ++i) { rk.A[i] = A[i]; rk.B[i] = B[i]; }
  const size_t lds = line_lds(W, true);
  int rc = OSBL_OK;
  auto go = [&](auto k) -> int {
    BCHK(hipFuncSetAttribute(reinterpret_cast<const void*>(k), hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds));
    k<<<1, 64 * W, lds, st>>>(in, Q, Q2, Qo, g.fs, ph, rk);
    BCHK(hipGetLastError());
    return OSBL_OK;
  };
  dispatch(conv, avg, [&](auto c, auto a) {
    constexpr int C = decltype(c)::value, V = decltype(a)::value;
    rc = mode == 0 ? go(&k_line_run<C, V, 0>) : go(&k_line_run<C, V, 1>);
  });
  return rc;
}

void launch_line_stage(int conv, int avg, int mode, const double* Q, double* Qo, double* Qn, const Grid& g,
                       const Phys& ph, const double* A, const double* B, int ns, int s, hipStream_t st) {
  const Inst in{g.n[0], g.idx(0, 0, 0), 1, 64, ph.dt, ph.inv_delta[0]};
  Coeffs rk{};
  rk.ns = ns;
  for (int i = 0; i < ns; ++i) { rk.A[i] = A[i]; rk.B[i] = B[i]; }
  const unsigned blocks = (unsigned)((g.n[0] + LINE_CELLS - 1) / LINE_CELLS);
  dispatch(conv, avg, [&](auto c, auto a) {
    constexpr int C = decltype(c)::value, V = decltype(a)::value;
    if (mode == 0) k_line_stage<C, V, 0><<<blocks, 64, 0, st>>>(in, Q, Qo, Qn, g.fs, ph, rk, s);
    else k_line_stage<C, V, 1><<<blocks, 64, 0, st>>>(in, Q, Qo, Qn, g.fs, ph, rk, s);
  });
}

}  // namespace osbl

extern "C" {

int osbl_batch_create(const osbl_config* base, int ninst, const int32_t* n, const double* delta, const double* dt,
                      const int64_t* nsteps, osbl_batch** out) {
  if (!base || !n || !delta || !dt || !nsteps || !out || ninst <= 0) return bfail(OSBL_E_ARG, "invalid argument");
  *out = nullptr;
  if (base->ndim != 1) return bfail(OSBL_E_ARG, "ensembles are 1-D");
  if (base->conv < OSBL_CONV_WENO_JS || base->conv > OSBL_CONV_TENO6)
    return bfail(OSBL_E_ARG, "ensembles use a characteristic scheme (WENO/TENO)");
  if (base->rk < OSBL_RK3 || base->rk > OSBL_RK4_LS) return bfail(OSBL_E_ARG, "unknown RK scheme");
  for (int s = 0; s < 2; ++s)
    if (base->bc[0][s] != OSBL_BC_EXTRAP0) return bfail(OSBL_E_ARG, "ensembles use extrapolation ends");
  auto* b = new osbl_batch();
  b->base = *base;
  b->ninst = ninst;
  b->ph.gama = base->gama;
  b->ph.gm1 = base->gama - 1.0;
  b->ph.igm1 = 1.0 / b->ph.gm1;
  b->ph.eps = base->eps;
  b->ph.teno_ct = base->teno_ct;
  b->mode_rk = base->rk == OSBL_RK3 ? 0 : 1;
  {
    double A[5], B[5];
    // same coefficients as the single-block runtime
    int ns;
    switch (base->rk) {
      case OSBL_RK3: ns = 3; A[0] = 2.0 / 3.0; A[1] = 5.0 / 12.0; A[2] = 3.0 / 5.0; B[0] = 1.0 / 4.0; B[1] = 3.0 / 20.0; B[2] = 3.0 / 5.0; break;
      case OSBL_RK3_LS: ns = 3; A[0] = 0.0; A[1] = -5.0 / 9.0; A[2] = -153.0 / 128.0; B[0] = 1.0 / 3.0; B[1] = 15.0 / 16.0; B[2] = 8.0 / 15.0; break;
      default: delete b; return bfail(OSBL_E_ARG, "ensembles support RungeKutta(3) and RungeKuttaLS(3)");
    }
    for (int i = 0; i < ns; ++i) { b->rk.A[i] = A[i]; b->rk.B[i] = B[i]; }
    b->rk.ns = ns;
  }
  long long off = BH;
  b->h_inst.resize(ninst);
  for (int i = 0; i < ninst; ++i) {
    if (n[i] < 8) { delete b; return bfail(OSBL_E_ARG, "instance with fewer than 8 points"); }
    if (!(delta[i] > 0.0) || !(dt[i] > 0.0) || nsteps[i] < 0) { delete b; return bfail(OSBL_E_ARG, "bad instance parameters"); }
    Inst& in = b->h_inst[i];
    in.n = n[i];
    in.off = (int)off;
    in.nsteps = (int)nsteps[i];
    in.dt = dt[i];
    in.inv_dx = 1.0 / delta[i];
    off += n[i] + 2 * BH;
    off = (off + 7) / 8 * 8 + BH;  // 64-byte aligned interiors
  }
  b->fs = (off + 63) / 64 * 64;
  if (b->fs * 3 >= (1LL << 31)) { delete b; return bfail(OSBL_E_ARG, "ensemble too large"); }
  b->order.resize(ninst);
  for (int i = 0; i < ninst; ++i) b->order[i] = i;
  std::stable_sort(b->order.begin(), b->order.end(), [&](int a, int c) {
    return (double)b->h_inst[a].n * b->h_inst[a].nsteps > (double)b->h_inst[c].n * b->h_inst[c].nsteps;
  });
  // staged mode segment lists
  std::vector<int> si, sc, pi, pp;
  for (int i = 0; i < ninst; ++i) {
    for (int c = 0; c < n[i]; c += LINE_CELLS) { si.push_back(i); sc.push_back(c); }
    for (int p = -BH; p < n[i] + BH; ++p) { pi.push_back(i); pp.push_back(p); }
  }
  b->nseg = (int)si.size();
  b->npts = (int)pi.size();
  auto fail_free = [&](int rc) { osbl_batch_destroy(b); return rc; };
  if (hipStreamCreateWithFlags(&b->stream, hipStreamNonBlocking) != hipSuccess) return fail_free(bfail(OSBL_E_HIP, "stream"));
  const size_t bytes = sizeof(double) * 3 * b->fs;
  if (hipMalloc((void**)&b->QA, bytes) != hipSuccess || hipMalloc((void**)&b->QB, bytes) != hipSuccess ||
      hipMalloc((void**)&b->Qo, bytes) != hipSuccess || hipMalloc((void**)&b->stage_buf, bytes) != hipSuccess ||
      hipHostMalloc((void**)&b->host_buf, sizeof(double) * 3 * *std::max_element(n, n + ninst)) != hipSuccess ||
      hipMalloc((void**)&b->d_inst, sizeof(Inst) * ninst) != hipSuccess ||
      hipMalloc((void**)&b->d_order, sizeof(int) * ninst) != hipSuccess ||
      hipMalloc((void**)&b->d_seg_inst, sizeof(int) * b->nseg) != hipSuccess ||
      hipMalloc((void**)&b->d_seg_c0, sizeof(int) * b->nseg) != hipSuccess ||
      hipMalloc((void**)&b->d_pt_inst, sizeof(int) * b->npts) != hipSuccess ||
      hipMalloc((void**)&b->d_pt_i, sizeof(int) * b->npts) != hipSuccess ||
      hipMalloc((void**)&b->d_step0, sizeof(int)) != hipSuccess)
    return fail_free(bfail(OSBL_E_NOMEM, "hipMalloc failed"));
  if (hipMemset(b->QA, 0, bytes) != hipSuccess || hipMemset(b->QB, 0, bytes) != hipSuccess ||
      hipMemset(b->Qo, 0, bytes) != hipSuccess ||
      hipMemcpy(b->d_order, b->order.data(), sizeof(int) * ninst, hipMemcpyHostToDevice) != hipSuccess ||
      hipMemcpy(b->d_seg_inst, si.data(), sizeof(int) * b->nseg, hipMemcpyHostToDevice) != hipSuccess ||
      hipMemcpy(b->d_seg_c0, sc.data(), sizeof(int) * b->nseg, hipMemcpyHostToDevice) != hipSuccess ||
      hipMemcpy(b->d_pt_inst, pi.data(), sizeof(int) * b->npts, hipMemcpyHostToDevice) != hipSuccess ||
      hipMemcpy(b->d_pt_i, pp.data(), sizeof(int) * b->npts, hipMemcpyHostToDevice) != hipSuccess)
    return fail_free(bfail(OSBL_E_HIP, "initialisation copy failed"));
  int rc = upload_instances(b);
  if (rc) return fail_free(rc);
  *out = b;
  return OSBL_OK;
}

void osbl_batch_destroy(osbl_batch* b) {
  if (!b) return;
  if (b->stream) (void)hipStreamSynchronize(b->stream);
  drop_chunks(b);
  for (void* p : {(void*)b->QA, (void*)b->QB, (void*)b->Qo, (void*)b->stage_buf, (void*)b->d_inst, (void*)b->d_order,
                  (void*)b->d_seg_inst, (void*)b->d_seg_c0, (void*)b->d_pt_inst, (void*)b->d_pt_i,
                  (void*)b->d_step0})
    if (p) (void)hipFree(p);
  if (b->host_buf) (void)hipHostFree(b->host_buf);
  if (b->stream) (void)hipStreamDestroy(b->stream);
  delete b;
}

int osbl_batch_set_state(osbl_batch* b, int inst, const double* host) {
  if (!b || !host || inst < 0 || inst >= b->ninst) return bfail(OSBL_E_ARG, "invalid argument");
  const Inst& in = b->h_inst[inst];
  for (int m = 0; m < 3; ++m)
    BCHK(hipMemcpy(b->QA + m * b->fs + in.off, host + (size_t)m * in.n, sizeof(double) * in.n, hipMemcpyHostToDevice));
  return OSBL_OK;
}

int osbl_batch_get_state(osbl_batch* b, int inst, double* host) {
  if (!b || !host || inst < 0 || inst >= b->ninst) return bfail(OSBL_E_ARG, "invalid argument");
  const Inst& in = b->h_inst[inst];
  // one kernel that writes to pinned memory and one wait: 512 instances one
  // by one took 21 ms with a blocking copy per variable
  std::lock_guard<std::mutex> lock(b->host_mu);
  k_batch_gather<<<(in.n + 255) / 256, 256, 0, b->stream>>>(b->QA + in.off, b->fs, in.n, b->host_buf);
  BCHK(hipGetLastError());
  BCHK(hipStreamSynchronize(b->stream));
  std::memcpy(host, b->host_buf, sizeof(double) * 3 * in.n);
  return OSBL_OK;
}

int osbl_batch_save(osbl_batch* b) {
  if (!b) return bfail(OSBL_E_ARG, "null");
  BCHK(hipMemcpyAsync(b->stage_buf, b->QA, sizeof(double) * 3 * b->fs, hipMemcpyDeviceToDevice, b->stream));
  return OSBL_OK;
}

int osbl_batch_restore(osbl_batch* b) {
  if (!b) return bfail(OSBL_E_ARG, "null");
  BCHK(hipMemcpyAsync(b->QA, b->stage_buf, sizeof(double) * 3 * b->fs, hipMemcpyDeviceToDevice, b->stream));
  return OSBL_OK;
}

int osbl_batch_run(osbl_batch* b, int mode, double* elapsed_ms) {
  if (!b) return bfail(OSBL_E_ARG, "null");
  hipEvent_t e0, e1;
  BCHK(hipEventCreate(&e0));
  BCHK(hipEventCreate(&e1));
  BCHK(hipEventRecord(e0, b->stream));
  int rc = mode == 0 ? run_persistent(b) : run_staged(b);
  if (rc) return rc;
  BCHK(hipEventRecord(e1, b->stream));
  BCHK(hipEventSynchronize(e1));
  float ms = 0.f;
  BCHK(hipEventElapsedTime(&ms, e0, e1));
  (void)hipEventDestroy(e0);
  (void)hipEventDestroy(e1);
  b->last_ms = ms;
  if (elapsed_ms) *elapsed_ms = ms;
  return OSBL_OK;
}

int osbl_batch_set_threads(osbl_batch* b, int nbuckets, const int32_t* max_n, const int32_t* threads) {
  if (!b || nbuckets <= 0 || !max_n || !threads) return bfail(OSBL_E_ARG, "invalid argument");
  for (int k = 0; k < nbuckets; ++k)
    if (threads[k] < 64 || threads[k] > 1024 || threads[k] % 64)
      return bfail(OSBL_E_ARG, "threads must be 64..1024, multiple of 64");
  b->bucket_n.assign(max_n, max_n + nbuckets);
  b->bucket_t.assign(threads, threads + nbuckets);
  b->bucket_n.back() = 1 << 30;
  return upload_instances(b);
}

int osbl_batch_set_graph_steps(osbl_batch* b, int steps) {
  if (!b || steps < 1) return bfail(OSBL_E_ARG, "invalid argument");
  if (steps != b->graph_steps) {
    BCHK(hipStreamSynchronize(b->stream));
    drop_chunks(b);
  }
  b->graph_steps = steps;
  return OSBL_OK;
}

}  // extern "C"
