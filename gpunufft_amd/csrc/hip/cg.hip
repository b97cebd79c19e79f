// Device-resident CG-SENSE solver on one plan (gnufft_cg_*).
//
// Solves (A^H A + alpha I) x = A^H y with the plain conjugate-gradient loop
// of the reference's demo reconstruction (matlab/demo/utils/cg_sense_2d.m:
// right-hand side :46-47 with useMulticoil, system matrix :51 and :99-102,
// iterations :63-82), where A is the plan's forward operator including
// coil sensitivities and density compensation. Vectors and scalars live in
// device memory; the scalar reductions are two-stage in double precision in
// a fixed order (deterministic); no iteration needs the host. One iteration
// (forward, adjoint, CG updates) is captured into a HIP graph after a warm-up
// and replayed.

#include <hip/hip_runtime.h>

#include <new>
#include <string>

#include "../../../include/gpunufft_hip.h"
#include "gnufft_internal.hpp"

namespace {

constexpr int kCgThreads = 256;
constexpr int kCgBlocks = 512;  // partial sums per reduction

int cg_fail(int code, const std::string& msg) {
  gnufft::set_last_error(msg);
  return code;
}

#define CG_HIP(expr)                                                                        \
  do {                                                                                      \
    hipError_t e_ = (expr);                                                                 \
    if (e_ != hipSuccess)                                                                   \
      return cg_fail(GNUFFT_ERR_DEVICE, std::string(#expr) + ": " + hipGetErrorString(e_)); \
  } while (0)

#define CG_ABI(expr)                  \
  do {                                \
    int rc_ = (expr);                 \
    if (rc_ != GNUFFT_OK) return rc_; \
  } while (0)

__device__ inline double block_sum(double v) {
  __shared__ double red[kCgThreads / 64];
  for (int o = 32; o >= 1; o >>= 1) v += __shfl_xor(v, o);
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  if (lane == 0) red[wave] = v;
  __syncthreads();
  double t = 0.0;
  if (threadIdx.x == 0)
    for (int w = 0; w < kCgThreads / 64; w++) t += red[w];
  return t;  // valid in thread 0
}

// Sum of part[0 .. kCgBlocks) in a fixed order, in every thread. Each block of
// a kernel that needs a sum forms it by itself (4 KB from the L2) instead of
// waiting for a kernel of one block: 4.4 us and a launch less, twice an
// iteration (240^2, 12 coils: 1354 -> 1295 us for ten iterations).
__device__ inline double partial_sum(const double* __restrict__ part) {
  __shared__ double total;
  double acc = 0.0;
  for (int i = threadIdx.x; i < kCgBlocks; i += kCgThreads) acc += part[i];
  acc = block_sum(acc);
  if (threadIdx.x == 0) total = acc;
  __syncthreads();
  acc = total;
  __syncthreads();  // (before the shared words are used again)
  return acc;
}

// Ap += alpha p; part[block] = sum Re(conj(p) Ap); the last iteration's rr_new
// becomes rr (its partial sums: nothing else touches them here)
__global__ void __launch_bounds__(kCgThreads) cg_pap_kernel(const float2* __restrict__ p,
                                                            float2* __restrict__ Ap, float alpha,
                                                            size_t n, double* __restrict__ part,
                                                            double* __restrict__ rr,
                                                            const double* __restrict__ rr_new) {
  if (threadIdx.x == 0) rr[blockIdx.x] = rr_new[blockIdx.x];
  double acc = 0.0;
  for (size_t i = (size_t)blockIdx.x * kCgThreads + threadIdx.x; i < n;
       i += (size_t)gridDim.x * kCgThreads) {
    const float2 a = p[i];
    float2 b = Ap[i];
    b.x += alpha * a.x;
    b.y += alpha * a.y;
    Ap[i] = b;
    acc += (double)a.x * b.x + (double)a.y * b.y;
  }
  acc = block_sum(acc);
  if (threadIdx.x == 0) part[blockIdx.x] = acc;
}

// a = rr / pAp; x += a p; r -= a Ap; part[block] = sum |r|^2 (rr, pap: partial sums)
__global__ void __launch_bounds__(kCgThreads) cg_step_kernel(float2* __restrict__ x,
                                                             float2* __restrict__ r,
                                                             const float2* __restrict__ p,
                                                             const float2* __restrict__ Ap,
                                                             const double* __restrict__ rr,
                                                             const double* __restrict__ pap, size_t n,
                                                             double* __restrict__ part) {
  const double rr_sum = partial_sum(rr), pap_sum = partial_sum(pap);
  const float a = pap_sum != 0.0 ? (float)(rr_sum / pap_sum) : 0.0f;
  double acc = 0.0;
  for (size_t i = (size_t)blockIdx.x * kCgThreads + threadIdx.x; i < n;
       i += (size_t)gridDim.x * kCgThreads) {
    const float2 pi = p[i], api = Ap[i];
    float2 xi = x[i], ri = r[i];
    xi.x += a * pi.x;
    xi.y += a * pi.y;
    ri.x -= a * api.x;
    ri.y -= a * api.y;
    x[i] = xi;
    r[i] = ri;
    acc += (double)ri.x * ri.x + (double)ri.y * ri.y;
  }
  acc = block_sum(acc);
  if (threadIdx.x == 0) part[blockIdx.x] = acc;
}

// p = r + (rr_new / rr) p (partial sums)
__global__ void __launch_bounds__(kCgThreads) cg_dir_kernel(float2* __restrict__ p,
                                                            const float2* __restrict__ r,
                                                            const double* __restrict__ rr,
                                                            const double* __restrict__ rr_new,
                                                            size_t n) {
  const double rr_sum = partial_sum(rr), new_sum = partial_sum(rr_new);
  const float b = rr_sum != 0.0 ? (float)(new_sum / rr_sum) : 0.0f;
  for (size_t i = (size_t)blockIdx.x * kCgThreads + threadIdx.x; i < n;
       i += (size_t)gridDim.x * kCgThreads) {
    const float2 ri = r[i];
    float2 pi = p[i];
    pi.x = ri.x + b * pi.x;
    pi.y = ri.y + b * pi.y;
    p[i] = pi;
  }
}

// x = 0; r = p = y; part[block] = sum |y|^2
__global__ void __launch_bounds__(kCgThreads) cg_init_kernel(float2* __restrict__ x,
                                                             float2* __restrict__ r,
                                                             float2* __restrict__ p,
                                                             const float2* __restrict__ y, size_t n,
                                                             double* __restrict__ part) {
  double acc = 0.0;
  for (size_t i = (size_t)blockIdx.x * kCgThreads + threadIdx.x; i < n;
       i += (size_t)gridDim.x * kCgThreads) {
    const float2 v = y[i];
    x[i] = make_float2(0.0f, 0.0f);
    r[i] = v;
    p[i] = v;
    acc += (double)v.x * v.x + (double)v.y * v.y;
  }
  acc = block_sum(acc);
  if (threadIdx.x == 0) part[blockIdx.x] = acc;
}

}  // namespace

struct gnufft_cg_s {
  gnufft_plan plan = nullptr;
  uint32_t coils = 0;
  uint32_t samples = 0;
  float alpha = 0.0f;
  size_t n = 0;       // image elements (coil-combined)
  float2* buf = nullptr;  // x, r, p, Ap, y (n each) then k ([coils][M])
  float2 *x = nullptr, *r = nullptr, *p = nullptr, *Ap = nullptr, *y = nullptr, *k = nullptr;
  double* s = nullptr;  // partial sums, kCgBlocks of each: |r|^2 before the step, Re(p^H Ap), |r|^2 after it
  double *rr = nullptr, *pap = nullptr, *rr_new = nullptr;
  hipGraph_t graph = nullptr;
  hipGraphExec_t exec = nullptr;
  uint64_t generation = 0;  // the plan's buffer generation the graph was captured at
  bool warm = false;
  // the solver's own stream (default priority, non-blocking: the legacy
  // null stream cannot be captured), ordered after / before the caller's
  // stream with events
  hipStream_t own = nullptr;
  hipEvent_t ev_in = nullptr, ev_out = nullptr;
};

namespace {

// A^H k. On odd grids the adjoint's rounding decides what CG returns, and the
// sums that do not depend on the samples' order are taken (sector_spread.hip).
int cg_adjoint(gnufft_cg c, const void* k, float2* out, hipStream_t s) {
  return gnufft::plan_adjoint(c->plan, k, out, c->coils, GNUFFT_STOP_DEAPODIZATION, gnufft::plan_odd_grid(c->plan), s);
}

// One CG iteration (the body of the captured graph).
int cg_iteration(gnufft_cg c, hipStream_t s) {
  CG_ABI(gnufft_forward(c->plan, c->p, c->k, c->coils, GNUFFT_STOP_DEAPODIZATION, s));
  CG_ABI(cg_adjoint(c, c->k, c->Ap, s));
  hipLaunchKernelGGL(cg_pap_kernel, dim3(kCgBlocks), dim3(kCgThreads), 0, s, c->p, c->Ap, c->alpha, c->n, c->pap,
                     c->rr, c->rr_new);
  hipLaunchKernelGGL(cg_step_kernel, dim3(kCgBlocks), dim3(kCgThreads), 0, s, c->x, c->r, c->p, c->Ap, c->rr,
                     c->pap, c->n, c->rr_new);
  hipLaunchKernelGGL(cg_dir_kernel, dim3(kCgBlocks), dim3(kCgThreads), 0, s, c->p, c->r, c->rr, c->rr_new, c->n);
  CG_HIP(hipGetLastError());
  return GNUFFT_OK;
}

void cg_free(gnufft_cg c) {
  if (c->exec) (void)hipGraphExecDestroy(c->exec);
  if (c->graph) (void)hipGraphDestroy(c->graph);
  if (c->buf) (void)hipFree(c->buf);
  if (c->s) (void)hipFree(c->s);
  if (c->ev_in) (void)hipEventDestroy(c->ev_in);
  if (c->ev_out) (void)hipEventDestroy(c->ev_out);
  if (c->own) (void)hipStreamDestroy(c->own);
  delete c;
}

}  // namespace

extern "C" {

int gnufft_cg_create(gnufft_cg* cg, gnufft_plan plan, uint32_t n_coils, float alpha) {
  if (!cg || !plan || n_coils == 0) return cg_fail(GNUFFT_ERR_INVALID_ARGUMENT, "cg_create: bad argument");
  *cg = nullptr;
  gnufft_plan_info info;
  CG_ABI(gnufft_plan_get_info(plan, &info));
  if (info.n_samples == 0) return cg_fail(GNUFFT_ERR_STATE, "cg_create: plan has no trajectory");
  if (info.n_sens_coils != n_coils)
    return cg_fail(GNUFFT_ERR_INVALID_ARGUMENT, "cg_create: plan needs sensitivities of n_coils coils");
  gnufft_cg c = new (std::nothrow) gnufft_cg_s();
  if (!c) return cg_fail(GNUFFT_ERR_OUT_OF_MEMORY, "cg_create: host allocation");
  c->plan = plan;
  c->coils = n_coils;
  c->samples = info.n_samples;
  c->alpha = alpha;
  c->n = (size_t)info.img_count;
  const size_t total = 5 * c->n + (size_t)n_coils * info.n_samples;
  if (hipMalloc(&c->buf, total * sizeof(float2)) != hipSuccess ||
      hipMalloc(&c->s, 3 * kCgBlocks * sizeof(double)) != hipSuccess) {
    cg_free(c);
    return cg_fail(GNUFFT_ERR_OUT_OF_MEMORY, "cg_create: device allocation");
  }
  if (hipStreamCreateWithFlags(&c->own, hipStreamNonBlocking) != hipSuccess ||
      hipEventCreateWithFlags(&c->ev_in, hipEventDisableTiming) != hipSuccess ||
      hipEventCreateWithFlags(&c->ev_out, hipEventDisableTiming) != hipSuccess) {
    cg_free(c);
    return cg_fail(GNUFFT_ERR_DEVICE, "cg_create: stream / event creation");
  }
  c->x = c->buf;
  c->r = c->x + c->n;
  c->p = c->r + c->n;
  c->Ap = c->p + c->n;
  c->y = c->Ap + c->n;
  c->k = c->y + c->n;
  c->rr = c->s;
  c->pap = c->rr + kCgBlocks;
  c->rr_new = c->pap + kCgBlocks;
  *cg = c;
  return GNUFFT_OK;
}

int gnufft_cg_destroy(gnufft_cg cg) {
  if (!cg) return GNUFFT_OK;
  (void)hipDeviceSynchronize();
  cg_free(cg);
  return GNUFFT_OK;
}

int gnufft_cg_solve(gnufft_cg c, const void* kdata, void* x_out, uint32_t iterations, int use_graph,
                    void* stream) {
  if (!c || !kdata || !x_out) return cg_fail(GNUFFT_ERR_INVALID_ARGUMENT, "cg_solve: null argument");
  {
    // the solver's vectors are sized for the plan's sample and coil counts
    gnufft_plan_info info;
    CG_ABI(gnufft_plan_get_info(c->plan, &info));
    if (info.n_samples != c->samples || info.n_sens_coils != c->coils)
      return cg_fail(GNUFFT_ERR_STATE,
                     "cg_solve: the plan's trajectory length or sensitivity coils changed since "
                     "cg_create; create a new solver");
  }
  // the work runs on the solver's stream, after the caller's stream's
  // earlier work and before its later work
  const hipStream_t caller = (hipStream_t)stream;
  const hipStream_t s = c->own;
  CG_HIP(hipEventRecord(c->ev_in, caller));
  CG_HIP(hipStreamWaitEvent(s, c->ev_in, 0));
  // right-hand side A^H y, then x = 0, r = p = A^H y, rr = |r|^2
  CG_ABI(cg_adjoint(c, kdata, c->y, s));
  hipLaunchKernelGGL(cg_init_kernel, dim3(kCgBlocks), dim3(kCgThreads), 0, s, c->x, c->r, c->p,
                     c->y, c->n, c->rr_new);
  CG_HIP(hipGetLastError());
  // The captured iteration holds the plan's device pointers (tables, work
  // grid, scratch, sensitivities). When any of them was freed or replaced
  // since the capture (set_trajectory, set_sens, a larger coil batch,
  // set_fft), the graph is dropped and captured again.
  if (use_graph && c->exec && c->generation != gnufft::plan_generation(c->plan)) {
    CG_HIP(hipStreamSynchronize(s));  // earlier replays may still run
    (void)hipGraphExecDestroy(c->exec);
    (void)hipGraphDestroy(c->graph);
    c->exec = nullptr;
    c->graph = nullptr;
    c->warm = false;
  }
  if (use_graph && !c->exec) {
    if (!c->warm) {
      // allocate the plan's work buffers and FFT plans outside the capture
      CG_ABI(gnufft_forward(c->plan, c->p, c->k, c->coils, GNUFFT_STOP_DEAPODIZATION, s));
      c->warm = true;
    }
    const uint64_t gen = gnufft::plan_generation(c->plan);
    CG_HIP(hipStreamBeginCapture(s, hipStreamCaptureModeThreadLocal));
    int rc = cg_iteration(c, s);
    hipGraph_t g = nullptr;
    hipError_t e = hipStreamEndCapture(s, &g);
    if (rc) {
      if (g) (void)hipGraphDestroy(g);
      return rc;
    }
    CG_HIP(e);
    if (gen != gnufft::plan_generation(c->plan)) {
      // a buffer was replaced while capturing: the graph may hold a freed pointer
      (void)hipGraphDestroy(g);
      return cg_fail(GNUFFT_ERR_STATE, "cg_solve: plan buffers changed during graph capture");
    }
    c->graph = g;
    CG_HIP(hipGraphInstantiate(&c->exec, c->graph, nullptr, nullptr, 0));
    c->generation = gen;
  }
  for (uint32_t it = 0; it < iterations; it++) {
    if (use_graph) {
      CG_HIP(hipGraphLaunch(c->exec, s));
    } else {
      CG_ABI(cg_iteration(c, s));
    }
  }
  CG_HIP(hipMemcpyAsync(x_out, c->x, c->n * sizeof(float2), hipMemcpyDeviceToDevice, s));
  CG_HIP(hipEventRecord(c->ev_out, s));
  CG_HIP(hipStreamWaitEvent(caller, c->ev_out, 0));
  return GNUFFT_OK;
}

}  // extern "C"
