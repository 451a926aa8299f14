// hmvm_krylov.hip -- BiCGSTAB on the device with the HIP HMVM as its operator.
//
// Restates the iteration of the reference's HACApK_bicgstab_lfmtx_hyp
// (src_hdump/m_HACApK_solve.f90:306-380): two HMVMs per iteration, vector
// updates and dot products between them.  Every scalar (alpha, zeta, beta,
// the residual norm, the stop state and the iteration count) stays in device
// memory, so one iteration is a fixed sequence of launches with no host
// synchronisation; with use_graph the iteration is captured once into a
// hipGraph and replayed.  A dot product is per-block partials, summed in one
// fixed tree by every block of the kernel that needs it, and therefore
// deterministic: the eager and the graph-replayed solve give the same bits.
//
// Stopping: the reference leaves its loop at the top of the first iteration
// whose ||r||/||b|| is below eps (m_HACApK_solve.f90:342).  Here the kernel
// that finds ||r|| sets a device stop word instead, and every later update
// kernel and scalar update returns at once, so the host may launch whole
// chunks of iterations between its read-backs and still get the reference's
// iterate and iteration count.  A zero divisor or a non-finite scalar sets
// the stop word to "breakdown" the same way.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <cstdio>
#include <cstring>
#include <mutex>

#include "hmvm_hip.h"
#include "hmvm_stage.hpp"
#include "hmvm_status.hpp"

namespace {

int hip_fail(const char *what, hipError_t e) {
  char m[512];
  std::snprintf(m, sizeof m, "%s failed: %s", what, hipGetErrorString(e));
  return hmvm::report_error(HMVM_ERR_HIP, m);
}

#define KRY_TRY(expr)                         \
  do {                                        \
    const hipError_t e_ = (expr);             \
    if (e_ != hipSuccess) return hip_fail(#expr, e_); \
  } while (0)

constexpr int kBlock = 256;
constexpr int kDotBlocks = 512;
constexpr size_t kScalarDoubles = 4 * kDotBlocks + 16;  // two arrays of partials, the scalars

// Device scalars.  A kernel's block 0 writes what later kernels need, in
// words of that kernel alone: every block of a kernel reads the words of the
// kernels before it and computes the same values from them, so no block waits
// for another.
enum {
  kBnorm = 0, kRho, kRnorm, kStopP, kItersP,  // bicg_p (kBnorm: the first one)
  kAlpha, kRhoOld, kStopT,                    // bicg_t
  kZeta, kStopU, kItersU,                     // bicg_update
  kNumScalars
};
// what bicg_state writes for the host
enum { kOutStop = 0, kOutIters, kOutRnorm, kOutBnorm, kNumOut };
static_assert(4 * kDotBlocks + kNumScalars + kNumOut <= kScalarDoubles && 2 + kNumOut <= hmvm::kStageTail,
              "work space of the scalars");
// stop words: 0 running, 1 converged, 2 breakdown; iterations counted once
// they have updated u

// Sums of (v0, v1) over the block's threads in a fixed tree, on every thread.
__device__ __forceinline__ double2 block_sum(double v0, double v1) {
  __shared__ double s0[kBlock], s1[kBlock];
  s0[threadIdx.x] = v0;
  s1[threadIdx.x] = v1;
  __syncthreads();
  for (int s = kBlock / 2; s > 0; s >>= 1) {
    if ((int)threadIdx.x < s) {
      s0[threadIdx.x] += s0[threadIdx.x + s];
      s1[threadIdx.x] += s1[threadIdx.x + s];
    }
    __syncthreads();
  }
  const double2 r = make_double2(s0[0], s1[0]);
  __syncthreads();  // the arrays may be used again
  return r;
}

__device__ __forceinline__ void put_partial(double *__restrict__ part, double2 d) {
  if (threadIdx.x == 0) {
    part[2 * blockIdx.x] = d.x;
    part[2 * blockIdx.x + 1] = d.y;
  }
}

// The dot products whose partials a kernel of as many blocks left, by every
// block that uses them: at most kDotBlocks pairs from the cache, against a
// launch of one block between producer and consumer (4.6 us each, four an
// iteration; N=20,000).
__device__ __forceinline__ double2 sum_partials(const double *__restrict__ part) {
  double x0 = 0, x1 = 0;
  for (int i = threadIdx.x; i < (int)gridDim.x; i += kBlock) {
    x0 += part[2 * i];
    x1 += part[2 * i + 1];
  }
  return block_sum(x0, x1);
}

// partial[block] = (sum a*b, sum a*c) over a grid-stride slice
__global__ __launch_bounds__(kBlock) void dot2_partial(int n, const double *__restrict__ a,
                                                       const double *__restrict__ b,
                                                       const double *__restrict__ c, double *__restrict__ part) {
  double x0 = 0, x1 = 0;
  for (int i = blockIdx.x * kBlock + threadIdx.x; i < n; i += gridDim.x * kBlock) {
    x0 += a[i] * b[i];
    x1 += a[i] * c[i];
  }
  put_partial(part, block_sum(x0, x1));
}

__device__ __forceinline__ bool below_tol(double rnorm, double bnorm, double tol) {
  return rnorm / (bnorm > 0.0 ? bnorm : 1.0) < tol;
}

// S = 0 (a kernel rather than a memset, so that no memset node enters a
// captured graph)
__global__ void bicg_scalars_zero(double *__restrict__ S) {
  if (threadIdx.x < kNumScalars) S[threadIdx.x] = 0.0;
}

// r = b - r (r holds A u on entry), shadow = r; partials (b,b), (r,r)
__global__ __launch_bounds__(kBlock) void bicg_init(int n, const double *__restrict__ b, double *__restrict__ r,
                                                    double *__restrict__ sh, double *__restrict__ part) {
  double x0 = 0, x1 = 0;
  for (int i = blockIdx.x * kBlock + threadIdx.x; i < n; i += gridDim.x * kBlock) {
    const double v = b[i] - r[i];
    r[i] = v;
    sh[i] = v;
    x0 += b[i] * b[i];
    x1 += v * v;
  }
  put_partial(part, block_sum(x0, x1));
}

// The state between two iterations, d = (b,b), (r,r) after the start or
// (s,r), (r,r) after an update: residual norm, stop word, rho = (s,r), beta.
struct Between {
  double bnorm, rho, rnorm, beta, stop;
};
__device__ __forceinline__ Between between(double2 d, double tol, const double *__restrict__ S) {
  Between w;
  const bool first = S[kItersU] == 0.0;
  w.bnorm = first ? sqrt(d.x) : S[kBnorm];
  w.rho = first ? d.y : d.x;  // the shadow is the first r
  w.rnorm = sqrt(d.y);
  w.beta = first ? 0.0 : S[kAlpha] / S[kZeta] * w.rho / S[kRhoOld];
  w.stop = below_tol(w.rnorm, w.bnorm, tol) ? 1.0  // the reference leaves the loop before beta is used
           : !first && (!isfinite(w.rnorm) || !isfinite(w.beta)) ? 2.0
                                                                 : 0.0;
  return w;
}

// p = r + beta*(p - zeta*Ap); p = r in the first iteration
__global__ __launch_bounds__(kBlock) void bicg_p(int n, const double *__restrict__ r, double *__restrict__ p,
                                                 const double *__restrict__ ap, const double *__restrict__ part,
                                                 double tol, double *__restrict__ S) {
  const bool first = S[kItersU] == 0.0, stopped = S[kStopU] != 0.0;  // uniform over the grid
  Between w{};
  if (!stopped) w = between(sum_partials(part), tol, S);
  if (blockIdx.x == 0 && threadIdx.x == 0) {
    S[kStopP] = stopped ? S[kStopU] : w.stop;
    S[kItersP] = S[kItersU];
    if (!stopped) {
      S[kRho] = w.rho;
      S[kRnorm] = w.rnorm;
      if (first) S[kBnorm] = w.bnorm;
    }
  }
  if (stopped || w.stop != 0.0) return;
  const double ze = S[kZeta];
  for (int i = blockIdx.x * kBlock + threadIdx.x; i < n; i += gridDim.x * kBlock)
    p[i] = first ? r[i] : r[i] + w.beta * (p[i] - ze * ap[i]);
}

// The state for the host, as the next bicg_p would find it.
__global__ __launch_bounds__(kBlock) void bicg_state(int nblk, const double *__restrict__ part, double tol,
                                                     const double *__restrict__ S, double *__restrict__ out) {
  double x0 = 0, x1 = 0;
  for (int i = threadIdx.x; i < nblk; i += kBlock) {  // sum_partials of the larger grid
    x0 += part[2 * i];
    x1 += part[2 * i + 1];
  }
  const double2 d = block_sum(x0, x1);
  if (threadIdx.x != 0) return;
  const bool stopped = S[kStopU] != 0.0;
  const Between w = between(d, tol, S);
  out[kOutStop] = stopped ? S[kStopU] : w.stop;
  out[kOutIters] = S[kItersU];
  out[kOutRnorm] = stopped ? S[kRnorm] : w.rnorm;
  out[kOutBnorm] = stopped ? S[kBnorm] : w.bnorm;
}

// alpha = rho/(s,Ap); t = r - alpha*Ap
__global__ __launch_bounds__(kBlock) void bicg_t(int n, const double *__restrict__ r, const double *__restrict__ ap,
                                                 double *__restrict__ t, const double *__restrict__ part,
                                                 double *__restrict__ S) {
  const bool stopped = S[kStopP] != 0.0;
  const double rho = S[kRho], al = rho / sum_partials(part).x;
  const double stop = stopped ? S[kStopP] : isfinite(al) ? 0.0 : 2.0;
  if (blockIdx.x == 0 && threadIdx.x == 0) {
    S[kStopT] = stop;
    if (!stopped) {
      S[kAlpha] = al;
      S[kRhoOld] = rho;
    }
  }
  if (stop != 0.0) return;
  for (int i = blockIdx.x * kBlock + threadIdx.x; i < n; i += gridDim.x * kBlock) t[i] = r[i] - al * ap[i];
}

// zeta = (At,t)/(At,At); u += alpha*p + zeta*t ; r = t - zeta*At; partials
// (s,r), (r,r)
__global__ __launch_bounds__(kBlock) void bicg_update(int n, double *__restrict__ u, const double *__restrict__ p,
                                                      const double *__restrict__ t, const double *__restrict__ at,
                                                      double *__restrict__ r, const double *__restrict__ sh,
                                                      const double *__restrict__ part, double *__restrict__ part_r,
                                                      double *__restrict__ S) {
  const bool stopped = S[kStopT] != 0.0;
  const double2 d = sum_partials(part);
  const double ze = d.x / d.y;
  const double stop = stopped ? S[kStopT] : isfinite(ze) ? 0.0 : 2.0;
  if (blockIdx.x == 0 && threadIdx.x == 0) {
    S[kStopU] = stop;
    S[kItersU] = S[kItersP] + (stop == 0.0 ? 1.0 : 0.0);
    if (!stopped) S[kZeta] = ze;
  }
  if (stop != 0.0) return;  // uniform over the grid
  const double al = S[kAlpha];
  double x0 = 0, x1 = 0;
  for (int i = blockIdx.x * kBlock + threadIdx.x; i < n; i += gridDim.x * kBlock) {
    u[i] = u[i] + al * p[i] + ze * t[i];
    const double v = t[i] - ze * at[i];
    r[i] = v;
    x0 += sh[i] * v;
    x1 += v * v;
  }
  put_partial(part_r, block_sum(x0, x1));
}

// Device vectors and scalars of one solve: b and u are the caller's (or
// copies of the caller's host vectors), the rest is work space.
struct Solver {
  int n = 0;
  double tol = 0;
  hmvm_plan *plan = nullptr;
  hipStream_t st = nullptr;
  const double *b = nullptr;
  double *u = nullptr, *r = nullptr, *sh = nullptr, *p = nullptr, *ap = nullptr, *t = nullptr, *at = nullptr,
         *part = nullptr, *part_r = nullptr, *S = nullptr;
  double *host_out = nullptr;  // pinned: where bicg_state writes (else behind S, and copied)
  // one grid for all kernels: a kernel sums as many partials as it has blocks
  dim3 grid() const { return dim3(std::min(kDotBlocks, (n + kBlock - 1) / kBlock)); }

  // Divides work space (6 n vectors, 2 arrays of partials, the scalars).
  void place(double *w) {
    const size_t m = (size_t)n;
    r = w;
    sh = w + m;
    p = w + 2 * m;
    ap = w + 3 * m;
    t = w + 4 * m;
    at = w + 5 * m;
    part = w + 6 * m;
    part_r = part + 2 * kDotBlocks;
    S = part_r + 2 * kDotBlocks;
  }
  // r = b - A u ; shadow = r ; norms (m_HACApK_solve.f90:326-339)
  int start() {
    hipLaunchKernelGGL(bicg_scalars_zero, dim3(1), dim3(64), 0, st, S);
    int rc = hmvm_plan_apply(plan, u, r, 0, st);
    if (rc) return rc;
    hipLaunchKernelGGL(bicg_init, grid(), dim3(kBlock), 0, st, n, b, r, sh, part_r);
    KRY_TRY(hipGetLastError());
    return HMVM_OK;
  }
  // one BiCGSTAB iteration (m_HACApK_solve.f90:341-372)
  int iterate() {
    hipLaunchKernelGGL(bicg_p, grid(), dim3(kBlock), 0, st, n, r, p, ap, part_r, tol, S);
    int rc = hmvm_plan_apply(plan, p, ap, 0, st);
    if (rc) return rc;
    hipLaunchKernelGGL(dot2_partial, grid(), dim3(kBlock), 0, st, n, sh, ap, ap, part);
    hipLaunchKernelGGL(bicg_t, grid(), dim3(kBlock), 0, st, n, r, ap, t, part, S);
    rc = hmvm_plan_apply(plan, t, at, 0, st);
    if (rc) return rc;
    hipLaunchKernelGGL(dot2_partial, grid(), dim3(kBlock), 0, st, n, at, t, at, part);
    hipLaunchKernelGGL(bicg_update, grid(), dim3(kBlock), 0, st, n, u, p, t, at, r, sh, part, part_r, S);
    KRY_TRY(hipGetLastError());
    return HMVM_OK;
  }
  int read_state(double *state) {
    double *out = host_out ? host_out : S + kNumScalars;
    hipLaunchKernelGGL(bicg_state, dim3(1), dim3(kBlock), 0, st, (int)grid().x, part_r, tol, S, out);
    KRY_TRY(hipGetLastError());
    if (!host_out) KRY_TRY(hipMemcpyAsync(state, out, sizeof(double) * kNumOut, hipMemcpyDeviceToHost, st));
    KRY_TRY(hipStreamSynchronize(st));
    if (host_out) std::memcpy(state, host_out, sizeof(double) * kNumOut);
    return HMVM_OK;
  }
};

// The solve loop shared by the entry points: start, then chunks of
// check_every iterations (eager, or replays of one captured iteration) until
// the stop word is set or max_iter iterations have been launched.  `timed`
// brackets the loop with events.
int solve(Solver &s, int max_iter, int use_graph, int check_every, bool timed, hmvm_krylov_result *res) {
  int rc = s.start();
  if (rc) return rc;
  double S0[kNumOut];
  // the graph is made while the device works on the start (N=20,000: 60 us
  // of the 100 to 150 us that capture and instantiation take); a start that
  // is already converged leaves it unused
  hipGraph_t graph = nullptr;
  hipGraphExec_t gexec = nullptr;
  if (use_graph && max_iter > 0) {
    KRY_TRY(hipStreamBeginCapture(s.st, hipStreamCaptureModeThreadLocal));
    rc = s.iterate();
    const hipError_t e = hipStreamEndCapture(s.st, &graph);
    if (rc || e != hipSuccess) {
      if (graph) (void)hipGraphDestroy(graph);
      return rc ? rc : hip_fail("hipStreamEndCapture", e);
    }
    const hipError_t ei = hipGraphInstantiate(&gexec, graph, nullptr, nullptr, 0);
    if (ei != hipSuccess) {
      (void)hipGraphDestroy(graph);
      return hip_fail("hipGraphInstantiate", ei);
    }
  }
  rc = s.read_state(S0);
  if (!rc && S0[kOutStop] != 0.0 && gexec) {  // no iteration to launch
    (void)hipGraphExecDestroy(gexec);
    gexec = nullptr;
  }
  if (rc) {
    if (gexec) (void)hipGraphExecDestroy(gexec);
    if (graph) (void)hipGraphDestroy(graph);
    return rc;
  }
  hipEvent_t e0 = nullptr, e1 = nullptr;
  if (timed) {
    (void)hipEventCreate(&e0);
    (void)hipEventCreate(&e1);
    (void)hipEventRecord(e0, s.st);
  }
  int launched = 0;
  while (launched < max_iter && S0[kOutStop] == 0.0) {
    const int chunk = check_every > 0 ? std::min(check_every, max_iter - launched) : max_iter - launched;
    for (int c = 0; c < chunk && !rc; c++) {
      if (gexec) {
        const hipError_t e = hipGraphLaunch(gexec, s.st);
        rc = e == hipSuccess ? HMVM_OK : hip_fail("hipGraphLaunch", e);
      } else
        rc = s.iterate();
    }
    if (rc) break;
    launched += chunk;
    if ((rc = s.read_state(S0))) break;
  }
  float ms = 0;
  if (timed) {
    (void)hipEventRecord(e1, s.st);
    if (hipEventSynchronize(e1) == hipSuccess) (void)hipEventElapsedTime(&ms, e0, e1);
    (void)hipEventDestroy(e0);
    (void)hipEventDestroy(e1);
  }
  if (gexec) (void)hipGraphExecDestroy(gexec);
  if (graph) (void)hipGraphDestroy(graph);
  if (rc) return rc;
  const double bnorm = S0[kOutBnorm] > 0 ? S0[kOutBnorm] : 1.0;
  res->iters = (int)S0[kOutIters];
  res->hmvms = 2 * res->iters + 1;
  res->relres = S0[kOutRnorm] / bnorm;
  res->ms_loop = ms;
  res->ms_per_iter = launched > 0 ? ms / launched : 0.0;
  res->graph_used = gexec ? 1 : 0;
  if (S0[kOutStop] == 2.0) {
    char m[256];
    std::snprintf(m, sizeof m, "BiCGSTAB broke down after %d iterations (zero divisor or non-finite scalar)",
                  res->iters);
    return hmvm::report_error(HMVM_ERR_BREAKDOWN, m);
  }
  return HMVM_OK;
}

}  // namespace

extern "C" int hmvm_bicgstab(hmvm_plan *plan, const double *b_host, double *u_host, int max_iter, double tol,
                             int use_graph, int check_every, hmvm_krylov_result *res) {
  hmvm::report_clear();
  if (!plan || !b_host || !u_host || !res || max_iter < 0 || check_every < 0)
    return hmvm::report_error(HMVM_ERR_ARG, "hmvm_bicgstab: NULL argument or negative count");
  std::memset(res, 0, sizeof(*res));
  hmvm_plan_info info;
  int rc = hmvm_plan_get_info(plan, &info);
  if (rc) return rc;
  Solver s;
  s.n = info.nd;
  s.tol = tol;
  s.plan = plan;
  const size_t nb = sizeof(double) * (size_t)s.n;
  // work space, b and u, in one allocation; the plan's stream
  struct Buffers {
    double *d = nullptr;
    hipStream_t st = nullptr;
    ~Buffers() {
      (void)hipStreamSynchronize(st);
      if (d) (void)hipFree(d);
    }
  } m;
  m.st = hmvm::plan_stream(plan);
  // b and u start on 16 bytes, on the device and in pinned memory: n rounded up to even
  const size_t n = (size_t)s.n, ne = n + n % 2, work = 6 * ne + kScalarDoubles;
  KRY_TRY(hipMalloc(&m.d, sizeof(double) * (work + 2 * ne)));
  s.st = m.st;
  s.place(m.d);
  double *b = m.d + work;
  s.b = b;
  s.u = b + ne;
  double *h = hmvm::plan_stage(plan);
  if (h) {
    std::memcpy(h, b_host, nb);
    std::memcpy(h + ne, u_host, nb);
    hmvm::stage_copy(b, h, ne + n, s.st);
    s.host_out = h + 2 * ne;
  } else {
    KRY_TRY(hipMemcpyAsync(b, b_host, nb, hipMemcpyHostToDevice, s.st));
    KRY_TRY(hipMemcpyAsync(s.u, u_host, nb, hipMemcpyHostToDevice, s.st));
  }
  rc = solve(s, max_iter, use_graph, check_every, true, res);
  if (rc == HMVM_OK || rc == HMVM_ERR_BREAKDOWN) {
    hipError_t e;
    if (h) {
      hmvm::stage_copy(h + ne, s.u, n, s.st);
      e = hipStreamSynchronize(s.st);
      if (e == hipSuccess) std::memcpy(u_host, h + ne, nb);
    } else {
      e = hipMemcpy(u_host, s.u, nb, hipMemcpyDeviceToHost);
    }
    if (e != hipSuccess) rc = hip_fail("hipMemcpy (u)", e);
  }
  return rc;
}

// ---- the allocation-free variant ----------------------------------------------
// Work space of hmvm_bicgstab_static: the six work vectors of a solve of at
// most kStaticMaxN unknowns, the dot partials and the scalars, in one array
// of the library's code object (48 MiB + 16 KiB; each device the library runs
// on holds its own copy until the process ends).  Every call on a device
// uses that device's copy: calls that overlap on one device race.
constexpr int kStaticMaxN = HMVM_BICGSTAB_STATIC_MAX_N;
constexpr size_t kScratchDoubles = 6 * (size_t)kStaticMaxN + kScalarDoubles;
static __device__ __align__(256) double scratch[kScratchDoubles];

namespace {

constexpr int kMaxDevices = 64;
std::mutex g_scratch_mu;
double *g_scratch_ptr[kMaxDevices] = {};

// The device address of `scratch` on the current device, resolved once per
// device (host code never passes the symbol's own name to a kernel: on the
// host it is only a stand-in).
int scratch_on_current_device(double **out) {
  int dev = -1;
  KRY_TRY(hipGetDevice(&dev));
  if (dev < 0 || dev >= kMaxDevices)
    return hmvm::report_error(HMVM_ERR_UNSUPPORTED, "hmvm_bicgstab_static: device index beyond 63");
  std::lock_guard<std::mutex> lock(g_scratch_mu);
  if (!g_scratch_ptr[dev]) {
    void *p = nullptr;
    KRY_TRY(hipGetSymbolAddress(&p, HIP_SYMBOL(scratch)));
    g_scratch_ptr[dev] = (double *)p;
  }
  *out = g_scratch_ptr[dev];
  return HMVM_OK;
}

}  // namespace

extern "C" int hmvm_bicgstab_static(hmvm_plan *plan, const double *d_b, double *d_u, int max_iter, double tol,
                                    int check_every, void *stream, hmvm_krylov_result *res) {
  hmvm::report_clear();
  if (!plan || !d_b || !d_u || !res || max_iter < 0 || check_every < 0)
    return hmvm::report_error(HMVM_ERR_ARG, "hmvm_bicgstab_static: NULL argument or negative count");
  std::memset(res, 0, sizeof(*res));
  hmvm_plan_info info;
  int rc = hmvm_plan_get_info(plan, &info);
  if (rc) return rc;
  if (info.nd > kStaticMaxN) {
    char m[256];
    std::snprintf(m, sizeof m, "hmvm_bicgstab_static: nd = %d exceeds the fixed work space (at most %d unknowns); "
                  "use hmvm_bicgstab", info.nd, kStaticMaxN);
    return hmvm::report_error(HMVM_ERR_ARG, m);
  }
  double *w = nullptr;
  if ((rc = scratch_on_current_device(&w))) return rc;
  Solver s;
  s.n = info.nd;
  s.tol = tol;
  s.plan = plan;
  s.st = (hipStream_t)stream;
  s.b = d_b;
  s.u = d_u;
  s.place(w);
  return solve(s, max_iter, 0, check_every, false, res);
}
