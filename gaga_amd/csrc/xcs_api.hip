// Host side of the recovery engine: kernels, resident plans, problem
// generation and the C ABI declared in include/gaga_amd.h.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <climits>
#include <cstdarg>
#include <cstdio>
#include <cstring>
#include <ctime>
#include <mutex>
#include <string>
#include <thread>
#include <array>
#include <vector>

#include "../../include/gaga_amd.h"
#include "xcs_split.h"
#include "xcs_sched.h"
#include "xcs_smvgen.h"
#include "xcs_subset.h"

using namespace xcs;

// --------------------------------------------------------- device memory --
// Device memory for the engine's buffers (one place to change placement).
static hipError_t dev_malloc(void **p, size_t bytes) { return hipMalloc(p, bytes); }

// Copies between device memory and the caller's (pageable) host memory.  From
// BOUNCE_MIN bytes on they go through pinned staging memory of the library's
// own (hipHostMalloc, two halves used in turn, kept for the life of the
// process) instead of the runtime's transfer path for large pageable copies,
// which would lock the caller's pages in place.  From BOUNCE_MIN bytes on,
// h2d returns once the data is on the device and d2h once it is in the
// caller's memory; below that both are hipMemcpyAsync on `st`.  st = nullptr:
// the null stream, synchronous at every size, as hipMemcpy.
constexpr size_t BOUNCE_MIN = (size_t)64 << 10, BOUNCE_HALF = (size_t)8 << 20;
static std::mutex g_bounce_mu;
static char *g_bounce = nullptr;
static hipEvent_t g_bounce_ev[2] = {nullptr, nullptr};

static hipError_t bounce_setup() {
  if (g_bounce) return hipSuccess;
  hipError_t e = hipHostMalloc((void **)&g_bounce, 2 * BOUNCE_HALF, hipHostMallocDefault);
  if (e != hipSuccess) {
    g_bounce = nullptr;
    return e;
  }
  for (hipEvent_t &ev : g_bounce_ev)
    if ((e = hipEventCreateWithFlags(&ev, hipEventDisableTiming)) != hipSuccess) return e;
  return hipSuccess;
}

static hipError_t h2d(void *dst, const void *src, size_t bytes, hipStream_t st) {
  if (bytes < BOUNCE_MIN)
    return st ? hipMemcpyAsync(dst, src, bytes, hipMemcpyHostToDevice, st)
              : hipMemcpy(dst, src, bytes, hipMemcpyHostToDevice);
  std::lock_guard<std::mutex> lock(g_bounce_mu);
  hipError_t e = bounce_setup();
  if (e != hipSuccess) return e;
  bool pending[2] = {false, false};
  int half = 0;
  for (size_t off = 0; off < bytes; off += BOUNCE_HALF, half ^= 1) {
    const size_t c = std::min(BOUNCE_HALF, bytes - off);
    if (pending[half] && (e = hipEventSynchronize(g_bounce_ev[half])) != hipSuccess) return e;
    char *b = g_bounce + half * BOUNCE_HALF;
    memcpy(b, (const char *)src + off, c);
    if (!st) {  // hipMemcpy's ordering against earlier device work
      if ((e = hipMemcpy((char *)dst + off, b, c, hipMemcpyHostToDevice)) != hipSuccess) return e;
      continue;
    }
    if ((e = hipMemcpyAsync((char *)dst + off, b, c, hipMemcpyHostToDevice, st)) != hipSuccess ||
        (e = hipEventRecord(g_bounce_ev[half], st)) != hipSuccess)
      return e;
    pending[half] = true;
  }
  for (int h = 0; h < 2; h++)
    if (pending[h] && (e = hipEventSynchronize(g_bounce_ev[h])) != hipSuccess) return e;
  return hipSuccess;
}

// `height` rows of `width` bytes from host src (row pitch spitch) to device dst
// (row pitch dpitch), staged as h2d is.
static hipError_t h2d_rows(void *dst, size_t dpitch, const void *src, size_t spitch, size_t width,
                           size_t height, hipStream_t st) {
  if (width * height < BOUNCE_MIN || width > BOUNCE_HALF)
    return st ? hipMemcpy2DAsync(dst, dpitch, src, spitch, width, height, hipMemcpyHostToDevice, st)
              : hipMemcpy2D(dst, dpitch, src, spitch, width, height, hipMemcpyHostToDevice);
  std::lock_guard<std::mutex> lock(g_bounce_mu);
  hipError_t e = bounce_setup();
  if (e != hipSuccess) return e;
  const size_t per = BOUNCE_HALF / width;  // rows per chunk
  bool pending[2] = {false, false};
  int half = 0;
  for (size_t r0 = 0; r0 < height; r0 += per, half ^= 1) {
    const size_t rc = std::min(per, height - r0);
    if (pending[half] && (e = hipEventSynchronize(g_bounce_ev[half])) != hipSuccess) return e;
    char *b = g_bounce + half * BOUNCE_HALF;
    for (size_t r = 0; r < rc; r++) memcpy(b + r * width, (const char *)src + (r0 + r) * spitch, width);
    if (!st) {
      if ((e = hipMemcpy2D((char *)dst + r0 * dpitch, dpitch, b, width, width, rc,
                           hipMemcpyHostToDevice)) != hipSuccess)
        return e;
      continue;
    }
    if ((e = hipMemcpy2DAsync((char *)dst + r0 * dpitch, dpitch, b, width, width, rc,
                              hipMemcpyHostToDevice, st)) != hipSuccess ||
        (e = hipEventRecord(g_bounce_ev[half], st)) != hipSuccess)
      return e;
    pending[half] = true;
  }
  for (int h = 0; h < 2; h++)
    if (pending[h] && (e = hipEventSynchronize(g_bounce_ev[h])) != hipSuccess) return e;
  return hipSuccess;
}

static hipError_t d2h(void *dst, const void *src, size_t bytes, hipStream_t st) {
  if (bytes < BOUNCE_MIN)
    return st ? hipMemcpyAsync(dst, src, bytes, hipMemcpyDeviceToHost, st)
              : hipMemcpy(dst, src, bytes, hipMemcpyDeviceToHost);
  std::lock_guard<std::mutex> lock(g_bounce_mu);
  hipError_t e = bounce_setup();
  if (e != hipSuccess) return e;
  if (!st) {  // hipMemcpy's ordering against earlier device work, chunk by chunk
    for (size_t off = 0; off < bytes; off += BOUNCE_HALF) {
      const size_t c = std::min(BOUNCE_HALF, bytes - off);
      if ((e = hipMemcpy(g_bounce, (const char *)src + off, c, hipMemcpyDeviceToHost)) != hipSuccess)
        return e;
      memcpy((char *)dst + off, g_bounce, c);
    }
    return hipSuccess;
  }
  // chunk j lands in half j % 2; chunk j - 1 is copied out while chunk j moves
  size_t prev_off = 0, prev_c = 0;
  int half = 0;
  for (size_t off = 0; off < bytes; off += BOUNCE_HALF, half ^= 1) {
    const size_t c = std::min(BOUNCE_HALF, bytes - off);
    if ((e = hipMemcpyAsync(g_bounce + half * BOUNCE_HALF, (const char *)src + off, c,
                            hipMemcpyDeviceToHost, st)) != hipSuccess ||
        (e = hipEventRecord(g_bounce_ev[half], st)) != hipSuccess)
      return e;
    if (prev_c) {
      if ((e = hipEventSynchronize(g_bounce_ev[half ^ 1])) != hipSuccess) return e;
      memcpy((char *)dst + prev_off, g_bounce + (half ^ 1) * BOUNCE_HALF, prev_c);
    }
    prev_off = off;
    prev_c = c;
  }
  if ((e = hipEventSynchronize(g_bounce_ev[half ^ 1])) != hipSuccess) return e;
  memcpy((char *)dst + prev_off, g_bounce + (half ^ 1) * BOUNCE_HALF, prev_c);
  return hipSuccess;
}

// ------------------------------------------------------------------ errors --
static thread_local std::string g_err;
static int set_err(int code, const char *fmt, ...) {
  char buf[512];
  va_list ap;
  va_start(ap, fmt);
  vsnprintf(buf, sizeof(buf), fmt, ap);
  va_end(ap);
  g_err = buf;
  return code;
}
#define HIP_TRY(expr)                                                                  \
  do {                                                                                 \
    hipError_t e_ = (expr);                                                            \
    if (e_ != hipSuccess)                                                              \
      return set_err(e_ == hipErrorOutOfMemory ? XCS_ENOMEM : XCS_EHIP, "%s: %s (%s:%d)", \
                     #expr, hipGetErrorString(e_), __FILE__, __LINE__);                \
  } while (0)
#define XCS_TRY(expr)        \
  do {                       \
    int r_ = (expr);         \
    if (r_ != XCS_OK) return r_; \
  } while (0)

#include "xcs_host.h"

// ----------------------------------------------------------------- kernels --
// One instance, the whole (cooperatively launched) grid is its team.
// The descriptor is copied to LDS: its fields then cannot alias the global
// vectors the solver writes, so the compiler keeps them in registers.
// spin_limit bounds every team-barrier wait (sleeps); on timeout the team
// abandons the instance (stop reason STOP_ABORTED, abort flag bar[2] set).
__global__ void __launch_bounds__(1024) solve_coop_kernel(const XProblem *P, int budget,
                                                          double *red, unsigned *bar,
                                                          long spin_limit) {
  __shared__ Lds L;
  __shared__ XProblem sP;
  if (threadIdx.x == 0) sP = *P;
  __syncthreads();
  Team t{(int)blockIdx.x, (int)gridDim.x, red, 0, bar};
  t.spin_limit = spin_limit;
  solve_instance(t, L, sP, budget);
}

// Team membership for the batched engine: c workgroups per team.  Workgroups
// are dispatched round-robin over the 8 XCDs (XCD = blockIdx % 8), so when the
// grid allows it a team is formed from workgroups of one XCD (shared L2).
__device__ __forceinline__ void batch_team(int c, int *team_id, int *rank) {
  const int b = blockIdx.x, nb = gridDim.x;
  if (c == 1) {
    *team_id = b;
    *rank = 0;
  } else if (nb % (8 * c) == 0) {
    const int xcd = b % 8, local = b / 8;
    *team_id = (local / c) * 8 + xcd;
    *rank = local % c;
  } else {
    *team_id = b / c;
    *rank = b % c;
  }
}

// The workgroup of rank 0 in this workgroup's team (see batch_team).
__device__ __forceinline__ int batch_team_leader(int c) {
  const int b = blockIdx.x, nb = gridDim.x;
  if (c == 1) return b;
  if (nb % (8 * c) == 0) {
    const int xcd = b % 8, local = b / 8;
    return (local / c) * c * 8 + xcd;
  }
  return (b / c) * c;
}

// Batched persistent form, two queues over the instances (largest first):
// teams of c workgroups take instances [0, n_big) from queue[0] and solve each
// with team-scoped barriers; when that range is used up each team dissolves
// and its workgroups take [n_big, count) one per workgroup from queue[1].  A
// team works in its leader's workspace and a lone workgroup in its own, so a
// dissolved workgroup never shares scratch with a team still running.
// TEAMS = false is the one-workgroup-per-instance form: the team queue is
// compiled out, which keeps its registers (and spills) out of the kernel.
// list (optional) maps queue positions to instances: a later launch of the
// tail schedule takes only the instances still running.
template <bool TEAMS>
__global__ void __launch_bounds__(1024) solve_batch_kernel(const XProblem *Ps, int count,
                                                           int n_big, int *queue,
                                                           const XWork *works, int *slots,
                                                           double *red, unsigned *bar, int c,
                                                           int budget, const int *list,
                                                           long spin_limit) {
  __shared__ Lds L;
  __shared__ XProblem sP;
  __shared__ int sidx;
  if (TEAMS && c > 1) {
    int team_id, rank;
    batch_team(c, &team_id, &rank);
    const int leader = batch_team_leader(c);
    Team t{rank, c, red + (size_t)team_id * 2 * RED_SLOTS * c, 0, bar + (size_t)team_id * BAR_WORDS};
    t.spin_limit = spin_limit;
    while (true) {
      if (rank == 0 && threadIdx.x == 0) slots[team_id] = atomicAdd(&queue[0], 1);
      t.sync();
      const int idx = slots[team_id];
      if (idx >= n_big) break;
      if (threadIdx.x == 0) {
        sP = Ps[list ? list[idx] : idx];
        attach_work(sP, works[leader]);
      }
      __syncthreads();
      solve_instance(t, L, sP, budget);
      t.sync();
      if (t.aborted) break;  // a team barrier timed out: the team stops taking instances
    }
  }
  Team t1{0, 1, nullptr, 0, nullptr};
  while (true) {
    if (threadIdx.x == 0) sidx = n_big + atomicAdd(&queue[1], 1);
    __syncthreads();
    const int idx = sidx;
    if (idx >= count) break;
    if (threadIdx.x == 0) {
      sP = Ps[list ? list[idx] : idx];
      attach_work(sP, works[blockIdx.x]);
    }
    __syncthreads();
    solve_instance(t1, L, sP, budget);
    __syncthreads();
  }
}

// y = A x_S (mode 0) or g = A^T r (mode 1) with the team operators.
__global__ void __launch_bounds__(1024) apply_coop_kernel(const XProblem *P, int transpose,
                                                          const float *in, float *out,
                                                          int cnt, double *red, unsigned *bar) {
  __shared__ Lds L;
  __shared__ XProblem sP;
  if (threadIdx.x == 0) sP = *P;
  __syncthreads();
  Team t{(int)blockIdx.x, (int)gridDim.x, red, 0, bar};
  if (transpose) {
    XG(float) o = (XG(float))out;
    op_AT(t, L, sP, (XG(const float))in, [&](int j, float g) { o[j] = g; });
  } else {
    op_A(t, L, sP, (XG(const float))in, (XG(float))out, cnt);
  }
}

// A^T y (transpose = 1) or A_S x (0: support from the planted-vector list in
// the team scratch is not available here, so only A^T is offered) for every
// instance of a batch, one workgroup per instance: the streaming product of the
// batched solver in isolation (bandwidth measurement).
__global__ void __launch_bounds__(1024) apply_batch_kernel(const XProblem *Ps, int count,
                                                           const XWork *works) {
  __shared__ Lds L;
  __shared__ XProblem sP;
  Team t{0, 1, nullptr, 0, nullptr};
  for (int idx = blockIdx.x; idx < count; idx += gridDim.x) {
    if (threadIdx.x == 0) {
      sP = Ps[idx];
      attach_work(sP, works[blockIdx.x]);
    }
    __syncthreads();
    XG(float) g = sP.grad;
    op_AT(t, L, sP, sP.y, [&](int j, float v) { g[j] = v; });
    __syncthreads();
  }
}

// y = A x_true for every instance of a batch, one workgroup per instance
// (the planted support is copied into the workgroup's support list first:
// the gen product gathers the columns it names).
__global__ void __launch_bounds__(1024) make_y_batch_kernel(const XProblem *Ps, int count,
                                                            const XWork *works,
                                                            const float *const *xt,
                                                            const int *const *sp) {
  __shared__ Lds L;
  __shared__ XProblem sP;
  Team t{0, 1, nullptr, 0, nullptr};
  for (int idx = blockIdx.x; idx < count; idx += gridDim.x) {
    if (threadIdx.x == 0) {
      sP = Ps[idx];
      attach_work(sP, works[blockIdx.x]);
    }
    __syncthreads();
    const int *s = sp[idx];
    for (int i = threadIdx.x; i < sP.k; i += blockDim.x) sP.supp[i] = s[i];
    __syncthreads();
    op_A(t, L, sP, (XG(const float))xt[idx], (XG(float))sP.y, sP.k);
    __syncthreads();
  }
}

// Start-of-solve reset of a batch: every x, every solver state, the work
// queue and the team barriers (a kernel, so it can sit in a captured graph).
__global__ void batch_reset_kernel(float *xs, size_t xs_len, int *st, size_t st_words, int *queue,
                                   unsigned *bar, size_t bar_words) {
  const size_t stride = (size_t)gridDim.x * blockDim.x;
  const size_t i0 = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
  for (size_t i = i0; i < xs_len; i += stride) xs[i] = 0.f;
  for (size_t i = i0; i < st_words; i += stride) st[i] = 0;
  for (size_t i = i0; i < bar_words; i += stride) bar[i] = 0u;
  if (i0 == 0) {
    queue[0] = 0;
    queue[1] = 0;
  }
}

// One FindSupportSet call with the team binning (functions.cu:397-436).
__global__ void __launch_bounds__(1024) find_support_coop_kernel(const XProblem *P,
                                                                 const float *v, XState *S_io,
                                                                 float slope, float intercept,
                                                                 double *red, unsigned *bar) {
  __shared__ Lds L;
  __shared__ XProblem sP;
  if (threadIdx.x == 0) sP = *P;
  __syncthreads();
  Team t{(int)blockIdx.x, (int)gridDim.x, red, 0, bar};
  XState S = *S_io;
  if (S.min_val > S.max_change) {
    if (t.rank == 0 && threadIdx.x == 0) {
      S_io->min_val = S.min_val - S.max_change;
      S_io->sum = -1;
    }
    return;
  }
  zero_counters(t, sP);
  t.sync();
  int kb;
  find_support_bin(t, L, sP, (XG(const float))v, sP.bins, S, slope, intercept, &kb);
  S.k_bin = kb;
  if (t.rank == 0 && threadIdx.x == 0) *S_io = S;
}

// A[i + j*lda] ~ N(0,1)/sqrt(m) from Philox4x32-10, key (seed, instance),
// counter (e mod 2^32, e div 2^32, STREAM_A, 0) with e = j*m + i; Box-Muller.
__global__ void gen_matrix_kernel(float *A, int m, int n, int lda, uint32_t seed, uint32_t inst) {
  const size_t total = (size_t)lda * n;
  const double s = 1.0 / sqrt((double)m);
  for (size_t idx = (size_t)blockIdx.x * blockDim.x + threadIdx.x; idx < total;
       idx += (size_t)gridDim.x * blockDim.x) {
    const int j = (int)(idx / lda), i = (int)(idx - (size_t)j * lda);
    float v = 0.f;
    if (i < m) {
      const uint64_t e = (uint64_t)j * (uint64_t)m + (uint64_t)i;
      uint32_t o[4];
      philox4x32_10((uint32_t)e, (uint32_t)(e >> 32), STREAM_A, 0u, seed, inst, o);
      const double z = sqrt(-2.0 * log(u01d(o[0]))) * cos(6.283185307179586476925286766559 * u01d(o[1]));
      v = (float)(z * s);
    }
    A[idx] = v;
  }
}

// DCT tables: tw[t] = exp(-2 pi i t / n), qw[q] = (cos, sin)(pi q / (2n)).
__global__ void dct_tables_kernel(float2 *tw, int n) {
  for (int t = blockIdx.x * blockDim.x + threadIdx.x; t < n; t += gridDim.x * blockDim.x) {
    double s, c;
    sincospi(-2.0 * (double)t / (double)n, &s, &c);
    tw[t] = make_float2((float)c, (float)s);
    sincospi((double)t / (2.0 * (double)n), &s, &c);
    tw[n + t] = make_float2((float)c, (float)s);
  }
}

// The inverse of a dct row list: pos[q] = -1 for every q < n (first launch),
// then pos[rows[i]] = i (second launch; the rows are distinct).
__global__ void dct_pos_fill_kernel(int *pos, int n) {
  for (int q = blockIdx.x * blockDim.x + threadIdx.x; q < n; q += gridDim.x * blockDim.x) pos[q] = -1;
}
__global__ void dct_pos_scatter_kernel(const int *rows, int m, int *pos) {
  for (int i = blockIdx.x * blockDim.x + threadIdx.x; i < m; i += gridDim.x * blockDim.x)
    pos[rows[i]] = i;
}
static int make_dct_pos(hipStream_t st, const int *rows, int m, int n, int *pos) {
  if (!rows || !pos) return set_err(XCS_EINVAL, "dct row map: rows or positions not allocated");
  hipLaunchKernelGGL(dct_pos_fill_kernel, dim3(std::min(4096, (n + 255) / 256)), dim3(256), 0, st,
                     pos, n);
  HIP_TRY(hipGetLastError());
  hipLaunchKernelGGL(dct_pos_scatter_kernel, dim3(std::min(4096, (m + 255) / 256)), dim3(256), 0,
                     st, rows, m, pos);
  HIP_TRY(hipGetLastError());
  return XCS_OK;
}

// ------------------------------------------------------------ host helpers --
static const char *const CSMPSP_OFF =
    "CSMPSP is switched off on the GPU in this build (a device fault in it is not yet explained)";
static int parse_alg(const char *alg) {
  if (!alg) return -1;
  if (!strcmp(alg, "NIHT")) return ALG_NIHT;
  if (!strcmp(alg, "HTP")) return ALG_HTP;
  if (!strcmp(alg, "CSMPSP")) return ALG_CSMPSP;
  if (!strcmp(alg, "CGIHT")) return ALG_CGIHT;
  // the reference's further greedy algorithms (gaga_gen.cu:65, 625-634)
  if (!strcmp(alg, "IHT")) return ALG_IHT;
  if (!strcmp(alg, "ThresholdSD")) return ALG_HTSD;
  if (!strcmp(alg, "ThresholdCG")) return ALG_HTCG;
  if (!strcmp(alg, "FIHT")) return ALG_FIHT;
  if (!strcmp(alg, "ALPS")) return ALG_ALPS;
  if (!strcmp(alg, "CGIHTprojected")) return ALG_CGIHTP;
  return -1;
}
static int parse_ens(const char *ens) {
  if (!ens) return -1;
  if (!strcmp(ens, "gen")) return ENS_GEN;
  if (!strcmp(ens, "smv")) return ENS_SMV;
  if (!strcmp(ens, "dct")) return ENS_DCT;
  return -1;
}
static int ilog2_exact(int n) {
  if (n <= 0 || (n & (n - 1))) return -1;
  int l = 0;
  while ((1 << l) < n) l++;
  return l;
}
static int round_up(int v, int a) { return (v + a - 1) / a * a; }

// Subsets (dct rows, planted supports) and planted values drawn on the device:
// jobs and plants are copied into the caller's device arrays dj / dp (sized for
// them), then one workgroup per subset and one per planted vector.  The host
// vectors may go out of scope on return (the copies are synchronous for them).
static int device_draws(hipStream_t st, const std::vector<SubsetJob> &jobs, SubsetJob *dj,
                        const std::vector<PlantJob> &plants, PlantJob *dp) {
  if (!jobs.empty()) {
    HIP_TRY(h2d(dj, jobs.data(), sizeof(SubsetJob) * jobs.size(), st));
    hipLaunchKernelGGL(subset_kernel, dim3((unsigned)std::min<size_t>(jobs.size(), 8192)), dim3(1024),
                       0, st, dj, (int)jobs.size());
    HIP_TRY(hipGetLastError());
  }
  if (!plants.empty()) {
    HIP_TRY(h2d(dp, plants.data(), sizeof(PlantJob) * plants.size(), st));
    hipLaunchKernelGGL(plant_kernel, dim3((unsigned)std::min<size_t>(plants.size(), 8192)), dim3(256),
                       0, st, dp, (int)plants.size());
    HIP_TRY(hipGetLastError());
  }
  HIP_TRY(hipStreamSynchronize(st));
  return XCS_OK;
}

// Device smv generation (the kernels above) into caller buffers: CSC (col_ptr
// n+1, rows and vals n*p) and CSR (row_ptr m+1, cols and rvals n*p).  tmp holds
// 4*m ints (counts and three scratch lists); flags[0] is a failure flag that
// accumulates over calls (zeroed once by the caller), flags[1] receives the
// number of empty rows the repair filled.
struct SmvOut {
  int *col_ptr, *rows, *row_ptr, *cols;
  float *vals, *rvals;
};
static int smv_check(int m, int n, int p, int ens) {
  if (ens < 1 || ens > 3) return set_err(XCS_EINVAL, "smv: matrixEnsemble must be 1, 2 or 3");
  if (p <= 0 || p > m) return set_err(XCS_EINVAL, "smv: need 0 < p <= m (p = %d, m = %d)", p, m);
  if (p > SMV_P_MAX) return set_err(XCS_EINVAL, "smv: the generator supports p <= %d", SMV_P_MAX);
  if ((long)n * p >= (long)INT_MAX) return set_err(XCS_EINVAL, "smv: n * p too large");
  return XCS_OK;
}
static int device_smv(hipStream_t st, int m, int n, int p, int ens, uint32_t seed, uint32_t inst,
                      const SmvOut &d, int *tmp, int *flags) {
  int *cnt = tmp, *first = tmp + m, *zl = tmp + 2 * (size_t)m, *don = tmp + 3 * (size_t)m;
  const float scale = 1.0f / sqrtf((float)p);
  HIP_TRY(hipMemsetAsync(cnt, 0, sizeof(int) * (size_t)m, st));
  hipLaunchKernelGGL(smv_columns_kernel, dim3((n + 255) / 256), dim3(256), 0, st, m, n, p, ens,
                     scale, seed, inst, d.rows, d.vals, cnt, flags);
  hipLaunchKernelGGL(smv_repair_kernel, dim3(1), dim3(1024), 0, st, m, n, p, d.rows, d.vals, cnt,
                     d.row_ptr, first, zl, don, flags + 1);
  HIP_TRY(hipMemsetAsync(first, 0, sizeof(int) * (size_t)m, st));
  hipLaunchKernelGGL(smv_fill_kernel, dim3((n + 256) / 256), dim3(256), 0, st, m, n, p, d.rows,
                     d.vals, d.row_ptr, first, d.col_ptr, d.cols, d.rvals);
  hipLaunchKernelGGL(smv_row_sort_kernel, dim3(m), dim3(64), 0, st, m, d.row_ptr, d.cols, d.rvals);
  HIP_TRY(hipGetLastError());
  return XCS_OK;
}
static const char *const SMV_FAIL =
    "smv generation: a column needed more than 2^20 draws (p too close to m)";

// ------------------------------------------------------------------- plans --
// Everything a solve starts from, in one launch: the descriptor, x = 0, a fresh
// state and cleared barrier words (a copy and three fills before: 4 of the
// runtime's calls, each with a launch of its own behind it).
__global__ void plan_reset_kernel(XProblem P, XProblem *d, unsigned *bar) {
  const int t = blockIdx.x * blockDim.x + threadIdx.x, stride = gridDim.x * blockDim.x;
  if (t == 0) *d = P;
  for (int i = t; i < P.n; i += stride) P.x[i] = 0.f;
  int *st = (int *)(XState *)P.st;
  for (int i = t; i < (int)(sizeof(XState) / sizeof(int)); i += stride) st[i] = 0;
  for (int i = t; i < BAR_WORDS; i += stride) bar[i] = 0u;
}

// Device memory of a plan: its vectors come out of one block (one allocation,
// one fill) as long as they fit, the rest one by one.  A given-problem call of
// 256 x 1024 made 23 allocations and as many fills, 0.2 ms of its 0.65.
constexpr size_t PLAN_SLAB_MAX = (size_t)16 << 20;

struct xcs_plan {
  int dev = 0;
  hipStream_t stream = nullptr;  // the lane's
  HostLane lane;
  char *slab = nullptr;
  size_t slab_left = 0;
  XProblem h{};         // host copy (device pointers)
  XProblem *d = nullptr;
  int team = 1, block = 256, mode = 0;
  int form = FORM_GENERAL;       // SolveForm the plan is laid out for
  const void *kernel = nullptr;  // and its kernel, where that is not solve_coop_kernel
  long spin_limit = BAR_SPIN_LIMIT;  // team-barrier wait bound (sleeps)
  double *red = nullptr;
  unsigned *bar = nullptr;
  std::vector<void *> allocs;
  std::vector<float> x_true;
  int k_planted = 0;
  float gen_ms = 0.f, last_ms = 0.f;
  XState last{};
  float *warm_g = nullptr;  // learned warm start: A^T y and the starting support
  int *warm_mask = nullptr;
  float *warm_score = nullptr;
  float *xt_dev = nullptr;  // the planted vector, where the plan was generated
  std::mutex pin_mu;  // held while a call uses the lane's staging memory
  ~xcs_plan() {
    // nothing of this plan may still run on memory that is about to be freed
    if (stream) (void)hipStreamSynchronize(stream);
    for (void *p : allocs) (void)hipFree(p);
    lane_put(&lane);
  }
  // The device is current: the plan's stream, events and staging memory.
  int open() {
    HIP_TRY(hipGetDevice(&dev));
    XCS_TRY(lane_get(&lane));
    stream = lane.stream;
    return XCS_OK;
  }
  // One cleared block for the allocations that follow.
  int reserve(size_t bytes) {
    if (bytes > PLAN_SLAB_MAX) return XCS_OK;
    char *q = nullptr;
    XCS_TRY(alloc(&q, bytes));
    slab = q;
    slab_left = bytes;
    return XCS_OK;
  }
  template <class T>
  int alloc(T **p, size_t count) {
    void *q = nullptr;
    const size_t bytes = std::max<size_t>(count, 1) * sizeof(T), need = (bytes + 255) / 256 * 256;
    if (need <= slab_left) {
      *p = (T *)slab;
      slab += need;
      slab_left -= need;
      return XCS_OK;
    }
    hipError_t e = dev_malloc(&q, bytes);
    if (e != hipSuccess)
      return set_err(XCS_ENOMEM, "hipMalloc(%zu bytes): %s", bytes, hipGetErrorString(e));
    allocs.push_back(q);
    e = hipMemsetAsync(q, 0, bytes, stream);
    if (e != hipSuccess) return set_err(XCS_EHIP, "hipMemsetAsync: %s", hipGetErrorString(e));
    *p = (T *)q;
    return XCS_OK;
  }
};

static int max_coop_blocks(int block, int *out) {
  int dev;
  HIP_TRY(hipGetDevice(&dev));
  int cus = 0;
  HIP_TRY(hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev));
  // every cooperative kernel must fit co-resident at the chosen grid size
  const void *kernels[] = {(const void *)solve_coop_kernel, (const void *)apply_coop_kernel,
                           (const void *)find_support_coop_kernel};
  int per = 1 << 30;
  for (const void *k : kernels) {
    int b = 0;
    HIP_TRY(hipOccupancyMaxActiveBlocksPerMultiprocessor(&b, k, block, 0));
    per = std::min(per, b);
  }
  if (per <= 0) return set_err(XCS_EINVAL, "block size %d does not fit on a CU", block);
  *out = per * cus;
  return XCS_OK;
}

static int use_device(int gpu) {
  int count = 0;
  hipError_t e = hipGetDeviceCount(&count);
  if (e != hipSuccess || count <= 0) return set_err(XCS_ENODEV, "no HIP device available");
  if (gpu < 0 || gpu >= count) gpu = 0;  // gaga_gen.cu:248-253 resets silently
  HIP_TRY(hipSetDevice(gpu));
  return XCS_OK;
}

// The timing variants exist for NIHT and HTP only (gaga_gen.cu:332-335: other
// algorithms run their plain form).
static int timing_fields(XProblem &P, int alg, int k, const xcs_options *o) {
  P.timing = (o->timing && (alg == ALG_NIHT || alg == ALG_HTP)) ? 1 : 0;
  P.supp_flag = P.timing ? o->supp_flag : 0;
  P.alpha0 = P.timing ? o->alpha : 0.25f;
  if (P.timing) {
    if (o->supp_flag < 0 || o->supp_flag > 3) return set_err(XCS_EINVAL, "supportFlag must be 0, 1, 2 or 3");
    if (!(o->alpha >= 0.f && o->alpha < 1.f)) return set_err(XCS_EINVAL, "alpha must be in [0, 1)");
    if (o->supp_flag >= 2 && k < 1) return set_err(XCS_EINVAL, "supportFlag 2 and 3 need k >= 1");
  }
  return XCS_OK;
}

static const void *resident_kernel(int alg, int block) {
  const bool s = block <= 512;
  switch (alg) {
    case ALG_NIHT:
      return s ? (const void *)solve_resident_kernel<ALG_NIHT, 512>
               : (const void *)solve_resident_kernel<ALG_NIHT, 1024>;
    case ALG_HTP:
      return s ? (const void *)solve_resident_kernel<ALG_HTP, 512>
               : (const void *)solve_resident_kernel<ALG_HTP, 1024>;
    case ALG_CGIHT:
      return s ? (const void *)solve_resident_kernel<ALG_CGIHT, 512>
               : (const void *)solve_resident_kernel<ALG_CGIHT, 1024>;
  }
  return nullptr;
}

// Whether the plan runs in the resident form (xcs_resident.h), and its geometry.
static int plan_resident(xcs_plan *pl, int alg, const xcs_options *o) {
  const XProblem &P = pl->h;
  const int block = o->block_size > 0 ? o->block_size : 512;
  int cus = 0, per = 0, dev = 0;
  HIP_TRY(hipGetDevice(&dev));
  HIP_TRY(hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev));
  const void *kernel = resident_kernel(alg, block);
  if (!kernel) return XCS_OK;
  HIP_TRY(hipOccupancyMaxActiveBlocksPerMultiprocessor(&per, kernel, block, 0));
  int team = o->team_size;
  if (team <= 0) {
    // Streaming A wants many workgroups, the three exchanges per iteration few:
    // the optimum grows with the square root of A's bytes.  Measured on MI355X,
    // ms per solve with 512 threads (256 and 1024 are slower at every size):
    // NIHT 256 x 1024 (1 MiB) 0.253 / 0.247 / 0.247 / 0.291 at 16 / 32 / 64 / 128
    // workgroups (general form: 0.9); CGIHT 1024 x 4096 (16 MiB) 0.439 / 0.341 /
    // 0.328 / 0.364 at 32 / 64 / 128 / 256; CGIHT 2048 x 8192 (64 MiB) 0.728 /
    // 0.569 / 0.551 at 64 / 128 / 256 (general form: 1.70).  HTP spends its time
    // in CG steps, whose products touch the support's columns only: half the team
    // (1001 x 5003: 0.343 / 0.357 / 0.426 at 64 / 128 / 256; general form 1.65).
    const double mib = 4.0 * P.lda * (double)P.n / (1 << 20);
    const double want = (alg == ALG_HTP ? 16.0 : 32.0) * std::sqrt(mib);
    team = 16;
    while (team < 256 && team * 1.42 < want) team *= 2;
  }
  if (team > per * cus || team > BAR_MAX_TEAM) return XCS_OK;
  if (!res_fits(alg, P.ens, P.n, P.lda, P.num_bins, P.timing, team)) return XCS_OK;
  pl->form = FORM_RESIDENT;
  pl->kernel = kernel;
  pl->team = team;
  pl->block = block;
  return XCS_OK;
}

static const void *split_kernel(int ens, int alg) {
  switch (alg) {
    case ALG_NIHT:
      return ens == ENS_DCT ? (const void *)solve_split_kernel<ENS_DCT, ALG_NIHT>
                            : (const void *)solve_split_kernel<ENS_SMV, ALG_NIHT>;
    case ALG_HTP:
      return ens == ENS_DCT ? (const void *)solve_split_kernel<ENS_DCT, ALG_HTP>
                            : (const void *)solve_split_kernel<ENS_SMV, ALG_HTP>;
    case ALG_CGIHT:
      return ens == ENS_DCT ? (const void *)solve_split_kernel<ENS_DCT, ALG_CGIHT>
                            : (const void *)solve_split_kernel<ENS_SMV, ALG_CGIHT>;
  }
  return nullptr;
}

// Whether the plan runs in the split form (xcs_split.h), and its geometry.
static int plan_split(xcs_plan *pl, int alg, const xcs_options *o) {
  const XProblem &P = pl->h;
  if (P.ens != ENS_SMV && P.ens != ENS_DCT) return XCS_OK;
  const void *kernel = split_kernel(P.ens, alg);
  const int block = o->block_size > 0 ? o->block_size : SP_THREADS;
  if (!kernel || block > SP_THREADS) return XCS_OK;
  int cus = 0, per = 0, dev = 0;
  HIP_TRY(hipGetDevice(&dev));
  HIP_TRY(hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev));
  HIP_TRY(hipOccupancyMaxActiveBlocksPerMultiprocessor(&per, kernel, block, 0));
  int team = o->team_size;
  if (team <= 0) {
    // As for the dense form the optimum grows with the square root of the size:
    // half of sqrt(n), in powers of two.  Measured on MI355X, ms per solve:
    // NIHT smv 1500 x 8000 0.238 / 0.253 / 0.273 at 16 / 32 / 64 workgroups; CGIHT smv
    // 6000 x 30011 0.357 / 0.324 / 0.384 at 32 / 64 / 128, NIHT 15000 x 65536 0.944 /
    // 0.921 / 1.158 at 64 / 128 / 256, CGIHT 2^15 x 2^18 2.93 / 1.91 / 1.76 at 64 /
    // 128 / 256 (general form 6.6); NIHT dct n = 2^17
    // 0.785 / 0.619 / 0.552 at 32 / 64 / 128; CGIHT dct n = 2^14 0.366 / 0.302 / 0.307
    // at 8 / 16 / 32; NIHT dct n = 2^20 1.66 at 256 (5.7; fewer do not fit its LDS).
    team = 2;
    while (team < 256 && 4.0 * team <= std::sqrt((double)P.n)) team *= 2;
    if (P.ens == ENS_DCT) {  // the factorisation allows up to half its rows
      const int n1 = P.log2n > 1 ? 1 << ((P.log2n - 1) / 2) : 1;
      team = std::min(team, n1 / 2);
    }
  }
  if (team > per * cus || team > BAR_MAX_TEAM) return XCS_OK;
  if (!split_fits(alg, P.ens, P.m, P.n, P.log2n, P.num_bins, P.timing, team, block)) return XCS_OK;
  pl->form = FORM_SPLIT;
  pl->kernel = kernel;
  pl->team = team;
  pl->block = block;
  return XCS_OK;
}

// Allocate workspace for (alg, ens, m, n) and fill the sizes in plan->h.
static int plan_alloc(xcs_plan *pl, int alg, int ens, int k, int m, int n, int p, int nz,
                      const xcs_options *o) {
  XProblem &P = pl->h;
  P.alg = alg;
  P.ens = ens;
  P.m = m;
  P.n = n;
  P.k = k;
  P.p = p;
  P.nz = nz;
  P.lda = round_up(m, 64);
  P.num_bins = o->num_bins > 0 ? o->num_bins : std::max(n / 20, 1000);
  P.maxiter = o->maxiter > 0 ? o->maxiter : ((alg == ALG_HTP || alg == ALG_CSMPSP) ? 300 : 5000);
  P.restart = o->restart;
  P.tol = o->tol_reference_default ? (float)(10 ^ (-4)) : o->tol;
  P.proj_frac_tol = o->proj_frac_tol > 0.f ? o->proj_frac_tol : 3.0f;  // gaga_gen.cu:190
  XCS_TRY(timing_fields(P, alg, k, o));
  P.log2n = ens == ENS_DCT ? ilog2_exact(n) : 0;
  pl->mode = o->mode;
  pl->spin_limit = o->barrier_spin_limit > 0 ? o->barrier_spin_limit : BAR_SPIN_LIMIT;
  // default workgroup size, measured on MI355X for one instance per cooperative
  // launch: 512 threads for every ensemble
  pl->block = o->block_size > 0 ? o->block_size : 512;
  if (pl->block % 64 || pl->block > 1024) return set_err(XCS_EINVAL, "block_size must be a multiple of 64 <= 1024");
  int maxb;
  XCS_TRY(max_coop_blocks(pl->block, &maxb));
  int team = o->team_size;
  if (team <= 0) {
    // The general form's team (solve_coop_kernel; plan_resident and plan_split
    // choose their own).  Bandwidth grows with the team, and so does the cost of its barriers
    // (8-10 team barriers or reductions per iteration).  Teams in proportion
    // to the bytes one product streams, capped where the measured optima on
    // MI355X (512-thread workgroups, CGIHT and NIHT) lie: gen 2048 x 8192 at
    // 64 workgroups (2.70 ms; 2.81 at 128; HTP, whose CG steps are gathers,
    // at 128: 7.79 against 8.44 ms at 64), gen 1024 x 4096 at 32-64, smv
    // n = 2^18 at 128 (18.3 ms), n = 2^15 at 32-64, dct n = 2^20 at 256
    // (22.6 ms; 26.8 at 128, 41.4 at 64, 30.6 at 512), dct n = 2^17 at 32.
    const double bytes = ens == ENS_GEN ? 4.0 * P.lda * (double)n
                         : ens == ENS_SMV ? 8.0 * nz : 24.0 * n;
    const double per = ens == ENS_GEN ? 5.0e5 : ens == ENS_SMV ? 1.15e5 : 1.0e5;
    const double cap = ens == ENS_GEN ? (alg == ALG_HTP ? 128.0 : 64.0)
                       : ens == ENS_SMV ? 128.0 : 256.0;
    team = (int)std::min<double>(cap, std::max(1.0, std::round(bytes / per)));
    // the dct FFT's passes split into a power of two of equal blocks: a team of
    // a power of two takes them in whole rounds (the nearest one, by ratio)
    if (ens == ENS_DCT) {
      int lo = 1;
      while (lo * 2 <= team) lo *= 2;
      team = (team * 3 >= lo * 4 && lo * 2 <= (int)cap) ? lo * 2 : lo;
    }
  }
  pl->team = std::min({team, maxb, BAR_MAX_TEAM});
  XCS_TRY(plan_resident(pl, alg, o));
  if (pl->form == FORM_GENERAL) XCS_TRY(plan_split(pl, alg, o));
  // CSMPSP is switched off on the device: two of its runs (a 4-workgroup team
  // and later a single workgroup) faulted the GPU and the cause is not yet
  // found; it stays off until it is.
  if (alg == ALG_CSMPSP) return set_err(XCS_EINVAL, CSMPSP_OFF);
  const size_t nn = (size_t)n, ml = (size_t)P.lda;
  // the allocations below and those that a generated or given problem adds (y, the
  // rows of a dct, a planted vector); the matrices have blocks of their own
  const size_t words = 9 * nn + (ens == ENS_DCT ? 7 * nn + ml : 0) + 6 * ml +
                       (ens == ENS_GEN ? 2 * (size_t)MAXCH * ml : 0) + P.num_bins + pl->team +
                       (P.timing ? 10 : 2) * ((size_t)P.maxiter + 2) +
                       4 * (size_t)RED_SLOTS * (pl->team + 1) + BAR_WORDS + std::max(k, 1);
  XCS_TRY(pl->reserve(4 * words + 32 * 256 + sizeof(XState) + sizeof(XProblem) + 1024));
  XCS_TRY(pl->alloc(&P.x, nn));
  XCS_TRY(pl->alloc(&P.thres, nn));
  XCS_TRY(pl->alloc(&P.grad, nn));
  XCS_TRY(pl->alloc(&P.gprev, nn));
  XCS_TRY(pl->alloc(&P.gprev_thres, nn));
  XCS_TRY(pl->alloc(&P.bins, nn));
  XCS_TRY(pl->alloc(&P.bins2, nn));
  XCS_TRY(pl->alloc(&P.resid, ml));
  XCS_TRY(pl->alloc(&P.resid_update, ml));
  XCS_TRY(pl->alloc(&P.resid2, ml));
  XCS_TRY(pl->alloc(&P.resid3, ml));
  XCS_TRY(pl->alloc(&P.counters, (size_t)P.num_bins + 64));
  XCS_TRY(pl->alloc(&P.supp, nn));
  XCS_TRY(pl->alloc(&P.wg_counts, (size_t)pl->team + 64));
  if (ens == ENS_GEN) XCS_TRY(pl->alloc(&P.partials, 2 * (size_t)MAXCH * ml));
  if (ens == ENS_DCT) {
    XCS_TRY(pl->alloc(&P.cwork, nn));
    int *pos;
    XCS_TRY(pl->alloc(&pos, nn));  // filled once the rows are known (make_dct_pos)
    xset(P.dct_pos, pos);
    float2 *tw;
    XCS_TRY(pl->alloc(&tw, 2 * nn));
    hipLaunchKernelGGL(dct_tables_kernel, dim3(std::min(4096, (n + 255) / 256)), dim3(256), 0,
                       pl->stream, tw, n);
    HIP_TRY(hipGetLastError());
    xset(P.twiddle, tw);
  }
  XCS_TRY(pl->alloc(&P.st, 1));
  XCS_TRY(pl->alloc(&P.trace_err, (size_t)P.maxiter + 2));
  XCS_TRY(pl->alloc(&P.trace_kbin, (size_t)P.maxiter + 2));
  if (P.timing) XCS_TRY(pl->alloc(&P.trace_ticks, 4 * ((size_t)P.maxiter + 2)));
  XCS_TRY(pl->alloc(&pl->red, (size_t)2 * RED_SLOTS * (pl->team + 1)));
  XCS_TRY(pl->alloc(&pl->bar, (size_t)BAR_WORDS));
  XCS_TRY(pl->alloc(&pl->d, 1));
  return XCS_OK;
}

static int plan_upload_desc(xcs_plan *pl) {
  HIP_TRY(h2d(pl->d, &pl->h, sizeof(XProblem), pl->stream));
  return XCS_OK;
}

static int launch_apply(xcs_plan *pl, int transpose, const float *in, float *out, int cnt) {
  HIP_TRY(hipMemsetAsync(pl->bar, 0, sizeof(unsigned) * BAR_WORDS, pl->stream));
  void *args[] = {(void *)&pl->d, (void *)&transpose, (void *)&in, (void *)&out, (void *)&cnt,
                  (void *)&pl->red, (void *)&pl->bar};
  HIP_TRY(hipLaunchCooperativeKernel((const void *)apply_coop_kernel, dim3(pl->team),
                                     dim3(pl->block), args, 0, pl->stream));
  return XCS_OK;
}

// y = A x for a device x whose support list (cnt entries, ascending) is d_supp, by the
// product the plan's solves use.
static int plan_make_y(xcs_plan *pl, const int *d_supp, int cnt, const float *d_x, float *d_y) {
  XProblem &P = pl->h;
  if (cnt)
    HIP_TRY(hipMemcpyAsync((int *)P.supp, d_supp, sizeof(int) * cnt, hipMemcpyDeviceToDevice,
                           pl->stream));
  XCS_TRY(plan_upload_desc(pl));
  if (pl->form == FORM_RESIDENT) {
    if (pl->block <= 512)
      hipLaunchKernelGGL(resident_y_kernel<512>, dim3(pl->team), dim3(pl->block), 0, pl->stream,
                         (const XProblem *)pl->d, d_x, cnt, d_y);
    else
      hipLaunchKernelGGL(resident_y_kernel<1024>, dim3(pl->team), dim3(pl->block), 0, pl->stream,
                         (const XProblem *)pl->d, d_x, cnt, d_y);
    HIP_TRY(hipGetLastError());
  } else if (pl->form == FORM_SPLIT) {
    HIP_TRY(hipMemsetAsync(pl->bar, 0, sizeof(unsigned) * BAR_WORDS, pl->stream));
    long limit = BAR_SPIN_LIMIT;
    int alg = P.alg;
    void *args[] = {(void *)&pl->d, (void *)&alg, (void *)&d_x, (void *)&d_y, (void *)&pl->bar, (void *)&limit};
    const void *kernel = P.ens == ENS_DCT ? (const void *)split_y_kernel<ENS_DCT>
                                          : (const void *)split_y_kernel<ENS_SMV>;
    HIP_TRY(hipLaunchCooperativeKernel(kernel, dim3(pl->team), dim3(pl->block), args, 0, pl->stream));
  } else {
    XCS_TRY(launch_apply(pl, 0, d_x, d_y, cnt));
  }
  HIP_TRY(hipStreamSynchronize(pl->stream));
  return XCS_OK;
}

// Build the CSC (fixed or general) and CSR device copies of an smv matrix.
static int plan_set_smv(xcs_plan *pl, const std::vector<int> &col_ptr, const std::vector<int> &rows,
                        const std::vector<float> &vals) {
  XProblem &P = pl->h;
  const int m = P.m, n = P.n, nz = (int)rows.size();
  std::vector<int> row_ptr((size_t)m + 1, 0), cols((size_t)nz);
  std::vector<float> rvals((size_t)nz);
  for (int e = 0; e < nz; e++) row_ptr[rows[e] + 1]++;
  for (int i = 0; i < m; i++) row_ptr[i + 1] += row_ptr[i];
  std::vector<int> fill(row_ptr.begin(), row_ptr.end() - 1);
  for (int j = 0; j < n; j++)
    for (int e = col_ptr[j]; e < col_ptr[j + 1]; e++) {
      const int pos = fill[rows[e]]++;
      cols[pos] = j;
      rvals[pos] = vals[e];
    }
  int *d_cp, *d_r, *d_rp, *d_c;
  float *d_v, *d_rv;
  XCS_TRY(pl->alloc(&d_cp, (size_t)n + 1));
  XCS_TRY(pl->alloc(&d_r, (size_t)nz));
  XCS_TRY(pl->alloc(&d_v, (size_t)nz));
  XCS_TRY(pl->alloc(&d_rp, (size_t)m + 1));
  XCS_TRY(pl->alloc(&d_c, (size_t)nz));
  XCS_TRY(pl->alloc(&d_rv, (size_t)nz));
  HIP_TRY(h2d(d_cp, col_ptr.data(), sizeof(int) * (n + 1), pl->stream));
  HIP_TRY(h2d(d_r, rows.data(), sizeof(int) * nz, pl->stream));
  HIP_TRY(h2d(d_v, vals.data(), sizeof(float) * nz, pl->stream));
  HIP_TRY(h2d(d_rp, row_ptr.data(), sizeof(int) * (m + 1), pl->stream));
  HIP_TRY(h2d(d_c, cols.data(), sizeof(int) * nz, pl->stream));
  HIP_TRY(h2d(d_rv, rvals.data(), sizeof(float) * nz, pl->stream));
  HIP_TRY(hipStreamSynchronize(pl->stream));
  xset(P.col_ptr, d_cp);
  xset(P.rows, d_r);
  xset(P.vals, d_v);
  xset(P.row_ptr, d_rp);
  xset(P.cols, d_c);
  xset(P.rvals, d_rv);
  P.nz = nz;
  return XCS_OK;
}

static int validate(int alg, int ens, int k, int m, int n) {
  if (alg < 0)
    return set_err(XCS_EINVAL, "algorithm must be one of NIHT, HTP, CSMPSP, CGIHT, IHT, "
                               "ThresholdSD, ThresholdCG, FIHT, ALPS, CGIHTprojected");
  if (ens < 0) return set_err(XCS_EINVAL, "ens must be either dct, gen, or smv.");
  if (m <= 0 || n <= 0 || k < 0) return set_err(XCS_EINVAL, "need m > 0, n > 0, k >= 0");
  if (ens == ENS_DCT && (ilog2_exact(n) < 1 || n > (1 << 22)))
    return set_err(XCS_EINVAL, "dct: n must be a power of two in [2, 2^22]");
  if (ens == ENS_DCT && m > n) return set_err(XCS_EINVAL, "dct: m must be <= n");
  return XCS_OK;
}

// Generate an instance into a fresh plan (seed, instance from opts).
static int plan_generate(xcs_plan *pl, int alg, int ens, int k, int m, int n, int p,
                         const xcs_options *o) {
  XCS_TRY(validate(alg, ens, k, m, n));
  if (k > n) return set_err(XCS_EINVAL, "k must be <= n");
  XCS_TRY(use_device(o->gpu_number));
  XCS_TRY(pl->open());
  HIP_TRY(hipEventRecord(pl->lane.e0, pl->stream));
  const uint32_t seed = o->seed, inst = o->instance;
  int *smv_tmp = nullptr;
  int nz = 0;
  if (ens == ENS_SMV) {
    XCS_TRY(smv_check(m, n, p, o->matrix_ensemble));
    nz = n * p;
  }
  XCS_TRY(plan_alloc(pl, alg, ens, k, m, n, p, nz, o));
  XProblem &P = pl->h;
  float *y;
  XCS_TRY(pl->alloc(&y, (size_t)P.lda));
  xset(P.y, y);
  if (ens == ENS_GEN) {
    float *A;
    XCS_TRY(pl->alloc(&A, (size_t)P.lda * n));
    const size_t total = (size_t)P.lda * n;
    const int blocks = (int)std::min<size_t>(65536, (total + 255) / 256);
    hipLaunchKernelGGL(gen_matrix_kernel, dim3(blocks), dim3(256), 0, pl->stream, A, m, n, P.lda,
                       seed, inst);
    HIP_TRY(hipGetLastError());
    xset(P.A, A);
  } else if (ens == ENS_SMV) {
    SmvOut d;
    XCS_TRY(pl->alloc(&d.col_ptr, (size_t)n + 1));
    XCS_TRY(pl->alloc(&d.rows, (size_t)nz));
    XCS_TRY(pl->alloc(&d.vals, (size_t)nz));
    XCS_TRY(pl->alloc(&d.row_ptr, (size_t)m + 1));
    XCS_TRY(pl->alloc(&d.cols, (size_t)nz));
    XCS_TRY(pl->alloc(&d.rvals, (size_t)nz));
    XCS_TRY(pl->alloc(&smv_tmp, 4 * (size_t)m + 2));
    XCS_TRY(device_smv(pl->stream, m, n, p, o->matrix_ensemble, seed, inst, d, smv_tmp,
                       smv_tmp + 4 * (size_t)m));
    xset(P.col_ptr, d.col_ptr);
    xset(P.rows, d.rows);
    xset(P.vals, d.vals);
    xset(P.row_ptr, d.row_ptr);
    xset(P.cols, d.cols);
    xset(P.rvals, d.rvals);
  }
  // the dct rows and the planted vector, drawn on the device
  std::vector<SubsetJob> jobs;
  if (ens == ENS_DCT) {
    int *d_rows;
    XCS_TRY(pl->alloc(&d_rows, (size_t)m));
    jobs.push_back(SubsetJob{n, m, seed, inst, STREAM_DCT_ROWS, d_rows});
    xset(P.dct_rows, d_rows);
  }
  int *d_supp;
  float *d_xt;
  XCS_TRY(pl->alloc(&d_supp, (size_t)std::max(k, 1)));
  XCS_TRY(pl->alloc(&d_xt, (size_t)n));
  jobs.push_back(SubsetJob{n, k, seed, inst, STREAM_SUPPORT, d_supp});
  const std::vector<PlantJob> plants = {PlantJob{k, o->vec_distribution, seed, inst, d_supp, d_xt, nullptr}};
  SubsetJob *dj;
  PlantJob *dp;
  XCS_TRY(pl->alloc(&dj, jobs.size()));
  XCS_TRY(pl->alloc(&dp, plants.size()));
  XCS_TRY(device_draws(pl->stream, jobs, dj, plants, dp));
  if (ens == ENS_DCT)
    XCS_TRY(make_dct_pos(pl->stream, (const int *)P.dct_rows, m, n, (int *)P.dct_pos));
  pl->k_planted = k;
  XCS_TRY(plan_make_y(pl, d_supp, k, d_xt, y));
  pl->x_true.resize((size_t)n);
  HIP_TRY(d2h(pl->x_true.data(), d_xt, sizeof(float) * n, nullptr));
  pl->xt_dev = d_xt;
  HIP_TRY(hipEventRecord(pl->lane.e1, pl->stream));
  HIP_TRY(hipEventSynchronize(pl->lane.e1));
  HIP_TRY(hipEventElapsedTime(&pl->gen_ms, pl->lane.e0, pl->lane.e1));
  if (smv_tmp) {
    int fl[2];
    HIP_TRY(d2h(fl, smv_tmp + 4 * (size_t)m, sizeof(fl), nullptr));
    if (fl[0]) return set_err(XCS_EINVAL, SMV_FAIL);
  }
  return XCS_OK;
}

static int launch_solve(xcs_plan *pl, int budget) {
  if (solve_form(pl->form, pl->h.warm != nullptr) != FORM_GENERAL) {
    void *args[] = {(void *)&pl->d, (void *)&budget, (void *)&pl->bar, (void *)&pl->spin_limit};
    HIP_TRY(hipLaunchCooperativeKernel(pl->kernel, dim3(pl->team), dim3(pl->block), args, 0, pl->stream));
    return XCS_OK;
  }
  void *args[] = {(void *)&pl->d, (void *)&budget, (void *)&pl->red, (void *)&pl->bar,
                  (void *)&pl->spin_limit};
  HIP_TRY(hipLaunchCooperativeKernel((const void *)solve_coop_kernel, dim3(pl->team),
                                     dim3(pl->block), args, 0, pl->stream));
  return XCS_OK;
}

// One solve; x_out (where not null) takes the solution.
static int plan_run(xcs_plan *pl, float *ms, float *x_out = nullptr) {
  XProblem &P = pl->h;
  // inputs stay resident
  hipLaunchKernelGGL(plan_reset_kernel, dim3(std::max(1, std::min(256, (P.n + 1023) / 1024))), dim3(256),
                     0, pl->stream, P, pl->d, pl->bar);
  HIP_TRY(hipGetLastError());
  HIP_TRY(hipEventRecord(pl->lane.e0, pl->stream));
  if (pl->mode == 1) {
    // plain form: one outer iteration per launch, host reads the stop flag
    // (an aborted team marks the instance done, so launching stops there too)
    int budget = 1;
    for (int launch = 0; launch < P.maxiter + 4; launch++) {
      XCS_TRY(launch_solve(pl, budget));
      int done = 0;
      HIP_TRY(d2h(&done, &P.st->done, sizeof(int), pl->stream));
      HIP_TRY(hipStreamSynchronize(pl->stream));
      if (done) break;
    }
  } else {
    int budget = P.maxiter + 4;
    XCS_TRY(launch_solve(pl, budget));
  }
  HIP_TRY(hipEventRecord(pl->lane.e1, pl->stream));
  // the state, the abort flag and a solution that the staging memory holds come
  // back in one launch behind the solve, for one synchronisation
  struct Back {
    XState st;
    unsigned abort_flag;
  };
  static_assert(sizeof(XState) % sizeof(float) == 0 && LANE_X + sizeof(Back) <= LANE_BYTES, "staging memory");
  Back *back = (Back *)(pl->lane.pin + LANE_X);
  const bool x_too = x_out && sizeof(float) * (size_t)P.n <= LANE_X;
  std::lock_guard<std::mutex> lock(pl->pin_mu);
  XferList L;
  L.add((XState *)P.st, &back->st, sizeof(XState) / sizeof(float));
  L.add(pl->bar + 2, &back->abort_flag, 1);
  if (x_too) L.add((float *)P.x, pl->lane.pin, P.n);
  HIP_TRY(xfer(L, pl->stream));
  HIP_TRY(hipStreamSynchronize(pl->stream));
  HIP_TRY(hipEventElapsedTime(&pl->last_ms, pl->lane.e0, pl->lane.e1));
  pl->last = back->st;
  if (back->abort_flag) return set_err(XCS_EHIP, "team barrier timed out (results invalid)");
  if (x_too)
    memcpy(x_out, pl->lane.pin, sizeof(float) * (size_t)P.n);
  else if (x_out)
    HIP_TRY(d2h(x_out, P.x, sizeof(float) * (size_t)P.n, pl->stream));
  if (ms) *ms = pl->last_ms;
  return XCS_OK;
}

// conv rate forms: results.cu:365-378 (generated) and gaga_gen.cu:735-742 (given)
static float conv_rate_results(const XState &S) {
  int temp = std::min(S.iter, 16);
  if (temp <= 1) return 0.0f;
  temp = temp - 1;
  const float root = 1 / (float)temp;
  temp = 15 - temp;
  return powf(S.prev[15] / S.prev[temp], root);
}
static float conv_rate_given(const XState &S) {
  int temp = std::min(S.iter, 16);
  if (temp == 0) return 0.0f;
  const float root = 1 / (float)temp;
  temp = 16 - temp;
  return powf(S.prev[15] / S.prev[temp], root);
}

static void host_norms(const std::vector<float> &xt, const float *xo, int k, float norms[3],
                       int support[4]) {
  double a1 = 0, a2 = 0, ai = 0, d1 = 0, d2 = 0, di = 0;
  int tp = 0, tn = 0;
  const int n = (int)xt.size();
  for (int i = 0; i < n; i++) {
    const double t = xt[i], o = xo[i], df = t - o;
    a1 += fabs(t);
    a2 += t * t;
    ai = std::max(ai, fabs(t));
    d1 += fabs(df);
    d2 += df * df;
    di = std::max(di, fabs(df));
    if (t != 0.0) {
      if (o != 0.0) tp++;
    } else if (o == 0.0) {
      tn++;
    }
  }
  if (norms) {
    norms[0] = (float)(d1 / a1);
    norms[1] = (float)(sqrt(d2) / sqrt(a2));
    norms[2] = (float)(di / ai);
  }
  if (support) {
    support[0] = tp;
    support[1] = k - tp;
    support[2] = tn;
    support[3] = n - k - tn;
  }
}

// f(0), ..., f(count - 1), each once, over up to 16 host threads (fewer for
// small counts); a thread that cannot be started has its share run here.
template <class F>
static void host_parallel_for(int count, F f) {
  const long hw = std::max(1u, std::thread::hardware_concurrency());
  const int nt = (int)std::max(1L, std::min({16L, hw, (long)(count + 31) / 32}));
  auto share = [&](int w) {
    for (int i = w; i < count; i += nt) f(i);
  };
  std::vector<std::thread> th;
  std::vector<int> here;
  for (int w = 1; w < nt; w++) {
    try {
      th.emplace_back(share, w);
    } catch (...) {
      here.push_back(w);
    }
  }
  share(0);
  for (int w : here) share(w);
  for (auto &t : th) t.join();
}

// ----------------------------------------------------------------- batches --
// Instance data lives in two arenas: one for the dense gen matrices (written
// in full by the generator, never cleared) and one for everything else
// (cleared once).  All solution vectors are contiguous (one reset, one copy
// back), and so are the solver states.
struct xcs_batch {
  int dev = 0;
  hipStream_t stream = nullptr;
  int alg = 0, count = 0, c = 1, block = 256, nteams = 0, grid = 0, budget = 0;
  int n_big = 0;  // instances [0, n_big) (queue order) go to teams of c workgroups
  bool exact = false;  // teams as configured, also where the chip has room for larger ones
  int ran_c = 0, ran_teams = 0;  // the last solve's first launch
  int resident = 0;  // workgroups resident at this block size (workspace sized for them)
  int *list = nullptr;  // queue slots of the instances a later phase of the tail schedule takes
  // tail schedule: phase 0 solves every instance on the configured geometry for at
  // most sched_budget[0] iterations; phase p > 0 gives the instances still running
  // teams of sched_team[p] workgroups for sched_budget[p] more (the last phase:
  // until done).  Empty: one launch, no budget beyond maxiter.
  std::vector<int> sched_team, sched_budget;
  std::vector<int> phase_instances;  // instances each phase of the last solve took
  // adaptive form of the schedule (one persistent launch, teams formed on the device)
  // instead of one launch per phase; counters and per-level queues
  bool adaptive = true;
  int split_team = 4;  // adaptive form: team size for phase-0 solves split at the end (< 2: off)
  int *sw = nullptr, *items = nullptr, *leads = nullptr;
  long spin_limit = BAR_SPIN_LIMIT;  // bound of every team-barrier and scheduler wait
  int red_stride = 0;  // doubles of reduction buffer per workgroup
  int n_max = 1, lda_max = 64, bins_max = 1000;
  bool any_dct = false;
  std::vector<XProblem> hP;  // queue order
  XProblem *dP = nullptr;
  float *xs = nullptr;       // every x, contiguous (queue order)
  size_t xs_len = 0;
  char *back = nullptr;      // pinned: the abort flag, then the states (batch_states)
  float *xs_host = nullptr;  // pinned copy of xs for the results (allocated on first use)
  std::vector<size_t> xoff;
  XState *sts = nullptr;
  // team workspace (depends on c and block)
  std::vector<void *> wallocs;
  XWork *dW = nullptr;
  int *slots = nullptr, *queue = nullptr;
  double *red = nullptr;
  unsigned *bar = nullptr;
  hipGraphExec_t graph = nullptr;
  std::vector<void *> allocs;
  std::vector<std::vector<float>> x_true;
  std::vector<int> ks;
  std::vector<XState> last;
  std::vector<int> order;  // order[q] = caller index of queue slot q
  std::vector<int> slot_of;  // slot_of[i] = queue slot of caller index i
  PinnedReadAhead ahead;           // solution vectors read in order
  unsigned long long *phase = nullptr;  // XCS_PHASE_TIMING builds only
  float gen_ms = 0.f, last_ms = 0.f;
  void drop_graph() {
    if (graph) (void)hipGraphExecDestroy(graph);
    graph = nullptr;
  }
  void drop_work() {
    for (void *q : wallocs) (void)hipFree(q);
    wallocs.clear();
  }
  ~xcs_batch() {
    // nothing of this batch may still run on memory that is about to be freed
    if (stream) (void)hipStreamSynchronize(stream);
    drop_graph();
    drop_work();
    for (void *q : allocs) (void)hipFree(q);
    if (xs_host) (void)hipHostFree(xs_host);
    if (back) (void)hipHostFree(back);
    if (stream) (void)hipStreamDestroy(stream);
  }
  int raw(void **q, size_t bytes, bool clear, std::vector<void *> &list) {
    void *r = nullptr;
    bytes = std::max<size_t>(bytes, 256);
    hipError_t e = dev_malloc(&r, bytes);
    if (e != hipSuccess)
      return set_err(XCS_ENOMEM, "hipMalloc(%zu bytes): %s", bytes, hipGetErrorString(e));
    list.push_back(r);
    if (clear) {
      e = hipMemsetAsync(r, 0, bytes, stream);
      if (e != hipSuccess) return set_err(XCS_EHIP, "hipMemsetAsync: %s", hipGetErrorString(e));
    }
    *q = r;
    return XCS_OK;
  }
  template <class T>
  int alloc(T **q, size_t cnt) {
    return raw((void **)q, cnt * sizeof(T), true, allocs);
  }
  template <class T>
  int walloc(T **q, size_t cnt) {
    return raw((void **)q, cnt * sizeof(T), true, wallocs);
  }
};

// The gen matrices of a batch in a series of device allocations of up to
// CHUNK bytes each (no matrix spans two) rather than one of tens of GB, which
// a fragmented device heap may refuse.  take() allocates the next chunk when
// the current one is full, sized for what is still to come.
struct ChunkArena {
  static constexpr size_t CHUNK = (size_t)2 << 30;
  char *base = nullptr;
  size_t used = 0, cap = 0, left = 0;  // left: bytes still to be taken overall
  static size_t up(size_t b) { return (b + 255) / 256 * 256; }
  template <class T>
  int take(xcs_batch *B, size_t cnt, T **out) {
    const size_t b = up(std::max<size_t>(cnt, 1) * sizeof(T));
    if (!base || used + b > cap) {
      if (b > left) return set_err(XCS_EINVAL, "internal: matrix arena overflow");
      const size_t want = std::max(b, std::min(CHUNK / b * b, left));
      XCS_TRY(B->raw((void **)&base, want, false, B->allocs));
      used = 0;
      cap = want;
    }
    *out = (T *)(base + used);
    used += b;
    left -= b;
    return XCS_OK;
  }
};

// Bump allocator over one device allocation (256-byte aligned pieces).
// take() returns nullptr once the capacity would be exceeded.
struct Arena {
  char *base = nullptr;
  size_t used = 0, cap = 0;
  static size_t up(size_t b) { return (b + 255) / 256 * 256; }
  template <class T>
  T *take(size_t cnt) {
    const size_t b = up(std::max<size_t>(cnt, 1) * sizeof(T));
    if (!base || used + b > cap) return nullptr;
    T *r = (T *)(base + used);
    used += b;
    return r;
  }
};

static int batch_occupancy(int block, int *per_cu, int *cus) {
  int dev;
  HIP_TRY(hipGetDevice(&dev));
  HIP_TRY(hipDeviceGetAttribute(cus, hipDeviceAttributeMultiprocessorCount, dev));
  // every form must fit co-resident at the chosen grid size
  int a = 0, b = 0;
  HIP_TRY(hipOccupancyMaxActiveBlocksPerMultiprocessor(&a, (const void *)solve_batch_kernel<false>,
                                                       block, 0));
  HIP_TRY(hipOccupancyMaxActiveBlocksPerMultiprocessor(&b, (const void *)solve_batch_kernel<true>,
                                                       block, 0));
  int s = 0;
  HIP_TRY(hipOccupancyMaxActiveBlocksPerMultiprocessor(&s, (const void *)solve_sched_kernel, block, 0));
  *per_cu = std::min({a, b, s});
  if (*per_cu <= 0) return set_err(XCS_EINVAL, "block size %d does not fit on a CU", block);
  return XCS_OK;
}

// Team geometry and per-team workspace for c workgroups of `block` threads.
// big < 0: every instance goes to a team of c workgroups; otherwise the
// `big` largest do and the rest run one per workgroup.
static int batch_configure(xcs_batch *B, int c, int block, int big = -1) {
  if (block % 64 || block < 64 || block > 1024)
    return set_err(XCS_EINVAL, "block_size must be a multiple of 64 in [64, 1024]");
  if (c < 1) return set_err(XCS_EINVAL, "team_size must be >= 1");
  if (B->alg == ALG_CSMPSP) c = 1;  // see plan_alloc: multi-workgroup CSMPSP is switched off
  int per_cu, cus;
  XCS_TRY(batch_occupancy(block, &per_cu, &cus));
  const int resident = per_cu * cus;
  if (c > resident) return set_err(XCS_EINVAL, "team_size %d exceeds %d resident workgroups", c, resident);
  int nteams = std::min(B->count, resident / c);
  if (c > 1 && nteams >= 8) nteams -= nteams % 8;  // whole teams per XCD
  HIP_TRY(hipStreamSynchronize(B->stream));
  B->drop_graph();
  B->drop_work();
  B->c = c;
  B->block = block;
  B->nteams = nteams;
  B->grid = nteams * c;
  B->n_big = c == 1 ? 0 : (big < 0 ? B->count : std::min(big, B->count));
  // scratch for every workgroup that can be resident at this block size (a team
  // uses its leader's), and team words for as many teams: any team size at this
  // block size then runs on the same allocation (the tail schedule changes it
  // between launches)
  const size_t T = (size_t)resident, ml = (size_t)B->lda_max;
  const size_t tmax = (size_t)std::min(resident, BAR_MAX_TEAM);
  B->resident = resident;
  int *cnt, *wgc;
  float *part;
  float2 *cw = nullptr;
  XCS_TRY(B->walloc(&cnt, T * ((size_t)B->bins_max + 64)));
  XCS_TRY(B->walloc(&wgc, T * (tmax + 64)));
  XCS_TRY(B->walloc(&part, T * 2 * MAXCH * ml));
  if (B->any_dct) XCS_TRY(B->walloc(&cw, T * (size_t)B->n_max));
  std::vector<XWork> hw(T);
  for (size_t t = 0; t < T; t++) {
    XWork &W = hw[t];
    xset(W.counters, cnt + t * ((size_t)B->bins_max + 64));
    xset(W.wg_counts, wgc + t * (tmax + 64));
    xset(W.partials, part + t * 2 * MAXCH * ml);
    xset(W.cwork, cw ? cw + t * (size_t)B->n_max : nullptr);
  }
  XCS_TRY(B->walloc(&B->dW, T));
  HIP_TRY(h2d(B->dW, hw.data(), sizeof(XWork) * T, B->stream));
  XCS_TRY(B->walloc(&B->slots, T));
  XCS_TRY(B->walloc(&B->queue, 64));
  XCS_TRY(B->walloc(&B->list, (size_t)std::max(B->count, 1)));
  // reduction buffer: room per workgroup for a team of tmax led by it (the adaptive
  // schedule's teams form from any workgroups; a static team of c uses c * 2 * RED_SLOTS
  // from its team index on)
  B->red_stride = 2 * RED_SLOTS * (int)tmax;
  XCS_TRY(B->walloc(&B->red, T * (size_t)B->red_stride));
  XCS_TRY(B->walloc(&B->bar, T * BAR_WORDS));
  HIP_TRY(hipStreamSynchronize(B->stream));  // hw goes out of scope
  return XCS_OK;
}

static int batch_generate(xcs_batch *B, int alg, int count, const int *ens, const int *k,
                          const int *m, const int *n, const int *p, const unsigned *inst,
                          const xcs_options *o) {
  if (alg < 0)
    return set_err(XCS_EINVAL, "algorithm must be one of NIHT, HTP, CSMPSP, CGIHT, IHT, "
                               "ThresholdSD, ThresholdCG, FIHT, ALPS, CGIHTprojected");
  if (alg == ALG_CSMPSP) return set_err(XCS_EINVAL, CSMPSP_OFF);
  if (count <= 0) return set_err(XCS_EINVAL, "count must be > 0");
  for (int i = 0; i < count; i++) {
    XCS_TRY(validate(alg, ens[i], k[i], m[i], n[i]));
    if (k[i] > n[i]) return set_err(XCS_EINVAL, "instance %d: k > n", i);
    if (ens[i] == ENS_SMV) {
      if (!p) return set_err(XCS_EINVAL, "instance %d: smv needs p", i);
      XCS_TRY(smv_check(m[i], n[i], p[i], o->matrix_ensemble));
    }
  }
  XCS_TRY(use_device(o->gpu_number));
  HIP_TRY(hipGetDevice(&B->dev));
  HIP_TRY(hipStreamCreateWithFlags(&B->stream, hipStreamNonBlocking));
  hipEvent_t e0, e1;
  HIP_TRY(hipEventCreate(&e0));
  HIP_TRY(hipEventCreate(&e1));
  HIP_TRY(hipEventRecord(e0, B->stream));
  B->alg = alg;
  B->count = count;
  for (int i = 0; i < count; i++) {
    B->n_max = std::max(B->n_max, n[i]);
    B->lda_max = std::max(B->lda_max, round_up(m[i], 64));
    B->bins_max = std::max(B->bins_max, o->num_bins > 0 ? o->num_bins : std::max(n[i] / 20, 1000));
    B->any_dct |= ens[i] == ENS_DCT;
  }
  XCS_TRY(batch_configure(B, o->team_size > 0 ? o->team_size : 1,
                          o->block_size > 0 ? o->block_size : 256));

  // descriptors; the dct rows, planted vectors and smv structure are drawn on
  // the device below
  std::vector<XProblem> hp((size_t)count);
  B->last.resize((size_t)count);
  int maxiter_max = 0, smv_m_max = 0;
  size_t small_bytes = 0, big_bytes = 0, vec_bytes = 0;
  std::vector<int> tw_n;
  for (int i = 0; i < count; i++) {
    XProblem &P = hp[i];
    memset(&P, 0, sizeof(P));
    P.alg = alg;
    P.ens = ens[i];
    P.m = m[i];
    P.n = n[i];
    P.k = k[i];
    P.p = ens[i] == ENS_SMV ? p[i] : 0;
    P.nz = P.n * P.p;
    P.lda = round_up(m[i], 64);
    P.num_bins = o->num_bins > 0 ? o->num_bins : std::max(n[i] / 20, 1000);
    P.maxiter = o->maxiter > 0 ? o->maxiter : ((alg == ALG_HTP || alg == ALG_CSMPSP) ? 300 : 5000);
    maxiter_max = std::max(maxiter_max, P.maxiter);
    P.restart = o->restart;
    P.tol = o->tol_reference_default ? (float)(10 ^ (-4)) : o->tol;
    P.proj_frac_tol = o->proj_frac_tol > 0.f ? o->proj_frac_tol : 3.0f;  // gaga_gen.cu:190
    XCS_TRY(timing_fields(P, alg, k[i], o));
    P.log2n = ens[i] == ENS_DCT ? ilog2_exact(n[i]) : 0;
    if (P.ens == ENS_SMV) smv_m_max = std::max(smv_m_max, P.m);
    // small arena: y, x_true, planted support, smv/dct structure
    small_bytes += Arena::up(4 * (size_t)P.lda) + Arena::up(4 * (size_t)P.n) +
                   Arena::up(4 * std::max<size_t>(P.k, 1));
    if (P.ens == ENS_SMV)
      small_bytes += Arena::up(4 * ((size_t)P.n + 1)) + Arena::up(4 * ((size_t)P.m + 1)) +
                     4 * Arena::up(4 * (size_t)P.nz);
    if (P.ens == ENS_DCT) {
      small_bytes += Arena::up(4 * (size_t)P.m) + Arena::up(4 * (size_t)P.n);
      if (std::find(tw_n.begin(), tw_n.end(), P.n) == tw_n.end()) {
        tw_n.push_back(P.n);
        small_bytes += Arena::up(16 * (size_t)P.n);
      }
    }
    if (P.ens == ENS_GEN) big_bytes += Arena::up(4 * (size_t)P.lda * P.n);
    // the instance's own vectors, kept from one iteration (and launch) to the next
    vec_bytes += 7 * Arena::up(4 * (size_t)P.n) + 4 * Arena::up(4 * (size_t)P.lda);
    B->xs_len += (size_t)P.n;
  }
  B->budget = maxiter_max + 4;
  B->spin_limit = o->barrier_spin_limit > 0 ? o->barrier_spin_limit : BAR_SPIN_LIMIT;

  // queue order: largest instances first (work-queue load balance)
  std::vector<int> order((size_t)count);
  for (int i = 0; i < count; i++) order[i] = i;
  auto cost = [&](int i) {
    const XProblem &P = hp[i];
    return P.ens == ENS_GEN ? (double)P.lda * P.n : P.ens == ENS_SMV ? 2.0 * P.nz : 6.0 * P.n;
  };
  std::stable_sort(order.begin(), order.end(), [&](int a, int b) { return cost(a) > cost(b); });
  B->order = order;
  B->slot_of.assign((size_t)count, 0);
  for (int q = 0; q < count; q++) B->slot_of[order[q]] = q;

  Arena small, vecs;
  ChunkArena big;
  small.cap = small_bytes;
  big.left = big_bytes;
  vecs.cap = vec_bytes;
  XCS_TRY(B->raw((void **)&small.base, small_bytes, true, B->allocs));
  XCS_TRY(B->raw((void **)&vecs.base, vec_bytes, true, B->allocs));
#define XCS_ARENA_OK(ptr) \
  if (!(ptr)) return set_err(XCS_EINVAL, "internal: instance arena overflow")
  XCS_TRY(B->alloc(&B->xs, B->xs_len));
  XCS_TRY(B->alloc(&B->sts, (size_t)count));
  int *smv_tmp = nullptr;
  if (smv_m_max > 0) XCS_TRY(B->alloc(&smv_tmp, 4 * (size_t)smv_m_max + 2));
  auto key_of = [&](int i) { return inst ? inst[i] : (uint32_t)i; };
  std::vector<std::pair<int, float2 *>> tw_cache;
  std::vector<size_t> xt_off((size_t)count);
  std::vector<const float *> xt_ptr((size_t)count);
  std::vector<const int *> sp_ptr((size_t)count);
  std::vector<SubsetJob> jobs;
  std::vector<PlantJob> plants;
  B->xoff.assign((size_t)count, 0);
  B->hP.resize((size_t)count);
  size_t xo = 0;
  for (int q = 0; q < count; q++) {
    const int i = order[q];
    XProblem P = hp[i];
    B->xoff[q] = xo;
    xset(P.x, B->xs + xo);
    xo += (size_t)P.n;
    xset(P.st, B->sts + q);
    float *y = small.take<float>(P.lda);
    float *xt = small.take<float>(P.n);
    int *sp = small.take<int>(P.k);
    XCS_ARENA_OK(y && xt && sp);
    xset(P.y, y);
    {
      float *fv[4];
      int *iv[3];
      float *mv[4];
      for (auto &v : fv) XCS_ARENA_OK((v = vecs.take<float>(P.n)));
      for (auto &v : iv) XCS_ARENA_OK((v = vecs.take<int>(P.n)));
      for (auto &v : mv) XCS_ARENA_OK((v = vecs.take<float>(P.lda)));
      xset(P.thres, fv[0]);
      xset(P.grad, fv[1]);
      xset(P.gprev, fv[2]);
      xset(P.gprev_thres, fv[3]);
      xset(P.bins, iv[0]);
      xset(P.bins2, iv[1]);
      xset(P.supp, iv[2]);
      xset(P.resid, mv[0]);
      xset(P.resid_update, mv[1]);
      xset(P.resid2, mv[2]);
      xset(P.resid3, mv[3]);
    }
    // planted vector (xt is zero: the arena is cleared once)
    jobs.push_back(SubsetJob{P.n, P.k, o->seed, key_of(i), STREAM_SUPPORT, sp});
    plants.push_back(PlantJob{P.k, o->vec_distribution, o->seed, key_of(i), sp, xt, nullptr});
    xt_ptr[q] = xt;
    sp_ptr[q] = sp;
    if (P.ens == ENS_GEN) {
      float *A = nullptr;
      XCS_TRY(big.take(B, (size_t)P.lda * P.n, &A));
      const size_t total = (size_t)P.lda * P.n;
      const int blocks = (int)std::min<size_t>(65536, (total + 255) / 256);
      hipLaunchKernelGGL(gen_matrix_kernel, dim3(blocks), dim3(256), 0, B->stream, A, P.m, P.n,
                         P.lda, o->seed, inst ? inst[i] : (uint32_t)i);
      HIP_TRY(hipGetLastError());
      xset(P.A, A);
    } else if (P.ens == ENS_SMV) {
      const int nz = P.nz;
      SmvOut d;
      d.col_ptr = small.take<int>((size_t)P.n + 1);
      d.rows = small.take<int>(nz);
      d.vals = small.take<float>(nz);
      d.row_ptr = small.take<int>((size_t)P.m + 1);
      d.cols = small.take<int>(nz);
      d.rvals = small.take<float>(nz);
      XCS_ARENA_OK(d.col_ptr && d.rows && d.vals && d.row_ptr && d.cols && d.rvals);
      // one scratch for every instance: the launches run in order on B->stream
      XCS_TRY(device_smv(B->stream, P.m, P.n, P.p, o->matrix_ensemble, o->seed, key_of(i), d,
                         smv_tmp, smv_tmp + 4 * (size_t)smv_m_max));
      xset(P.col_ptr, d.col_ptr);
      xset(P.rows, d.rows);
      xset(P.vals, d.vals);
      xset(P.row_ptr, d.row_ptr);
      xset(P.cols, d.cols);
      xset(P.rvals, d.rvals);
    } else {
      int *d_rows = small.take<int>(P.m);
      int *d_pos = small.take<int>(P.n);
      XCS_ARENA_OK(d_rows && d_pos);
      jobs.push_back(SubsetJob{P.n, P.m, o->seed, key_of(i), STREAM_DCT_ROWS, d_rows});
      xset(P.dct_rows, d_rows);
      xset(P.dct_pos, d_pos);
      float2 *tw = nullptr;
      for (auto &e : tw_cache)
        if (e.first == P.n) tw = e.second;
      if (!tw) {
        tw = small.take<float2>(2 * (size_t)P.n);
        XCS_ARENA_OK(tw);
        hipLaunchKernelGGL(dct_tables_kernel, dim3(std::min(4096, (P.n + 255) / 256)), dim3(256), 0,
                           B->stream, tw, P.n);
        HIP_TRY(hipGetLastError());
        tw_cache.push_back({P.n, tw});
      }
      xset(P.twiddle, tw);
    }
    B->hP[q] = P;
  }
#undef XCS_ARENA_OK
  // dct rows, planted supports and values, one workgroup per subset
  SubsetJob *dj;
  PlantJob *dp;
  XCS_TRY(B->alloc(&dj, jobs.size()));
  XCS_TRY(B->alloc(&dp, plants.size()));
  XCS_TRY(device_draws(B->stream, jobs, dj, plants, dp));
  // (B->hP holds the device pointers; hp[] is the pre-arena description)
  for (const XProblem &P : B->hP)
    if (P.ens == ENS_DCT)
      XCS_TRY(make_dct_pos(B->stream, (const int *)P.dct_rows, P.m, P.n, (int *)P.dct_pos));
  // host copies of the planted vectors for the results (queue order)
  B->x_true.assign((size_t)count, std::vector<float>());
  B->ks.assign((size_t)count, 0);
  for (int q = 0; q < count; q++) {
    B->x_true[q].resize((size_t)B->hP[q].n);
    B->ks[q] = B->hP[q].k;
    HIP_TRY(d2h(B->x_true[q].data(), xt_ptr[q], 4 * (size_t)B->hP[q].n, B->stream));
  }
#ifdef XCS_PHASE_TIMING
  XCS_TRY(B->alloc(&B->phase, 32));
  for (XProblem &P : B->hP) xset(P.phase_ticks, B->phase);
#endif
  XCS_TRY(B->alloc(&B->dP, (size_t)count));
  HIP_TRY(h2d(B->dP, B->hP.data(), sizeof(XProblem) * count, B->stream));
  // y = A x_true for every instance, one workgroup each
  const float **d_xt;
  const int **d_sp;
  XCS_TRY(B->alloc(&d_xt, (size_t)count));
  XCS_TRY(B->alloc(&d_sp, (size_t)count));
  HIP_TRY(h2d(d_xt, xt_ptr.data(), sizeof(void *) * count, B->stream));
  HIP_TRY(h2d(d_sp, sp_ptr.data(), sizeof(void *) * count, B->stream));
  const int ygrid = std::min(count, B->nteams);  // one team workspace per workgroup
  hipLaunchKernelGGL(make_y_batch_kernel, dim3(ygrid), dim3(B->block), 0, B->stream, B->dP, count,
                     B->dW, d_xt, d_sp);
  HIP_TRY(hipGetLastError());
  HIP_TRY(hipEventRecord(e1, B->stream));
  HIP_TRY(hipEventSynchronize(e1));
  HIP_TRY(hipEventElapsedTime(&B->gen_ms, e0, e1));
  (void)hipEventDestroy(e0);
  (void)hipEventDestroy(e1);
  if (smv_tmp) {
    int fl = 0;
    HIP_TRY(d2h(&fl, smv_tmp + 4 * (size_t)smv_m_max, sizeof(int), nullptr));
    if (fl) return set_err(XCS_EINVAL, SMV_FAIL);
  }
  return XCS_OK;
}

// Reset, then solve: the two launches of one batched solve, on B->stream.
// budget: iterations per instance in this launch.
static int batch_enqueue(xcs_batch *B, int budget, int c, int grid) {
  B->ran_c = c;
  B->ran_teams = grid / c;
  const int rgrid = (int)std::min<size_t>(4096, (B->xs_len + 255) / 256 + 1);
  hipLaunchKernelGGL(batch_reset_kernel, dim3(rgrid), dim3(256), 0, B->stream, B->xs, B->xs_len,
                     (int *)B->sts, sizeof(XState) / sizeof(int) * (size_t)B->count, B->queue,
                     B->bar, (size_t)BAR_WORDS * B->resident);
  HIP_TRY(hipGetLastError());
  const int *list = nullptr;
  void *args[] = {(void *)&B->dP, (void *)&B->count, (void *)&B->n_big, (void *)&B->queue,
                  (void *)&B->dW, (void *)&B->slots, (void *)&B->red, (void *)&B->bar,
                  (void *)&c, (void *)&budget, (void *)&list, (void *)&B->spin_limit};
  if (c > 1) {
    HIP_TRY(hipLaunchCooperativeKernel((const void *)solve_batch_kernel<true>, dim3(grid),
                                       dim3(B->block), args, 0, B->stream));
  } else {
    HIP_TRY(hipLaunchKernel((const void *)solve_batch_kernel<false>, dim3(grid),
                            dim3(B->block), args, 0, B->stream));
  }
  return XCS_OK;
}
static int batch_enqueue(xcs_batch *B, int budget) {
  return batch_enqueue(B, budget, B->c, B->grid);
}

// Single-workgroup teams: the reset and the persistent solve are captured
// once into a HIP graph and replayed.  Multi-workgroup teams need the
// cooperative launch (co-residency of a team's workgroups), which is issued
// directly.
static int batch_capture(xcs_batch *B) {
  B->drop_graph();
  if (B->c > 1) return XCS_OK;
  hipGraph_t g = nullptr;
  HIP_TRY(hipStreamBeginCapture(B->stream, hipStreamCaptureModeThreadLocal));
  const int rc = batch_enqueue(B, B->sched_budget.empty() ? B->budget : B->sched_budget[0]);
  const hipError_t e = hipStreamEndCapture(B->stream, &g);
  if (rc != XCS_OK) {
    if (g) (void)hipGraphDestroy(g);
    return rc;
  }
  if (e != hipSuccess) return set_err(XCS_EHIP, "hipStreamEndCapture: %s", hipGetErrorString(e));
  const hipError_t e2 = hipGraphInstantiate(&B->graph, g, nullptr, nullptr, 0);
  (void)hipGraphDestroy(g);
  if (e2 != hipSuccess) {
    B->graph = nullptr;
    return set_err(XCS_EHIP, "hipGraphInstantiate: %s", hipGetErrorString(e2));
  }
  return XCS_OK;
}

// A later phase of the tail schedule: the `cnt` instances at queue positions
// B->list[0, cnt) on teams of c workgroups (whole teams per XCD where they
// fit), at most `budget` more iterations each.  Cooperative launch for c > 1.
static int batch_enqueue_phase(xcs_batch *B, int cnt, int c, int budget) {
  c = std::max(1, std::min(c, std::min(B->resident, BAR_MAX_TEAM)));
  const int nteams = batch_teams(B->resident, cnt, c);
  const int grid = nteams * c, n_big = c > 1 ? cnt : 0;
  hipLaunchKernelGGL(batch_reset_kernel, dim3(64), dim3(256), 0, B->stream, B->xs, (size_t)0,
                     (int *)B->sts, (size_t)0, B->queue, B->bar, (size_t)BAR_WORDS * nteams);
  HIP_TRY(hipGetLastError());
  const int *list = B->list;
  void *args[] = {(void *)&B->dP, (void *)&cnt, (void *)&n_big, (void *)&B->queue, (void *)&B->dW,
                  (void *)&B->slots, (void *)&B->red, (void *)&B->bar, (void *)&c,
                  (void *)&budget, (void *)&list, (void *)&B->spin_limit};
  if (c > 1) {
    HIP_TRY(hipLaunchCooperativeKernel((const void *)solve_batch_kernel<true>, dim3(grid),
                                       dim3(B->block), args, 0, B->stream));
  } else {
    HIP_TRY(hipLaunchKernel((const void *)solve_batch_kernel<false>, dim3(grid), dim3(B->block),
                            args, 0, B->stream));
  }
  return XCS_OK;
}

// The solver states of queue slots [0, cnt) and whether a team's abort word (word
// 2 of its barrier words) is set, straight into pinned memory.
__global__ void __launch_bounds__(256) batch_back_kernel(const int *st, int words, const unsigned *bar,
                                                         int teams, int *out, int *aborted) {
  for (int i = blockIdx.x * 256 + threadIdx.x; i < words; i += gridDim.x * 256) out[i] = st[i];
  if (blockIdx.x == 0) {
    int bad = 0;
    for (int t = threadIdx.x; t < teams; t += 256) bad |= bar[(size_t)t * BAR_WORDS + 2] != 0u;
    bad = __syncthreads_or(bad);
    if (threadIdx.x == 0) *aborted = bad;
  }
}

// B->last of slots [0, cnt) after what the stream holds, in one launch and one
// synchronisation; an aborted team is an error.  (A strided copy of the abort words
// into pageable memory moved one word at a time: 5 ms for 512 teams.)
static int batch_states(xcs_batch *B, int cnt) {
  if (!B->back)
    HIP_TRY(hipHostMalloc((void **)&B->back, sizeof(XState) * (size_t)B->count + 64, hipHostMallocDefault));
  XState *st = (XState *)(B->back + 64);
  const int words = (int)(sizeof(XState) / sizeof(int)) * cnt;
  hipLaunchKernelGGL(batch_back_kernel, dim3(std::max(1, std::min(64, (words + 1023) / 1024))), dim3(256), 0,
                     B->stream, (const int *)B->sts, words, (const unsigned *)B->bar, B->resident, (int *)st,
                     (int *)B->back);
  HIP_TRY(hipGetLastError());
  HIP_TRY(hipStreamSynchronize(B->stream));
  std::copy(st, st + cnt, B->last.begin());
  if (*(int *)B->back) return set_err(XCS_EHIP, "team barrier timed out (results invalid)");
  return XCS_OK;
}

// The adaptive form of the tail schedule: one cooperative launch of every
// resident workgroup; level l of the schedule is phase l's team size and budget.
static int batch_run_adaptive(xcs_batch *B, float *ms) {
  const int levels = (int)B->sched_budget.size();
  SchedLevels lv{};
  lv.n = levels;
  for (int l = 0; l < levels; l++) {
    lv.c[l] = l ? std::max(1, std::min(B->sched_team[l], std::min(B->resident, BAR_MAX_TEAM))) : 1;
    lv.budget[l] = l + 1 == levels ? B->budget : B->sched_budget[l];
  }
  B->ran_c = 1;
  B->ran_teams = B->resident;
  lv.split_c = B->split_team >= 2 ? std::min(B->split_team, std::min(B->resident, BAR_MAX_TEAM)) : 0;
  // a partly formed team per level must never hold every workgroup
  const int chk = sched_levels_check(lv, B->resident);
  if (chk == -1)
    return set_err(XCS_EINVAL, "adaptive schedule: at most %d phases (%d with splitting)",
                   SCHED_MAX_LEVELS, SCHED_MAX_LEVELS - 1);
  if (chk != 0)
    return set_err(XCS_EINVAL, "adaptive schedule: the later phases' team sizes minus one (and the "
                               "split team's) must add up to fewer than the %d resident workgroups",
                   B->resident);
  if (!B->sw) {
    XCS_TRY(B->alloc(&B->sw, (size_t)SCHED_WORDS));
    XCS_TRY(B->alloc(&B->items, (size_t)SCHED_MAX_LEVELS * B->count));
    XCS_TRY(B->alloc(&B->leads, (size_t)SCHED_MAX_LEVELS * B->count));
  }
  hipEvent_t e0, e1;
  HIP_TRY(hipEventCreate(&e0));
  HIP_TRY(hipEventCreate(&e1));
  HIP_TRY(hipEventRecord(e0, B->stream));
  const int rgrid = (int)std::min<size_t>(4096, (B->xs_len + 255) / 256 + 1);
  hipLaunchKernelGGL(batch_reset_kernel, dim3(rgrid), dim3(256), 0, B->stream, B->xs, B->xs_len,
                     (int *)B->sts, sizeof(XState) / sizeof(int) * (size_t)B->count, B->queue,
                     B->bar, (size_t)BAR_WORDS * B->resident);
  HIP_TRY(hipGetLastError());
  hipLaunchKernelGGL(sched_reset_kernel, dim3(64), dim3(256), 0, B->stream, B->sw, B->items, B->leads,
                     B->count, levels + 1);
  HIP_TRY(hipGetLastError());
  void *args[] = {(void *)&B->dP, (void *)&B->count, (void *)&B->dW, (void *)&B->red,
                  (void *)&B->red_stride, (void *)&B->bar, (void *)&B->sw, (void *)&B->items,
                  (void *)&B->leads, (void *)&lv, (void *)&B->spin_limit};
  HIP_TRY(hipLaunchCooperativeKernel((const void *)solve_sched_kernel, dim3(B->resident),
                                     dim3(B->block), args, 0, B->stream));
  HIP_TRY(hipEventRecord(e1, B->stream));
  HIP_TRY(hipEventSynchronize(e1));
  HIP_TRY(hipEventElapsedTime(&B->last_ms, e0, e1));
  (void)hipEventDestroy(e0);
  (void)hipEventDestroy(e1);
  std::vector<int> sw((size_t)SCHED_WORDS);
  HIP_TRY(d2h(sw.data(), B->sw, sizeof(int) * sw.size(), B->stream));
  XCS_TRY(batch_states(B, B->count));
  if (sw[SW_ABORT * SCHED_LINE]) return set_err(XCS_EHIP, "scheduler wait timed out (results invalid)");
  B->phase_instances.assign(1, B->count);
  for (int l = 1; l < levels; l++) B->phase_instances.push_back(sw[(SW_TAIL + l) * SCHED_LINE]);
  B->phase_instances.push_back(lv.split_c >= 2 ? sw[(SW_TAIL + levels) * SCHED_LINE] : 0);
  if (ms) *ms = B->last_ms;
  return XCS_OK;
}

// Algorithmic bytes of one product of queue slot q's instance.
static double batch_bytes1(const xcs_batch *B, int q) {
  const XProblem &P = B->hP[q];
  return P.ens == ENS_GEN ? 4.0 * P.lda * (double)P.n : P.ens == ENS_SMV ? 8.0 * P.nz : 24.0 * P.n;
}

// The geometry of a solve on teams without a tail schedule.
static BatchPick batch_pick(const xcs_batch *B) {
  double most = 0.0, most1 = 0.0;
  for (int q = 0; q < B->n_big; q++) most = std::max(most, batch_bytes1(B, q));
  for (int q = B->n_big; q < B->count; q++) most1 = std::max(most1, batch_bytes1(B, q));
  return batch_pick(B->count, B->n_big, B->c, B->resident, BAR_MAX_TEAM, most, most1, !B->exact);
}
static bool batch_picks(const xcs_batch *B) { return B->c > 1 && B->sched_budget.empty() && B->n_big > 0; }

static int batch_run(xcs_batch *B, float *ms) {
  if (B->adaptive && B->c == 1 && B->sched_budget.size() >= 2) return batch_run_adaptive(B, ms);
  if (B->c == 1 && !B->graph) XCS_TRY(batch_capture(B));
  hipEvent_t e0, e1;
  HIP_TRY(hipEventCreate(&e0));
  HIP_TRY(hipEventCreate(&e1));
  HIP_TRY(hipEventRecord(e0, B->stream));
  if (B->graph) {
    HIP_TRY(hipGraphLaunch(B->graph, B->stream));
  } else if (batch_picks(B)) {
    const BatchPick p = batch_pick(B);
    XCS_TRY(batch_enqueue(B, B->budget, p.c, p.teams * p.c));
  } else {
    XCS_TRY(batch_enqueue(B, B->sched_budget.empty() ? B->budget : B->sched_budget[0]));
  }
  B->phase_instances.assign(1, B->count);
  // the tail schedule: the instances still running go to larger teams
  for (size_t ph = 1; ph < B->sched_budget.size(); ph++) {
    XCS_TRY(batch_states(B, B->count));
    std::vector<int> run;
    for (int q = 0; q < B->count; q++)
      if (!B->last[q].done) run.push_back(q);
    if (run.empty()) break;
    B->phase_instances.push_back((int)run.size());
    HIP_TRY(h2d(B->list, run.data(), sizeof(int) * run.size(), B->stream));
    const int budget = ph + 1 == B->sched_budget.size() ? B->budget : B->sched_budget[ph];
    XCS_TRY(batch_enqueue_phase(B, (int)run.size(), B->sched_team[ph], budget));
  }
  HIP_TRY(hipEventRecord(e1, B->stream));
  HIP_TRY(hipEventSynchronize(e1));
  HIP_TRY(hipEventElapsedTime(&B->last_ms, e0, e1));
  (void)hipEventDestroy(e0);
  (void)hipEventDestroy(e1);
  XCS_TRY(batch_states(B, B->count));
  if (ms) *ms = B->last_ms;
  return XCS_OK;
}

// ---------------------------------------------------------------- autotune --
// Candidate team geometries are timed on the batch itself with every
// instance capped at `probe_iters` iterations (0: full solves); the fastest
// is kept.  Results are cached in a text file, one line per batch signature:
//   <signature> <team_size> <block> <probe_ms>
static std::string batch_signature(const xcs_batch *B, int probe_iters) {
  std::vector<SigInstance> inst;
  inst.reserve(B->hP.size());
  for (const XProblem &P : B->hP) inst.push_back(SigInstance{P.ens, P.n, P.lda, P.nz});
  return batch_signature_text(B->alg, inst, probe_iters);
}

static int batch_tune(xcs_batch *B, int probe_iters, const char *cache_path, int verbose,
                      int *team_out, int *block_out, int *big_out, float *ms_out) {
  const std::string sig = batch_signature(B, probe_iters);
  if (cache_path && *cache_path) {
    FILE *f = fopen(cache_path, "r");
    if (f) {
      char key[1024];
      int c, b, big;
      float t;
      bool hit = false;
      while (fscanf(f, "%1023s %d %d %d %f", key, &c, &b, &big, &t) == 5)
        if (sig == key) {
          hit = true;
          *team_out = c;
          *block_out = b;
          *big_out = big;
          *ms_out = t;
        }
      fclose(f);
      if (hit) {
        XCS_TRY(batch_configure(B, *team_out, *block_out, *big_out));
        return XCS_OK;
      }
    }
  }
  const int saved_budget = B->budget;
  const int budget = probe_iters > 0 ? probe_iters : saved_budget;
  static const int blocks[] = {256, 512, 1024};
  static const int teams[] = {1, 2, 4, 8};
  // teams for every instance, or for the largest 1/16, 1/8, 1/4 only
  const int splits[] = {-1, B->count / 16, B->count / 8, B->count / 4};
  float best = 1e30f;
  int best_c = B->c, best_b = B->block, best_big = -1;
  // what the candidates so far ran as: where the chip has room for larger teams,
  // several of them come to the same launch, which is timed once
  std::vector<std::array<int, 4>> timed;
  for (int bi = 0; bi < 3; bi++)
    for (int ti = 0; ti < 4; ti++)
      for (int si = 0; si < 4; si++) {
        const int c = teams[ti], blk = blocks[bi], big = splits[si];
        if (c == 1 && si > 0) continue;
        if (c > 1 && si > 0 && big < 1) continue;
        int per_cu, cus;
        XCS_TRY(batch_occupancy(blk, &per_cu, &cus));
        if (c > 1 && per_cu * cus / c < 8) continue;
        XCS_TRY(batch_configure(B, c, blk, big));
        const BatchPick as = batch_picks(B) ? batch_pick(B) : BatchPick{B->c, B->nteams};
        const std::array<int, 4> key = {as.c, as.teams, blk, B->n_big};
        if (std::find(timed.begin(), timed.end(), key) != timed.end()) continue;
        timed.push_back(key);
        B->budget = budget;
        float ms = 0.f;
        const int rc = batch_run(B, &ms);
        B->budget = saved_budget;
        if (rc != XCS_OK) return rc;
        if (verbose) {
          fprintf(stderr, "tune: team %d (ran %d) block %4d team instances %5d: %9.2f ms\n", c, B->ran_c,
                  blk, B->n_big, ms);
          fflush(stderr);
        }
        if (ms < best) {
          best = ms;
          best_c = c;
          best_b = blk;
          best_big = big;
        }
      }
  B->budget = saved_budget;
  XCS_TRY(batch_configure(B, best_c, best_b, best_big));
  *team_out = best_c;
  *block_out = best_b;
  *big_out = best_big;
  *ms_out = best;
  if (cache_path && *cache_path) {
    FILE *f = fopen(cache_path, "a");
    if (f) {
      fprintf(f, "%s %d %d %d %.4f\n", sig.c_str(), best_c, best_b, best_big, best);
      fclose(f);
    }
  }
  return XCS_OK;
}

// ------------------------------------------------------------------ C ABI --
extern "C" {

const char *xcs_last_error(void) { return g_err.c_str(); }
const char *xcs_version(void) { return "gaga_amd 0.1 (gfx950)"; }

int xcs_options_default(const char *alg, const char *ens, int n, xcs_options *o) {
  if (!o) return set_err(XCS_EINVAL, "opts is NULL");
  const int a = parse_alg(alg), e = parse_ens(ens);
  if (a < 0) return set_err(XCS_EINVAL, "unknown algorithm '%s'", alg ? alg : "(null)");
  if (e < 0) return set_err(XCS_EINVAL, "ens must be either dct, gen, or smv.");
  memset(o, 0, sizeof(*o));
  o->tol = 1e-4f;  // the documented intent (gagaOptions.m); see tol_reference_default
  o->tol_reference_default = 0;
  o->maxiter = (a == ALG_HTP || a == ALG_CSMPSP) ? 300 : 5000;  // gaga_gen.cu:191-192
  o->num_bins = std::max(n / 20, 1000);                       // gaga_gen.cu:180
  o->restart = 0;
  o->seed = 0;
  o->instance = 0;
  o->vec_distribution = 1;                       // binary
  o->matrix_ensemble = e == ENS_SMV ? 3 : 1;     // smv default 'expander' (gaga_smv.cu:241)
  o->gpu_number = 0;
  o->mode = 0;
  o->team_size = 0;
  o->block_size = 0;
  o->proj_frac_tol = 3.0f;  // gaga_gen.cu:190, gaga_smv.cu:256, gaga_dct.cu:180
  o->timing = 0;            // gaga_gen.cu:185
  o->supp_flag = 0;         // gaga_gen.cu:187
  o->alpha = 0.25f;         // gaga_gen.cu:186
  o->barrier_spin_limit = 0;
  return XCS_OK;
}

int xcs_plan_create(const char *alg, const char *ens, int k, int m, int n, int p,
                    const xcs_options *opts, xcs_plan **out) {
  if (!out || !opts) return set_err(XCS_EINVAL, "NULL argument");
  *out = nullptr;
  xcs_plan *pl = new xcs_plan();
  int r = plan_generate(pl, parse_alg(alg), parse_ens(ens), k, m, n, p, opts);
  if (r != XCS_OK) {
    delete pl;
    return r;
  }
  *out = pl;
  return XCS_OK;
}

int xcs_plan_solve(xcs_plan *pl, float *ms) {
  if (!pl) return set_err(XCS_EINVAL, "NULL plan");
  HIP_TRY(hipSetDevice(pl->dev));
  return plan_run(pl, ms);
}

int xcs_plan_results(xcs_plan *pl, float norms[3], int *iterations, int support[4],
                     float *conv_rate, int *stop_reason, float *x_out, float *x_true) {
  if (!pl) return set_err(XCS_EINVAL, "NULL plan");
  HIP_TRY(hipSetDevice(pl->dev));
  const int n = pl->h.n;
  const bool x_pin = x_out && sizeof(float) * (size_t)n <= LANE_X;
  const bool planted = pl->xt_dev && (norms || support);
  if (x_pin || planted) {
    std::lock_guard<std::mutex> lock(pl->pin_mu);
    float *xh = x_pin ? (float *)pl->lane.pin : nullptr;
    NormPart *part = (NormPart *)(pl->lane.pin + LANE_X);
    const int wgs = norm_wgs(n);
    static_assert(LANE_X + NORM_WGS * sizeof(NormPart) <= LANE_BYTES, "staging memory");
    if (planted) {
      hipLaunchKernelGGL(norms_kernel, dim3(wgs), dim3(256), 0, pl->stream, (const float *)(float *)pl->h.x,
                         (const float *)pl->xt_dev, n, xh, part);
      HIP_TRY(hipGetLastError());
    } else {
      XferList L;
      L.add((float *)pl->h.x, xh, n);
      HIP_TRY(xfer(L, pl->stream));
    }
    HIP_TRY(hipStreamSynchronize(pl->stream));
    if (planted) norms_finish(part, wgs, n, pl->k_planted, norms, support);
    if (x_pin) memcpy(x_out, xh, sizeof(float) * (size_t)n);
  }
  if (x_out && !x_pin) HIP_TRY(d2h(x_out, pl->h.x, sizeof(float) * (size_t)n, pl->stream));
  if (iterations) *iterations = pl->last.iter;
  if (conv_rate) *conv_rate = conv_rate_results(pl->last);
  if (stop_reason) *stop_reason = pl->last.stop_reason;
  if (x_true && !pl->x_true.empty()) memcpy(x_true, pl->x_true.data(), sizeof(float) * n);
  return XCS_OK;
}

int xcs_plan_trace(xcs_plan *pl, int *k_bin, float *resid_norm, int len) {
  if (!pl) return set_err(XCS_EINVAL, "NULL plan");
  HIP_TRY(hipSetDevice(pl->dev));
  len = std::min(len, pl->h.maxiter + 2);
  if (k_bin) HIP_TRY(d2h(k_bin, pl->h.trace_kbin, sizeof(int) * len, nullptr));
  if (resid_norm)
    HIP_TRY(d2h(resid_norm, pl->h.trace_err, sizeof(float) * len, nullptr));
  return XCS_OK;
}

int xcs_plan_apply_timed(xcs_plan *pl, int transpose, int reps, float *ms_per, double *bytes) {
  if (!pl || reps <= 0 || !ms_per) return set_err(XCS_EINVAL, "bad arguments");
  HIP_TRY(hipSetDevice(pl->dev));
  XProblem &P = pl->h;
  // input: the planted product y (A^T y) or the planted vector's support (A x_S)
  const float *in = transpose ? (const float *)P.y : (const float *)P.thres;
  float *out = transpose ? (float *)P.grad : (float *)P.resid2;
  int cnt = 0;
  if (!transpose) {
    std::vector<int> supp;
    for (int j = 0; j < P.n; j++)
      if (!pl->x_true.empty() && pl->x_true[j] != 0.f) supp.push_back(j);
    cnt = (int)supp.size();
    HIP_TRY(h2d((void *)P.thres, pl->x_true.data(), sizeof(float) * P.n, pl->stream));
    if (cnt)
      HIP_TRY(h2d((void *)P.supp, supp.data(), sizeof(int) * cnt, pl->stream));
  }
  XCS_TRY(plan_upload_desc(pl));
  XCS_TRY(launch_apply(pl, transpose, in, out, cnt));  // warm-up
  hipEvent_t e0, e1;
  HIP_TRY(hipEventCreate(&e0));
  HIP_TRY(hipEventCreate(&e1));
  HIP_TRY(hipEventRecord(e0, pl->stream));
  for (int r = 0; r < reps; r++) XCS_TRY(launch_apply(pl, transpose, in, out, cnt));
  HIP_TRY(hipEventRecord(e1, pl->stream));
  HIP_TRY(hipEventSynchronize(e1));
  float ms = 0.f;
  HIP_TRY(hipEventElapsedTime(&ms, e0, e1));
  (void)hipEventDestroy(e0);
  (void)hipEventDestroy(e1);
  *ms_per = ms / reps;
  if (bytes) {
    const double m = P.m, n = P.n;
    if (P.ens == ENS_GEN)
      *bytes = transpose ? 4.0 * m * n + 4.0 * m + 4.0 * n : 4.0 * m * cnt + 8.0 * cnt + 4.0 * m;
    else if (P.ens == ENS_SMV)
      *bytes = 8.0 * P.nz + 4.0 * m + 4.0 * n;
    else
      *bytes = 4.0 * n + 8.0 * m;
  }
  return XCS_OK;
}

int xcs_plan_bytes(xcs_plan *pl, double *bytes) {
  if (!pl || !bytes) return set_err(XCS_EINVAL, "NULL argument");
  *bytes = pl->last.mat_bytes;
  return XCS_OK;
}

int xcs_plan_form(xcs_plan *pl, int *form, int *support_bits, int *rows_staged, int *columns_staged) {
  if (!pl) return set_err(XCS_EINVAL, "NULL plan");
  HIP_TRY(hipSetDevice(pl->dev));
  const XProblem &P = pl->h;
  int bits = 0, rows = 0, cols = 0;
  if (pl->form == FORM_SPLIT && P.ens == ENS_SMV && (support_bits || rows_staged || columns_staged)) {
    const SplitGeom G = split_geom(P.ens, P.alg, P.m, P.n, P.log2n, P.num_bins, pl->team);
    bits = G.filter;
    if (rows_staged || columns_staged) {
      std::vector<int> rp((size_t)P.m + 1), cp((size_t)P.n + 1);
      HIP_TRY(d2h(rp.data(), P.row_ptr, sizeof(int) * rp.size(), nullptr));
      HIP_TRY(d2h(cp.data(), P.col_ptr, sizeof(int) * cp.size(), nullptr));
      for (int w = 0; w < pl->team; w++) {
        const int j0 = (int)std::min<long>(P.n, (long)w * G.nl), i0 = (int)std::min<long>(P.m, (long)w * G.rl);
        const int nlv = std::min(G.nl, P.n - j0), rlv = std::min(G.rl, P.m - i0);
        const SplitStage T = split_stage(G, P.n, rlv, nlv, rp[i0 + rlv] - rp[i0], cp[j0 + nlv] - cp[j0]);
        rows += T.rows;
        cols += T.cols;
      }
    }
  }
  if (form) *form = pl->form;
  if (support_bits) *support_bits = bits;
  if (rows_staged) *rows_staged = rows;
  if (columns_staged) *columns_staged = cols;
  return XCS_OK;
}

int xcs_plan_geometry(xcs_plan *pl, int *team_size, int *block_size) {
  if (!pl || !team_size || !block_size) return set_err(XCS_EINVAL, "NULL argument");
  *team_size = pl->team;
  *block_size = pl->block;
  return XCS_OK;
}

void xcs_plan_destroy(xcs_plan *pl) { delete pl; }

// The per-solve results line of File_output (dct), File_output_smv and
// File_output_gen (GAGA/gaga/functions.cu:34-80): keys, order, separators and
// number formats as the reference prints them, so its processing scripts
// (CGIHTcode/code/process_{gen,smv,dct}_data.m, a whitespace textscan) read it
// unchanged.  smv prints band_percentage 0.00 (this build draws no banded
// supports) and noise_level 0.0000 (no noise), as the reference's noiseless
// path does (results.cu:350).
static int results_line(std::string &out, const char *alg, int ens, int k, int m, int n, int p,
                        int mat_ens, int vec_dist, const float *e, const float *t, int iters,
                        float rate, const int *sp, unsigned int seed) {
  const char *tag = ens == ENS_GEN ? "gen" : ens == ENS_SMV ? "smv" : "dct";
  char b[1024];
  int w = snprintf(b, sizeof(b), "%s_S_%s output: k %d, m %d, n %d, vecDistribution %d ", alg, tag,
                   k, m, n, vec_dist);
  if (ens == ENS_SMV)
    w += snprintf(b + w, sizeof(b) - w, "nonzeros_per_column %d matrixEnsemble %d ", p, mat_ens);
  else if (ens == ENS_GEN)
    w += snprintf(b + w, sizeof(b) - w, "matrixEnsemble %d ", mat_ens);
  w += snprintf(b + w, sizeof(b) - w,
                "errorl1 %0.7e errorl2 %0.7e errorlinf %0.7e timeALG %0.7e timeIter %0.7e "
                "timeTotal %0.7e iterations %d converge_rate %0.7e TruePos %d FalsePos %d "
                "TrueNeg %d FalseNeg %d ",
                e[0], e[1], e[2], t[0], t[1], t[2], iters, rate, sp[0], sp[1], sp[2], sp[3]);
  if (ens == ENS_SMV)
    w += snprintf(b + w, sizeof(b) - w, "seed %u band_percentage %1.2f noise_level %2.4f \n", seed,
                  0.0f, 0.0f);
  else
    w += snprintf(b + w, sizeof(b) - w, "seed %u \n", seed);
  if (w <= 0 || w >= (int)sizeof(b)) return set_err(XCS_EINVAL, "results line too long");
  out.assign(b, (size_t)w);
  return XCS_OK;
}

// The timing variants' results text (File_output_timings*, functions.cu:82-212):
// the line with alpha and supp_flag (smv: NonzerosPerCol and matrixEnsemble at its
// end, gen: matrixEnsemble), then one line per iteration (HTP adds its CG steps and
// CG time).
static int results_timing_text(std::string &out, const char *alg, int a, int ens, int k, int m,
                               int n, int p, int mat_ens, int vec_dist, const float *e,
                               const float *t, int iters, float rate, const int *sp,
                               unsigned int seed, float alpha, int supp_flag, const float *ti,
                               const float *ts, const int *cg, const float *tcg) {
  const char *tag = ens == ENS_GEN ? "gen" : ens == ENS_SMV ? "smv" : "dct";
  char b[1024];
  int w = snprintf(b, sizeof(b),
                   "%s_S_%s output: k %d, m %d, n %d, vecDistribution %d "
                   "errorl1 %0.7e errorl2 %0.7e errorlinf %0.7e timeALG %0.7e timeIter %0.7e "
                   "timeTotal %0.7e iterations %d converge_rate %0.7e TruePos %d FalsePos %d "
                   "TrueNeg %d FalseNeg %d seed %u alpha %0.7e ",
                   alg, tag, k, m, n, vec_dist, e[0], e[1], e[2], t[0], t[1], t[2], iters, rate,
                   sp[0], sp[1], sp[2], sp[3], seed, alpha);
  if (ens == ENS_SMV)
    w += snprintf(b + w, sizeof(b) - w, "supp_flag %d NonzerosPerCol %d matrixEnsemble %d \n",
                  supp_flag, p, mat_ens);
  else if (ens == ENS_GEN)
    w += snprintf(b + w, sizeof(b) - w, "supp_flag %d matrixEnsemble %d \n", supp_flag, mat_ens);
  else
    w += snprintf(b + w, sizeof(b) - w, "supp_flag %d \n", supp_flag);
  if (w <= 0 || w >= (int)sizeof(b)) return set_err(XCS_EINVAL, "results line too long");
  out.assign(b, (size_t)w);
  for (int j = 0; j < iters; j++) {
    char l[256];
    int lw;
    if (a == ALG_HTP)
      lw = snprintf(l, sizeof(l),
                    "iteration %d time_iteration %0.7e time_supp_set %0.7e cg_per_iteration %0.0f "
                    "time_for_cg %0.7e\n",
                    j, ti[j], ts[j], (float)cg[j], tcg[j]);
    else
      lw = snprintf(l, sizeof(l), "iteration %d time_iteration %0.7e time_supp_set %0.7e\n", j,
                    ti[j], ts[j]);
    out.append(l, (size_t)lw);
  }
  return XCS_OK;
}

static int timing_args_ok(int a, int iters, const float *ti, const float *ts, const int *cg,
                          const float *tcg) {
  if (a != ALG_NIHT && a != ALG_HTP) return set_err(XCS_EINVAL, "timing results exist for NIHT and HTP");
  if (iters < 0) return set_err(XCS_EINVAL, "iterations < 0");
  if (iters > 0 && (!ti || !ts || (a == ALG_HTP && (!cg || !tcg))))
    return set_err(XCS_EINVAL, "NULL per-iteration array");
  return XCS_OK;
}

int xcs_results_timing_text(char *buf, size_t buf_len, const char *alg, const char *ens, int k,
                            int m, int n, int p, int matrix_ensemble, int vec_distribution,
                            const float norms[3], const float times[3], int iterations,
                            float conv_rate, const int support[4], unsigned int seed, float alpha,
                            int supp_flag, const float *time_iteration, const float *time_supp_set,
                            const int *cg_per_iteration, const float *time_for_cg) {
  const int a = parse_alg(alg), e = parse_ens(ens);
  if (a < 0 || e < 0) return set_err(XCS_EINVAL, "unknown algorithm or ensemble");
  if (!buf || !norms || !times || !support) return set_err(XCS_EINVAL, "NULL argument");
  XCS_TRY(timing_args_ok(a, iterations, time_iteration, time_supp_set, cg_per_iteration, time_for_cg));
  std::string text;
  XCS_TRY(results_timing_text(text, alg, a, e, k, m, n, p, matrix_ensemble, vec_distribution, norms,
                              times, iterations, conv_rate, support, seed, alpha, supp_flag,
                              time_iteration, time_supp_set, cg_per_iteration, time_for_cg));
  if (text.size() + 1 > buf_len)
    return set_err(XCS_EINVAL, "buffer of %zu bytes holds no %zu-byte text", buf_len, text.size() + 1);
  memcpy(buf, text.c_str(), text.size() + 1);
  return (int)text.size();
}

int xcs_results_timing_append(const char *dir, const char *alg, const char *ens, int k, int m,
                              int n, int p, int matrix_ensemble, int vec_distribution,
                              const float norms[3], const float times[3], int iterations,
                              float conv_rate, const int support[4], unsigned int seed,
                              float alpha, int supp_flag, const float *time_iteration,
                              const float *time_supp_set, const int *cg_per_iteration,
                              const float *time_for_cg) {
  const int a = parse_alg(alg), e = parse_ens(ens);
  if (a < 0 || e < 0) return set_err(XCS_EINVAL, "unknown algorithm or ensemble");
  if (!norms || !times || !support) return set_err(XCS_EINVAL, "NULL argument");
  XCS_TRY(timing_args_ok(a, iterations, time_iteration, time_supp_set, cg_per_iteration, time_for_cg));
  std::string text;
  XCS_TRY(results_timing_text(text, alg, a, e, k, m, n, p, matrix_ensemble, vec_distribution, norms,
                              times, iterations, conv_rate, support, seed, alpha, supp_flag,
                              time_iteration, time_supp_set, cg_per_iteration, time_for_cg));
  // gpu_timings_data_<ens>YYYYMMDD.txt (results.cu:1540-1560 and twins)
  const time_t now = time(nullptr);
  struct tm tmv;
  localtime_r(&now, &tmv);
  char name[64];
  snprintf(name, sizeof(name), "gpu_timings_data_%s%d%02d%02d.txt", ens, tmv.tm_year + 1900,
           tmv.tm_mon + 1, tmv.tm_mday);
  std::string path = (dir && *dir) ? std::string(dir) + "/" + name : std::string(name);
  FILE *f = fopen(path.c_str(), "a+");
  if (!f) return set_err(XCS_EINVAL, "cannot open %s for appending", path.c_str());
  const bool ok = fputs(text.c_str(), f) >= 0;
  if (fclose(f) != 0 || !ok) return set_err(XCS_EINVAL, "cannot write %s", path.c_str());
  return XCS_OK;
}

int xcs_plan_times(xcs_plan *pl, float times[3]) {
  if (!pl || !times) return set_err(XCS_EINVAL, "NULL argument");
  // as xcs_cs_generate reports them: solve, solve per iteration, solve + generation (ms)
  times[0] = pl->last_ms;
  times[1] = pl->last.iter > 0 ? pl->last_ms / (float)pl->last.iter : 0.f;
  times[2] = pl->last_ms + pl->gen_ms;
  return XCS_OK;
}

int xcs_results_line(char *buf, size_t buf_len, const char *alg, const char *ens, int k, int m,
                     int n, int p, int matrix_ensemble, int vec_distribution, const float norms[3],
                     const float times[3], int iterations, float conv_rate, const int support[4],
                     unsigned int seed) {
  const int a = parse_alg(alg), e = parse_ens(ens);
  if (a < 0 || e < 0) return set_err(XCS_EINVAL, "unknown algorithm or ensemble");
  if (!buf || !norms || !times || !support) return set_err(XCS_EINVAL, "NULL argument");
  std::string line;
  XCS_TRY(results_line(line, alg, e, k, m, n, p, matrix_ensemble, vec_distribution, norms, times,
                       iterations, conv_rate, support, seed));
  if (line.size() + 1 > buf_len)
    return set_err(XCS_EINVAL, "buffer of %zu bytes holds no %zu-byte line", buf_len,
                   line.size() + 1);
  memcpy(buf, line.c_str(), line.size() + 1);
  return (int)line.size();
}

int xcs_results_append(const char *dir, const char *alg, const char *ens, int k, int m, int n,
                       int p, int matrix_ensemble, int vec_distribution, const float norms[3],
                       const float times[3], int iterations, float conv_rate,
                       const int support[4], unsigned int seed) {
  const int a = parse_alg(alg), e = parse_ens(ens);
  if (a < 0 || e < 0) return set_err(XCS_EINVAL, "unknown algorithm or ensemble");
  if (!norms || !times || !support) return set_err(XCS_EINVAL, "NULL argument");
  std::string line;
  XCS_TRY(results_line(line, alg, e, k, m, n, p, matrix_ensemble, vec_distribution, norms, times,
                       iterations, conv_rate, support, seed));
  // gpu_data_<ens>YYYYMMDD.txt from the local date (results.cu:509-525)
  const time_t now = time(nullptr);
  struct tm tmv;
  localtime_r(&now, &tmv);
  char name[64];
  snprintf(name, sizeof(name), "gpu_data_%s%d%02d%02d.txt", ens, tmv.tm_year + 1900,
           tmv.tm_mon + 1, tmv.tm_mday);
  std::string path = (dir && *dir) ? std::string(dir) + "/" + name : std::string(name);
  FILE *f = fopen(path.c_str(), "a+");
  if (!f) return set_err(XCS_EINVAL, "cannot open %s for appending", path.c_str());
  const bool ok = fputs(line.c_str(), f) >= 0;
  if (fclose(f) != 0 || !ok) return set_err(XCS_EINVAL, "cannot write %s", path.c_str());
  return XCS_OK;
}

int xcs_cs_generate(const char *alg, const char *ens, int k, int m, int n, int p,
                    const xcs_options *opts, float norms[3], float times[3], int *iterations,
                    int support[4], float *conv_rate, float *x_out, float *x_true) {
  xcs_options o;
  if (opts)
    o = *opts;
  else
    XCS_TRY(xcs_options_default(alg, ens, n, &o));
  xcs_plan *pl = nullptr;
  XCS_TRY(xcs_plan_create(alg, ens, k, m, n, p, &o, &pl));
  float ms = 0.f;
  int r = xcs_plan_solve(pl, &ms);
  if (r == XCS_OK)
    r = xcs_plan_results(pl, norms, iterations, support, conv_rate, nullptr, x_out, x_true);
  if (r == XCS_OK && times) {
    times[0] = ms;
    times[1] = pl->last.iter > 0 ? ms / (float)pl->last.iter : 0.f;
    times[2] = ms + pl->gen_ms;
  }
  xcs_plan_destroy(pl);
  return r;
}

// Shared tail of the solve-given-problem forms.
static int given_solve(xcs_plan *pl, const float *y, float *x_out, int *iterations,
                       float *conv_rate) {
  XProblem &P = pl->h;
  float *d_y;
  XCS_TRY(pl->alloc(&d_y, (size_t)P.lda));
  HIP_TRY(h2d(d_y, y, sizeof(float) * P.m, pl->stream));
  xset(P.y, d_y);
  XCS_TRY(plan_run(pl, nullptr, x_out));
  if (iterations) *iterations = pl->last.iter;
  if (conv_rate) *conv_rate = conv_rate_given(pl->last);
  return XCS_OK;
}

static int given_begin(xcs_plan *pl, int gpu) {
  XCS_TRY(use_device(gpu));
  return pl->open();
}

int xcs_cs_gen(const char *alg, const float *y, const float *A, int m, int n, int k,
               const xcs_options *opts, float *x_out, int *iterations, float *conv_rate) {
  const int a = parse_alg(alg);
  XCS_TRY(validate(a, ENS_GEN, k, m, n));
  if (!y || !A) return set_err(XCS_EINVAL, "NULL y or A");
  xcs_options o;
  if (opts)
    o = *opts;
  else
    XCS_TRY(xcs_options_default(alg, "gen", n, &o));
  xcs_plan pl;
  XCS_TRY(given_begin(&pl, o.gpu_number));
  XCS_TRY(plan_alloc(&pl, a, ENS_GEN, k, m, n, 0, 0, &o));
  float *dA;
  XCS_TRY(pl.alloc(&dA, (size_t)pl.h.lda * n));
  HIP_TRY(h2d_rows(dA, sizeof(float) * pl.h.lda, A, sizeof(float) * m, sizeof(float) * m, n, pl.stream));
  xset(pl.h.A, dA);
  return given_solve(&pl, y, x_out, iterations, conv_rate);
}

}  // extern "C"

// ------------------------------------------------------- allocation-free form --
// Scratch of the allocation-free gen solve (xcs_cs_gen_noalloc): one copy per GPU,
// held until the process ends.  Host code never uses the array's name as an
// address: it asks hipGetSymbolAddress for this device's copy once per device
// (noalloc_scratch) and passes that pointer to the kernels.
constexpr size_t NOALLOC_SCRATCH_BYTES = 4u << 20;
static __device__ __align__(256) unsigned char scratch[NOALLOC_SCRATCH_BYTES];

constexpr int NOALLOC_MAX_DEVICES = 64;
static std::mutex g_scratch_mu;
static void *g_scratch_ptr[NOALLOC_MAX_DEVICES];

// This device's copy of `scratch` (the device must be current).
static int noalloc_scratch(int dev, unsigned char **out) {
  if (dev < 0 || dev >= NOALLOC_MAX_DEVICES)
    return set_err(XCS_EINVAL, "device %d beyond the %d the allocation-free form tracks", dev,
                   NOALLOC_MAX_DEVICES);
  std::lock_guard<std::mutex> lock(g_scratch_mu);
  if (!g_scratch_ptr[dev]) {
    void *p = nullptr;
    HIP_TRY(hipGetSymbolAddress(&p, HIP_SYMBOL(scratch)));
    if (!p) return set_err(XCS_EHIP, "hipGetSymbolAddress(scratch) returned NULL");
    g_scratch_ptr[dev] = p;
  }
  *out = (unsigned char *)g_scratch_ptr[dev];
  return XCS_OK;
}

// The solver workspace of one gen instance carved out of the scratch buffer
// (256-byte aligned pieces).  Returns the bytes used, or 0 when it does not fit.
static size_t noalloc_layout(unsigned char *base, int n, int lda, int num_bins, XProblem &P,
                             float **y) {
  size_t off = 0;
  auto take = [&](size_t bytes) {
    unsigned char *p = base + off;
    off += (bytes + 255) / 256 * 256;
    return p;
  };
  const size_t fn = sizeof(float) * (size_t)n, in = sizeof(int) * (size_t)n;
  const size_t fm = sizeof(float) * (size_t)lda;
  *y = (float *)take(fm);
  xset(P.thres, (float *)take(fn));
  xset(P.grad, (float *)take(fn));
  xset(P.gprev, (float *)take(fn));
  xset(P.gprev_thres, (float *)take(fn));
  xset(P.bins, (int *)take(in));
  xset(P.bins2, (int *)take(in));
  xset(P.supp, (int *)take(in));
  xset(P.resid, (float *)take(fm));
  xset(P.resid_update, (float *)take(fm));
  xset(P.resid2, (float *)take(fm));
  xset(P.resid3, (float *)take(fm));
  xset(P.counters, (int *)take(sizeof(int) * ((size_t)num_bins + 64)));
  xset(P.wg_counts, (int *)take(sizeof(int) * 64));
  xset(P.partials, (float *)take(2 * (size_t)MAXCH * fm));
  xset(P.st, (XState *)take(sizeof(XState)));
  return off <= NOALLOC_SCRATCH_BYTES ? off : 0;
}

// y (zero padded to lda), x = 0 and a fresh solver state, in one kernel (no
// memset nodes, so the sequence can sit in a captured graph).
__global__ void noalloc_prep_kernel(const float *y_in, int m, int lda, float *y, float *x, int n,
                                    int *st, int st_words) {
  const int stride = gridDim.x * blockDim.x;
  for (int i = blockIdx.x * blockDim.x + threadIdx.x; i < lda; i += stride)
    y[i] = i < m ? y_in[i] : 0.f;
  for (int j = blockIdx.x * blockDim.x + threadIdx.x; j < n; j += stride) x[j] = 0.f;
  for (int w = blockIdx.x * blockDim.x + threadIdx.x; w < st_words; w += stride) st[w] = 0;
}

// One instance solved by one workgroup (the batched engine's single-workgroup
// form); the descriptor comes by value.
__global__ void __launch_bounds__(1024) solve_one_kernel(XProblem P, int budget) {
  __shared__ Lds L;
  __shared__ XProblem sP;
  if (threadIdx.x == 0) sP = P;
  __syncthreads();
  Team t{0, 1, nullptr, 0, nullptr};
  solve_instance(t, L, sP, budget);
}

extern "C" {

int xcs_cs_gen_noalloc(const char *alg, const float *d_y, const float *d_A, int lda, int m, int n,
                       int k, const xcs_options *opts, float *d_x_out, int *iterations,
                       float *conv_rate, void *stream) {
  const int a = parse_alg(alg);
  XCS_TRY(validate(a, ENS_GEN, k, m, n));
  if (a == ALG_CSMPSP) return set_err(XCS_EINVAL, CSMPSP_OFF);
  if (!d_y || !d_A || !d_x_out) return set_err(XCS_EINVAL, "NULL y, A or x_out");
  if (k > n) return set_err(XCS_EINVAL, "k must be <= n");
  if (lda < m || lda % 64)
    return set_err(XCS_EINVAL, "lda must be a multiple of 64 and >= m (lda = %d, m = %d)", lda, m);
  if (((uintptr_t)d_A | (uintptr_t)d_y | (uintptr_t)d_x_out) % 16)
    return set_err(XCS_EINVAL, "A, y and x_out must be 16-byte aligned device pointers");
  if (n > XCS_NOALLOC_MAX_N || lda > XCS_NOALLOC_MAX_LDA)
    return set_err(XCS_EINVAL, "the allocation-free form takes n <= %d and lda <= %d (n = %d, lda = %d)",
                   XCS_NOALLOC_MAX_N, XCS_NOALLOC_MAX_LDA, n, lda);
  xcs_options o;
  if (opts)
    o = *opts;
  else
    XCS_TRY(xcs_options_default(alg, "gen", n, &o));
  XProblem P{};
  P.alg = a;
  P.ens = ENS_GEN;
  P.m = m;
  P.n = n;
  P.k = k;
  P.lda = lda;
  P.num_bins = o.num_bins > 0 ? o.num_bins : std::max(n / 20, 1000);
  if (P.num_bins > XCS_NOALLOC_MAX_BINS)
    return set_err(XCS_EINVAL, "the allocation-free form takes numBins <= %d", XCS_NOALLOC_MAX_BINS);
  P.maxiter = o.maxiter > 0 ? o.maxiter : ((a == ALG_HTP) ? 300 : 5000);
  P.restart = o.restart;
  P.tol = o.tol_reference_default ? (float)(10 ^ (-4)) : o.tol;
  P.proj_frac_tol = o.proj_frac_tol > 0.f ? o.proj_frac_tol : 3.0f;
  XCS_TRY(timing_fields(P, a, k, &o));
  const int block = o.block_size > 0 ? o.block_size : 256;
  if (block % 64 || block > 1024) return set_err(XCS_EINVAL, "block_size must be a multiple of 64 <= 1024");
  XCS_TRY(use_device(o.gpu_number));
  int dev = 0;
  HIP_TRY(hipGetDevice(&dev));
  unsigned char *base = nullptr;
  XCS_TRY(noalloc_scratch(dev, &base));
  float *y = nullptr;
  if (!noalloc_layout(base, n, lda, P.num_bins, P, &y))
    return set_err(XCS_EINVAL, "the instance needs more than the %zu bytes of scratch",
                   NOALLOC_SCRATCH_BYTES);
  xset(P.A, d_A);
  xset(P.y, y);
  xset(P.x, d_x_out);
  hipStream_t st = (hipStream_t)stream;
  const int words = (int)(sizeof(XState) / sizeof(int));
  hipLaunchKernelGGL(noalloc_prep_kernel, dim3(std::min(64, (std::max(n, lda) + 255) / 256)),
                     dim3(256), 0, st, d_y, m, lda, y, d_x_out, n, (int *)(XState *)P.st, words);
  HIP_TRY(hipGetLastError());
  hipLaunchKernelGGL(solve_one_kernel, dim3(1), dim3(block), 0, st, P, P.maxiter + 4);
  HIP_TRY(hipGetLastError());
  if (iterations || conv_rate) {
    XState S;
    HIP_TRY(d2h(&S, (XState *)P.st, sizeof(XState), st));
    HIP_TRY(hipStreamSynchronize(st));
    if (iterations) *iterations = S.iter;
    if (conv_rate) *conv_rate = conv_rate_given(S);
  }
  return XCS_OK;
}

int xcs_cs_smv(const char *alg, const float *y, const int *rows, const int *cols,
               const float *vals, int nz, int m, int n, int k, const xcs_options *opts,
               float *x_out, int *iterations, float *conv_rate) {
  const int a = parse_alg(alg);
  XCS_TRY(validate(a, ENS_SMV, k, m, n));
  if (!y || !rows || !cols || !vals || nz <= 0) return set_err(XCS_EINVAL, "bad smv arrays");
  // 1-based triplets -> 0-based CSC sorted by (col, row)
  std::vector<int> cp((size_t)n + 1, 0), rr((size_t)nz);
  std::vector<float> vv((size_t)nz);
  for (int e = 0; e < nz; e++) {
    const int r = rows[e] - 1, c = cols[e] - 1;
    if (r < 0 || r >= m || c < 0 || c >= n)
      return set_err(XCS_EINVAL, "smv entry %d out of range (row %d, col %d)", e, rows[e], cols[e]);
    cp[c + 1]++;
  }
  for (int j = 0; j < n; j++) cp[j + 1] += cp[j];
  std::vector<int> order((size_t)nz);
  for (int e = 0; e < nz; e++) order[e] = e;
  std::stable_sort(order.begin(), order.end(), [&](int a_, int b_) {
    if (cols[a_] != cols[b_]) return cols[a_] < cols[b_];
    return rows[a_] < rows[b_];
  });
  for (int q = 0; q < nz; q++) {
    rr[q] = rows[order[q]] - 1;
    vv[q] = vals[order[q]];
  }
  xcs_options o;
  if (opts)
    o = *opts;
  else
    XCS_TRY(xcs_options_default(alg, "smv", n, &o));
  xcs_plan pl;
  XCS_TRY(given_begin(&pl, o.gpu_number));
  XCS_TRY(plan_alloc(&pl, a, ENS_SMV, k, m, n, 0, nz, &o));
  XCS_TRY(plan_set_smv(&pl, cp, rr, vv));
  return given_solve(&pl, y, x_out, iterations, conv_rate);
}

int xcs_cs_dct(const char *alg, const float *y, const int *rows, int k, int m, int n,
               const xcs_options *opts, float *x_out, int *iterations, float *conv_rate) {
  const int a = parse_alg(alg);
  XCS_TRY(validate(a, ENS_DCT, k, m, n));
  if (!y || !rows) return set_err(XCS_EINVAL, "NULL y or rows");
  std::vector<int> r0((size_t)m);
  std::vector<char> seen((size_t)n, 0);
  for (int i = 0; i < m; i++) {
    r0[i] = rows[i] - 1;
    if (r0[i] < 0 || r0[i] >= n) return set_err(XCS_EINVAL, "dct row %d out of range", rows[i]);
    if (seen[r0[i]]++) return set_err(XCS_EINVAL, "dct row %d given twice (rows must be distinct)", rows[i]);
  }
  xcs_options o;
  if (opts)
    o = *opts;
  else
    XCS_TRY(xcs_options_default(alg, "dct", n, &o));
  xcs_plan pl;
  XCS_TRY(given_begin(&pl, o.gpu_number));
  XCS_TRY(plan_alloc(&pl, a, ENS_DCT, k, m, n, 0, 0, &o));
  int *d_rows;
  XCS_TRY(pl.alloc(&d_rows, (size_t)m));
  HIP_TRY(h2d(d_rows, r0.data(), sizeof(int) * m, pl.stream));
  xset(pl.h.dct_rows, d_rows);
  XCS_TRY(make_dct_pos(pl.stream, d_rows, m, n, (int *)pl.h.dct_pos));
  return given_solve(&pl, y, x_out, iterations, conv_rate);
}

int xcs_find_support_set(const float *v, int n, int k, int num_bins, float slope, float intercept,
                         float max_change, float *min_val, float *alpha, int *max_bin, int *k_bin,
                         int *bins, int *sum) {
  if (!v || !min_val || !alpha || !max_bin || !k_bin || !bins || !sum || n <= 0 || num_bins <= 0)
    return set_err(XCS_EINVAL, "bad arguments");
  if (*max_bin > num_bins) return set_err(XCS_EINVAL, "max_bin > num_bins");
  xcs_options o;
  XCS_TRY(xcs_options_default("NIHT", "gen", n, &o));
  o.num_bins = num_bins;
  xcs_plan pl;
  XCS_TRY(given_begin(&pl, 0));
  XCS_TRY(plan_alloc(&pl, ALG_NIHT, ENS_GEN, k, 1, n, 0, 0, &o));
  float *dv;
  XCS_TRY(pl.alloc(&dv, (size_t)n));
  HIP_TRY(h2d(dv, v, sizeof(float) * n, pl.stream));
  XState S{};
  S.min_val = *min_val;
  S.max_change = max_change;
  S.alpha_bin = *alpha;
  S.max_bin = *max_bin;
  S.k_bin = *k_bin;
  HIP_TRY(h2d(pl.h.st, &S, sizeof(S), pl.stream));
  XCS_TRY(plan_upload_desc(&pl));
  void *args[] = {(void *)&pl.d, (void *)&dv, (void *)&pl.h.st, (void *)&slope,
                  (void *)&intercept, (void *)&pl.red, (void *)&pl.bar};
  HIP_TRY(hipLaunchCooperativeKernel((const void *)find_support_coop_kernel, dim3(pl.team),
                                     dim3(pl.block), args, 0, pl.stream));
  HIP_TRY(hipStreamSynchronize(pl.stream));
  HIP_TRY(d2h(&S, pl.h.st, sizeof(S), nullptr));
  *min_val = S.min_val;
  *alpha = S.alpha_bin;
  *max_bin = S.max_bin;
  *k_bin = S.k_bin;
  *sum = S.sum;
  if (S.sum >= 0) HIP_TRY(d2h(bins, pl.h.bins, sizeof(int) * n, nullptr));
  return XCS_OK;
}

int xcs_apply(const char *ens, int transpose, int m, int n, const float *A, const int *col_ptr,
              const int *rows, const float *vals, const int *dct_rows, const float *in,
              float *out) {
  const int e = parse_ens(ens);
  XCS_TRY(validate(ALG_NIHT, e, 0, m, n));
  if (!in || !out) return set_err(XCS_EINVAL, "NULL in/out");
  xcs_options o;
  XCS_TRY(xcs_options_default("NIHT", ens, n, &o));
  xcs_plan pl;
  XCS_TRY(given_begin(&pl, 0));
  int nz = 0;
  if (e == ENS_SMV) {
    if (!col_ptr || !rows || !vals) return set_err(XCS_EINVAL, "smv arrays required");
    nz = col_ptr[n];
  }
  XCS_TRY(plan_alloc(&pl, ALG_NIHT, e, 0, m, n, 0, nz, &o));
  XProblem &P = pl.h;
  if (e == ENS_GEN) {
    if (!A) return set_err(XCS_EINVAL, "A required");
    float *dA;
    XCS_TRY(pl.alloc(&dA, (size_t)P.lda * n));
    HIP_TRY(h2d_rows(dA, sizeof(float) * P.lda, A, sizeof(float) * m, sizeof(float) * m, n, pl.stream));
    xset(P.A, dA);
  } else if (e == ENS_SMV) {
    std::vector<int> cp(col_ptr, col_ptr + n + 1), rr(rows, rows + nz);
    std::vector<float> vv(vals, vals + nz);
    for (int q = 0; q < nz; q++)
      if (rr[q] < 0 || rr[q] >= m) return set_err(XCS_EINVAL, "smv row out of range");
    XCS_TRY(plan_set_smv(&pl, cp, rr, vv));
  } else {
    if (!dct_rows) return set_err(XCS_EINVAL, "dct rows required");
    std::vector<char> seen((size_t)n, 0);
    for (int i = 0; i < m; i++) {
      if (dct_rows[i] < 0 || dct_rows[i] >= n) return set_err(XCS_EINVAL, "dct row out of range");
      if (seen[dct_rows[i]]++) return set_err(XCS_EINVAL, "dct rows must be distinct");
    }
    int *dr;
    XCS_TRY(pl.alloc(&dr, (size_t)m));
    HIP_TRY(h2d(dr, dct_rows, sizeof(int) * m, pl.stream));
    xset(P.dct_rows, dr);
    XCS_TRY(make_dct_pos(pl.stream, dr, m, n, (int *)P.dct_pos));
  }
  const int lin = transpose ? m : n, lout = transpose ? n : m;
  float *din, *dout;
  XCS_TRY(pl.alloc(&din, (size_t)std::max(lin, P.lda)));
  XCS_TRY(pl.alloc(&dout, (size_t)std::max(lout, P.lda)));
  HIP_TRY(h2d(din, in, sizeof(float) * lin, pl.stream));
  int cnt = 0;
  if (!transpose) {
    std::vector<int> supp;
    for (int j = 0; j < n; j++)
      if (in[j] != 0.f) supp.push_back(j);
    cnt = (int)supp.size();
    if (cnt) HIP_TRY(h2d(P.supp, supp.data(), sizeof(int) * cnt, pl.stream));
  }
  XCS_TRY(plan_upload_desc(&pl));
  XCS_TRY(launch_apply(&pl, transpose, din, dout, cnt));
  HIP_TRY(hipStreamSynchronize(pl.stream));
  HIP_TRY(d2h(out, dout, sizeof(float) * lout, nullptr));
  return XCS_OK;
}

int xcs_generate_gen(int m, int n, unsigned int seed, unsigned int instance, float *A) {
  if (m <= 0 || n <= 0 || !A) return set_err(XCS_EINVAL, "bad arguments");
  XCS_TRY(use_device(0));
  xcs_plan pl;
  XCS_TRY(pl.open());
  float *dA;
  XCS_TRY(pl.alloc(&dA, (size_t)m * n));
  const size_t total = (size_t)m * n;
  const int blocks = (int)std::min<size_t>(65536, (total + 255) / 256);
  hipLaunchKernelGGL(gen_matrix_kernel, dim3(blocks), dim3(256), 0, pl.stream, dA, m, n, m, seed,
                     instance);
  HIP_TRY(hipGetLastError());
  HIP_TRY(hipStreamSynchronize(pl.stream));
  HIP_TRY(d2h(A, dA, sizeof(float) * total, nullptr));
  return XCS_OK;
}


int xcs_plan_timings(xcs_plan *pl, float *iter_ms, float *supp_ms, int *cg_iters, float *cg_ms,
                     int len) {
  if (!pl || len < 0) return set_err(XCS_EINVAL, "bad arguments");
  if (!pl->h.trace_ticks) return set_err(XCS_EINVAL, "the plan was not created with timing on (NIHT or HTP)");
  len = std::min(len, pl->h.maxiter + 2);
  HIP_TRY(hipSetDevice(pl->dev));
  std::vector<unsigned long long> t(4 * (size_t)len);
  if (len) HIP_TRY(d2h(t.data(), pl->h.trace_ticks, sizeof(unsigned long long) * t.size(), nullptr));
  int khz = 0;
  HIP_TRY(hipDeviceGetAttribute(&khz, hipDeviceAttributeWallClockRate, pl->dev));
  if (khz <= 0) return set_err(XCS_EHIP, "wall clock rate unavailable");
  const double per_ms = (double)khz;
  for (int i = 0; i < len; i++) {
    if (iter_ms) iter_ms[i] = (float)(t[4 * i + 0] / per_ms);
    if (supp_ms) supp_ms[i] = (float)(t[4 * i + 1] / per_ms);
    if (cg_iters) cg_iters[i] = (int)t[4 * i + 2];
    if (cg_ms) cg_ms[i] = (float)(t[4 * i + 3] / per_ms);
  }
  return XCS_OK;
}

int xcs_generate_smv(int m, int n, int p, int ens, unsigned int seed, unsigned int instance,
                     int *rows, float *vals, int *row_ptr, int *cols, float *rvals, int *empty) {
  if (!rows || !vals) return set_err(XCS_EINVAL, "NULL argument");
  XCS_TRY(smv_check(m, n, p, ens));
  XCS_TRY(use_device(0));
  xcs_plan pl;
  XCS_TRY(pl.open());
  const size_t nz = (size_t)n * p;
  SmvOut d;
  int *tmp;
  XCS_TRY(pl.alloc(&d.col_ptr, (size_t)n + 1));
  XCS_TRY(pl.alloc(&d.rows, nz));
  XCS_TRY(pl.alloc(&d.vals, nz));
  XCS_TRY(pl.alloc(&d.row_ptr, (size_t)m + 1));
  XCS_TRY(pl.alloc(&d.cols, nz));
  XCS_TRY(pl.alloc(&d.rvals, nz));
  XCS_TRY(pl.alloc(&tmp, 4 * (size_t)m + 2));
  XCS_TRY(device_smv(pl.stream, m, n, p, ens, seed, instance, d, tmp, tmp + 4 * (size_t)m));
  HIP_TRY(hipStreamSynchronize(pl.stream));
  int fl[2];
  HIP_TRY(d2h(fl, tmp + 4 * (size_t)m, sizeof(fl), nullptr));
  if (fl[0]) return set_err(XCS_EINVAL, SMV_FAIL);
  HIP_TRY(d2h(rows, d.rows, sizeof(int) * nz, nullptr));
  HIP_TRY(d2h(vals, d.vals, sizeof(float) * nz, nullptr));
  if (row_ptr) HIP_TRY(d2h(row_ptr, d.row_ptr, sizeof(int) * ((size_t)m + 1), nullptr));
  if (cols) HIP_TRY(d2h(cols, d.cols, sizeof(int) * nz, nullptr));
  if (rvals) HIP_TRY(d2h(rvals, d.rvals, sizeof(float) * nz, nullptr));
  if (empty) *empty = fl[1];
  return XCS_OK;
}

int xcs_batch_create(const char *alg, int count, const int *ens, const int *k, const int *m,
                     const int *n, const int *p, const unsigned int *instance,
                     const xcs_options *opts, xcs_batch **out) {
  if (!out || !opts || !ens || !k || !m || !n) return set_err(XCS_EINVAL, "NULL argument");
  *out = nullptr;
  xcs_batch *B = new xcs_batch();
  int r = batch_generate(B, parse_alg(alg), count, ens, k, m, n, p, instance, opts);
  if (r != XCS_OK) {
    delete B;
    return r;
  }
  *out = B;
  return XCS_OK;
}

int xcs_batch_solve(xcs_batch *B, float *ms) {
  if (!B) return set_err(XCS_EINVAL, "NULL batch");
  HIP_TRY(hipSetDevice(B->dev));
  ReadAhead::Writing writing(B->ahead);
  return batch_run(B, ms);
}

int xcs_batch_results(xcs_batch *B, float *norms, int *iterations, int *stop_reason,
                      float *conv_rate) {
  if (!B) return set_err(XCS_EINVAL, "NULL batch");
  HIP_TRY(hipSetDevice(B->dev));
  if (norms) {
    if (!B->xs_host) {
      const hipError_t e = hipHostMalloc((void **)&B->xs_host, sizeof(float) * B->xs_len, hipHostMallocDefault);
      if (e != hipSuccess) {
        B->xs_host = nullptr;
        return set_err(XCS_ENOMEM, "hipHostMalloc(%zu bytes): %s", sizeof(float) * B->xs_len,
                       hipGetErrorString(e));
      }
    }
    HIP_TRY(hipMemcpy(B->xs_host, B->xs, sizeof(float) * B->xs_len, hipMemcpyDeviceToHost));
    // instances are independent and each is one sequential loop, so the split
    // over threads does not change any value
    const float *xo = B->xs_host;
    host_parallel_for(B->count, [&](int q) {
      host_norms(B->x_true[q], xo + B->xoff[q], B->ks[q], norms + 3 * (size_t)B->order[q], nullptr);
    });
  }
  for (int q = 0; q < B->count; q++) {
    const int i = B->order[q];
    if (iterations) iterations[i] = B->last[q].iter;
    if (stop_reason) stop_reason[i] = B->last[q].stop_reason;
    if (conv_rate) conv_rate[i] = conv_rate_results(B->last[q]);
  }
  return XCS_OK;
}

int xcs_batch_x(xcs_batch *B, int idx, float *x_out, float *x_true) {
  if (!B || idx < 0 || idx >= B->count) return set_err(XCS_EINVAL, "bad batch index");
  HIP_TRY(hipSetDevice(B->dev));
  const int q = B->slot_of[idx];
  const XProblem &P = B->hP[q];
  float *const out[2] = {x_out, nullptr};
  auto piece = [B](int i, int, const float **src, long *n) {
    const int s = B->slot_of[i];
    *src = B->xs + B->xoff[s];
    *n = B->hP[s].n;
  };
  if (x_out && !B->ahead.read(idx, B->count, 1, piece, out, B->stream))
    HIP_TRY(d2h(x_out, B->xs + B->xoff[q], sizeof(float) * P.n, nullptr));
  if (x_true) memcpy(x_true, B->x_true[q].data(), sizeof(float) * P.n);
  return XCS_OK;
}

int xcs_batch_configure(xcs_batch *B, int team_size, int block_size, int big_count) {
  if (!B) return set_err(XCS_EINVAL, "NULL batch");
  HIP_TRY(hipSetDevice(B->dev));
  ReadAhead::Writing writing(B->ahead);
  return batch_configure(B, team_size, block_size, big_count);
}

int xcs_batch_schedule(xcs_batch *B, int phases, const int *team_sizes, const int *budgets) {
  if (!B) return set_err(XCS_EINVAL, "NULL batch");
  if (phases < 0 || phases == 1 || phases > 16 || (phases && (!team_sizes || !budgets)))
    return set_err(XCS_EINVAL, "a tail schedule has 0 or 2..16 phases");
  for (int p = 0; p + 1 < phases; p++)
    if (budgets[p] < 1) return set_err(XCS_EINVAL, "phase budgets must be >= 1");
  for (int p = 1; p < phases; p++)
    if (team_sizes[p] < 1) return set_err(XCS_EINVAL, "phase team sizes must be >= 1");
  if (B->alg == ALG_CSMPSP) return set_err(XCS_EINVAL, CSMPSP_OFF);
  HIP_TRY(hipSetDevice(B->dev));
  ReadAhead::Writing writing(B->ahead);
  HIP_TRY(hipStreamSynchronize(B->stream));
  B->drop_graph();
  B->sched_team.assign(team_sizes, team_sizes + phases);
  B->sched_budget.assign(budgets, budgets + phases);
  return XCS_OK;
}

#ifdef XCS_SCHED_TRACE
// Instrumented builds only: the adaptive schedule's job records of the last solve
// (7 x 8-byte-aligned fields each, as SchedTraceRec); *n = records written.
extern "C" int xcs_sched_trace_read(void *out, int max, int *n) {
  int cnt = 0;
  HIP_TRY(hipDeviceSynchronize());
  HIP_TRY(hipMemcpyFromSymbol(&cnt, HIP_SYMBOL(sched_trace_count), sizeof(int)));
  cnt = std::min(cnt, std::min(max, SCHED_TRACE_MAX));
  if (cnt > 0)
    HIP_TRY(hipMemcpyFromSymbol(out, HIP_SYMBOL(sched_trace_buf), sizeof(SchedTraceRec) * cnt));
  *n = cnt;
  return XCS_OK;
}
#endif

int xcs_batch_schedule_mode(xcs_batch *B, int adaptive, int split_team) {
  if (!B) return set_err(XCS_EINVAL, "NULL batch");
  if (adaptive != 0 && adaptive != 1) return set_err(XCS_EINVAL, "mode must be 0 or 1");
  if (split_team < 0 || split_team > BAR_MAX_TEAM)
    return set_err(XCS_EINVAL, "split_team must be in [0, %d]", BAR_MAX_TEAM);
  HIP_TRY(hipSetDevice(B->dev));
  ReadAhead::Writing writing(B->ahead);
  HIP_TRY(hipStreamSynchronize(B->stream));
  B->drop_graph();
  B->adaptive = adaptive != 0;
  B->split_team = split_team;
  return XCS_OK;
}

int xcs_batch_phase_counts(xcs_batch *B, int *counts, int phases) {
  if (!B || !counts || phases < 0) return set_err(XCS_EINVAL, "bad arguments");
  for (int p = 0; p < phases; p++)
    counts[p] = p < (int)B->phase_instances.size() ? B->phase_instances[p] : 0;
  return XCS_OK;
}

int xcs_batch_tune(xcs_batch *B, int probe_iters, const char *cache_path, int verbose,
                   int *team_size, int *block_size, int *big_count, float *probe_ms) {
  if (!B || !team_size || !block_size || !big_count || !probe_ms)
    return set_err(XCS_EINVAL, "NULL argument");
  if (probe_iters < 0) return set_err(XCS_EINVAL, "probe_iters must be >= 0");
  HIP_TRY(hipSetDevice(B->dev));
  ReadAhead::Writing writing(B->ahead);
  return batch_tune(B, probe_iters, cache_path, verbose, team_size, block_size, big_count,
                    probe_ms);
}

int xcs_batch_info(xcs_batch *B, int *teams, int *team_size, int *block, float *gen_ms) {
  if (!B) return set_err(XCS_EINVAL, "NULL batch");
  if (teams) *teams = B->nteams;
  if (team_size) *team_size = B->c;
  if (block) *block = B->block;
  if (gen_ms) *gen_ms = B->gen_ms;
  return XCS_OK;
}

int xcs_batch_ran(xcs_batch *B, int *teams, int *team_size) {
  if (!B) return set_err(XCS_EINVAL, "NULL batch");
  if (!B->ran_c) return set_err(XCS_EINVAL, "the batch has not been solved");
  if (teams) *teams = B->ran_teams;
  if (team_size) *team_size = B->ran_c;
  return XCS_OK;
}

int xcs_batch_exact(xcs_batch *B, int exact) {
  if (!B) return set_err(XCS_EINVAL, "NULL batch");
  B->exact = exact != 0;
  return XCS_OK;
}

int xcs_batch_apply_timed(xcs_batch *B, int reps, float *ms_per, double *bytes) {
  if (!B || reps <= 0 || !ms_per) return set_err(XCS_EINVAL, "bad arguments");
  HIP_TRY(hipSetDevice(B->dev));
  ReadAhead::Writing writing(B->ahead);
  int per_cu, cus;
  XCS_TRY(batch_occupancy(B->block, &per_cu, &cus));
  const int grid = std::min(B->count, B->nteams);  // works[] has one entry per team
  hipEvent_t e0, e1;
  HIP_TRY(hipEventCreate(&e0));
  HIP_TRY(hipEventCreate(&e1));
  hipLaunchKernelGGL(apply_batch_kernel, dim3(grid), dim3(B->block), 0, B->stream, B->dP, B->count, B->dW);
  HIP_TRY(hipGetLastError());
  HIP_TRY(hipEventRecord(e0, B->stream));
  for (int r = 0; r < reps; r++)
    hipLaunchKernelGGL(apply_batch_kernel, dim3(grid), dim3(B->block), 0, B->stream, B->dP, B->count, B->dW);
  HIP_TRY(hipGetLastError());
  HIP_TRY(hipEventRecord(e1, B->stream));
  HIP_TRY(hipEventSynchronize(e1));
  float ms = 0.f;
  HIP_TRY(hipEventElapsedTime(&ms, e0, e1));
  (void)hipEventDestroy(e0);
  (void)hipEventDestroy(e1);
  *ms_per = ms / reps;
  if (bytes) {
    double s = 0.0;
    for (const XProblem &P : B->hP) {
      const double m = P.m, n = P.n;
      s += P.ens == ENS_GEN ? 4.0 * m * n + 4.0 * m + 4.0 * n
           : P.ens == ENS_SMV ? 8.0 * P.nz + 4.0 * m + 4.0 * n : 4.0 * n + 8.0 * m;
    }
    *bytes = s;
  }
  return XCS_OK;
}

int xcs_batch_bytes(xcs_batch *B, double *bytes) {
  if (!B || !bytes) return set_err(XCS_EINVAL, "NULL argument");
  double s = 0.0;
  for (const XState &S : B->last) s += S.mat_bytes;
  *bytes = s;
  return XCS_OK;
}

void xcs_batch_destroy(xcs_batch *B) { delete B; }

// Phase tick counters of the instrumented build (zeros otherwise).
int xcs_batch_phase_ticks(xcs_batch *B, unsigned long long *out32) {
  if (!B || !out32) return set_err(XCS_EINVAL, "NULL argument");
  memset(out32, 0, 32 * sizeof(unsigned long long));
  if (B->phase)
    HIP_TRY(d2h(out32, B->phase, 32 * sizeof(unsigned long long), nullptr));
  return XCS_OK;
}

}  // extern "C"

// ------------------------------------------------------------ calibration --
// Plain streaming copy of known size (float4 loads and stores): the reference
// point for reading HBM traffic counters (FETCH_SIZE, WRITE_SIZE).
__global__ void stream_copy_kernel(const float4 *in, float4 *out, long n4) {
  for (long e = (long)blockIdx.x * blockDim.x + threadIdx.x; e < n4;
       e += (long)gridDim.x * blockDim.x)
    out[e] = in[e];
}

// Streaming read: every block sums its share of float4s (non-temporal loads,
// four in flight per lane) and writes one value, so nothing is optimised away.
__global__ void __launch_bounds__(1024) stream_read_kernel(const float4 *in, long n4, float *out) {
  float acc = 0.f;
  const long stride = (long)gridDim.x * blockDim.x;
  long e = (long)blockIdx.x * blockDim.x + threadIdx.x;
  for (; e + 3 * stride < n4; e += 4 * stride) {
    float4 v[4];
#pragma unroll
    for (int u = 0; u < 4; u++) v[u] = load_nt((XG(const float4))(in + e + u * stride));
#pragma unroll
    for (int u = 0; u < 4; u++) acc += (v[u].x + v[u].y) + (v[u].z + v[u].w);
  }
  for (; e < n4; e += stride) {
    const float4 v = in[e];
    acc += (v.x + v.y) + (v.z + v.w);
  }
  acc = wave_sum(acc);
  __shared__ float part[MAX_WAVES];
  if ((threadIdx.x & (WAVE - 1)) == 0) part[threadIdx.x / WAVE] = acc;
  __syncthreads();
  if (threadIdx.x == 0) {
    float s = 0.f;
    for (int w = 0; w < (int)blockDim.x / WAVE; w++) s += part[w];
    out[blockIdx.x] = s;
  }
}

extern "C" int xcs_stream_read(long bytes, int reps, float *ms_per) {
  if (bytes <= 0 || bytes % 16 || reps <= 0 || !ms_per) return set_err(XCS_EINVAL, "bad arguments");
  XCS_TRY(use_device(0));
  int dev = 0, cus = 0;
  HIP_TRY(hipGetDevice(&dev));
  HIP_TRY(hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev));
  const int grid = 2 * cus;
  void *a = nullptr, *o = nullptr;
  HIP_TRY(dev_malloc(&a, (size_t)bytes));
  hipError_t e = hipMalloc(&o, sizeof(float) * grid);
  if (e != hipSuccess) {
    (void)hipFree(a);
    return set_err(XCS_ENOMEM, "hipMalloc: %s", hipGetErrorString(e));
  }
  (void)hipMemset(a, 0, (size_t)bytes);
  hipEvent_t e0, e1;
  (void)hipEventCreate(&e0);
  (void)hipEventCreate(&e1);
  const long n4 = bytes / 16;
  hipLaunchKernelGGL(stream_read_kernel, dim3(grid), dim3(1024), 0, 0, (const float4 *)a, n4, (float *)o);
  (void)hipEventRecord(e0, 0);
  for (int r = 0; r < reps; r++)
    hipLaunchKernelGGL(stream_read_kernel, dim3(grid), dim3(1024), 0, 0, (const float4 *)a, n4, (float *)o);
  (void)hipEventRecord(e1, 0);
  e = hipEventSynchronize(e1);
  float ms = 0.f;
  (void)hipEventElapsedTime(&ms, e0, e1);
  (void)hipEventDestroy(e0);
  (void)hipEventDestroy(e1);
  (void)hipFree(a);
  (void)hipFree(o);
  if (e != hipSuccess) return set_err(XCS_EHIP, "read: %s", hipGetErrorString(e));
  *ms_per = ms / reps;
  return XCS_OK;
}

extern "C" int xcs_stream_copy(long bytes, int reps, float *ms_per) {
  if (bytes <= 0 || bytes % 16 || reps <= 0 || !ms_per) return set_err(XCS_EINVAL, "bad arguments");
  XCS_TRY(use_device(0));
  void *a = nullptr, *b = nullptr;
  HIP_TRY(dev_malloc(&a, (size_t)bytes));
  hipError_t e = dev_malloc(&b, (size_t)bytes);
  if (e != hipSuccess) {
    (void)hipFree(a);
    return set_err(XCS_ENOMEM, "hipMalloc: %s", hipGetErrorString(e));
  }
  (void)hipMemset(a, 0, (size_t)bytes);
  hipEvent_t e0, e1;
  (void)hipEventCreate(&e0);
  (void)hipEventCreate(&e1);
  const long n4 = bytes / 16;
  hipLaunchKernelGGL(stream_copy_kernel, dim3(4096), dim3(256), 0, 0, (const float4 *)a, (float4 *)b, n4);
  (void)hipEventRecord(e0, 0);
  for (int r = 0; r < reps; r++)
    hipLaunchKernelGGL(stream_copy_kernel, dim3(4096), dim3(256), 0, 0, (const float4 *)a, (float4 *)b, n4);
  (void)hipEventRecord(e1, 0);
  e = hipEventSynchronize(e1);
  float ms = 0.f;
  (void)hipEventElapsedTime(&ms, e0, e1);
  (void)hipEventDestroy(e0);
  (void)hipEventDestroy(e1);
  (void)hipFree(a);
  (void)hipFree(b);
  if (e != hipSuccess) return set_err(XCS_EHIP, "copy: %s", hipGetErrorString(e));
  *ms_per = ms / reps;
  return XCS_OK;
}

// --------------------------------------------------- many right-hand sides --
#include "xcs_mfma.h"
#include "xcs_mrhs.h"
#include "xcs_mlp.h"
