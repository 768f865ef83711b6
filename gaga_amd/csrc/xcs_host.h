// Host side of a call: streams with staging memory that calls share, small
// transfers in one launch, and the read-back of many solution vectors.
#pragma once
#include "xcs_readahead.h"

// ------------------------------------------------------------------ copies --
// Up to XFER_MAX pieces of floats copied by one launch, either way between
// device memory and pinned host memory.  Bounded by the link and the launch
// (about 10 us with its synchronisation on MI355X), where each hipMemcpy of the
// same sizes takes 11-17 us; a piece whose two ends are 16-byte aligned moves as
// float4.
constexpr int XFER_MAX = 128;
struct XferList {
  int cnt = 0;
  struct Piece {
    const float *src;
    float *dst;
    long n;
  } p[XFER_MAX];
  void add(const void *src, void *dst, long n) { p[cnt++] = Piece{(const float *)src, (float *)dst, n}; }
};

__global__ void __launch_bounds__(256) xfer_kernel(XferList L) {
  const float *src = L.p[blockIdx.y].src;
  float *dst = L.p[blockIdx.y].dst;
  const long n = L.p[blockIdx.y].n;
  const long t = (long)blockIdx.x * 256 + threadIdx.x, stride = (long)gridDim.x * 256;
  long done = 0;
  if (!(((uintptr_t)src | (uintptr_t)dst) & 15)) {
    const long q = n >> 2;
    for (long i = t; i < q; i += stride)
      reinterpret_cast<float4 *>(dst)[i] = reinterpret_cast<const float4 *>(src)[i];
    done = q << 2;
  }
  for (long i = done + t; i < n; i += stride) dst[i] = src[i];
}

// Enqueue the list (at least one piece) on `st`.
static hipError_t xfer(const XferList &L, hipStream_t st) {
  long most = 0;
  for (int i = 0; i < L.cnt; i++) most = std::max(most, L.p[i].n);
  // 1024 floats a workgroup and pass, about 256 workgroups in all
  const long want = std::max(1L, std::min((most + 1023) / 1024, (long)(256 + L.cnt - 1) / L.cnt));
  hipLaunchKernelGGL(xfer_kernel, dim3((unsigned)want, (unsigned)L.cnt), dim3(256), 0, st, L);
  return hipGetLastError();
}

// ------------------------------------------------------------------- lanes --
// What one plan (or one given-problem call) needs of the runtime: a stream, two
// timing events and pinned memory for its state and small solution vectors.
// Creating and destroying the stream alone takes about 70 us on MI355X and the
// pinned block as long again, of a given-problem call that solves in 250; so an idle lane
// goes back to a pool, at most LANES_IDLE of them, and a lane beyond those is
// destroyed.  A lane belongs to one plan at a time and is idle on the device
// when it comes back.
constexpr int LANES_IDLE = 4;
constexpr size_t LANE_X = (size_t)256 << 10, LANE_BYTES = LANE_X + (16 << 10);
struct HostLane {
  int dev = -1;
  hipStream_t stream = nullptr;
  hipEvent_t e0 = nullptr, e1 = nullptr;
  char *pin = nullptr;
  void destroy() {
    if (e0) (void)hipEventDestroy(e0);
    if (e1) (void)hipEventDestroy(e1);
    if (pin) (void)hipHostFree(pin);
    if (stream) (void)hipStreamDestroy(stream);
    *this = HostLane{};
  }
};
static std::mutex g_lane_mu;
static HostLane g_lanes[LANES_IDLE];

// A lane of the current device.
static int lane_get(HostLane *out) {
  int dev = 0;
  HIP_TRY(hipGetDevice(&dev));
  {
    std::lock_guard<std::mutex> lock(g_lane_mu);
    for (HostLane &l : g_lanes)
      if (l.stream && l.dev == dev) {
        *out = l;
        l = HostLane{};
        return XCS_OK;
      }
  }
  HostLane l;
  l.dev = dev;
  hipError_t e = hipStreamCreateWithFlags(&l.stream, hipStreamNonBlocking);
  if (e == hipSuccess) e = hipEventCreate(&l.e0);
  if (e == hipSuccess) e = hipEventCreate(&l.e1);
  if (e == hipSuccess) e = hipHostMalloc((void **)&l.pin, LANE_BYTES, hipHostMallocDefault);
  if (e != hipSuccess) {
    l.destroy();
    return set_err(XCS_EHIP, "stream, events or staging memory: %s", hipGetErrorString(e));
  }
  *out = l;
  return XCS_OK;
}

// Give a lane back.  A lane whose stream reports an error is not used again.
static void lane_put(HostLane *l) {
  if (!l->stream) return;
  if (hipStreamSynchronize(l->stream) == hipSuccess) {
    std::lock_guard<std::mutex> lock(g_lane_mu);
    for (HostLane &q : g_lanes)
      if (!q.stream) {
        q = *l;
        *l = HostLane{};
        return;
      }
  }
  l->destroy();
}

// ----------------------------------------------------------- solution norms --
// x (n floats) to `xh` where given, and this workgroup's share of the sums that
// the relative errors and the support counts are made of: l1, l2 squared and
// maximum of xt and of xt - x in 64 bits, true positives and true negatives.
// The workgroups' shares are added on the host in their order, so the values
// do not depend on timing.  On MI355X n = 2^20: one thread of the host 1.5 ms
// (a chain of 64-bit additions), this launch about 20 us.
constexpr int NORM_WGS = 64;
struct NormPart {
  double a1, a2, ai, d1, d2, di;
  int tp, tn, pad[2];
};
static_assert(sizeof(NormPart) == 64, "one line per workgroup");

__global__ void __launch_bounds__(256) norms_kernel(const float *x, const float *xt, int n, float *xh,
                                                    NormPart *part) {
  double a1 = 0, a2 = 0, ai = 0, d1 = 0, d2 = 0, di = 0;
  int tp = 0, tn = 0;
  for (int i = blockIdx.x * 256 + threadIdx.x; i < n; i += gridDim.x * 256) {
    const float xf = x[i], tf = xt[i];
    const double t = tf, o = xf, df = t - o;
    if (xh) xh[i] = xf;
    a1 += fabs(t);
    a2 += t * t;
    ai = ai < fabs(t) ? fabs(t) : ai;
    d1 += fabs(df);
    d2 += df * df;
    di = di < fabs(df) ? fabs(df) : di;
    if (t != 0.0) {
      if (o != 0.0) tp++;
    } else if (o == 0.0) {
      tn++;
    }
  }
  for (int s = 32; s; s >>= 1) {
    a1 += __shfl_xor(a1, s);
    a2 += __shfl_xor(a2, s);
    d1 += __shfl_xor(d1, s);
    d2 += __shfl_xor(d2, s);
    const double u = __shfl_xor(ai, s), v = __shfl_xor(di, s);
    ai = ai < u ? u : ai;
    di = di < v ? v : di;
    tp += __shfl_xor(tp, s);
    tn += __shfl_xor(tn, s);
  }
  __shared__ NormPart w[4];
  if ((threadIdx.x & 63) == 0) w[threadIdx.x >> 6] = NormPart{a1, a2, ai, d1, d2, di, tp, tn, {0, 0}};
  __syncthreads();
  if (threadIdx.x) return;
  NormPart r = w[0];
  for (int q = 1; q < 4; q++) {
    r.a1 += w[q].a1;
    r.a2 += w[q].a2;
    r.d1 += w[q].d1;
    r.d2 += w[q].d2;
    r.ai = r.ai < w[q].ai ? w[q].ai : r.ai;
    r.di = r.di < w[q].di ? w[q].di : r.di;
    r.tp += w[q].tp;
    r.tn += w[q].tn;
  }
  part[blockIdx.x] = r;
}

static int norm_wgs(int n) { return std::max(1, std::min(NORM_WGS, (n + 2047) / 2048)); }

static void norms_finish(const NormPart *p, int cnt, int n, int k, float norms[3], int support[4]) {
  NormPart r = p[0];
  for (int q = 1; q < cnt; q++) {
    r.a1 += p[q].a1;
    r.a2 += p[q].a2;
    r.d1 += p[q].d1;
    r.d2 += p[q].d2;
    r.ai = std::max(r.ai, p[q].ai);
    r.di = std::max(r.di, p[q].di);
    r.tp += p[q].tp;
    r.tn += p[q].tn;
  }
  if (norms) {
    norms[0] = (float)(r.d1 / r.a1);
    norms[1] = (float)(sqrt(r.d2) / sqrt(r.a2));
    norms[2] = (float)(r.di / r.ai);
  }
  if (support) {
    support[0] = r.tp;
    support[1] = k - r.tp;
    support[2] = r.tn;
    support[3] = n - k - r.tn;
  }
}

// -------------------------------------------------------------- read ahead --
// The window's memory and transfers (xcs_readahead.h) on a stream.
static float *pinned_alloc(size_t bytes) {
  void *p = nullptr;
  if (hipHostMalloc(&p, bytes, hipHostMallocDefault) == hipSuccess) return (float *)p;
  (void)hipGetLastError();
  return nullptr;
}
static void pinned_free(float *p) { (void)hipHostFree(p); }
struct PinnedReadAhead : ReadAhead {
  PinnedReadAhead() : ReadAhead(pinned_alloc, pinned_free) {}
  // Row i of `count` rows: see ReadAhead::get.
  template <class F>
  bool read(int i, int count, int pieces, F piece, float *const out[2], hipStream_t st) {
    static_assert(2 * READ_ROWS <= XFER_MAX, "one launch a window");
    XferList L;
    return get(
        i, count, pieces, piece, out, [&](const float *src, float *dst, long n) { L.add(src, dst, n); },
        [&] { return xfer(L, st) == hipSuccess && hipStreamSynchronize(st) == hipSuccess; });
  }
};
