// One dense (gen) instance on a team of workgroups with the solver's n-vectors
// resident in every workgroup's LDS: NIHT, HTP and CGIHT.
//
// What bounded the single instance before was not the matrix but the team
// barriers: the general solver (xcs_solver.h) splits every n-vector over the
// team, so an iteration crosses about twelve barriers and reductions of 4.5 to
// 6 us each (the agent-scope fences that write back and invalidate the L2s
// among them) around 15-20 us of matrix streaming.  Here every workgroup keeps
// all of x, the gradient and the direction in its LDS and repeats the cheap n-vector
// work (updates, binning, the k-bin walk, the support list) for itself, so only
// the two matrix products are split and three exchanges per iteration remain:
//   1. the residual rows (each workgroup forms A x_S for its own rows, all
//      support columns, so no partial sums cross workgroups) with |r|^2;
//   2. the gradient entries (each wave forms A^T r for its own columns);
//   3. |A d|^2 of the step direction (each workgroup its own rows).
// An exchange is one hop (rt_allreduce below) and moves its vector with
// device-scope stores and loads that go past the L2s, so it needs no fence.
// HTP's CG steps live on the support: A^T reads the support's columns only and
// a step takes two exchanges.
// Measured on MI355X: CGIHT 2048 x 8192 (15 iterations) 1.70 -> 0.55 ms, 37 us an
// iteration, of which A^T r takes 7.4 and the exchanges 12; NIHT 256 x 1024 0.9 -> 0.25
// ms; HTP 1001 x 5003 1.65 -> 0.34 ms (plan_resident has the team sizes).
//
// The arithmetic is that of the general solver except for the order of sums.
#pragma once
#include "xcs_solver.h"

namespace xcs {

constexpr int RES_LDS = 144 * 1024;  // bytes of LDS for the vectors below (of 160 KB per CU)
constexpr int RES_TCAP = 256;        // rows of A x a workgroup can own
constexpr int RES_QB = 4;            // float4 row groups of one gather block (at most)

__host__ __device__ inline size_t res_up16(size_t b) { return (b + 15) & ~(size_t)15; }
// LDS bytes of an instance: x, g, p, r, histogram, two masks, support list.
__host__ __device__ inline size_t res_lds_bytes(int n, int lda, int num_bins) {
  return 3 * res_up16(4 * (size_t)n) + res_up16(4 * (size_t)lda) + res_up16(4 * (size_t)num_bins) +
         2 * res_up16(8 * ((size_t)n / 64 + 1)) + res_up16(2 * (size_t)n);
}
// Whether the resident form can take an instance.  n < 65536: list entries are
// 16 bits wide.
inline bool res_fits(int alg, int ens, int n, int lda, int num_bins, int timing, int team) {
  return ens == ENS_GEN && (alg == ALG_NIHT || alg == ALG_HTP || alg == ALG_CGIHT) && !timing &&
         team > 1 && n < 65536 && lda <= RES_TCAP * team &&
         res_lds_bytes(n, lda, num_bins) <= (size_t)RES_LDS;
}

// ------------------------------------------------------ wave reductions ----
// Cross-lane sums and maxima by DPP moves (a few cycles a step where a shuffle
// through the LDS crossbar takes ~100); the result is read from lane 63 into a
// scalar register, so it is uniform for the compiler too.
template <int CTRL, int ROWS>
__device__ __forceinline__ int dpp_i(int v) {
  return __builtin_amdgcn_update_dpp(0, v, CTRL, ROWS, 0xf, false);
}
template <int CTRL, int ROWS>
__device__ __forceinline__ float dpp_f(float v) {
  return __int_as_float(dpp_i<CTRL, ROWS>(__float_as_int(v)));
}
template <int CTRL, int ROWS>
__device__ __forceinline__ double dpp_d(double v) {
  const unsigned long long b = (unsigned long long)__double_as_longlong(v);
  const unsigned lo = (unsigned)dpp_i<CTRL, ROWS>((int)(unsigned)b);
  const unsigned hi = (unsigned)dpp_i<CTRL, ROWS>((int)(unsigned)(b >> 32));
  return __longlong_as_double((long long)(((unsigned long long)hi << 32) | lo));
}
__device__ __forceinline__ double lane_d(double v, int l) {
  const unsigned long long b = (unsigned long long)__double_as_longlong(v);
  const unsigned lo = (unsigned)__builtin_amdgcn_readlane((int)(unsigned)b, l);
  const unsigned hi = (unsigned)__builtin_amdgcn_readlane((int)(unsigned)(b >> 32), l);
  return __longlong_as_double((long long)(((unsigned long long)hi << 32) | lo));
}
__device__ __forceinline__ float lane_f(float v, int l) {
  return __int_as_float(__builtin_amdgcn_readlane(__float_as_int(v), l));
}
// Lanes that a step does not reach add 0 (update_dpp's old value).
constexpr int DPP_SHR1 = 0x111, DPP_SHR2 = 0x112, DPP_SHR4 = 0x114, DPP_SHR8 = 0x118;
constexpr int DPP_ROR4 = 0x124, DPP_ROR8 = 0x128, DPP_ROR1 = 0x121, DPP_ROR2 = 0x122;
constexpr int DPP_BCAST15 = 0x142, DPP_BCAST31 = 0x143;
__device__ __forceinline__ double wsum_d(double v) {
  v += dpp_d<DPP_SHR1, 0xf>(v);
  v += dpp_d<DPP_SHR2, 0xf>(v);
  v += dpp_d<DPP_SHR4, 0xf>(v);
  v += dpp_d<DPP_SHR8, 0xf>(v);
  v += dpp_d<DPP_BCAST15, 0xa>(v);
  v += dpp_d<DPP_BCAST31, 0xc>(v);
  return lane_d(v, 63);
}
// Maximum of non-negative values (0 is the identity).
__device__ __forceinline__ double wmax_d(double v) {
  v = fmax(v, dpp_d<DPP_SHR1, 0xf>(v));
  v = fmax(v, dpp_d<DPP_SHR2, 0xf>(v));
  v = fmax(v, dpp_d<DPP_SHR4, 0xf>(v));
  v = fmax(v, dpp_d<DPP_SHR8, 0xf>(v));
  v = fmax(v, dpp_d<DPP_BCAST15, 0xa>(v));
  v = fmax(v, dpp_d<DPP_BCAST31, 0xc>(v));
  return lane_d(v, 63);
}
__device__ __forceinline__ float wsum_f(float v) {
  v += dpp_f<DPP_SHR1, 0xf>(v);
  v += dpp_f<DPP_SHR2, 0xf>(v);
  v += dpp_f<DPP_SHR4, 0xf>(v);
  v += dpp_f<DPP_SHR8, 0xf>(v);
  v += dpp_f<DPP_BCAST15, 0xa>(v);
  v += dpp_f<DPP_BCAST31, 0xc>(v);
  return lane_f(v, 63);
}
__device__ __forceinline__ float wmax_f(float v) {
  v = fmaxf(v, dpp_f<DPP_SHR1, 0xf>(v));
  v = fmaxf(v, dpp_f<DPP_SHR2, 0xf>(v));
  v = fmaxf(v, dpp_f<DPP_SHR4, 0xf>(v));
  v = fmaxf(v, dpp_f<DPP_SHR8, 0xf>(v));
  v = fmaxf(v, dpp_f<DPP_BCAST15, 0xa>(v));
  v = fmaxf(v, dpp_f<DPP_BCAST31, 0xc>(v));
  return lane_f(v, 63);
}
// Inclusive prefix sums over the lanes.
__device__ __forceinline__ int wscan_i(int v) {
  v += dpp_i<DPP_SHR1, 0xf>(v);
  v += dpp_i<DPP_SHR2, 0xf>(v);
  v += dpp_i<DPP_SHR4, 0xf>(v);
  v += dpp_i<DPP_SHR8, 0xf>(v);
  v += dpp_i<DPP_BCAST15, 0xa>(v);
  v += dpp_i<DPP_BCAST31, 0xc>(v);
  return v;
}

// Workgroup sums of ND doubles and maxima of NM non-negative floats, the same
// bits in every thread (and, on the same data, in every workgroup).  One
// __syncthreads: consecutive calls alternate between two banks of LDS slots,
// and a bank is written again only after the barrier of the call between.
struct WgSlots {
  double d[2][3][MAX_WAVES];
  float m[2][2][MAX_WAVES];
};
template <int ND, int NM>
__device__ __forceinline__ void wg_reduce(WgSlots &W, int &bank, double (&d)[ND ? ND : 1],
                                          float (&m)[NM ? NM : 1]) {
  const int lane = threadIdx.x & (WAVE - 1), wave = threadIdx.x / WAVE;
  const int nw = blockDim.x / WAVE;
  bank ^= 1;
#pragma unroll
  for (int k = 0; k < ND; k++) {
    const double s = wsum_d(d[k]);
    if (lane == 0) W.d[bank][k][wave] = s;
  }
#pragma unroll
  for (int k = 0; k < NM; k++) {
    const float s = wmax_f(m[k]);
    if (lane == 0) W.m[bank][k][wave] = s;
  }
  __syncthreads();
#pragma unroll
  for (int k = 0; k < ND; k++) d[k] = wsum_d(lane < nw ? W.d[bank][k][lane] : 0.0);
#pragma unroll
  for (int k = 0; k < NM; k++) m[k] = wmax_f(lane < nw ? W.m[bank][k][lane] : 0.f);
}

// ------------------------------------------------------------- exchange ----
__device__ __forceinline__ void st_dev(XG(float) p, float v) {
  __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ float ld_dev(XG(const float) p) {
  return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
// src (16-byte aligned, len floats) to LDS, read past the L2s, 8 bytes a load,
// four loads in flight per thread.
__device__ __forceinline__ void ld_dev_vec(float *dst, XG(const float) src, int len) {
  XG(const unsigned long long) s8 = reinterpret_cast<XG(const unsigned long long)>(src);
  unsigned long long *d8 = reinterpret_cast<unsigned long long *>(dst);
  const int h = len >> 1, nt = blockDim.x;
  for (int e0 = threadIdx.x; e0 < h; e0 += 4 * nt) {
    unsigned long long v[4];
#pragma unroll
    for (int u = 0; u < 4; u++)
      if (e0 + u * nt < h)
        v[u] = __hip_atomic_load(s8 + e0 + u * nt, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
#pragma unroll
    for (int u = 0; u < 4; u++)
      if (e0 + u * nt < h) d8[e0 + u * nt] = v[u];
  }
  if ((len & 1) && threadIdx.x == 0) dst[len - 1] = ld_dev(src + len - 1);
}

// The team's words (BAR_WORDS of a plan, zero before its first launch): word 1
// the tag of the last exchange (launch to launch), word 2 the abort flag, from
// word BAR_LINE on two banks of tagged 64-bit words, [word][rank].
struct RTeam {
  int rank, size;
  unsigned *bar;
  unsigned tag;
  long spin_limit;
  int aborted;
};
constexpr int RT_KMAX = 4;  // doubles per exchange
static_assert(BAR_LINE + 2 * (2 * (2 * RT_KMAX) * BAR_MAX_TEAM) <= BAR_WORDS, "exchange words");
struct RtSlots {
  double part[RT_KMAX][MAX_WAVES];
  double out[RT_KMAX];
  int bad;
};

// Barrier over the team that sums K doubles (one partial per thread; double k is
// maximised instead where bit k of MAXES is set, non-negative values): one hop.
// Every wave first waits for its own device-scope stores (vmcnt), so what the
// workgroup published before the call has arrived when its words do.  Each
// workgroup posts its partials as 64-bit words of tag and half a double (one
// word with the tag alone for K = 0); wave 0 of every workgroup polls all words
// of all workgroups until they carry the tag and adds them in a fixed order, so
// all workgroups hold the same bits.  A word and its tag arrive together, so no
// fence orders them.  Two banks by the tag's parity: a workgroup posts tag
// t + 2 only after every workgroup has read tag t.  Measured: 2.5 / 2.9 / 3.4 us
// at 64 / 128 / 256 workgroups, against 2.8 / 3.8 / 5.7 for the two-hop flag
// barrier with its fences (4.5-6 us in a solve).  Waits are bounded as in
// team_barrier.
template <int K, int MAXES = 0>
__device__ __forceinline__ void rt_allreduce(RTeam &t, RtSlots &X, const double (&v)[K ? K : 1],
                                             double (&out)[K ? K : 1]) {
  constexpr int KK = K ? K : 1, W = K ? 2 * K : 1;
  const int lane = threadIdx.x & (WAVE - 1), wave = threadIdx.x / WAVE;
  const int nw = blockDim.x / WAVE;
#pragma unroll
  for (int k = 0; k < KK; k++) out[k] = 0.0;
  if (t.aborted) return;  // uniform
  if (K) {
#pragma unroll
    for (int k = 0; k < K; k++) {
      const double s = (MAXES >> k & 1) ? wmax_d(v[k]) : wsum_d(v[k]);
      if (lane == 0) X.part[k][wave] = s;
    }
  }
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
  __syncthreads();
  t.tag++;
  if (wave == 0) {
    const unsigned long long T = (unsigned long long)t.tag << 32;
    unsigned long long *bank = reinterpret_cast<unsigned long long *>(t.bar + BAR_LINE) +
                               (size_t)(t.tag & 1u) * (2 * RT_KMAX) * BAR_MAX_TEAM;
    unsigned long long mine = T;
    if (K) {
#pragma unroll
      for (int k = 0; k < K; k++) {
        const double part = lane < nw ? X.part[k][lane] : 0.0;
        const double s = (MAXES >> k & 1) ? wmax_d(part) : wsum_d(part);
        const unsigned long long b = (unsigned long long)__double_as_longlong(s);
        if ((lane >> 1) == k) mine = T | ((lane & 1) ? (b >> 32) : (b & 0xFFFFFFFFull));
      }
    }
    if (lane < W)
      __hip_atomic_store(&bank[(size_t)lane * t.size + t.rank], mine, __ATOMIC_RELAXED,
                         __HIP_MEMORY_SCOPE_AGENT);
    double acc[KK];
#pragma unroll
    for (int k = 0; k < KK; k++) acc[k] = 0.0;
    int bad = 0;
    for (int r0 = 0; r0 < t.size && !bad; r0 += WAVE) {
      const int r = r0 + lane;
      unsigned long long w[W];
      long spins = 0;
      while (true) {
        bool ok = true;
#pragma unroll
        for (int q = 0; q < W; q++) {
          w[q] = T;
          if (r < t.size)
            w[q] = __hip_atomic_load(&bank[(size_t)q * t.size + r], __ATOMIC_RELAXED,
                                     __HIP_MEMORY_SCOPE_AGENT);
          ok = ok && (unsigned)(w[q] >> 32) == t.tag;
        }
        if (__all(ok)) break;
        if (++spins > t.spin_limit ||
            ((spins & 1023) == 0 &&
             __hip_atomic_load(&t.bar[2], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) != 0u)) {
          bad = 1;  // wave-uniform: the count, and one word read by the whole wave
          break;
        }
      }
      if (K && !bad && r < t.size) {
#pragma unroll
        for (int k = 0; k < K; k++) {
          const double b = __longlong_as_double(
              (long long)((w[(2 * k + 1) % W] << 32) | (w[(2 * k) % W] & 0xFFFFFFFFull)));
          acc[k] = (MAXES >> k & 1) ? fmax(acc[k], b) : acc[k] + b;
        }
      }
    }
    if (K) {
#pragma unroll
      for (int k = 0; k < K; k++) {
        const double s = (MAXES >> k & 1) ? wmax_d(acc[k]) : wsum_d(acc[k]);
        if (lane == 0) X.out[k] = s;
      }
    }
    if (lane == 0) {
      X.bad = bad;
      if (bad) __hip_atomic_store(&t.bar[2], 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    }
  }
  __syncthreads();
  if (K) {
#pragma unroll
    for (int k = 0; k < K; k++) out[k] = X.out[k];
  }
  if (X.bad) t.aborted = 1;  // uniform in the workgroup
}

// ------------------------------------------------------------ the state ----
// The residual history of the stop rules is kept with entry i in lane i < 16 of
// every wave (each wave keeps its own copy: pushes and the rules are a few DPP
// moves and ballots, uniform, without barriers).
__device__ __forceinline__ float hist_push(float h, float v) {
  const int lane = threadIdx.x & (WAVE - 1);
  const float nx = __shfl_down(h, 1);
  return lane < 15 ? nx : v;
}
// max16 of the entries, as the reference's scan takes it (they are finite when
// the rules are asked: a NaN residual ends the solve by itself).
__device__ __forceinline__ float hist_max(float h) {
  const int lane = threadIdx.x & (WAVE - 1);
  float v = lane < 16 ? h : lane_f(h, 0);
#pragma unroll
  for (int o = 1; o < 16; o <<= 1) v = fmaxf(v, __shfl_xor(v, o));
  return lane_f(v, 0);
}

// LDS views of a resident solve.
struct Res {
  float *x, *g, *p, *r;
  int *hist;
  unsigned long long *mask, *mask2;  // support bits now, and scratch for the next
  unsigned short *list;              // support, ascending
  float (*tile)[RES_TCAP];           // this workgroup's rows of the last products
  float (*wsum)[4 * RES_QB];         // per 16-lane row of each wave: a gather block's sums
  WgSlots *slots;
  RtSlots *rt;
  int bank;
  int cnt;         // support size
  int row0, rows;  // this workgroup's rows of A x
};
// Team-uniform scalars (registers).
struct ResS {
  int k_bin, sum, max_bin, beta_to_zero, supp_change;
  float alpha_bin, min_val, max_change, max_value, slope, mu;
  double bytes;
};

// Rows of A x per workgroup: whole float4 groups.  Workgroups are dealt to the
// 8 XCDs round robin, so rank w and w + 8 share an L2: they get adjacent tiles,
// whose columns share 128-byte lines when a tile is narrower than a line.
__device__ __forceinline__ void res_rows(int rank, int size, int lda, int *row0, int *rows) {
  const int T = ((lda + size - 1) / size + 3) / 4 * 4;
  int tile = rank;
  if (size % 16 == 0) {
    const int q = rank >> 3, xcd = rank & 7;
    tile = (q & 1) + 2 * (xcd + 8 * (q >> 1));
  }
  *row0 = min(lda, tile * T);
  *rows = min(T, lda - *row0);
}

template <int CTRL>
__device__ __forceinline__ void add_ror(float4 &a) {
  a.x += dpp_f<CTRL, 0xf>(a.x);
  a.y += dpp_f<CTRL, 0xf>(a.y);
  a.z += dpp_f<CTRL, 0xf>(a.z);
  a.w += dpp_f<CTRL, 0xf>(a.w);
}
// Sum of the lanes with equal lane % qb within each row of 16 lanes.
__device__ __forceinline__ void row_fold(float4 &a, int qb) {
  if (qb <= 8) add_ror<DPP_ROR8>(a);
  if (qb <= 4) add_ror<DPP_ROR4>(a);
  if (qb <= 2) add_ror<DPP_ROR2>(a);
  if (qb <= 1) add_ror<DPP_ROR1>(a);
}
__device__ __forceinline__ void fma4(float4 &c, const float4 &a, float w) {
  c.x = fmaf(a.x, w, c.x);
  c.y = fmaf(a.y, w, c.y);
  c.z = fmaf(a.z, w, c.z);
  c.w = fmaf(a.w, w, c.w);
}

// tile[v0 ...] = rows [row0, row0 + rows) of A u for the support columns (two
// vectors u0, u1 for NV = 2), u indexed by column in LDS.  Lanes take qb float4
// row groups of as many columns as fit, four columns in flight per lane; a
// lane's columns are summed in ascending order, then its row of 16 lanes, then
// the rows in order.  The support is small (about k) or, with Gaussian signals,
// now and then most of n: both are read here in one pass without partial sums
// in memory.  Starts after and ends with __syncthreads.
template <int NV>
__device__ __forceinline__ void res_gather(Res &R, XG(const float) A, int lda, const float *u0,
                                           const float *u1) {
  const int nq = R.rows >> 2, lq = lda >> 2;
  int qb = 1;
  while (qb < nq && qb < RES_QB) qb *= 2;
  const int lane = threadIdx.x & (WAVE - 1);
  const int nrow = blockDim.x / 16, row = threadIdx.x / 16;
  const int slots = blockDim.x / qb, slot = threadIdx.x / qb;
  constexpr int U = 4;
  for (int q0 = 0; q0 < nq; q0 += qb) {
    const int q = q0 + (lane & (qb - 1));
    float4 a0 = make_float4(0.f, 0.f, 0.f, 0.f), a1 = a0;
    if (q < nq) {
      XG(const float4) base = reinterpret_cast<XG(const float4)>(A + R.row0) + q;
      for (int s = slot; s < R.cnt; s += U * slots) {
        float4 a[U];
        float w0[U], w1[U];
#pragma unroll
        for (int u = 0; u < U; u++) {
          const bool ok = s + u * slots < R.cnt;
          const int j = R.list[ok ? s + u * slots : s];
          a[u] = base[(size_t)j * lq];
          w0[u] = ok ? u0[j] : 0.f;
          if (NV == 2) w1[u] = ok ? u1[j] : 0.f;
        }
#pragma unroll
        for (int u = 0; u < U; u++) {
          fma4(a0, a[u], w0[u]);
          if (NV == 2) fma4(a1, a[u], w1[u]);
        }
      }
    }
    row_fold(a0, qb);
    if (NV == 2) row_fold(a1, qb);
    if ((lane & 15) < qb) {
      *reinterpret_cast<float4 *>(&R.wsum[row][4 * (lane & 15)]) = a0;
      if (NV == 2) *reinterpret_cast<float4 *>(&R.wsum[4 * MAX_WAVES + row][4 * (lane & 15)]) = a1;
    }
    __syncthreads();
    for (int e = threadIdx.x; e < NV * 4 * qb; e += blockDim.x) {
      const int v = e / (4 * qb), i = e - v * 4 * qb;
      if (4 * q0 + i < R.rows) {
        float s = 0.f;
#pragma unroll 8
        for (int w = 0; w < nrow; w++) s += R.wsum[v * 4 * MAX_WAVES + w][i];
        R.tile[v][4 * q0 + i] = s;
      }
    }
    __syncthreads();
  }
}

// Two columns' dot products with r (LDS) by one wave: loads of both issue
// together, 4 float4 per lane and column.
__device__ __forceinline__ void res_dot2(const float4 *r4, XG(const float4) c0, XG(const float4) c1,
                                         int nq, int lane, float *g0, float *g1) {
  constexpr int U = 4;
  float s00 = 0.f, s01 = 0.f, s10 = 0.f, s11 = 0.f;
  for (int q = lane; q < nq; q += U * WAVE) {
    float4 a0[U], a1[U];
#pragma unroll
    for (int u = 0; u < U; u++) {
      const int qq = q + u * WAVE;
      const bool ok = qq < nq;
      a0[u] = ok ? load_nt(c0 + qq) : make_float4(0.f, 0.f, 0.f, 0.f);
      a1[u] = ok ? load_nt(c1 + qq) : make_float4(0.f, 0.f, 0.f, 0.f);
    }
#pragma unroll
    for (int u = 0; u < U; u++) {
      const int qq = q + u * WAVE;
      const float4 b = qq < nq ? r4[qq] : make_float4(0.f, 0.f, 0.f, 0.f);
      if (u & 1) {
        s01 = dot4(a0[u], b, s01);
        s11 = dot4(a1[u], b, s11);
      } else {
        s00 = dot4(a0[u], b, s00);
        s10 = dot4(a1[u], b, s10);
      }
    }
  }
  *g0 = wsum_f(s00 + s01);
  *g1 = wsum_f(s10 + s11);
}

// g = A^T r for this workgroup's columns (all columns, or the support's only,
// by list position), published to gx; the exchange that follows makes it
// readable.  Neighbouring support columns go to different workgroups.
template <bool SUPP>
__device__ __forceinline__ void res_AT(const RTeam &t, const Res &R, const XProblem &P,
                                       XG(float) gx) {
  const int lane = threadIdx.x & (WAVE - 1), nw = blockDim.x / WAVE;
  const int wave = threadIdx.x / WAVE, GW = t.size * nw, lda = P.lda;
  const int end = SUPP ? R.cnt : P.n;
  const int step = SUPP ? GW : 1;  // distance of a wave's two columns
  for (int s = SUPP ? wave * t.size + t.rank : 2 * (t.rank * nw + wave); s < end; s += 2 * GW) {
    const bool two = s + step < end;
    const int j0 = SUPP ? R.list[s] : s, j1 = two ? (SUPP ? R.list[s + step] : s + 1) : j0;
    float g0, g1;
    res_dot2(reinterpret_cast<const float4 *>(R.r),
             reinterpret_cast<XG(const float4)>(P.A + (size_t)j0 * lda),
             reinterpret_cast<XG(const float4)>(P.A + (size_t)j1 * lda), lda >> 2, lane, &g0, &g1);
    if (lane == 0) st_dev(gx + s, g0);
    if (lane == 1 && two) st_dev(gx + s + step, g1);
  }
}

__device__ __forceinline__ bool res_in(const Res &R, int j) {
  return (R.mask[j >> 6] >> (j & 63)) & 1ull;
}

// Support list and count from the mask (visible): every wave scans the words'
// counts for itself, then writes the entries of its own words.  Returns whether
// an entry of mask2 is missing in mask.  Ends with __syncthreads.
__device__ __forceinline__ bool res_list(Res &R, int n) {
  const int lane = threadIdx.x & (WAVE - 1), wave = threadIdx.x / WAVE;
  const int nw = blockDim.x / WAVE, words = (n + 63) >> 6;
  int base = 0;
  bool left = false;
  for (int b = 0; b < words; b += WAVE) {
    const unsigned long long m = b + lane < words ? R.mask[b + lane] : 0ull;
    const unsigned long long o = b + lane < words ? R.mask2[b + lane] : 0ull;
    left = left || (o & ~m);
    const int c = __popcll(m);
    const int incl = wscan_i(c);
    // this wave writes words b + wave, b + wave + nw, ...
    for (int w = wave; w < WAVE && b + w < words; w += nw) {
      const unsigned mlo = (unsigned)__builtin_amdgcn_readlane((int)(unsigned)m, w);
      const unsigned mhi = (unsigned)__builtin_amdgcn_readlane((int)(unsigned)(m >> 32), w);
      const unsigned long long mw = ((unsigned long long)mhi << 32) | mlo;
      const int pos = base + __builtin_amdgcn_readlane(incl, w) - __popcll(mw);
      if ((mw >> lane) & 1ull)
        R.list[pos + __popcll(mw & ((1ull << lane) - 1ull))] = (unsigned short)(64 * (b + w) + lane);
    }
    base += __builtin_amdgcn_readlane(incl, 63);
  }
  R.cnt = base;
  __syncthreads();
  return __any(left);
}

// FindSupportSet's binning branch on x (functions.cu:404-428) with max |x| =
// S.max_value, then the threshold, the mask and the list, all in this
// workgroup's LDS.  The k-bin walk is done by every wave for itself (a chunk of
// bins per lane, a scan over the lanes).  The histogram is zero on entry and
// zeroed again.  Starts with the wave's own x entries only; ends with
// __syncthreads.  Returns whether an entry left the support.
__device__ __forceinline__ bool res_rebin(Res &R, const XProblem &P, ResS &S) {
  const int n = P.n, nt = blockDim.x, lane = threadIdx.x & (WAVE - 1);
  S.slope = (float)(P.num_bins - 1) / S.max_value;
  const float slope = S.slope, inter = S.max_value;
  const int mb = S.max_bin;
  for (int j = threadIdx.x; j < n; j += nt) {
    const float v = R.x[j];
    const int b = linear_bin(v, slope, inter);
    if ((double)fabsf(v) > (double)inter * .000001 && b < mb) atomicAdd(&R.hist[b], 1);
  }
  __syncthreads();
  int kb = -1, sum = 0;
  if (P.k > 0) {  // the k-bin walk (functions.cu:414-420)
    const int chunk = ((mb + WAVE - 1) / WAVE) | 1;  // odd: lanes on distinct banks
    const int lo = min(mb, lane * chunk), hi = min(mb, lo + chunk);
    int c = 0;
    for (int b = lo; b < hi; b++) c += R.hist[b];
    const int incl = wscan_i(c);
    const unsigned long long cross = __ballot(incl >= P.k);
    if (cross == 0ull) {  // never reaches k
      kb = mb - 1;
      sum = __builtin_amdgcn_readlane(incl, 63);
    } else {
      const int l = __ffsll((unsigned long long)cross) - 1;
      int acc = incl - c, b = lo;
      if (lane == l)
        for (; b < hi; b++) {
          acc += R.hist[b];
          if (acc >= P.k) break;
        }
      kb = __builtin_amdgcn_readlane(b, l);
      sum = __builtin_amdgcn_readlane(acc, l);
    }
  }
  if (sum < P.k) {
    S.alpha_bin = S.alpha_bin * 0.5f;
    S.max_bin = (int)((float)P.num_bins * (1.0f - S.alpha_bin));
  }
  S.min_val = __fsub_rn(inter, __fdiv_rn((float)(kb + 1), slope));
  S.sum = sum;
  S.k_bin = kb;
  unsigned long long *m = R.mask2;
  for (int j0 = 0; j0 < n; j0 += nt) {  // whole waves: j0 and nt are multiples of 64
    const int j = j0 + threadIdx.x;
    const bool in = j < n && linear_bin(R.x[j], slope, inter) <= kb;
    if (j < n && !in) R.x[j] = 0.f;
    const unsigned long long bits = __ballot(in);
    if (lane == 0 && j < n) m[j >> 6] = bits;
  }
  __syncthreads();
  for (int b = threadIdx.x; b < P.num_bins; b += nt) R.hist[b] = 0;
  R.mask2 = R.mask;
  R.mask = m;
  return res_list(R, n);
}

// r = y - (rows of A x in tile[0]) published to rx; returns the thread's part of |r|^2.
__device__ __forceinline__ double res_publish_resid(const Res &R, const XProblem &P, XG(float) rx) {
  double e2 = 0.0;
  for (int i = threadIdx.x; i < R.rows; i += blockDim.x) {
    const float v = __fsub_rn(P.y[R.row0 + i], R.tile[0][i]);
    st_dev(rx + R.row0 + i, v);
    e2 += (double)v * (double)v;
  }
  return e2;
}
// Row `v` of the tile published to rx; returns the thread's part of its norm squared.
__device__ __forceinline__ double res_publish_tile(const Res &R, int v, XG(float) rx) {
  double a2 = 0.0;
  for (int i = threadIdx.x; i < R.rows; i += blockDim.x) {
    const float w = R.tile[v][i];
    st_dev(rx + R.row0 + i, w);
    a2 += (double)w * (double)w;
  }
  return a2;
}

// Algorithmic bytes of A^T r on cnt columns.
__device__ __forceinline__ double res_at_supp_bytes(const XProblem &P, int cnt) {
  return 4.0 * P.m * cnt + 4.0 * P.m + 4.0 * cnt;
}

// r (LDS) <- the published residual; dst (LDS) <- A^T r, all entries.
__device__ __forceinline__ void res_gradient(RTeam &t, Res &R, const XProblem &P, ResS &S,
                                             XG(float) rx, XG(float) gx, float *dst) {
  double z[1] = {0.0};
  if (rx) {
    ld_dev_vec(R.r, rx, P.lda);
    __syncthreads();
  }
  S.bytes += op_bytes(P, true, 0);
  res_AT<false>(t, R, P, gx);
  rt_allreduce<0>(t, *R.rt, z, z);
  ld_dev_vec(dst, gx, P.n);
  __syncthreads();
}

// CG projection on the support (cg_projection of xcs_solver.h): direction in p,
// CG residual in g, both on the support only.  Returns errCG.
__device__ __forceinline__ float res_cg_projection(RTeam &t, Res &R, const XProblem &P, ResS &S,
                                                   XG(float) rx, XG(float) gx, int max_steps) {
  const float tolCG = P.tol * P.tol;
  const float tol2 = 10.0f * tolCG;
  const int nt = blockDim.x;
  float dummy[1];
  S.bytes += op_bytes(P, false, R.cnt);
  res_gather<1>(R, P.A, P.lda, R.x, nullptr);
  float errCG;
  {
    double v[1] = {res_publish_resid(R, P, rx)}, o[1];
    rt_allreduce<1>(t, *R.rt, v, o);
    errCG = (float)o[0];
  }
  float hist = (threadIdx.x & (WAVE - 1)) == 15 ? errCG : 0.f, evo = 1.f, diff = 1.f;
  float mu_old = 0.f, alpha = 0.f;
  double a2 = 0.0;
  // step -1 forms the first direction; step it >= 0 is CG step it.  Each: r (the
  // residual, then A d) in LDS, A^T r on the support, the new direction, then
  // one pass over the support's columns for the residual (steps >= 0) and A d.
  for (int it = -1; !t.aborted; it++) {
    if (it >= 0) {
      if (!((errCG > tolCG) & (it < max_steps) & (diff > tol2))) break;
      alpha = (float)a2;
      alpha = (S.mu < 1000.0f * alpha) ? S.mu / alpha : 0.f;
    }
    ld_dev_vec(R.r, rx, P.lda);
    __syncthreads();
    S.bytes += res_at_supp_bytes(P, R.cnt);
    res_AT<true>(t, R, P, gx);
    {
      double z[1] = {0.0};
      rt_allreduce<0>(t, *R.rt, z, z);
    }
    double g2[1] = {0.0};
    for (int s = threadIdx.x; s < R.cnt; s += nt) {
      const int j = R.list[s];
      const float th = ld_dev(gx + s);
      const float gp = it < 0 ? th : fmaf(-alpha, th, R.g[j]);
      R.g[j] = gp;
      g2[0] += (double)gp * (double)gp;
    }
    wg_reduce<1, 0>(*R.slots, R.bank, g2, dummy);
    mu_old = S.mu;
    S.mu = (float)g2[0];
    const float beta = it < 0 ? 0.f : (S.mu < 1000.0f * mu_old) ? S.mu / mu_old : 0.f;
    for (int s = threadIdx.x; s < R.cnt; s += nt) {
      const int j = R.list[s];
      if (it < 0) {
        R.p[j] = R.g[j];
      } else {
        R.x[j] = fmaf(alpha, R.p[j], R.x[j]);
        R.p[j] = __fadd_rn(__fmul_rn(beta, R.p[j]), R.g[j]);
      }
    }
    __syncthreads();
    double v[2] = {0.0, 0.0}, o[2];
    // the last allowed step needs no next A d
    const bool next = it + 1 < max_steps;
    S.bytes += op_bytes(P, false, R.cnt) + (it >= 0 && next ? 8.0 * R.cnt + 4.0 * P.m : 0.0);
    if (it < 0) {
      if (!((errCG > tolCG) & (diff > tol2))) break;  // no step will be taken
      res_gather<1>(R, P.A, P.lda, R.p, nullptr);
      v[1] = res_publish_tile(R, 0, rx);
    } else {
      if (next)
        res_gather<2>(R, P.A, P.lda, R.x, R.p);
      else
        res_gather<1>(R, P.A, P.lda, R.x, nullptr);
      for (int i = threadIdx.x; i < R.rows; i += nt) {
        const float e = __fsub_rn(P.y[R.row0 + i], R.tile[0][i]);
        v[0] += (double)e * (double)e;
      }
      if (next) v[1] = res_publish_tile(R, 1, rx);
    }
    rt_allreduce<2>(t, *R.rt, v, o);
    a2 = o[1];
    if (it >= 0) {
      errCG = (float)o[0];
      hist = hist_push(hist, errCG);
      evo = hist_push(evo, __fsub_rn(lane_f(hist, 14), lane_f(hist, 15)));
      diff = hist_max(evo);
    }
  }
  return errCG;
}

// The stop rules of should_continue and stop_update (xcs_solver.h) on the lane
// history.
struct ResStop {
  float err, err_start, diff;
  int iter, fail, cycle;
};
__device__ __forceinline__ bool res_continue(const ResStop &S, const XProblem &P, int *reason) {
  if (!(S.err > P.tol)) { *reason = 0; return false; }
  if (!(S.iter < P.maxiter)) { *reason = 1; return false; }
  if (!(S.err < 100.0f * S.err_start)) { *reason = 2; return false; }
  if (!((double)S.diff > .01 * (double)P.tol)) { *reason = 3; return false; }
  if (S.fail != 0) { *reason = 4; return false; }
  if (!S.cycle) { *reason = 5; return false; }
  return true;
}
__device__ __forceinline__ void res_stop_update(ResStop &S, float prev, float *evo, int fail_after) {
  const float last = lane_f(prev, 15);
  *evo = hist_push(*evo, __fsub_rn(lane_f(prev, 14), last));
  S.diff = hist_max(*evo);
  const unsigned long long same = __ballot(prev == last) & 0x7FFFull;
  if (same && S.iter > 4) S.cycle = 0;
  if (S.iter > fail_after) {
    const float root = 1 / 15.0f;
    float rate = last / lane_f(prev, 0);
    rate = powf(rate, root);
    if (rate > 0.999f) S.fail = 1;
  }
}

// One instance by the whole (cooperatively launched) grid: at most `budget`
// outer iterations from the saved state.  MAXT: the largest workgroup (512 lets
// the compiler use 256 registers: no spills).
template <int ALG, int MAXT>
__global__ void __launch_bounds__(MAXT) solve_resident_kernel(const XProblem *Pp, int budget,
                                                              unsigned *bar, long spin_limit) {
  constexpr bool CG = ALG == ALG_CGIHT;
  __shared__ __attribute__((aligned(16))) unsigned char lds[RES_LDS];
  __shared__ XProblem sP;
  __shared__ float tile[2][RES_TCAP];
  __shared__ __attribute__((aligned(16))) float wsum[2 * 4 * MAX_WAVES][4 * RES_QB];
  __shared__ WgSlots slots;
  __shared__ RtSlots rt;
  if (threadIdx.x == 0) sP = *Pp;
  __syncthreads();
  const XProblem &P = sP;
  if (P.st->done) return;
  const int lane = threadIdx.x & (WAVE - 1), nt = blockDim.x;
  const int n = P.n;
  RTeam t{(int)blockIdx.x, (int)gridDim.x, bar, bar[1], spin_limit, 0};
  XG(float) rx = P.resid;  // exchange buffers
  XG(float) gx = P.grad;
  Res R;
  {
    unsigned char *q = lds;
    auto take = [&](size_t b) {
      unsigned char *r = q;
      q += res_up16(b);
      return r;
    };
    R.x = (float *)take(4 * (size_t)n);
    R.g = (float *)take(4 * (size_t)n);
    R.p = (float *)take(4 * (size_t)n);
    R.r = (float *)take(4 * (size_t)P.lda);
    R.hist = (int *)take(4 * (size_t)P.num_bins);
    R.mask = (unsigned long long *)take(8 * ((size_t)n / 64 + 1));
    R.mask2 = (unsigned long long *)take(8 * ((size_t)n / 64 + 1));
    R.list = (unsigned short *)take(2 * (size_t)n);
  }
  R.tile = tile;
  R.wsum = wsum;
  R.slots = &slots;
  R.rt = &rt;
  R.bank = 0;
  R.cnt = 0;
  res_rows(t.rank, t.size, P.lda, &R.row0, &R.rows);
  for (int b = threadIdx.x; b < P.num_bins; b += nt) R.hist[b] = 0;
  for (int w = threadIdx.x; w <= n / 64; w += nt) R.mask[w] = R.mask2[w] = 0ull;
  float prev = 0.f, evo = 1.f;  // the history, entry i in lane i
  ResS S;
  ResStop Q;
  float dummyf[1];
  double dummyd[1];
  // trace (rank 0): iteration idx selected its support at kb with residual e
  auto trace = [&](int idx, int kb, float e) {
    if (t.rank == 0 && threadIdx.x == 0) {
      if (P.trace_kbin) P.trace_kbin[idx] = kb;
      if (P.trace_err) P.trace_err[idx] = e;
    }
  };
  bool zero = false;
  if (P.st->initialized) {  // a continued solve: state, x, direction and support from memory
    XG(const XState) st = P.st;
    S.k_bin = st->k_bin;
    S.sum = st->sum;
    S.max_bin = st->max_bin;
    S.beta_to_zero = st->beta_to_zero;
    S.supp_change = st->supp_change;
    S.alpha_bin = st->alpha_bin;
    S.min_val = st->min_val;
    S.max_change = st->max_change;
    S.max_value = st->max_value;
    S.slope = st->slope;
    S.mu = st->mu;
    S.bytes = st->mat_bytes;
    Q.err = st->err;
    Q.err_start = st->err_start;
    Q.diff = st->diff;
    Q.iter = st->iter;
    Q.fail = st->fail;
    Q.cycle = st->cycle;
    if (lane < 16) {
      prev = st->prev[lane];
      evo = st->evo[lane];
    }
    __syncthreads();  // masks zeroed
    for (int j0 = 0; j0 < n; j0 += nt) {
      const int j = j0 + threadIdx.x;
      const bool ok = j < n;
      if (ok) {
        R.x[j] = P.x[j];
        R.p[j] = P.gprev[j];
      }
      const unsigned long long m = __ballot(ok && P.bins[ok ? j : 0] <= S.k_bin);
      if (lane == 0 && ok) R.mask[j >> 6] = m;
    }
    __syncthreads();
    (void)res_list(R, n);
  } else {
    // common initialisation (algorithms.cu:1284-1358 and equivalents)
    S.k_bin = S.sum = 0;
    S.alpha_bin = 0.25f;
    S.max_bin = (int)((float)P.num_bins * (1.0f - S.alpha_bin));
    S.min_val = 0.f;
    S.max_change = ALG == ALG_HTP ? 0.0f : 1.0f;
    S.slope = S.mu = 0.f;
    S.beta_to_zero = 1;
    S.supp_change = 1;
    S.bytes = 0.0;
    Q.diff = 1.f;
    Q.iter = 0;
    Q.fail = 0;
    Q.cycle = 1;
    double e2[1] = {0.0};
    for (int i = threadIdx.x; i < P.lda; i += nt) {
      const float r = P.y[i];
      R.r[i] = r;
      e2[0] += (double)r * (double)r;
    }
    for (int j = threadIdx.x; j < n; j += nt) R.p[j] = 0.f;
    __syncthreads();
    res_gradient(t, R, P, S, nullptr, gx, R.x);
    float xm[1] = {0.f};
    for (int j = threadIdx.x; j < n; j += nt) xm[0] = fmaxf(xm[0], fabsf(R.x[j]));
    wg_reduce<1, 1>(slots, R.bank, e2, xm);
    Q.err = Q.err_start = (float)sqrt(e2[0]);
    S.max_value = xm[0];
    zero = S.max_value == 0.f;  // A^T y == 0: x = 0 is returned
    if (!zero) {
      (void)res_rebin(R, P, S);
      trace(0, S.k_bin, Q.err);
      if (CG) {
        // r^0 and its gradient as the first direction (algorithms.cu:3762-3808)
        S.bytes += op_bytes(P, false, R.cnt);
        res_gather<1>(R, P.A, P.lda, R.x, nullptr);
        double v[1] = {res_publish_resid(R, P, rx)}, o[1];
        rt_allreduce<1>(t, rt, v, o);
        Q.err = (float)sqrt(o[0]);
        if (lane == 15) prev = Q.err;
        res_gradient(t, R, P, S, rx, gx, R.p);
        evo = hist_push(evo, __fsub_rn(0.f, Q.err));
      }
    }
  }
  int reason = 0;
  while (!zero && budget > 0 && !t.aborted && res_continue(Q, P, &reason)) {
    budget--;
    const bool uncg = CG && !P.restart && S.supp_change;
    // residual rows; UnrestrictedCG (functions.cu:1107-1220) forms A p_old,S in the
    // same pass (tile[1]) as A x
    S.bytes += op_bytes(P, false, R.cnt) + (uncg ? 8.0 * R.cnt + 4.0 * P.m : 0.0);
    if (uncg)
      res_gather<2>(R, P.A, P.lda, R.x, R.p);
    else
      res_gather<1>(R, P.A, P.lda, R.x, nullptr);
    float norm;  // |r| at the start of the iteration
    {
      double v[1] = {res_publish_resid(R, P, rx)}, o[1];
      rt_allreduce<1>(t, rt, v, o);
      norm = (float)sqrt(o[0]);
    }
    res_gradient(t, R, P, S, rx, gx, R.g);
    float mx[2] = {0.f, 0.f};  // max |direction|, max |x|
    float step;
    const float *dir = CG ? R.p : R.g;
    if (!uncg) {
      // RestrictedSD (NIHT, HTP: functions.cu:659-745) and the restricted CG step
      // with support evolution (functions.cu:1004-1102)
      double th2[1] = {0.0};
      for (int s = threadIdx.x; s < R.cnt; s += nt) {
        const float th = R.g[R.list[s]];
        th2[0] += (double)th * (double)th;
      }
      wg_reduce<1, 0>(slots, R.bank, th2, dummyf);
      if (CG) {
        float beta = 0.f;
        const float mu_new = (float)th2[0];
        if (S.beta_to_zero != 1) beta = (mu_new < 1000.0f * S.mu) ? mu_new / S.mu : 0.f;
        S.mu = mu_new;
        for (int j = threadIdx.x; j < n; j += nt)
          R.p[j] = __fadd_rn(__fmul_rn(beta, R.p[j]), R.g[j]);
        __syncthreads();
      }
      S.bytes += op_bytes(P, false, R.cnt);
      res_gather<1>(R, P.A, P.lda, dir, nullptr);
      double v[1] = {0.0}, o[1];
      for (int i = threadIdx.x; i < R.rows; i += nt) v[0] += (double)tile[0][i] * (double)tile[0][i];
      rt_allreduce<1>(t, rt, v, o);
      if (CG) {
        const float a = (float)o[0];
        step = (S.mu < 1000.0f * a) ? S.mu / a : 0.f;
      } else {
        const float err = (float)sqrt(o[0]);
        const float mu = (float)sqrt(th2[0]);
        step = mu / err;
        step = (mu < 400.0f * err) ? step * step : 0.f;
      }
    } else {
      // A g_S into tile[0]; A p_old,S stays in tile[1]
      S.bytes += op_bytes(P, false, R.cnt);
      res_gather<1>(R, P.A, P.lda, R.g, nullptr);
      float beta = 0.f;
      if (S.beta_to_zero != 1) {
        double v[2] = {0.0, 0.0}, o[2];
        for (int i = threadIdx.x; i < R.rows; i += nt) {
          const double ap = tile[1][i], ag = tile[0][i];
          v[0] += ap * ag;
          v[1] += ap * ap;
        }
        rt_allreduce<2>(t, rt, v, o);
        beta = -((float)o[0]) / (float)o[1];
      }
      double an[2] = {0.0, 0.0}, ad[1] = {0.0}, o[1];
      for (int j = threadIdx.x; j < n; j += nt) {
        const float g = R.g[j];
        const float gp = __fadd_rn(__fmul_rn(beta, R.p[j]), g);
        R.p[j] = gp;
        if (res_in(R, j)) {
          an[0] += (double)gp * (double)g;
          an[1] += (double)g * (double)g;
        }
      }
      for (int i = threadIdx.x; i < R.rows; i += nt) {
        const float r = __fadd_rn(__fmul_rn(beta, tile[1][i]), tile[0][i]);
        ad[0] += (double)r * (double)r;
      }
      wg_reduce<2, 0>(slots, R.bank, an, dummyf);
      rt_allreduce<1>(t, rt, ad, o);
      step = (float)an[0] / (float)o[0];
      S.mu = (float)an[1];
    }
    for (int j = threadIdx.x; j < n; j += nt) {
      const float d = dir[j];
      const float xn = fmaf(step, d, R.x[j]);
      R.x[j] = xn;
      mx[0] = fmaxf(mx[0], fabsf(d));
      mx[1] = fmaxf(mx[1], fabsf(xn));
    }
    wg_reduce<0, 2>(slots, R.bank, dummyd, mx);
    S.max_change = 2.0f * step * mx[0];
    // support update (the skip rule of FindSupportSet, functions.cu:400-403)
    if (CG) S.beta_to_zero = 0;
    if (S.min_val <= S.max_change) {
      S.max_value = mx[1];
      const bool left = res_rebin(R, P, S);
      if (CG) {
        S.supp_change = left ? 1 : 0;
        if (left && P.restart) S.beta_to_zero = 1;
      }
    } else {
      S.supp_change = CG ? 0 : S.supp_change;
      S.min_val = S.min_val - S.max_change;
      for (int j = threadIdx.x; j < n; j += nt)
        if (!res_in(R, j)) R.x[j] = 0.f;
      __syncthreads();
    }
    prev = hist_push(prev, norm);
    Q.err = norm;
    if (ALG == ALG_HTP) {
      Q.err = sqrtf(res_cg_projection(t, R, P, S, rx, gx, 15));
      prev = hist_push(prev, Q.err);
    }
    res_stop_update(Q, prev, &evo, ALG == ALG_HTP ? 125 : 749);
    Q.iter++;
    trace(Q.iter, S.k_bin, Q.err);
  }
  int done = 0;
  if (t.aborted) {
    done = 1;
    reason = STOP_ABORTED;
  } else if (zero || !res_continue(Q, P, &reason)) {
    done = 1;
    if (zero) reason = 0;
  }
  __syncthreads();
  for (int j = t.rank * nt + threadIdx.x; j < n; j += t.size * nt) {
    P.x[j] = R.x[j];
    P.gprev[j] = R.p[j];
    P.bins[j] = res_in(R, j) ? S.k_bin : S.k_bin + 1;
  }
  if (t.rank == 0 && threadIdx.x < 16) {
    XG(XState) st = P.st;
    st->prev[threadIdx.x] = prev;
    st->evo[threadIdx.x] = evo;
    if (threadIdx.x == 0) {
      st->initialized = 1;
      st->done = done;
      st->stop_reason = done ? reason : 0;
      st->iter = Q.iter;
      st->k_bin = S.k_bin;
      st->max_bin = S.max_bin;
      st->sum = S.sum;
      st->supp_count = R.cnt;
      st->beta_to_zero = S.beta_to_zero;
      st->supp_change = S.supp_change;
      st->fail = Q.fail;
      st->cycle = Q.cycle;
      st->alpha_bin = S.alpha_bin;
      st->min_val = S.min_val;
      st->max_change = S.max_change;
      st->max_value = S.max_value;
      st->slope = S.slope;
      st->mu = S.mu;
      st->err = Q.err;
      st->err_start = Q.err_start;
      st->diff = Q.diff;
      st->mat_bytes = S.bytes;
      bar[1] = t.tag;
    }
  }
}

// y = A x of a generated instance (x in memory, its support ascending in P.supp)
// by the solve's own product in the solve's geometry, so that the planted vector
// leaves no residual: with y from the general form's product, whose sums round
// differently, a solve cannot come below about ||y|| 2^-23 (CGIHT 1024 x 4096: 7e-7
// of 7).  One launch of the team, no exchanges.
template <int MAXT>
__global__ void __launch_bounds__(MAXT) resident_y_kernel(const XProblem *Pp, const float *x, int cnt,
                                                          float *y) {
  __shared__ __attribute__((aligned(16))) unsigned char lds[RES_LDS];
  __shared__ XProblem sP;
  __shared__ float tile[2][RES_TCAP];
  __shared__ __attribute__((aligned(16))) float wsum[2 * 4 * MAX_WAVES][4 * RES_QB];
  if (threadIdx.x == 0) sP = *Pp;
  __syncthreads();
  const XProblem &P = sP;
  Res R;
  R.x = (float *)lds;
  R.list = (unsigned short *)(lds + res_up16(4 * (size_t)P.n));
  R.tile = tile;
  R.wsum = wsum;
  R.cnt = cnt;
  res_rows(blockIdx.x, gridDim.x, P.lda, &R.row0, &R.rows);
  for (int s = threadIdx.x; s < cnt; s += blockDim.x) {
    const int j = P.supp[s];
    R.list[s] = (unsigned short)j;
    R.x[j] = x[j];
  }
  __syncthreads();
  res_gather<1>(R, P.A, P.lda, R.x, nullptr);
  for (int i = threadIdx.x; i < R.rows; i += blockDim.x) y[R.row0 + i] = tile[0][i];
}

}  // namespace xcs
