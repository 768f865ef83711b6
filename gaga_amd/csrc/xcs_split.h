// One sparse (smv) or subsampled-DCT instance on a team of workgroups with the
// solver's vectors split over the workgroups' LDS: NIHT, HTP and CGIHT.
//
// At these sizes (n up to 2^20) no workgroup can hold whole vectors as the dense
// resident form does.  Here workgroup w owns a slice of the n-vectors (x, the
// gradient, the direction) and a slice of the m-vectors, both in its LDS; every
// elementwise step, the thresholds and the norms work on them without memory
// traffic.  What crosses workgroups moves inside one-hop exchanges
// (rt_allreduce), about seven per iteration where the general form crosses
// about twelve fenced barriers, and each carries the scalar sums pending at
// that point:
//   * one per matrix product: smv publishes the operand (device-scope stores),
//     then gathers it through the L2s (one cache invalidation per workgroup); the
//     DCT publishes its half-transformed data (below);
//   * the step length, max |x| and the histogram of the support selection.
//
// smv: the matrix entries of the own rows and columns do not change during a solve
// and stay in LDS as far as it has room, and the operand of every A product is
// zero off the support, so a row's entries are tested against the support's bits
// (all n of them in LDS, exchanged once per selection) and only the few that hit
// are gathered.  An iteration of 2^15 x 2^18 (CGIHT, 256 workgroups) 76 -> 51 us: A x
// gathers 28 -> 6 us, A^T r 10.7 -> 6.2; what is left is six exchanges (20 us), the
// A^T gather's random loads and the selection (5).
//
// DCT: a transform of n reals is an FFT of N = n / 2 complex values by N = N1 N2
// (half the work and half the exchanged bytes of the complex transform of the
// real data).  Forward: workgroups transform columns (residues mod N2 of the
// packed index), exchange, transform rows (residues mod N1 of the output index).
// The inverse runs the same steps backwards, so a workgroup's outputs of one
// product are exactly its inputs of the next: x lives as the packed time slots of the
// owned residues mod N2, y and the residual as the coefficient slots of the
// owned residues mod N1 (r and -r together: the real transform pairs k with
// N - k), and the one exchange per product is the transpose in the middle.  The
// column transforms are decimation in time from bit-reversed slots and the row
// transforms decimation in frequency into them, so no permutation is ever made.
//
// Measured on MI355X: smv 2^15 x 2^18 CGIHT 6.6 -> 1.75 ms (34 iterations), dct
// n = 2^20 NIHT 5.7 -> 1.66 ms (20 iterations); a DCT product costs about 15 us
// there where the complex transform in fenced passes took 65 (plan_split has
// the other sizes and the teams).
// The arithmetic is that of the general solver except for the order of sums and
// the factorisation of the transform.
#pragma once
#include "xcs_resident.h"

namespace xcs {

constexpr int SP_THREADS = 512;       // workgroup size (at most)
constexpr int SP_LDS = 150 * 1024;    // bytes of LDS for the slices and tables
constexpr int SP_HIST = 4096;         // histogram bins held in LDS
constexpr int SP_PAD = 64;            // slices of n-vectors: multiples of a wave

// Twiddles of a length-2^b transform held in LDS: what its radix-4 butterflies read.
__host__ __device__ inline size_t sp_twiddles(int b) { return b < 2 ? 1 : (size_t)3 << (b - 2); }
// Histogram bins held in LDS: all of them or none.
__host__ __device__ inline int sp_hist(int num_bins) { return num_bins <= SP_HIST ? num_bins : 0; }
// Layout of an instance over `size` workgroups.
struct SplitGeom {
  int nl, rl;          // floats per workgroup of an n-vector and of an m-vector
  int b1, b2;          // dct: N1 = 2^b1 rows, N2 = 2^b2 columns
  size_t lds;          // bytes
  bool filter;         // smv: room for the support bits of all columns besides
};
__host__ __device__ inline SplitGeom split_geom(int ens, int alg, int m, int n, int log2n,
                                                int num_bins, int size) {
  SplitGeom G{};
  const int vecs = alg == ALG_HTP ? 4 : 3;
  if (ens == ENS_DCT) {
    const int ln = log2n - 1;
    G.b1 = ln / 2;
    G.b2 = ln - G.b1;
    G.nl = G.rl = n / size;
    G.lds = res_up16(8 * sp_twiddles(G.b1)) + res_up16(8 * sp_twiddles(G.b2)) +
            res_up16((size_t)G.rl / 8 + 8);
  } else {
    G.nl = ((n + size - 1) / size + SP_PAD - 1) / SP_PAD * SP_PAD;
    G.rl = ((m + size - 1) / size + 3) / 4 * 4;
  }
  G.lds += vecs * res_up16(4 * (size_t)G.nl) + 3 * res_up16(4 * (size_t)G.rl) +
           res_up16((size_t)G.nl / 8 + 8) + res_up16(4 * (size_t)sp_hist(num_bins));
  G.filter = ens == ENS_SMV && G.lds + res_up16((size_t)n / 8 + 8) <= (size_t)SP_LDS;
  return G;
}
// smv with the support bits in LDS: what LDS has left takes the own rows' columns (rn
// entries of rlv rows), then the own columns' rows and values (cn entries of nlv).
struct SplitStage {
  bool rows, cols;
};
__host__ __device__ inline SplitStage split_stage(const SplitGeom &G, int n, int rlv, int nlv, int rn, int cn) {
  SplitStage T{false, false};
  if (!G.filter) return T;
  size_t left = (size_t)SP_LDS - G.lds - res_up16((size_t)n / 8 + 8);
  T.rows = left >= res_up16(4 * ((size_t)rlv + 1 + rn + 8));
  if (T.rows) left -= res_up16(4 * ((size_t)rlv + 1)) + res_up16(4 * (size_t)rn);
  T.cols = left >= res_up16(4 * ((size_t)nlv + 1 + 2 * (size_t)cn + 12));
  return T;
}
inline bool split_fits(int alg, int ens, int m, int n, int log2n, int num_bins, int timing,
                       int team, int block) {
  if ((alg != ALG_NIHT && alg != ALG_HTP && alg != ALG_CGIHT) || timing || team < 2 ||
      block > SP_THREADS || num_bins > n)
    return false;
  if (ens == ENS_DCT) {
    if (log2n < 6 || n > (1 << 20) || (team & (team - 1))) return false;
    const int N1 = 1 << ((log2n - 1) / 2);
    if (team > N1 / 2 || n / team < 64) return false;
  } else if (ens != ENS_SMV) {
    return false;
  }
  return split_geom(ens, alg, m, n, log2n, num_bins, team).lds <= (size_t)SP_LDS;
}

// ------------------------------------------------------------ the state ----
struct Sp {
  float *x, *g, *p, *q;        // n-slices (q: HTP only)
  float *y, *t0, *t1;          // m-slices (dct: all owned coefficients, unsampled ones zero)
  int *hist;                   // zero between uses
  unsigned long long *mask;    // support bits of the n-slice
  unsigned long long *rmask;   // dct: sampled bits of the m-slice
  const float2 *w1, *w2;       // dct: w_N1^k and w_N2^k, k < 3/4 of the length
  WgSlots *slots;
  RtSlots *rt;
  int bank, par;               // wg_reduce bank, histogram parity
  int mid;                     // dct: parity of the exchange buffer
  int nl, nlv, rl, rlv;        // slice lengths and how much of them is in range
  int j0, i0;                  // smv: first column and row
  unsigned long long *fmask;   // smv: the support bits of all columns, or null (not enough LDS)
  bool fnew;                   // smv: the own bits have changed since fmask was read
  // smv: the own rows' and columns' entries, where LDS has room for them (else null);
  // pointers relative to the first entry
  const int *lrp, *lcols, *lcp, *lrows;
  const float *lvals;
  int rbase;                   // first entry of the own rows
  int b1, b2;
};

__device__ __forceinline__ bool sp_in(const Sp &R, int i) {
  return (R.mask[i >> 6] >> (i & 63)) & 1ull;
}
__device__ __forceinline__ void st_dev_w(XG(unsigned long long) p, unsigned long long v) {
  __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ unsigned long long ld_dev_w(XG(const unsigned long long) p) {
  return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ void st_dev2(XG(float2) p, float2 v) {
  st_dev_w(reinterpret_cast<XG(unsigned long long)>(p),
           ((unsigned long long)__float_as_uint(v.y) << 32) | (unsigned long long)__float_as_uint(v.x));
}
__device__ __forceinline__ float2 ld_dev2(XG(const float2) p) {
  const unsigned long long b = ld_dev_w(reinterpret_cast<XG(const unsigned long long)>(p));
  return make_float2(__uint_as_float((unsigned)b), __uint_as_float((unsigned)(b >> 32)));
}

// ------------------------------------------------------------------ smv ----
// dst[r] = sum over the entries of row (column) first + r, r < cnt, of
// val * v[idx], LPR lanes per row: a lane takes every LPR-th entry, eight loads
// in flight, then the lanes' sums.  NV vectors share the index loads.  ptr, idx
// and val are in memory or in LDS.
template <int LPR, int NV, class PI, class PV>
__device__ __forceinline__ void sp_gather_l(PI ptr, PI idx, PV val, int first, int cnt,
                                            XG(const float) v0, XG(const float) v1, float *d0,
                                            float *d1) {
  const int sub = threadIdx.x % LPR;
  for (int r = threadIdx.x / LPR; r < cnt; r += blockDim.x / LPR) {
    const int e0 = ptr[first + r], e1 = ptr[first + r + 1];
    float s0 = 0.f, s1 = 0.f;
    for (int e = e0 + sub; e < e1; e += 8 * LPR) {
      int c[8];
      float a[8], x0[8], x1[8];
#pragma unroll
      for (int u = 0; u < 8; u++) {
        const int ee = e + u * LPR < e1 ? e + u * LPR : e;  // a valid entry either way
        c[u] = idx[ee];
        a[u] = val[ee];
      }
#pragma unroll
      for (int u = 0; u < 8; u++) {
        x0[u] = v0[c[u]];
        if (NV == 2) x1[u] = v1[c[u]];
      }
#pragma unroll
      for (int u = 0; u < 8; u++)
        if (e + u * LPR < e1) {
          s0 = fmaf(a[u], x0[u], s0);
          if (NV == 2) s1 = fmaf(a[u], x1[u], s1);
        }
    }
#pragma unroll
    for (int o = 1; o < LPR; o <<= 1) {
      s0 += __shfl_xor(s0, o);
      if (NV == 2) s1 += __shfl_xor(s1, o);
    }
    if (sub == 0) {
      d0[r] = s0;
      if (NV == 2) d1[r] = s1;
    }
  }
}
// One vector, one lane per row, two rows at a time, and only the loads of
// entries that exist.
template <class PI, class PV>
__device__ __forceinline__ void sp_gather_pair(PI ptr, PI idx, PV val, int first, int cnt,
                                               XG(const float) v, float *d) {
  const int nt = blockDim.x;
  for (int r = threadIdx.x; r < cnt; r += 2 * nt) {
    const int rb = r + nt < cnt ? r + nt : r;
    const int ea = ptr[first + r], ea1 = ptr[first + r + 1];
    const int eb = ptr[first + rb], eb1 = rb == r ? eb : ptr[first + rb + 1];
    float s[2] = {0.f, 0.f};
    for (int o = 0; o < max(ea1 - ea, eb1 - eb); o += 8) {
      int c[2][8];
      float a[2][8], x[2][8];
#pragma unroll
      for (int h = 0; h < 2; h++)
#pragma unroll
        for (int u = 0; u < 8; u++) {
          const int e = (h ? eb : ea) + o + u;
          c[h][u] = -1;
          a[h][u] = 0.f;
          if (e < (h ? eb1 : ea1)) {
            c[h][u] = idx[e];
            a[h][u] = val[e];
          }
        }
#pragma unroll
      for (int h = 0; h < 2; h++)
#pragma unroll
        for (int u = 0; u < 8; u++) {
          x[h][u] = 0.f;
          if (c[h][u] >= 0) x[h][u] = v[c[h][u]];
        }
#pragma unroll
      for (int h = 0; h < 2; h++)
#pragma unroll
        for (int u = 0; u < 8; u++)
          if (c[h][u] >= 0) s[h] = fmaf(a[h][u], x[h][u], s[h]);
    }
    d[r] = s[0];
    if (rb != r) d[rb] = s[1];
  }
}
template <int NV, class PI, class PV>
__device__ __forceinline__ void sp_gather(PI ptr, PI idx, PV val, int first, int cnt, int avg,
                                          XG(const float) v0, XG(const float) v1, float *d0,
                                          float *d1) {
  // as many lanes as leave each about eight entries; two rows at a time where a
  // thread has that many (A^T r of 2^15 x 2^18: 7.8 us one by one, 6.2 in pairs; of
  // 2^15 x 2^20, from memory, an iteration 227 and 199 us; with a single row a thread the
  // pairs are slower, 2.7 against 1.4 us at 3001 x 30011)
  if (avg > 32)
    sp_gather_l<8, NV>(ptr, idx, val, first, cnt, v0, v1, d0, d1);
  else if (avg > 12)
    sp_gather_l<4, NV>(ptr, idx, val, first, cnt, v0, v1, d0, d1);
  else if (NV == 1 && cnt > (int)blockDim.x)
    sp_gather_pair(ptr, idx, val, first, cnt, v0, d0);
  else
    sp_gather_l<1, NV>(ptr, idx, val, first, cnt, v0, v1, d0, d1);
  __syncthreads();
}
// The same sums for operands that are zero outside the support, whose bits are
// in LDS: a lane tests its entries' bits (up to 64 at a time), then reads value
// and operand of the few that are set, two in flight.  An entry costs two LDS
// reads instead of a random load through the L2, which is what bounds the
// product: smv 2^15 x 2^18 (1.8 million entries, k = 3277) 12 us unfiltered, under
// 3 filtered.  The lanes per row fill the workgroup in one pass over the rows.
template <int NV, class PI>
__device__ __forceinline__ void sp_gather_supp(PI ptr, PI idx, XG(const float) val, int first,
                                               int cnt, const unsigned long long *mask,
                                               XG(const float) v0, XG(const float) v1, float *d0,
                                               float *d1) {
  int lpr = 1;
  while (lpr < 16 && 2 * lpr * cnt <= (int)blockDim.x) lpr *= 2;
  const unsigned *mw = reinterpret_cast<const unsigned *>(mask);
  const int sub = threadIdx.x & (lpr - 1), nr = blockDim.x / lpr;
  for (int r = threadIdx.x / lpr; r < cnt; r += nr) {
    const int e0 = ptr[first + r], e1 = ptr[first + r + 1];
    float s0 = 0.f, s1 = 0.f;
    for (int e = e0 + sub; e < e1; e += 64 * lpr) {
      unsigned long long hits = 0ull;
      for (int u0 = 0; u0 < 64 && e + u0 * lpr < e1; u0 += 8) {
        int c[8];
#pragma unroll
        for (int u = 0; u < 8; u++) c[u] = idx[min(e + (u0 + u) * lpr, e1 - 1)];
        unsigned h = 0;
#pragma unroll
        for (int u = 0; u < 8; u++)
          if (e + (u0 + u) * lpr < e1) h |= ((mw[c[u] >> 5] >> (c[u] & 31)) & 1u) << u;
        hits |= (unsigned long long)h << u0;
      }
      while (hits) {
        const int ea = e + (__ffsll(hits) - 1) * lpr;
        hits &= hits - 1;
        const bool two = hits != 0ull;
        const int eb = two ? e + (__ffsll(hits) - 1) * lpr : ea;
        hits &= hits - 1;
        const int ca = idx[ea], cb = idx[eb];
        const float aa = val[ea], ab = val[eb], xa = v0[ca], xb = v0[cb];
        float pa = 0.f, pb = 0.f;
        if (NV == 2) {
          pa = v1[ca];
          pb = v1[cb];
        }
        s0 = fmaf(aa, xa, s0);
        if (NV == 2) s1 = fmaf(aa, pa, s1);
        if (two) {
          s0 = fmaf(ab, xb, s0);
          if (NV == 2) s1 = fmaf(ab, pb, s1);
        }
      }
    }
    for (int o = 1; o < lpr; o <<= 1) {
      s0 += __shfl_xor(s0, o);
      if (NV == 2) s1 += __shfl_xor(s1, o);
    }
    if (sub == 0) {
      d0[r] = s0;
      if (NV == 2) d1[r] = s1;
    }
  }
  __syncthreads();
}

// ------------------------------------------------------------------ dct ----
template <int SIGN>
__device__ __forceinline__ float2 sp_tw(float2 w) {  // tables hold the forward sign
  return SIGN > 0 ? make_float2(w.x, -w.y) : w;
}
// Radix-4 butterflies (three twiddle products for four points where two radix-2
// stages take four) and fused multiply-adds (two roundings a component where
// separate products take three): the packed transform passes over the spectrum once
// more than the general form's (xcs_fft.h), and with that form's butterflies its
// products came out 4-5% further from 64 bits than they; with these 5-10% nearer,
// and their projection on the support, which is what reaches x, 12-27% nearer.
__device__ __forceinline__ float2 sp_cmul(float2 a, float2 b) {
  return make_float2(fmaf(a.x, b.x, -__fmul_rn(a.y, b.y)), fmaf(a.x, b.y, __fmul_rn(a.y, b.x)));
}
__device__ __forceinline__ float2 sp_add(float2 a, float2 b) {
  return make_float2(__fadd_rn(a.x, b.x), __fadd_rn(a.y, b.y));
}
__device__ __forceinline__ float2 sp_sub(float2 a, float2 b) {
  return make_float2(__fsub_rn(a.x, b.x), __fsub_rn(a.y, b.y));
}
// a + s i b with s = SIGN (the quarter turn of the transform's direction).
template <int SIGN>
__device__ __forceinline__ float2 sp_turn(float2 a, float2 b) {
  return SIGN > 0 ? make_float2(__fsub_rn(a.x, b.y), __fadd_rn(a.y, b.x))
                  : make_float2(__fadd_rn(a.x, b.y), __fsub_rn(a.y, b.x));
}
// cnt sequences of length 2^lb, contiguous in f, in place: decimation in time
// from bit-reversed to natural order.
template <int SIGN>
__device__ __forceinline__ void sp_dit(float2 *f, const float2 *tw, int lb, int cnt) {
  const int len = 1 << lb;
  int lh = 0;
  for (; lh + 2 <= lb; lh += 2) {
    const int h = 1 << lh, lq = lb - 2, s2 = len >> (lh + 2);
    for (int b = threadIdx.x; b < (cnt << lq); b += blockDim.x) {
      const int sq = b >> lq, bb = b & ((1 << lq) - 1);
      const int pos = bb & (h - 1), base = (sq << lb) + ((bb >> lh) << (lh + 2)) + pos;
      const int e = pos * s2;
      const float2 x0 = f[base], t1 = sp_cmul(f[base + h], sp_tw<SIGN>(tw[2 * e]));
      const float2 t2 = sp_cmul(f[base + 2 * h], sp_tw<SIGN>(tw[e]));
      const float2 t3 = sp_cmul(f[base + 3 * h], sp_tw<SIGN>(tw[3 * e]));
      const float2 u = sp_add(x0, t1), v = sp_sub(x0, t1), c = sp_add(t2, t3), d = sp_sub(t2, t3);
      f[base] = sp_add(u, c);
      f[base + h] = sp_turn<SIGN>(v, d);
      f[base + 2 * h] = sp_sub(u, c);
      f[base + 3 * h] = sp_turn<-SIGN>(v, d);
    }
    __syncthreads();
  }
  if (lh < lb) {
    const int h = 1 << lh;
    for (int b = threadIdx.x; b < (cnt << lh); b += blockDim.x) {
      const int sq = b >> lh, pos = b & (h - 1), i0 = (sq << lb) + pos;
      const float2 u = f[i0], v = sp_cmul(f[i0 + h], sp_tw<SIGN>(tw[pos]));
      f[i0] = sp_add(u, v);
      f[i0 + h] = sp_sub(u, v);
    }
    __syncthreads();
  }
}
// The same from natural to bit-reversed order: decimation in frequency.
template <int SIGN>
__device__ __forceinline__ void sp_dif(float2 *f, const float2 *tw, int lb, int cnt) {
  const int len = 1 << lb;
  int lh = lb;  // log2 of twice the next stage's span
  if (lb & 1) {
    const int h = len >> 1;
    lh--;
    for (int b = threadIdx.x; b < (cnt << lh); b += blockDim.x) {
      const int sq = b >> lh, pos = b & (h - 1), i0 = (sq << lb) + pos;
      const float2 u = f[i0], v = f[i0 + h];
      f[i0] = sp_add(u, v);
      f[i0 + h] = sp_cmul(sp_sub(u, v), sp_tw<SIGN>(tw[pos]));
    }
    __syncthreads();
  }
  for (; lh >= 2; lh -= 2) {
    const int l2 = lh - 2, h = 1 << l2, lq = lb - 2;  // spans 2h, then h
    const int s1 = len >> (l2 + 2);
    for (int b = threadIdx.x; b < (cnt << lq); b += blockDim.x) {
      const int sq = b >> lq, bb = b & ((1 << lq) - 1);
      const int pos = bb & (h - 1), base = (sq << lb) + ((bb >> l2) << lh) + pos;
      const int e = pos * s1;
      const float2 x0 = f[base], x1 = f[base + h], x2 = f[base + 2 * h], x3 = f[base + 3 * h];
      const float2 u = sp_add(x0, x2), v = sp_sub(x0, x2), c = sp_add(x1, x3), d = sp_sub(x1, x3);
      f[base] = sp_add(u, c);
      f[base + h] = sp_cmul(sp_sub(u, c), sp_tw<SIGN>(tw[2 * e]));
      f[base + 2 * h] = sp_cmul(sp_turn<SIGN>(v, d), sp_tw<SIGN>(tw[e]));
      f[base + 3 * h] = sp_cmul(sp_turn<-SIGN>(v, d), sp_tw<SIGN>(tw[3 * e]));
    }
    __syncthreads();
  }
}
__device__ __forceinline__ int sp_rev(int v, int bits) {
  return bits ? (int)(__brev((unsigned)v) >> (32 - bits)) : 0;
}
// Residue mod N1 of coefficient class a of workgroup `rank` (classes come in
// pairs r, N1 - r; 0 is paired with N1 / 2), h pairs per workgroup.
__device__ __forceinline__ int sp_class(int rank, int h, int a, int N1) {
  const int r = rank * h + (a >> 1);
  return (a & 1) ? (r ? N1 - r : N1 >> 1) : r;
}
// Global coefficient index k (of N) of coefficient slot e.
__device__ __forceinline__ int sp_coef(const Sp &R, int rank, int size, int e) {
  const int N1 = 1 << R.b1, h = (N1 / size) >> 1;
  const int a = e >> R.b2, k2 = sp_rev(e & ((1 << R.b2) - 1), R.b2);
  return sp_class(rank, h, a, N1) + (k2 << R.b1);
}
// z index (time order of the transform) of float f of a packed time slice.
__device__ __forceinline__ int sp_time(const Sp &R, int rank, int size, int f) {
  const int e = f >> 1, N2 = 1 << R.b2, cb = N2 / size;
  const int c = rank * cb + (e >> R.b1);
  const int s = c + (sp_rev(e & ((1 << R.b1) - 1), R.b1) << R.b2);
  return 2 * s + (f & 1);
}
// Calls f(eA, eB, k) for every pair of slots holding coefficients k and N - k
// (0 < k < N / 2 or its mirror), and f0(e) / fh(e) for k = 0 and k = N / 2.
template <class F, class F0, class FH>
__device__ __forceinline__ void sp_pairs(const Sp &R, int rank, int size, F &&f, F0 &&f0, FH &&fh) {
  const int N1 = 1 << R.b1, N2 = 1 << R.b2, h = (N1 / size) >> 1;
  for (int w = threadIdx.x; w < h * N2; w += blockDim.x) {
    const int b = w >> R.b2, e = w & (N2 - 1);
    const int r = rank * h + b;
    const int sa = (2 * b) << R.b2, sb = sa + N2;
    const int k2 = sp_rev(e, R.b2);
    if (r) {
      f(sa + e, sb + ((N2 - 1) ^ e), r + (k2 << R.b1));
    } else {
      // class 0: k2 with N2 - k2; class N1 / 2: k2 with N2 - 1 - k2
      if (k2 == 0) {
        f0(sa + e);
      } else if (k2 < (N2 >> 1)) {
        f(sa + e, sa + sp_rev(N2 - k2, R.b2), k2 << R.b1);
      } else if (k2 == (N2 >> 1)) {
        fh(sa + e);
      }
      if (k2 < (N2 >> 1)) f(sb + e, sb + ((N2 - 1) ^ e), (N1 >> 1) + (k2 << R.b1));
    }
  }
}

// ------------------------------------------------------------- products ----
// One product: publish the operand, one exchange that also reduces K pending
// doubles, consume.  Buffers of consecutive products differ (smv: the two
// directions; dct: parity), so no workgroup overwrites what a slower one reads.
template <int ENS>
struct SpOp;

template <>
struct SpOp<ENS_SMV> {
  // d0 = A s0 (and d1 = A s1); operands cut to the support where m is set, zero
  // outside it where not
  template <int NV, int K, int MAXES = 0>
  static __device__ __forceinline__ void A(RTeam &t, Sp &R, const XProblem &P, const float *s0,
                                           bool m0, const float *s1, bool m1, float *d0, float *d1,
                                           const double (&v)[K ? K : 1], double (&o)[K ? K : 1]) {
    XG(float) b0 = P.thres;
    XG(float) b1 = P.gprev_thres;
    for (int i = threadIdx.x; i < R.nlv; i += blockDim.x) {
      const bool in = (m0 || m1) ? sp_in(R, i) : true;
      st_dev(b0 + R.j0 + i, (m0 && !in) ? 0.f : s0[i]);
      if (NV == 2) st_dev(b1 + R.j0 + i, (m1 && !in) ? 0.f : s1[i]);
    }
    // the support bits go along the first time after they have changed (P.bins is
    // written at the end of a solve and read at the start of a continued one)
    const bool bits = R.fmask && R.fnew;
    XG(unsigned long long) fw = reinterpret_cast<XG(unsigned long long)>(P.bins);
    if (bits)
      for (int w = threadIdx.x; 64 * w < R.nlv; w += blockDim.x)
        st_dev_w(fw + (R.j0 >> 6) + w, R.mask[w]);
    rt_allreduce<K, MAXES>(t, *R.rt, v, o);
    if (threadIdx.x < WAVE) __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "agent");
    if (bits) {
      ld_dev_vec((float *)R.fmask, reinterpret_cast<XG(const float)>(P.bins), 2 * ((P.n + 63) >> 6));
      R.fnew = false;
    }
    __syncthreads();
    XG(const float) v0 = b0;
    XG(const float) v1 = b1;
    if (R.lcols)
      sp_gather_supp<NV>(R.lrp, R.lcols, P.rvals + R.rbase, 0, R.rlv, R.fmask, v0, v1, d0, d1);
    else if (R.fmask)
      sp_gather_supp<NV>(P.row_ptr, P.cols, P.rvals, R.i0, R.rlv, R.fmask, v0, v1, d0, d1);
    else
      sp_gather<NV>(P.row_ptr, P.cols, P.rvals, R.i0, R.rlv, P.nz / P.m, v0, v1, d0, d1);
  }
  // d = A^T s
  template <int K, int MAXES = 0>
  static __device__ __forceinline__ void AT(RTeam &t, Sp &R, const XProblem &P, float *s, float *d,
                                            const double (&v)[K ? K : 1], double (&o)[K ? K : 1]) {
    XG(float) b = P.resid;
    for (int i = threadIdx.x; i < R.rlv; i += blockDim.x) st_dev(b + R.i0 + i, s[i]);
    rt_allreduce<K, MAXES>(t, *R.rt, v, o);
    if (threadIdx.x < WAVE) __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "agent");
    __syncthreads();
    XG(const float) r = b;
    if (R.lrows)
      sp_gather<1>(R.lcp, R.lrows, R.lvals, 0, R.nlv, P.nz / P.n, r, r, d, nullptr);
    else
      sp_gather<1>(P.col_ptr, P.rows, P.vals, R.j0, R.nlv, P.nz / P.n, r, r, d, nullptr);
  }
};

template <>
struct SpOp<ENS_DCT> {
  static __device__ __forceinline__ XG(float2) buf(const XProblem &P, int parity, int v) {
    if (parity == 0) return P.cwork + (v ? (size_t)(P.n >> 1) : (size_t)0);
    return reinterpret_cast<XG(float2)>(v ? P.gprev_thres : P.thres);
  }
  template <int NV, int K, int MAXES = 0>
  static __device__ __forceinline__ void A(RTeam &t, Sp &R, const XProblem &P, const float *s0,
                                           bool m0, const float *s1, bool m1, float *d0, float *d1,
                                           const double (&v)[K ? K : 1], double (&o)[K ? K : 1]) {
    const int n = P.n, N1 = 1 << R.b1, N2 = 1 << R.b2, nc = R.nl >> 1;
    const int cb = N2 / t.size, c0 = t.rank * cb, lcb = 31 - __clz(cb);
    XG(const float2) tw = P.twiddle;
    for (int i = threadIdx.x; i < R.nl; i += blockDim.x) {
      const bool in = (m0 || m1) ? sp_in(R, i) : true;
      d0[i] = (m0 && !in) ? 0.f : s0[i];
      if (NV == 2) d1[i] = (m1 && !in) ? 0.f : s1[i];
    }
    __syncthreads();
    sp_dit<-1>((float2 *)d0, R.w1, R.b1, cb);
    if (NV == 2) sp_dit<-1>((float2 *)d1, R.w1, R.b1, cb);
    for (int e = threadIdx.x; e < nc; e += blockDim.x) {
      const int cl = e & (cb - 1), k1 = e >> lcb, c = c0 + cl;
      const float2 w = tw[(2 * c * k1) & (n - 1)];
      const size_t at = ((size_t)k1 << R.b2) + c;
      st_dev2(buf(P, R.mid, 0) + at, sp_cmul(((float2 *)d0)[(cl << R.b1) + k1], w));
      if (NV == 2) st_dev2(buf(P, R.mid, 1) + at, sp_cmul(((float2 *)d1)[(cl << R.b1) + k1], w));
    }
    rt_allreduce<K, MAXES>(t, *R.rt, v, o);
    const int h = (N1 / t.size) >> 1;
    for (int e = threadIdx.x; e < nc; e += blockDim.x) {
      const int r = sp_class(t.rank, h, e >> R.b2, N1);
      const size_t at = ((size_t)r << R.b2) + (e & (N2 - 1));
      ((float2 *)d0)[e] = ld_dev2(buf(P, R.mid, 0) + at);
      if (NV == 2) ((float2 *)d1)[e] = ld_dev2(buf(P, R.mid, 1) + at);
    }
    R.mid ^= 1;
    __syncthreads();
    sp_dif<-1>((float2 *)d0, R.w2, R.b2, 2 * h);
    coefs(t, R, P, (float2 *)d0);
    if (NV == 2) {
      sp_dif<-1>((float2 *)d1, R.w2, R.b2, 2 * h);
      coefs(t, R, P, (float2 *)d1);
    }
    __syncthreads();
  }
  // Packed spectrum to DCT-II coefficients: slot k becomes (X_k, X_{n-k}), slot
  // 0 (X_0, X_N); unsampled coefficients become 0.
  static __device__ __forceinline__ void coefs(const RTeam &t, const Sp &R, const XProblem &P,
                                               float2 *f) {
    const int n = P.n, N = n >> 1;
    XG(const float2) tw = P.twiddle;
    XG(const float2) qw = P.twiddle + n;
    const float w0 = (float)sqrt(1.0 / (double)n), w = (float)sqrt(2.0 / (double)n);
    auto put = [&](int e, float2 c, float2 q) {
      const unsigned long long bits = R.rmask[e >> 5] >> ((2 * e) & 63);
      f[e] = make_float2(
          (bits & 1) ? __fmul_rn(w, fmaf(c.x, q.x, __fmul_rn(c.y, q.y))) : 0.f,
          (bits & 2) ? __fmul_rn(w, fmaf(c.x, q.y, -__fmul_rn(c.y, q.x))) : 0.f);
    };
    sp_pairs(
        R, t.rank, t.size,
        [&](int ea, int eb, int k) {
          const float2 a = f[ea], b = f[eb];
          // E = (a + conj b) / 2, D = (a - conj b) / 2, C_k = E - i w_n^k D
          const float2 E = make_float2(0.5f * __fadd_rn(a.x, b.x), 0.5f * __fsub_rn(a.y, b.y));
          const float2 D = make_float2(0.5f * __fsub_rn(a.x, b.x), 0.5f * __fadd_rn(a.y, b.y));
          const float2 c = tw[k];
          put(ea, make_float2(fmaf(c.x, D.y, fmaf(c.y, D.x, E.x)), fmaf(-c.x, D.x, fmaf(c.y, D.y, E.y))), qw[k]);
          // C_{N-k} = conj(E + i w_n^k D)
          put(eb, make_float2(fmaf(-c.x, D.y, fmaf(-c.y, D.x, E.x)), -fmaf(c.x, D.x, fmaf(-c.y, D.y, E.y))),
              qw[N - k]);
        },
        [&](int e) {
          const float2 a = f[e];
          const unsigned long long bits = R.rmask[e >> 5] >> ((2 * e) & 63);
          f[e] = make_float2((bits & 1) ? __fmul_rn(w0, __fadd_rn(a.x, a.y)) : 0.f,
                             (bits & 2) ? __fmul_rn(w, __fmul_rn(__fsub_rn(a.x, a.y), qw[N].x)) : 0.f);
        },
        [&](int e) {
          const float2 a = f[e];
          put(e, make_float2(a.x, -a.y), qw[N >> 1]);
        });
  }
  // The inverse's packed spectrum from coefficient slots, in place.
  static __device__ __forceinline__ void spectrum(const RTeam &t, const Sp &R, const XProblem &P,
                                                  float2 *f) {
    const int n = P.n, N = n >> 1;
    XG(const float2) tw = P.twiddle;
    XG(const float2) qw = P.twiddle + n;
    const float w0 = (float)sqrt(1.0 / (double)n), w = (float)sqrt(2.0 / (double)n);
    // H = w / 2 ((a cos + b sin) + i (a sin - b cos))
    auto half = [&](float2 d, float2 q) {
      return make_float2(0.5f * __fmul_rn(w, fmaf(d.x, q.x, __fmul_rn(d.y, q.y))),
                         0.5f * __fmul_rn(w, fmaf(d.x, q.y, -__fmul_rn(d.y, q.x))));
    };
    sp_pairs(
        R, t.rank, t.size,
        [&](int ea, int eb, int k) {
          const float2 a = half(f[ea], qw[k]), b = half(f[eb], qw[N - k]);
          const float2 S = make_float2(__fadd_rn(a.x, b.x), __fsub_rn(a.y, b.y));
          const float2 D = make_float2(__fsub_rn(a.x, b.x), __fadd_rn(a.y, b.y));
          const float2 c = tw[k];  // u = e^{2 pi i k / n} D = conj(c) D
          f[ea] = make_float2(fmaf(-c.x, D.y, fmaf(c.y, D.x, S.x)), fmaf(c.x, D.x, fmaf(c.y, D.y, S.y)));  // S + i u
          f[eb] = make_float2(fmaf(c.x, D.y, fmaf(-c.y, D.x, S.x)), fmaf(c.x, D.x, fmaf(c.y, D.y, -S.y)));  // conj S + i conj u
        },
        [&](int e) {
          const float2 d = f[e];
          const float h0 = __fmul_rn(w0, d.x), hN = __fmul_rn(w, __fmul_rn(d.y, qw[N].x));
          f[e] = make_float2(__fadd_rn(h0, hN), __fsub_rn(h0, hN));
        },
        [&](int e) {
          const float2 H = half(f[e], qw[N >> 1]);
          f[e] = make_float2(2.0f * H.x, -2.0f * H.y);
        });
  }
  // d = A^T s; s is destroyed
  template <int K, int MAXES = 0>
  static __device__ __forceinline__ void AT(RTeam &t, Sp &R, const XProblem &P, float *s, float *d,
                                            const double (&v)[K ? K : 1], double (&o)[K ? K : 1]) {
    const int n = P.n, N1 = 1 << R.b1, N2 = 1 << R.b2, nc = R.nl >> 1;
    const int cb = N2 / t.size, c0 = t.rank * cb;
    const int rb = N1 / t.size, h = rb >> 1, lrb = 31 - __clz(rb);
    XG(const float2) tw = P.twiddle;
    XG(float2) mid = buf(P, R.mid, 0);
    __syncthreads();
    spectrum(t, R, P, (float2 *)s);
    __syncthreads();
    sp_dit<1>((float2 *)s, R.w2, R.b2, rb);
    // mid'[q2][position of the class]: a workgroup's classes lie side by side
    for (int e = threadIdx.x; e < nc; e += blockDim.x) {
      const int a = e & (rb - 1), q2 = e >> lrb;
      const int r = sp_class(t.rank, h, a, N1);
      const float2 w = tw[(2 * r * q2) & (n - 1)];
      st_dev2(mid + ((size_t)q2 << R.b1) + t.rank * rb + a,
              sp_cmul(((float2 *)s)[(a << R.b2) + q2], make_float2(w.x, -w.y)));
    }
    rt_allreduce<K, MAXES>(t, *R.rt, v, o);
    for (int e = threadIdx.x; e < nc; e += blockDim.x) {
      const int cl = e >> R.b1, pos = e & (N1 - 1);
      const int r = sp_class(pos >> lrb, h, pos & (rb - 1), N1);
      ((float2 *)d)[(cl << R.b1) + r] = ld_dev2(mid + ((size_t)(c0 + cl) << R.b1) + pos);
    }
    R.mid ^= 1;
    __syncthreads();
    sp_dif<1>((float2 *)d, R.w1, R.b1, cb);
  }
};

// ------------------------------------------------------ support selection --
// One hop that gathers an int per workgroup (thread 0's) and returns, to every
// thread, the first workgroup at which the running sum reaches k (-1: none),
// the sum before it and the total.
__device__ __forceinline__ int rt_crossing(RTeam &t, int mine, int k, int *before, int *total) {
  __shared__ int s_res[4];
  *before = *total = 0;
  if (t.aborted) return -1;
  t.tag++;
  __syncthreads();
  if (threadIdx.x < WAVE) {
    const int lane = threadIdx.x;
    const unsigned long long T = (unsigned long long)t.tag << 32;
    unsigned long long *bank = reinterpret_cast<unsigned long long *>(t.bar + BAR_LINE) +
                               (size_t)(t.tag & 1u) * (2 * RT_KMAX) * BAR_MAX_TEAM;
    if (lane == 0)
      __hip_atomic_store(&bank[t.rank], T | (unsigned)mine, __ATOMIC_RELAXED,
                         __HIP_MEMORY_SCOPE_AGENT);
    int run = 0, wc = -1, pre = 0, bad = 0;
    for (int r0 = 0; r0 < t.size && !bad; r0 += WAVE) {
      const int r = r0 + lane;
      unsigned long long w;
      long spins = 0;
      while (true) {
        w = T;
        if (r < t.size)
          w = __hip_atomic_load(&bank[r], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        if (__all((unsigned)(w >> 32) == t.tag)) break;
        if (++spins > t.spin_limit ||
            ((spins & 1023) == 0 &&
             __hip_atomic_load(&t.bar[2], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) != 0u)) {
          bad = 1;
          break;
        }
      }
      const int c = r < t.size ? (int)(unsigned)w : 0;
      const int incl = run + wscan_i(c);
      const unsigned long long cross = __ballot(incl >= k);
      if (wc < 0 && cross) {
        const int l = __ffsll(cross) - 1;
        wc = r0 + l;
        pre = __builtin_amdgcn_readlane(incl - c, l);
      }
      run = __builtin_amdgcn_readlane(incl, 63);
    }
    if (lane == 0) {
      s_res[0] = wc;
      s_res[1] = pre;
      s_res[2] = run;
      s_res[3] = bad;
      if (bad) __hip_atomic_store(&t.bar[2], 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    }
  }
  __syncthreads();
  *before = s_res[1];
  *total = s_res[2];
  if (s_res[3]) t.aborted = 1;
  return s_res[0];
}

__device__ __forceinline__ int ld_dev_i(XG(const int) p) {
  return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

// The first bin of [base, base + len) at which before + the running count
// reaches k, read by `cnt(b)`: every wave walks for itself.  *sum: the count.
template <class Cnt>
__device__ __forceinline__ int sp_walk(Cnt &&cnt, int base, int len, int before, int k, int *sum) {
  const int lane = threadIdx.x & (WAVE - 1);
  const int chunk = ((len + WAVE - 1) / WAVE) | 1;
  const int lo = min(len, lane * chunk), hi = min(len, lo + chunk);
  int c = 0;
  for (int b = lo; b < hi; b++) c += cnt(base + b);
  const int incl = before + wscan_i(c);
  const unsigned long long cross = __ballot(incl >= k);
  if (cross == 0ull) {
    *sum = __builtin_amdgcn_readlane(incl, 63);
    return base + len - 1;
  }
  const int l = __ffsll(cross) - 1;
  int acc = incl - c, b = lo;
  if (lane == l)
    for (; b < hi; b++) {
      acc += cnt(base + b);
      if (acc >= k) break;
    }
  *sum = __builtin_amdgcn_readlane(acc, l);
  return base + __builtin_amdgcn_readlane(b, l);
}

// FindSupportSet's binning branch (functions.cu:404-428) on the team's x with
// max |x| = S.max_value, the threshold and the mask of the own slice.  Returns
// the thread's part of the number of mask words from which an entry left.
// Counters: two arrays used in turn, each workgroup zeroing its part of the
// other one meanwhile.  Up to SP_HIST bins are counted in LDS first and read
// back whole by every workgroup; beyond that only entries above the bins' lower
// end are counted at all (a few times k), straight into memory, each workgroup
// sums its share of the bins and one more hop finds the share with the crossing.
__device__ __forceinline__ double sp_rebin(RTeam &t, Sp &R, const XProblem &P, ResS &S) {
  const int nt = blockDim.x, lane = threadIdx.x & (WAVE - 1);
  S.slope = (float)(P.num_bins - 1) / S.max_value;
  const float slope = S.slope, inter = S.max_value;
  const int mb = S.max_bin, nb = P.num_bins;
  XG(int) cur = R.par ? P.bins2 : P.counters;
  XG(int) other = R.par ? P.counters : P.bins2;
  R.par ^= 1;
  const int cb = (nb + t.size - 1) / t.size, lo = min(nb, t.rank * cb), hi = min(nb, lo + cb);
  for (int b = lo + threadIdx.x; b < hi; b += nt)
    __hip_atomic_store(other + b, 0, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  const bool lds = nb <= SP_HIST;
  for (int i = threadIdx.x; i < R.nlv; i += nt) {
    const float v = R.x[i];
    const int b = linear_bin(v, slope, inter);
    if ((double)fabsf(v) > (double)inter * .000001 && b < mb) {
      if (lds)
        atomicAdd(&R.hist[b], 1);
      else
        __hip_atomic_fetch_add(cur + b, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    }
  }
  if (lds) {
    __syncthreads();
    for (int b = threadIdx.x; b < mb; b += nt)
      if (R.hist[b])
        __hip_atomic_fetch_add(cur + b, R.hist[b], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  }
  double z[1] = {0.0};
  rt_allreduce<0>(t, *R.rt, z, z);
  int kb = -1, sum = 0;
  if (P.k > 0) {
    if (lds) {
      for (int b = threadIdx.x; b < mb; b += nt) R.hist[b] = ld_dev_i(cur + b);
      __syncthreads();
      kb = sp_walk([&](int b) { return R.hist[b]; }, 0, mb, 0, P.k, &sum);
      __syncthreads();
    } else {
      int c = 0;  // this workgroup's share, by its first wave
      if (threadIdx.x < WAVE) {
        for (int b = lo + lane; b < min(hi, mb); b += WAVE) c += ld_dev_i(cur + b);
        c = __builtin_amdgcn_readlane(wscan_i(c), 63);
      }
      int before, total;
      const int wc = rt_crossing(t, c, P.k, &before, &total);
      if (wc < 0) {
        kb = mb - 1;
        sum = total;
      } else {
        const int base = min(mb, wc * cb);
        kb = sp_walk([&](int b) { return ld_dev_i(cur + b); }, base, min(mb, base + cb) - base,
                     before, P.k, &sum);
      }
    }
  }
  if (lds)
    for (int b = threadIdx.x; b < mb; b += nt) R.hist[b] = 0;
  if (sum < P.k) {
    S.alpha_bin = S.alpha_bin * 0.5f;
    S.max_bin = (int)((float)nb * (1.0f - S.alpha_bin));
  }
  S.min_val = __fsub_rn(inter, __fdiv_rn((float)(kb + 1), slope));
  S.sum = sum;
  S.k_bin = kb;
  double left = 0.0;
  for (int j0 = 0; j0 < R.nl; j0 += nt) {
    const int i = j0 + threadIdx.x;
    const bool in = i < R.nlv && linear_bin(R.x[i], slope, inter) <= kb;
    if (i < R.nlv && !in) R.x[i] = 0.f;
    const unsigned long long bits = __ballot(in);
    if (lane == 0 && i < R.nl) {
      if (R.mask[i >> 6] & ~bits) left = 1.0;
      R.mask[i >> 6] = bits;
    }
  }
  R.fnew = true;
  __syncthreads();
  return left;
}

// sum of squares of a thread's share of a slice
__device__ __forceinline__ double sp_sq(const float *v, int len) {
  double a = 0.0;
  for (int i = threadIdx.x; i < len; i += blockDim.x) a += (double)v[i] * (double)v[i];
  return a;
}
// t0 = y - t0; the thread's part of its norm squared
__device__ __forceinline__ double sp_resid(const Sp &R) {
  double e2 = 0.0;
  for (int i = threadIdx.x; i < R.rlv; i += blockDim.x) {
    const float r = __fsub_rn(R.y[i], R.t0[i]);
    R.t0[i] = r;
    e2 += (double)r * (double)r;
  }
  return e2;
}

// CG projection on the support (cg_projection of xcs_solver.h): direction in p,
// CG residual in g, both zero off the support.  Returns errCG.
template <int ENS>
__device__ __forceinline__ float sp_cg_projection(RTeam &t, Sp &R, const XProblem &P, ResS &S,
                                                  int max_steps) {
  typedef SpOp<ENS> Op;
  const float tolCG = P.tol * P.tol;
  const float tol2 = 10.0f * tolCG;
  const int nt = blockDim.x;
  double z[1] = {0.0}, v1[1], o1[1], v2[2], o2[2];
  const double bA = op_bytes(P, false, 0), bT = op_bytes(P, true, 0);
  S.bytes += bA + bT;
  Op::template A<1, 0>(t, R, P, R.x, false, nullptr, false, R.t0, nullptr, z, z);
  v1[0] = sp_resid(R);
  Op::template AT<1>(t, R, P, R.t0, R.g, v1, o1);
  float errCG = (float)o1[0];
  v1[0] = 0.0;
  for (int i = threadIdx.x; i < R.nlv; i += nt) {
    const float th = sp_in(R, i) ? R.g[i] : 0.f;
    R.g[i] = th;
    R.p[i] = th;
    v1[0] += (double)th * (double)th;
  }
  rt_allreduce<1>(t, *R.rt, v1, o1);
  S.mu = (float)o1[0];
  float hist = (threadIdx.x & (WAVE - 1)) == 15 ? errCG : 0.f, evo = 1.f, diff = 1.f;
  float *ad = R.t0;  // A d
  double a2 = 0.0;
  for (int it = 0; !t.aborted && ((errCG > tolCG) & (it < max_steps) & (diff > tol2)); it++) {
    if (it == 0) {
      S.bytes += bA;
      Op::template A<1, 0>(t, R, P, R.p, false, nullptr, false, R.t0, nullptr, z, z);
      v1[0] = sp_sq(R.t0, R.rlv);
      rt_allreduce<1>(t, *R.rt, v1, o1);
      a2 = o1[0];
    }
    float alpha = (float)a2;
    alpha = (S.mu < 1000.0f * alpha) ? S.mu / alpha : 0.f;
    S.bytes += bT;
    Op::template AT<0>(t, R, P, ad, R.q, z, z);
    v1[0] = 0.0;
    for (int i = threadIdx.x; i < R.nlv; i += nt) {
      const float th = sp_in(R, i) ? R.q[i] : 0.f;
      const float gp = fmaf(-alpha, th, R.g[i]);
      R.g[i] = gp;
      v1[0] += (double)gp * (double)gp;
    }
    rt_allreduce<1>(t, *R.rt, v1, o1);
    float beta = S.mu;
    S.mu = (float)o1[0];
    beta = (S.mu < 1000.0f * beta) ? S.mu / beta : 0.f;
    for (int i = threadIdx.x; i < R.nlv; i += nt) {
      R.x[i] = fmaf(alpha, R.p[i], R.x[i]);
      R.p[i] = __fadd_rn(__fmul_rn(beta, R.p[i]), R.g[i]);
    }
    // the new residual and, unless this was the last allowed step, the next A d
    const bool next = it + 1 < max_steps;
    S.bytes += next ? 2.0 * bA : bA;
    __syncthreads();
    if (next) {
      Op::template A<2, 0>(t, R, P, R.x, false, R.p, false, R.t0, R.t1, z, z);
      v2[1] = sp_sq(R.t1, R.rlv);
    } else {
      Op::template A<1, 0>(t, R, P, R.x, false, nullptr, false, R.t0, nullptr, z, z);
      v2[1] = 0.0;
    }
    ad = R.t1;
    v2[0] = sp_resid(R);
    rt_allreduce<2>(t, *R.rt, v2, o2);
    errCG = (float)o2[0];
    a2 = o2[1];
    hist = hist_push(hist, errCG);
    evo = hist_push(evo, __fsub_rn(lane_f(hist, 14), lane_f(hist, 15)));
    diff = hist_max(evo);
  }
  return errCG;
}

// Index of element i of the n-slice in the caller's vectors.
template <int ENS>
__device__ __forceinline__ int sp_column(const Sp &R, const RTeam &t, int n, int i) {
  if (ENS != ENS_DCT) return R.j0 + i;
  const int z = sp_time(R, t.rank, t.size, i);
  return z < n / 2 ? 2 * z : 2 * (n - 1 - z) + 1;
}
// The workgroup's slices in LDS for an instance of `alg`, with y (slots and rt are
// the kernel's own); the smv entries are staged by the solve.
template <int ENS>
__device__ __forceinline__ SplitGeom sp_open(Sp &R, const RTeam &t, const XProblem &P, int alg,
                                             unsigned char *lds) {
  const int lane = threadIdx.x & (WAVE - 1), nt = blockDim.x, n = P.n;
  const SplitGeom G = split_geom(ENS, alg, P.m, n, P.log2n, P.num_bins, t.size);
  {
    unsigned char *q = lds;
    auto take = [&](size_t b) {
      unsigned char *r = q;
      q += res_up16(b);
      return r;
    };
    R.nl = G.nl;
    R.rl = G.rl;
    R.b1 = G.b1;
    R.b2 = G.b2;
    R.x = (float *)take(4 * (size_t)G.nl);
    R.g = (float *)take(4 * (size_t)G.nl);
    R.p = (float *)take(4 * (size_t)G.nl);
    R.q = alg == ALG_HTP ? (float *)take(4 * (size_t)G.nl) : nullptr;
    R.y = (float *)take(4 * (size_t)G.rl);
    R.t0 = (float *)take(4 * (size_t)G.rl);
    R.t1 = (float *)take(4 * (size_t)G.rl);
    R.mask = (unsigned long long *)take((size_t)G.nl / 8 + 8);
    R.hist = (int *)take(4 * (size_t)sp_hist(P.num_bins));
    R.rmask = nullptr;
    R.w1 = R.w2 = nullptr;
    if (ENS == ENS_DCT) {
      R.rmask = (unsigned long long *)take((size_t)G.rl / 8 + 8);
      float2 *w1 = (float2 *)take(8 * sp_twiddles(G.b1));
      float2 *w2 = (float2 *)take(8 * sp_twiddles(G.b2));
      for (int k = threadIdx.x; k < (int)sp_twiddles(G.b1); k += nt)
        w1[k] = P.twiddle[(size_t)k << (P.log2n - G.b1)];
      for (int k = threadIdx.x; k < (int)sp_twiddles(G.b2); k += nt)
        w2[k] = P.twiddle[(size_t)k << (P.log2n - G.b2)];
      R.w1 = w1;
      R.w2 = w2;
    }
  }
  R.fmask = nullptr;
  R.fnew = true;
  R.lrp = R.lcols = R.lcp = R.lrows = nullptr;
  R.lvals = nullptr;
  R.rbase = 0;
  if (G.filter) R.fmask = (unsigned long long *)(lds + G.lds);
  R.bank = R.par = R.mid = 0;
  // slices: smv contiguous columns and rows, dct the owned packed slots
  R.j0 = min(n, t.rank * G.nl);
  R.i0 = min(P.m, t.rank * G.rl);
  R.nlv = ENS == ENS_DCT ? G.nl : min(G.nl, n - R.j0);
  R.rlv = ENS == ENS_DCT ? G.rl : min(G.rl, P.m - R.i0);
  if (ENS == ENS_DCT) {
    for (int j0 = 0; j0 < R.rl; j0 += nt) {
      const int i = j0 + threadIdx.x;
      int pos = -1;
      if (i < R.rl) {
        const int k = sp_coef(R, t.rank, t.size, i >> 1);
        pos = P.dct_pos[(i & 1) ? (k ? n - k : n >> 1) : k];
        R.y[i] = pos >= 0 ? P.y[pos] : 0.f;
      }
      const unsigned long long bits = __ballot(pos >= 0);
      if (lane == 0 && i < R.rl) R.rmask[i >> 6] = bits;
    }
  } else {
    for (int i = threadIdx.x; i < R.rlv; i += nt) R.y[i] = P.y[R.i0 + i];
  }
  return G;
}

// One instance by the whole (cooperatively launched) grid: at most `budget`
// outer iterations from the saved state.
template <int ENS, int ALG>
__global__ void __launch_bounds__(SP_THREADS) solve_split_kernel(const XProblem *Pp, int budget,
                                                                 unsigned *bar, long spin_limit) {
  typedef SpOp<ENS> Op;
  constexpr bool CG = ALG == ALG_CGIHT;
  __shared__ __attribute__((aligned(16))) unsigned char lds[SP_LDS];
  __shared__ XProblem sP;
  __shared__ WgSlots slots;
  __shared__ RtSlots rt;
  if (threadIdx.x == 0) sP = *Pp;
  __syncthreads();
  const XProblem &P = sP;
  if (P.st->done) return;
  const int lane = threadIdx.x & (WAVE - 1), nt = blockDim.x, n = P.n;
  RTeam t{(int)blockIdx.x, (int)gridDim.x, bar, bar[1], spin_limit, 0};
  Sp R;
  const SplitGeom G = sp_open<ENS>(R, t, P, ALG, lds);
  R.slots = &slots;
  R.rt = &rt;
  auto column = [&](int i) { return sp_column<ENS>(R, t, n, i); };
  if (ENS == ENS_SMV && G.filter) {
    // the matrix entries do not change during a solve
    unsigned char *q = lds + G.lds + res_up16((size_t)n / 8 + 8);
    auto take = [&](int words) {
      unsigned char *r = q;
      q += res_up16(4 * (size_t)words);
      return r;
    };
    R.rbase = P.row_ptr[R.i0];
    const int rn = P.row_ptr[R.i0 + R.rlv] - R.rbase;
    const int cbase = P.col_ptr[R.j0], cn = P.col_ptr[R.j0 + R.nlv] - cbase;
    const SplitStage T = split_stage(G, n, R.rlv, R.nlv, rn, cn);
    if (T.rows) {
      int *rp = (int *)take(R.rlv + 1), *cols = (int *)take(rn);
      for (int i = threadIdx.x; i <= R.rlv; i += nt) rp[i] = P.row_ptr[R.i0 + i] - R.rbase;
      for (int e = threadIdx.x; e < rn; e += nt) cols[e] = P.cols[R.rbase + e];
      R.lrp = rp;
      R.lcols = cols;
    }
    if (T.cols) {
      int *cp = (int *)take(R.nlv + 1), *rows = (int *)take(cn);
      float *vals = (float *)take(cn);
      for (int i = threadIdx.x; i <= R.nlv; i += nt) cp[i] = P.col_ptr[R.j0 + i] - cbase;
      for (int e = threadIdx.x; e < cn; e += nt) {
        rows[e] = P.rows[cbase + e];
        vals[e] = P.vals[cbase + e];
      }
      R.lcp = cp;
      R.lrows = rows;
      R.lvals = vals;
    }
  }
  for (int b = threadIdx.x; b < sp_hist(P.num_bins); b += nt) R.hist[b] = 0;
  for (int w = threadIdx.x; w <= R.nl / 64; w += nt) R.mask[w] = 0ull;
  {  // both counter arrays start at zero (read after the first exchanges)
    const int cb = (P.num_bins + t.size - 1) / t.size, lo = t.rank * cb;
    for (int b = lo + threadIdx.x; b < min(P.num_bins, lo + cb); b += nt) {
      __hip_atomic_store(P.counters + b, 0, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      __hip_atomic_store(P.bins2 + b, 0, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    }
  }
  float prev = 0.f, evo = 1.f;
  ResS S;
  ResStop Q;
  double z[1] = {0.0}, v1[1], o1[1];
  const double bA = op_bytes(P, false, 0), bT = op_bytes(P, true, 0);
  auto trace = [&](int idx, int kb, float e) {
    if (t.rank == 0 && threadIdx.x == 0) {
      if (P.trace_kbin) P.trace_kbin[idx] = kb;
      if (P.trace_err) P.trace_err[idx] = e;
    }
  };
  bool zero = false;
  double left = 0.0;  // support words an entry left at the last selection (this thread's)
  if (P.st->initialized) {
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
    if (CG && S.supp_change) left = threadIdx.x == 0 ? 1.0 : 0.0;
    __syncthreads();
    for (int j0 = 0; j0 < R.nl; j0 += nt) {
      const int i = j0 + threadIdx.x;
      const bool ok = i < R.nlv;
      const int j = ok ? column(i) : 0;
      if (ok) {
        R.x[i] = P.x[j];
        R.p[i] = P.gprev[j];
      }
      const unsigned long long bits = __ballot(ok && P.bins[j] <= S.k_bin);
      if (lane == 0 && i < R.nl) R.mask[i >> 6] = bits;
    }
    rt_allreduce<0>(t, rt, z, z);  // counters zero everywhere
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
    S.bytes = bT;
    Q.diff = 1.f;
    Q.iter = 0;
    Q.fail = 0;
    Q.cycle = 1;
    __syncthreads();
    v1[0] = sp_sq(R.y, R.rlv);
    for (int i = threadIdx.x; i < R.rlv; i += nt) R.t0[i] = R.y[i];
    for (int i = threadIdx.x; i < R.nl; i += nt) R.p[i] = 0.f;
    Op::template AT<1>(t, R, P, R.t0, R.x, v1, o1);
    Q.err = Q.err_start = (float)sqrt(o1[0]);
    v1[0] = 0.0;
    for (int i = threadIdx.x; i < R.nlv; i += nt) v1[0] = fmax(v1[0], (double)fabsf(R.x[i]));
    rt_allreduce<1, 1>(t, rt, v1, o1);
    S.max_value = (float)o1[0];
    zero = S.max_value == 0.f;  // A^T y == 0: x = 0 is returned
    if (!zero) {
      (void)sp_rebin(t, R, P, S);
      trace(0, S.k_bin, Q.err);
      if (CG) {
        // r^0 and its gradient as the first direction (algorithms.cu:3762-3808)
        S.bytes += bA + bT;
        Op::template A<1, 0>(t, R, P, R.x, false, nullptr, false, R.t0, nullptr, z, z);
        v1[0] = sp_resid(R);
        Op::template AT<1>(t, R, P, R.t0, R.p, v1, o1);
        Q.err = (float)sqrt(o1[0]);
        if (lane == 15) prev = Q.err;
        evo = hist_push(evo, __fsub_rn(0.f, Q.err));
        left = threadIdx.x == 0 ? 1.0 : 0.0;  // supp_change = 1
      }
    }
  }
  int reason = 0;
  while (!zero && budget > 0 && !t.aborted && res_continue(Q, P, &reason)) {
    budget--;
    // residual rows; the exchange brings whether the last selection lost an entry
    S.bytes += bA + bT;
    if (CG) {
      v1[0] = left;
      Op::template A<1, 1>(t, R, P, R.x, false, nullptr, false, R.t0, nullptr, v1, o1);
      S.supp_change = o1[0] > 0.0 ? 1 : 0;
      if (S.supp_change && P.restart && Q.iter > 0) S.beta_to_zero = 1;
    } else {
      Op::template A<1, 0>(t, R, P, R.x, false, nullptr, false, R.t0, nullptr, z, z);
    }
    v1[0] = sp_resid(R);
    Op::template AT<1>(t, R, P, R.t0, R.g, v1, o1);
    const float norm = (float)sqrt(o1[0]);  // |r| at the start of the iteration
    const bool uncg = CG && !P.restart && S.supp_change;
    const float *dir = CG ? R.p : R.g;
    float step, dmax;
    if (!uncg) {
      // RestrictedSD (NIHT, HTP: functions.cu:659-745) and the restricted CG step
      // with support evolution (functions.cu:1004-1102)
      double w2[2] = {0.0, 0.0}, r2[2];
      for (int i = threadIdx.x; i < R.nlv; i += nt) {
        const float g = R.g[i];
        if (sp_in(R, i)) w2[0] += (double)g * (double)g;
        w2[1] = fmax(w2[1], (double)fabsf(g));
      }
      S.bytes += bA;
      if (CG) {
        v1[0] = w2[0];
        rt_allreduce<1>(t, rt, v1, o1);
        float beta = 0.f;
        const float mu_new = (float)o1[0];
        if (S.beta_to_zero != 1) beta = (mu_new < 1000.0f * S.mu) ? mu_new / S.mu : 0.f;
        S.mu = mu_new;
        w2[1] = 0.0;
        for (int i = threadIdx.x; i < R.nlv; i += nt) {
          const float gp = __fadd_rn(__fmul_rn(beta, R.p[i]), R.g[i]);
          R.p[i] = gp;
          w2[1] = fmax(w2[1], (double)fabsf(gp));
        }
        __syncthreads();
        Op::template A<1, 0>(t, R, P, R.p, true, nullptr, false, R.t0, nullptr, z, z);
        w2[0] = sp_sq(R.t0, R.rlv);
        rt_allreduce<2, 2>(t, rt, w2, r2);
        const float a = (float)r2[0];
        step = (S.mu < 1000.0f * a) ? S.mu / a : 0.f;
        dmax = (float)r2[1];
      } else {
        Op::template A<1, 2, 2>(t, R, P, R.g, true, nullptr, false, R.t0, nullptr, w2, r2);
        v1[0] = sp_sq(R.t0, R.rlv);
        rt_allreduce<1>(t, rt, v1, o1);
        const float err = (float)sqrt(o1[0]);
        const float mu = (float)sqrt(r2[0]);
        step = mu / err;
        step = (mu < 400.0f * err) ? step * step : 0.f;
        dmax = (float)r2[1];
      }
    } else {
      // UnrestrictedCG (functions.cu:1107-1220): A p_old,S and A g_S together
      S.bytes += 2.0 * bA;
      Op::template A<2, 0>(t, R, P, R.p, true, R.g, true, R.t0, R.t1, z, z);
      float beta = 0.f;
      if (S.beta_to_zero != 1) {
        double v2[2] = {0.0, 0.0}, o2[2];
        for (int i = threadIdx.x; i < R.rlv; i += nt) {
          const double ap = R.t0[i], ag = R.t1[i];
          v2[0] += ap * ag;
          v2[1] += ap * ap;
        }
        rt_allreduce<2>(t, rt, v2, o2);
        beta = -((float)o2[0]) / (float)o2[1];
      }
      double v4[4] = {0.0, 0.0, 0.0, 0.0}, o4[4];  // p.g_S, |g_S|^2, |A p_S|^2, max |p|
      for (int i = threadIdx.x; i < R.nlv; i += nt) {
        const float g = R.g[i];
        const float gp = __fadd_rn(__fmul_rn(beta, R.p[i]), g);
        R.p[i] = gp;
        v4[3] = fmax(v4[3], (double)fabsf(gp));
        if (sp_in(R, i)) {
          v4[0] += (double)gp * (double)g;
          v4[1] += (double)g * (double)g;
        }
      }
      for (int i = threadIdx.x; i < R.rlv; i += nt) {
        const float r = __fadd_rn(__fmul_rn(beta, R.t0[i]), R.t1[i]);
        v4[2] += (double)r * (double)r;
      }
      rt_allreduce<4, 8>(t, rt, v4, o4);
      step = (float)o4[0] / (float)o4[2];
      S.mu = (float)o4[1];
      dmax = (float)o4[3];
    }
    double xm[1] = {0.0};
    for (int i = threadIdx.x; i < R.nlv; i += nt) {
      const float xn = fmaf(step, dir[i], R.x[i]);
      R.x[i] = xn;
      xm[0] = fmax(xm[0], (double)fabsf(xn));
    }
    S.max_change = 2.0f * step * dmax;
    // support update (the skip rule of FindSupportSet, functions.cu:400-403)
    if (CG) S.beta_to_zero = 0;
    if (S.min_val <= S.max_change) {
      rt_allreduce<1, 1>(t, rt, xm, o1);
      S.max_value = (float)o1[0];
      left = sp_rebin(t, R, P, S);
    } else {
      left = 0.0;
      S.min_val = S.min_val - S.max_change;
      for (int i = threadIdx.x; i < R.nlv; i += nt)
        if (!sp_in(R, i)) R.x[i] = 0.f;
      __syncthreads();
    }
    prev = hist_push(prev, norm);
    Q.err = norm;
    if (ALG == ALG_HTP) {
      Q.err = sqrtf(sp_cg_projection<ENS>(t, R, P, S, 15));
      prev = hist_push(prev, Q.err);
    }
    res_stop_update(Q, prev, &evo, ALG == ALG_HTP ? 125 : 749);
    Q.iter++;
    trace(Q.iter, S.k_bin, Q.err);
  }
  if (CG && !zero) {  // the saved state's supp_change (and restart), pending from the last selection
    v1[0] = left;
    rt_allreduce<1>(t, rt, v1, o1);
    S.supp_change = o1[0] > 0.0 ? 1 : 0;
    if (S.supp_change && P.restart) S.beta_to_zero = 1;
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
  for (int i = threadIdx.x; i < R.nlv; i += nt) {
    const int j = column(i);
    P.x[j] = R.x[i];
    P.gprev[j] = R.p[i];
    P.bins[j] = sp_in(R, i) ? S.k_bin : S.k_bin + 1;
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
      st->supp_count = S.sum;
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

// y = A x of a generated instance (x in memory) by the solve's own product in the
// solve's geometry (see resident_y_kernel): the planted vector leaves no residual.
// dct 2^20, m = 2^18 + 1: with the general form's y an NIHT solve to 1e-5 stalled at
// 1.15e-5 for 32 iterations, with this one it takes 16.
template <int ENS>
__global__ void __launch_bounds__(SP_THREADS) split_y_kernel(const XProblem *Pp, int alg, const float *x,
                                                             float *y, unsigned *bar, long spin_limit) {
  __shared__ __attribute__((aligned(16))) unsigned char lds[SP_LDS];
  __shared__ XProblem sP;
  __shared__ WgSlots slots;
  __shared__ RtSlots rt;
  if (threadIdx.x == 0) sP = *Pp;
  __syncthreads();
  const XProblem &P = sP;
  const int n = P.n;
  RTeam t{(int)blockIdx.x, (int)gridDim.x, bar, bar[1], spin_limit, 0};
  Sp R;
  (void)sp_open<ENS>(R, t, P, alg, lds);
  R.slots = &slots;
  R.rt = &rt;
  for (int j0 = 0; j0 < R.nl; j0 += blockDim.x) {
    const int i = j0 + threadIdx.x;
    const float v = i < R.nlv ? x[sp_column<ENS>(R, t, n, i)] : 0.f;
    if (i < R.nl) R.x[i] = v;
    const unsigned long long bits = __ballot(v != 0.f);
    if ((threadIdx.x & (WAVE - 1)) == 0 && i < R.nl) R.mask[i >> 6] = bits;
  }
  __syncthreads();
  double z[1] = {0.0};
  SpOp<ENS>::template A<1, 0>(t, R, P, R.x, false, nullptr, false, R.t0, nullptr, z, z);
  for (int i = threadIdx.x; i < R.rlv; i += blockDim.x) {
    if (ENS == ENS_DCT) {
      const int k = sp_coef(R, t.rank, t.size, i >> 1), pos = P.dct_pos[(i & 1) ? (k ? n - k : n >> 1) : k];
      if (pos >= 0) y[pos] = R.t0[i];
    } else {
      y[R.i0 + i] = R.t0[i];
    }
  }
}

}  // namespace xcs
