// Team-level greedy recovery: ensemble operators and the four algorithms.
//
// Every routine here is executed by all threads of all workgroups of a team
// (see xcs_device.h).  Scalars live in registers and are computed redundantly
// and identically by every thread, so control flow is uniform.  Vectors live
// in global memory; "strided ownership" means index i of a length-L vector is
// handled by team thread i mod gsize, so chained elementwise passes need no
// barrier.  Barriers (t.sync) are placed where another thread's writes are read.
//
// Reference semantics followed (file:line in the reference):
//   NIHT    GAGA/gaga/algorithms.cu:1274-1441, RestrictedSD functions.cu:659-745
//   HTP     algorithms.cu:2491-2716, RestrictedCG functions.cu:922-1000
//   CSMPSP  algorithms.cu:3372-3674
//   CGIHT   algorithms.cu:3689-3942, functions.cu:1004-1102 (restricted step),
//           functions.cu:1107-1220 (unrestricted step)
//   support selection functions.cu:374-436, kernels.cu:64-81, 135-193
// Inner products: per-thread partials in FP32 (residual norms in FP64), the
// cross-thread combination in FP64, rounded to FP32 for the step logic; the
// residual-norm history is FP32 like the reference's.
#pragma once
#include "xcs_device.h"
#include "xcs_engine.h"
#include "xcs_fft.h"

namespace xcs {

// ------------------------------------------------------------ gen ----------
// Columns whose loads the gather issues together (per lane, one float4 each)
// and float4 loads per lane and column the dense A^T r keeps in flight.
#ifndef XCS_GATHER_U
#define XCS_GATHER_U 4
#endif
#ifndef XCS_AT_U
#define XCS_AT_U 4
#endif
constexpr int GATHER_U = XCS_GATHER_U;

// out[i] = sum_{s < cnt} A[i, supp[s]] * v[supp[s]]   (gen_matvec_sparse,
// GAGA/Matrices/gen_gpu.cu:79-132, as a deterministic two-phase gather).
// The support indices and values are staged in LDS so every column load is
// independent; work items are (256-row tile, chunk of cs support columns);
// chunk partials are summed in a fixed order.  out is written with strided
// ownership.  Reads v: caller makes it visible.  NV = 2 forms A v0 and A v1
// over the same support in one pass over its columns (each output with the
// arithmetic of its own NV = 1 pass: same chunks, same order).  Supports of
// more than GATHER_BLOCK entries are gathered block by block (the partials
// hold one block), each block's sum added to out in block order.
template <int NV>
__device__ void gen_A_multi(Team &t, Lds &L, const XProblem &P, XG(const float) v0,
                            XG(float) out0, XG(const float) v1, XG(float) out1, int cnt) {
  const int lane = threadIdx.x & (WAVE - 1);
  const int lda = P.lda, nq = lda >> 2;
  XG(const float) A = P.A;
  XG(float) part = P.partials;
  const int row_tiles = (nq + WAVE - 1) / WAVE;
#ifdef XCS_PHASE_TIMING
  if (P.phase_ticks && t.rank == 0 && threadIdx.x == 0) {
    atomicMax(&P.phase_ticks[22], (unsigned long long)cnt);
    atomicAdd(&P.phase_ticks[23], (unsigned long long)cnt);
    atomicAdd(&P.phase_ticks[24], 1ull);
  }
#endif
  PHASE_BEGIN();
  const int nblk = gather_blocks(cnt);
  for (int blk = 0; blk < nblk; blk++) {
    const int b0 = blk * GATHER_BLOCK;
    const int bcnt = min(cnt - b0, GATHER_BLOCK);
    XG(const int) supp = P.supp + b0;
    const GatherGeom G = gather_geom(bcnt);
    const int cs = G.cs, nch = G.nch, cpp = G.cpp;
    if (blk > 0) t.sync();  // the previous block's partials have been summed everywhere
    for (int ch0 = 0; ch0 < nch; ch0 += cpp) {
      const int s_base = ch0 * cs;
      const int s_cnt = min(bcnt - s_base, cpp * cs);
      const int ch_cnt = min(nch - ch0, cpp);
      for (int i = threadIdx.x; i < s_cnt; i += blockDim.x) {
        const int j = supp[s_base + i];
        L.g.j[i] = j;
        L.g.v[i] = v0[j];
        if (NV == 2) L.g.w[i] = v1[j];
      }
      __syncthreads();
      PHASE(P, t, 18);
      const int items = row_tiles * ch_cnt;
      for (int it = t.gwave(); it < items; it += t.nwaves()) {
        const int rt = it % row_tiles, ch = it / row_tiles;
        const int q = rt * WAVE + lane;
        if (q < nq) {
          float4 acc = make_float4(0.f, 0.f, 0.f, 0.f);
          float4 acc2 = make_float4(0.f, 0.f, 0.f, 0.f);
          const int s0 = ch * cs, s1 = min(s_cnt, s0 + cs);
          int s = s0;
          for (; s + GATHER_U <= s1; s += GATHER_U) {
            float4 a[GATHER_U];
            float xv[GATHER_U], xw[GATHER_U];
#pragma unroll
            for (int u = 0; u < GATHER_U; u++) {
              a[u] = reinterpret_cast<XG(const float4)>(A + (size_t)L.g.j[s + u] * lda)[q];
              xv[u] = L.g.v[s + u];
              if (NV == 2) xw[u] = L.g.w[s + u];
            }
#pragma unroll
            for (int u = 0; u < GATHER_U; u++) {
              acc.x = fmaf(a[u].x, xv[u], acc.x);
              acc.y = fmaf(a[u].y, xv[u], acc.y);
              acc.z = fmaf(a[u].z, xv[u], acc.z);
              acc.w = fmaf(a[u].w, xv[u], acc.w);
              if (NV == 2) {
                acc2.x = fmaf(a[u].x, xw[u], acc2.x);
                acc2.y = fmaf(a[u].y, xw[u], acc2.y);
                acc2.z = fmaf(a[u].z, xw[u], acc2.z);
                acc2.w = fmaf(a[u].w, xw[u], acc2.w);
              }
            }
          }
          for (; s < s1; s++) {
            const float4 a = reinterpret_cast<XG(const float4)>(A + (size_t)L.g.j[s] * lda)[q];
            const float xv = L.g.v[s];
            acc.x = fmaf(a.x, xv, acc.x);
            acc.y = fmaf(a.y, xv, acc.y);
            acc.z = fmaf(a.z, xv, acc.z);
            acc.w = fmaf(a.w, xv, acc.w);
            if (NV == 2) {
              const float xw = L.g.w[s];
              acc2.x = fmaf(a.x, xw, acc2.x);
              acc2.y = fmaf(a.y, xw, acc2.y);
              acc2.z = fmaf(a.z, xw, acc2.z);
              acc2.w = fmaf(a.w, xw, acc2.w);
            }
          }
          reinterpret_cast<XG(float4)>(part + (size_t)(ch0 + ch) * lda)[q] = acc;
          if (NV == 2) reinterpret_cast<XG(float4)>(part + (size_t)(MAXCH + ch0 + ch) * lda)[q] = acc2;
        }
      }
      PHASE(P, t, 19);
      __syncthreads();
      PHASE(P, t, 20);
    }
    t.sync();
    for (int i = t.gtid(); i < P.m; i += t.gsize()) {
      float s = 0.f;
      for (int c = 0; c < nch; c++) s += part[(size_t)c * lda + i];
      out0[i] = blk ? out0[i] + s : s;
      if (NV == 2) {
        float s2 = 0.f;
        for (int c = 0; c < nch; c++) s2 += part[(size_t)(MAXCH + c) * lda + i];
        out1[i] = blk ? out1[i] + s2 : s2;
      }
    }
  }
  PHASE(P, t, 21);
}
__device__ void gen_A(Team &t, Lds &L, const XProblem &P, XG(const float) v, XG(float) out,
                      int cnt) {
  gen_A_multi<1>(t, L, P, v, out, nullptr, nullptr, cnt);
}

// g = A^T r, dense (gen_matvec on the transpose, gen_gpu.cu:33-74, 161-171),
// reading the single column-major copy of A.  Each wave streams two columns
// at a time (four float4 per lane per column in flight, non-temporal: A is
// read once per product) against the residual staged in LDS.
// epi(j, g_j) is called once per column by lane 0 of the owning wave.
typedef float xcs_v4f __attribute__((ext_vector_type(4)));
__device__ __forceinline__ float4 load_nt(XG(const float4) p) {
  const xcs_v4f v = __builtin_nontemporal_load(reinterpret_cast<XG(const xcs_v4f)>(p));
  return make_float4(v.x, v.y, v.z, v.w);
}
__device__ __forceinline__ float dot4(float4 a, float4 b, float acc) {
  acc = fmaf(a.x, b.x, acc);
  acc = fmaf(a.y, b.y, acc);
  acc = fmaf(a.z, b.z, acc);
  return fmaf(a.w, b.w, acc);
}
template <class Epi>
__device__ void gen_AT(Team &t, Lds &L, const XProblem &P, XG(const float) r, Epi &&epi) {
  const int lane = threadIdx.x & (WAVE - 1);
  const int lda = P.lda, n = P.n, nq = lda >> 2;
  XG(const float) A = P.A;
  XG(const float4) r4 = reinterpret_cast<XG(const float4)>(r);
  const bool lds = lda <= RLDS;
  if (lds) {
    for (int q = threadIdx.x; q < nq; q += blockDim.x) L.s.r[q] = r4[q];
    __syncthreads();
  }
  const int gw = t.gwave(), GW = t.nwaves();
  constexpr int U = XCS_AT_U;
  for (int j0 = 2 * gw; j0 < n; j0 += 2 * GW) {
    const bool two = j0 + 1 < n;
    XG(const float4) c0 = reinterpret_cast<XG(const float4)>(A + (size_t)j0 * lda);
    XG(const float4) c1 = reinterpret_cast<XG(const float4)>(A + (size_t)(two ? j0 + 1 : j0) * lda);
    float s00 = 0.f, s01 = 0.f, s10 = 0.f, s11 = 0.f;
    for (int q = lane; q < nq; q += U * WAVE) {
      float4 a0[U], a1[U], b[U];
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
        float4 rv = make_float4(0.f, 0.f, 0.f, 0.f);
        if (qq < nq) {
          if (lds)
            rv = L.s.r[qq];
          else
            rv = r4[qq];
        }
        b[u] = rv;
      }
#pragma unroll
      for (int u = 0; u < U; u += 2) {
        s00 = dot4(a0[u], b[u], s00);
        s01 = dot4(a0[u + 1], b[u + 1], s01);
        s10 = dot4(a1[u], b[u], s10);
        s11 = dot4(a1[u + 1], b[u + 1], s11);
      }
    }
    const float g0 = wave_sum(s00 + s01);
    const float g1 = wave_sum(s10 + s11);
    if (lane == 0) {
      epi(j0, g0);
      if (two) epi(j0 + 1, g1);
    }
  }
  if (lds) __syncthreads();
}

// ------------------------------------------------------------ smv ----------
// sum over e in [e0, e1) of val[e] * vec[idx[e]], one fmaf per entry in index
// order.  Whole groups of 8 entries issue their index, value and gathered loads
// together, so the latencies overlap (a row holds nz/m entries, 56 at n = 2^18
// and m = n/8); the rest go one by one.  (Predicating a last partial group
// instead measured slower: smv 2^18 CGIHT 20.1 against 14.6 ms.)
__device__ __forceinline__ float gather_dot(XG(const int) idx, XG(const float) val,
                                            XG(const float) vec, int e0, int e1) {
  float s = 0.f;
  int e = e0;
  for (; e + 8 <= e1; e += 8) {
    int c[8];
    float a[8], x[8];
#pragma unroll
    for (int q = 0; q < 8; q++) {
      c[q] = idx[e + q];
      a[q] = val[e + q];
    }
#pragma unroll
    for (int q = 0; q < 8; q++) x[q] = vec[c[q]];
#pragma unroll
    for (int q = 0; q < 8; q++) s = fmaf(a[q], x[q], s);
  }
  for (; e < e1; e++) s = fmaf(val[e], vec[idx[e]], s);
  return s;
}

// y = A v over the CSR copy (sparse_matvec, GAGA/Matrices/smv_gpu.cu:29-37,
// as a deterministic row gather instead of atomics).  Strided ownership.
__device__ void smv_A(Team &t, const XProblem &P, XG(const float) v, XG(float) out) {
  for (int i = t.gtid(); i < P.m; i += t.gsize())
    out[i] = gather_dot(P.cols, P.rvals, v, P.row_ptr[i], P.row_ptr[i + 1]);
}
// g = A^T r over CSC (sparse_matvecT, smv_gpu.cu:40-47): column gather.
template <class Epi>
__device__ void smv_AT(Team &t, const XProblem &P, XG(const float) r, Epi &&epi) {
  for (int j = t.gtid(); j < P.n; j += t.gsize())
    epi(j, gather_dot(P.rows, P.vals, r, P.col_ptr[j], P.col_ptr[j + 1]));
}

// --------------------------------------------------------- dispatch --------
// Algorithmic bytes of one operator application (what the roofline is quoted
// against): gen A_S x_S reads |S| columns (4m|S| + 8|S|) and writes y (4m);
// gen A^T r reads A once (4mn) plus r and g; smv reads values + row indices
// (8 nz) plus both vectors; dct reads x and writes the m samples (4n + 8m).
__device__ __forceinline__ double op_bytes(const XProblem &P, bool transpose, int cnt) {
  const double m = P.m, n = P.n;
  if (P.ens == ENS_GEN)
    return transpose ? 4.0 * m * n + 4.0 * m + 4.0 * n : 4.0 * m * cnt + 8.0 * cnt + 4.0 * m;
  if (P.ens == ENS_SMV) return 8.0 * P.nz + 4.0 * m + 4.0 * n;
  return 4.0 * n + 8.0 * m;
}

// out = A v_S.  v must be zero off the support for smv/dct (it always is:
// callers pass thresholded vectors).  Strided ownership of out.
__device__ void op_A(Team &t, Lds &L, const XProblem &P, XG(const float) v, XG(float) out,
                     int cnt) {
  if (P.ens == ENS_GEN)
    gen_A(t, L, P, v, out, cnt);
  else if (P.ens == ENS_SMV)
    smv_A(t, P, v, out);
  else
    dct_A(t, L, P, v, out);
}
template <class Epi>
__device__ void op_AT(Team &t, Lds &L, const XProblem &P, XG(const float) r, Epi &&epi) {
  if (P.ens == ENS_GEN)
    gen_AT(t, L, P, r, epi);
  else if (P.ens == ENS_SMV)
    smv_AT(t, P, r, epi);
  else
    dct_AT(t, L, P, r, epi);
}

// Operator applications of the solver, with algorithmic-byte accounting.
__device__ __forceinline__ void opA(Team &t, Lds &L, const XProblem &P, XState &S,
                                    XG(const float) v, XG(float) out) {
  S.mat_bytes += op_bytes(P, false, S.supp_count);
  op_A(t, L, P, v, out, S.supp_count);
}
template <class Epi>
__device__ __forceinline__ void opAT(Team &t, Lds &L, const XProblem &P, XState &S,
                                     XG(const float) r, Epi &&epi) {
  S.mat_bytes += op_bytes(P, true, 0);
  op_AT(t, L, P, r, epi);
}

// ------------------------------------------------------ support state ------
// LinearBinning over v (kernels.cu:135-146); counters must be zero and
// visible.  Ends with a team barrier (counters complete).
__device__ void team_binning(Team &t, Lds &L, const XProblem &P, XG(const float) v, XG(int) bins,
                             int max_bin, float slope, float intercept) {
  // the histogram in LDS when it fits the whole union (free while binning:
  // 12288 bins, smv n = 2^18 included), else straight into the counters
  int *hist = reinterpret_cast<int *>(&L);
  constexpr int HCAP = (int)(sizeof(Lds) / sizeof(int));
  const bool lds = max_bin <= HCAP;
  if (lds) {
    __syncthreads();  // no wave still reads what an operator left in the union
    for (int b = threadIdx.x; b < max_bin; b += blockDim.x) hist[b] = 0;
    __syncthreads();
  }
  for (int i = t.gtid(); i < P.n; i += t.gsize()) {
    const float temp = fabsf(v[i]);
    int b;
    if ((double)temp > (double)intercept * .000001) {
      b = (int)fmaxf(0.0f, __fmul_rn(slope, __fsub_rn(intercept, temp)));
      if (b < max_bin) {
        if (lds)
          atomicAdd(&hist[b], 1);
        else
          atomicAdd(&P.counters[b], 1);
      }
    } else {
      b = (int)__fmaf_rn(slope, intercept, 1.0f);
    }
    bins[i] = b;
  }
  if (lds) {
    __syncthreads();
    for (int b = threadIdx.x; b < max_bin; b += blockDim.x)
      if (hist[b]) atomicAdd(&P.counters[b], hist[b]);
  }
  t.sync();
}

// Zero the histogram counters (strided); caller syncs before binning.
__device__ void zero_counters(Team &t, const XProblem &P) {
  for (int b = t.gtid(); b < P.num_bins; b += t.gsize()) P.counters[b] = 0;
}

// FindSupportSet's binning branch (functions.cu:404-428) on vector v whose
// bins go to `bins`; scalars in S.  Caller zeroed counters and synced.
__device__ void find_support_bin(Team &t, Lds &L, const XProblem &P, XG(const float) v,
                                 XG(int) bins,
                                 XState &S, float slope, float intercept, int *k_bin_out) {
  team_binning(t, L, P, v, bins, S.max_bin, slope, intercept);
  int kb, sum;
  kbin_select(P.counters, S.max_bin, P.k, &kb, &sum, (int *)&L, (int)(sizeof(Lds) / sizeof(int)));
  if (sum < P.k) {
    S.alpha_bin = S.alpha_bin * 0.5f;
    S.max_bin = (int)((float)P.num_bins * (1.0f - S.alpha_bin));
  }
  S.min_val = __fsub_rn(intercept, __fdiv_rn((float)(kb + 1), slope));
  S.sum = sum;
  *k_bin_out = kb;
}

// Ascending support list {i : in(i)} into P.supp; returns its length
// (uniform; 0 once the team has aborted).  Requires what `in` reads to be visible;
// ends with supp visible.
template <class In>
__device__ int build_support_if(Team &t, const XProblem &P, In &&in) {
  const int n = P.n;
  const int per = (n + t.size - 1) / t.size;
  const int lo = min(n, t.rank * per), hi = min(n, lo + per);
  // each wave takes a contiguous part of the workgroup's range (whole rounds of
  // 64) and finds its members by ballot: one count pass, one workgroup step for
  // the waves' offsets, one pass that writes
  const int lane = threadIdx.x & (WAVE - 1), wave = threadIdx.x / WAVE;
  const int nw = blockDim.x / WAVE;
  const int wper = ((hi - lo + nw - 1) / nw + WAVE - 1) / WAVE * WAVE;
  const int wlo = min(hi, lo + wave * wper), whi = min(hi, wlo + wper);
  int c = 0;
  for (int base = wlo; base < whi; base += WAVE) {
    const int i = base + lane;
    c += __popcll(__ballot(i < whi && in(i)));
  }
  __shared__ int s_wc[MAX_WAVES];
  if (lane == 0) s_wc[wave] = c;
  __syncthreads();
  int wave_off = 0, wg_total = 0;
  for (int w = 0; w < nw; w++) {
    if (w < wave) wave_off += s_wc[w];
    wg_total += s_wc[w];
  }
  int offset = 0, total = wg_total;
  if (t.size > 1) {
    if (threadIdx.x == 0) P.wg_counts[t.rank] = wg_total;
    t.sync();
    // a wait timed out: the counts may be an earlier, longer instance's, which would
    // place the list's entries past its end
    if (t.aborted) return 0;
    int before = 0, all = 0;
    for (int w = threadIdx.x; w < t.size; w += blockDim.x) {
      const int v = P.wg_counts[w];
      all += v;
      if (w < t.rank) before += v;
    }
    int vv[2] = {before, all};
    // workgroup sums (integer: exact, order free)
    __shared__ int sb[2][MAX_WAVES];
    vv[0] = wave_sum_i(vv[0]);
    vv[1] = wave_sum_i(vv[1]);
    if (lane == 0) {
      sb[0][wave] = vv[0];
      sb[1][wave] = vv[1];
    }
    __syncthreads();
    offset = 0;
    total = 0;
    for (int w = 0; w < nw; w++) {
      offset += sb[0][w];
      total += sb[1][w];
    }
    __syncthreads();
  }
  int pos = offset + wave_off;
  for (int base = wlo; base < whi; base += WAVE) {
    const int i = base + lane;
    const bool f = i < whi && in(i);
    const unsigned long long mask = __ballot(f);
    if (f) P.supp[pos + __popcll(mask & ((1ull << lane) - 1ull))] = i;
    pos += __popcll(mask);
  }
  t.sync();
  return total;
}

// Support list {i : bins[i] <= k_bin}.
__device__ int build_support(Team &t, const XProblem &P, int k_bin) {
  return build_support_if(t, P, [&](int i) { return P.bins[i] <= k_bin; });
}

// ------------------------------------------------------------ helpers ------
__device__ __forceinline__ void push16(float *h, float v) {
#pragma unroll
  for (int j = 0; j < 15; j++) h[j] = h[j + 1];
  h[15] = v;
}
__device__ __forceinline__ float max16(const float *h) {
  float mx = h[0];
#pragma unroll
  for (int j = 1; j < 16; j++)
    if (h[j] > mx) mx = h[j];
  return mx;
}

// resid = y - A x_S ; returns the FP64 partial of ||resid||^2 (strided).
__device__ double residual(Team &t, Lds &L, const XProblem &P, XState &S, XG(float) resid,
                           XG(float) tmp) {
  opA(t, L, P, S, P.x, tmp);
  double e2 = 0.0;
  for (int i = t.gtid(); i < P.m; i += t.gsize()) {
    const float r = __fsub_rn(P.y[i], tmp[i]);
    resid[i] = r;
    e2 += (double)r * (double)r;
  }
  return e2;
}

template <int K>
__device__ __forceinline__ void reduce(Team &t, double (&v)[K], const int (&op)[K]) {
  team_reduce<double, K>(t, v, op);
}

// ------------------------------------------------------------ steps --------
// RestrictedSD_S_* (functions.cu:473-745): returns maxChange; *xmax gets the
// thread partial of max|x_new|.
__device__ float step_restricted_sd(Team &t, Lds &L, const XProblem &P, XState &S, float *xmax) {
  const int kb = S.k_bin;
  double e2 = residual(t, L, P, S, P.resid, P.resid_update);
  {
    double v[1] = {e2};
    const int op[1] = {0};
    reduce(t, v, op);
    push16(S.prev, (float)sqrt(v[0]));
  }
  float gmax = 0.f, th2 = 0.f;
  opAT(t, L, P, S, P.resid, [&](int j, float g) {
    P.grad[j] = g;
    const float th = (P.bins[j] <= kb) ? g : 0.f;
    P.thres[j] = th;
    th2 = fmaf(th, th, th2);
    gmax = fmaxf(gmax, fabsf(g));
  });
  t.sync();
  opA(t, L, P, S, P.thres, P.resid_update);
  float a2 = 0.f;
  for (int i = t.gtid(); i < P.m; i += t.gsize()) a2 = fmaf(P.resid_update[i], P.resid_update[i], a2);
  double v[3] = {a2, th2, gmax};
  const int op[3] = {0, 0, 1};
  reduce(t, v, op);
  const float err = (float)sqrt(v[0]);
  float mu = (float)sqrt(v[1]);
  if (mu < 400.0f * err) {
    mu = mu / err;
    mu = mu * mu;
  } else {
    mu = 0.f;
  }
  float xm = 0.f;
  for (int i = t.gtid(); i < P.n; i += t.gsize()) {
    const float xn = fmaf(mu, P.grad[i], P.x[i]);
    P.x[i] = xn;
    xm = fmaxf(xm, fabsf(xn));
  }
  *xmax = xm;
  return 2.0f * mu * (float)v[2];
}

// RestrictedCG_S_* (functions.cu:752-1000): one CG step on the support.
// grad = search direction, gprev = CG residual, S.mu carries <r,r>.
// Pushes the squared residual onto hist.
__device__ void step_restricted_cg(Team &t, Lds &L, const XProblem &P, XState &S, float *hist,
                                   bool ad_ready = false, bool fuse_next = false) {
  const int kb = S.k_bin;
  if (ad_ready) {
    // A d was formed by the previous step's two-output pass (into resid3)
    for (int i = t.gtid(); i < P.m; i += t.gsize()) P.resid[i] = P.resid3[i];
  } else {
    opA(t, L, P, S, P.grad, P.resid);
  }
  float a2 = 0.f;
  for (int i = t.gtid(); i < P.m; i += t.gsize()) a2 = fmaf(P.resid[i], P.resid[i], a2);
  float alpha;
  {
    double v[1] = {a2};
    const int op[1] = {0};
    reduce(t, v, op);
    alpha = (float)v[0];
  }
  if (S.mu < 1000.0f * alpha)
    alpha = S.mu / alpha;
  else
    alpha = 0.f;
  for (int i = t.gtid(); i < P.n; i += t.gsize()) P.x[i] = fmaf(alpha, P.grad[i], P.x[i]);
  float gp2 = 0.f;
  opAT(t, L, P, S, P.resid, [&](int j, float g) {
    const float th = (P.bins[j] <= kb) ? g : 0.f;
    const float gp = fmaf(-alpha, th, P.gprev[j]);
    P.gprev[j] = gp;
    gp2 = fmaf(gp, gp, gp2);
  });
  float beta = S.mu;
  {
    double v[1] = {gp2};
    const int op[1] = {0};
    reduce(t, v, op);
    S.mu = (float)v[0];
  }
  if (S.mu < 1000.0f * beta)
    beta = S.mu / beta;
  else
    beta = 0.f;
  for (int i = t.gtid(); i < P.n; i += t.gsize())
    P.grad[i] = __fadd_rn(__fmul_rn(beta, P.grad[i]), P.gprev[i]);
  t.sync();
  double e2;
  if (fuse_next) {
    // gen: A x for the residual and A d for the next step in one pass over the
    // support's columns (each output as its own pass would form it)
    S.mat_bytes += op_bytes(P, false, S.supp_count) + 8.0 * S.supp_count + 4.0 * P.m;
    gen_A_multi<2>(t, L, P, P.x, P.resid_update, P.grad, P.resid3, S.supp_count);
    e2 = 0.0;
    for (int i = t.gtid(); i < P.m; i += t.gsize()) {
      const float r = __fsub_rn(P.y[i], P.resid_update[i]);
      P.resid[i] = r;
      e2 += (double)r * (double)r;
    }
  } else {
    e2 = residual(t, L, P, S, P.resid, P.resid_update);
  }
  double v[1] = {e2};
  const int op[1] = {0};
  reduce(t, v, op);
  push16(hist, (float)v[0]);
}

// CG projection on the current support shared by HTP and CSMPSP
// (algorithms.cu:2607-2669, 3431-3488, 3548-3604).  Returns errCG.
__device__ float cg_projection(Team &t, Lds &L, const XProblem &P, XState &S, bool fixed_diff,
                               int max_steps = 15, int *iters = nullptr) {
  const int kb = S.k_bin;
  float hist[16], evo[16];
#pragma unroll
  for (int j = 0; j < 16; j++) {
    hist[j] = 0.f;
    evo[j] = 1.f;
  }
  hist[15] = S.prev[15];
  float diffCG = 1.f;
  const float tolCG = P.tol * P.tol;
  const float tol2 = 10.0f * tolCG;
  double e2 = residual(t, L, P, S, P.resid, P.resid_update);
  t.sync();
  float g2 = 0.f;
  opAT(t, L, P, S, P.resid, [&](int j, float g) {
    const float th = (P.bins[j] <= kb) ? g : 0.f;
    P.grad[j] = th;
    P.gprev[j] = th;
    g2 = fmaf(th, th, g2);
  });
  double v[2] = {g2, e2};
  const int op[2] = {0, 0};
  reduce(t, v, op);
  S.mu = (float)v[0];
  float errCG = (float)v[1];
  hist[15] = errCG;
  int iterCG = 0;
  const bool gen = P.ens == ENS_GEN;
  while ((errCG > tolCG) & (iterCG < max_steps) & (diffCG > tol2)) {
    // gen: each step but the last allowed one also forms the next step's A d
    step_restricted_cg(t, L, P, S, hist, gen && iterCG > 0, gen && iterCG + 1 < max_steps);
    errCG = hist[15];
    iterCG++;
#pragma unroll
    for (int j = 0; j < 15; j++) evo[j] = evo[j + 1];
    evo[15] = hist[14] - hist[15];
    diffCG = fixed_diff ? 10.0f : max16(evo);
  }
  if (iters) *iters = iterCG;
  return errCG;
}

// RestrictedCGwithSupportEvolution_S_* (functions.cu:1004-1102).
__device__ float step_cg_restricted(Team &t, Lds &L, const XProblem &P, XState &S, float *xmax) {
  const int kb = S.k_bin;
  PHASE_BEGIN();
  double e2 = residual(t, L, P, S, P.resid, P.resid_update);
  PHASE(P, t, 0);
  {
    double v[1] = {e2};
    const int op[1] = {0};
    reduce(t, v, op);
    push16(S.prev, (float)sqrt(v[0]));
  }
  PHASE(P, t, 1);
  float th2 = 0.f;
  opAT(t, L, P, S, P.resid, [&](int j, float g) {
    P.grad[j] = g;
    const float th = (P.bins[j] <= kb) ? g : 0.f;
    P.thres[j] = th;
    th2 = fmaf(th, th, th2);
  });
  PHASE(P, t, 2);
  float beta;
  {
    double v[1] = {th2};
    const int op[1] = {0};
    reduce(t, v, op);
    const float mu_new = (float)v[0];
    if (S.beta_to_zero == 1) {
      beta = 0.f;
      S.mu = mu_new;
    } else {
      beta = S.mu;
      S.mu = mu_new;
      if (S.mu < 1000.0f * beta)
        beta = S.mu / beta;
      else
        beta = 0.f;
    }
  }
  float pmax = 0.f;
  for (int i = t.gtid(); i < P.n; i += t.gsize()) {
    const float gp = __fadd_rn(__fmul_rn(beta, P.gprev[i]), P.grad[i]);
    P.gprev[i] = gp;
    P.gprev_thres[i] = (P.bins[i] <= kb) ? gp : 0.f;
    pmax = fmaxf(pmax, fabsf(gp));
  }
  t.sync();
  PHASE(P, t, 3);
  opA(t, L, P, S, P.gprev_thres, P.resid_update);
  PHASE(P, t, 4);
  float a2 = 0.f;
  for (int i = t.gtid(); i < P.m; i += t.gsize()) a2 = fmaf(P.resid_update[i], P.resid_update[i], a2);
  double v[2] = {a2, pmax};
  const int op[2] = {0, 1};
  reduce(t, v, op);
  float alpha = (float)v[0];
  if (S.mu < 1000.0f * alpha)
    alpha = S.mu / alpha;
  else
    alpha = 0.f;
  float xm = 0.f;
  for (int i = t.gtid(); i < P.n; i += t.gsize()) {
    const float xn = fmaf(alpha, P.gprev[i], P.x[i]);
    P.x[i] = xn;
    xm = fmaxf(xm, fabsf(xn));
  }
  *xmax = xm;
  PHASE(P, t, 5);
  return 2.0f * alpha * (float)v[1];
}

// UnrestrictedCG_S_* (functions.cu:1107-1220).
__device__ float step_cg_unrestricted(Team &t, Lds &L, const XProblem &P, XState &S, float *xmax) {
  const int kb = S.k_bin;
  PHASE_BEGIN();
  // resid_update = -(A x - y).  gen: A x and A p_old_S (the previous direction on the
  // current support, final at this point) share one pass over the support's columns
  const bool fused = P.ens == ENS_GEN;
  if (fused) {
    S.mat_bytes += op_bytes(P, false, S.supp_count) + 8.0 * S.supp_count + 4.0 * P.m;
    gen_A_multi<2>(t, L, P, P.x, P.resid_update, P.gprev_thres, P.resid, S.supp_count);
  } else {
    opA(t, L, P, S, P.x, P.resid_update);
  }
  PHASE(P, t, 15);
  double e2 = 0.0;
  for (int i = t.gtid(); i < P.m; i += t.gsize()) {
    const float r = -__fsub_rn(P.resid_update[i], P.y[i]);
    P.resid_update[i] = r;
    e2 += (double)r * (double)r;
  }
  {
    double v[1] = {e2};
    const int op[1] = {0};
    reduce(t, v, op);
    push16(S.prev, (float)sqrt(v[0]));
  }
  PHASE(P, t, 6);
  opAT(t, L, P, S, P.resid_update, [&](int j, float g) {
    P.grad[j] = g;
    P.thres[j] = (P.bins[j] <= kb) ? g : 0.f;
  });
  t.sync();
  PHASE(P, t, 7);
  if (!fused) opA(t, L, P, S, P.gprev_thres, P.resid);
  t.sync();
  PHASE(P, t, 8);
  opA(t, L, P, S, P.thres, P.resid_update);
  PHASE(P, t, 9);
  float beta = 0.f;
  if (S.beta_to_zero != 1) {
    float num = 0.f, den = 0.f;
    for (int i = t.gtid(); i < P.m; i += t.gsize()) {
      num = fmaf(P.resid[i], P.resid_update[i], num);
      den = fmaf(P.resid[i], P.resid[i], den);
    }
    double v[2] = {num, den};
    const int op[2] = {0, 0};
    reduce(t, v, op);
    beta = -((float)v[0]) / (float)v[1];
  }
  float pmax = 0.f, an = 0.f, mu2 = 0.f, ad = 0.f;
  for (int i = t.gtid(); i < P.n; i += t.gsize()) {
    const float gp = __fadd_rn(__fmul_rn(beta, P.gprev[i]), P.grad[i]);
    P.gprev[i] = gp;
    const float gpt = (P.bins[i] <= kb) ? gp : 0.f;
    P.gprev_thres[i] = gpt;
    pmax = fmaxf(pmax, fabsf(gp));
    const float th = P.thres[i];
    an = fmaf(gpt, th, an);
    mu2 = fmaf(th, th, mu2);
  }
  for (int i = t.gtid(); i < P.m; i += t.gsize()) {
    const float r = __fadd_rn(__fmul_rn(beta, P.resid[i]), P.resid_update[i]);
    P.resid[i] = r;
    ad = fmaf(r, r, ad);
  }
  double v[4] = {an, ad, pmax, mu2};
  const int op[4] = {0, 0, 1, 0};
  reduce(t, v, op);
  PHASE(P, t, 10);
  float alpha = (float)v[0] / (float)v[1];
  float xm = 0.f;
  for (int i = t.gtid(); i < P.n; i += t.gsize()) {
    const float xn = fmaf(alpha, P.gprev[i], P.x[i]);
    P.x[i] = xn;
    xm = fmaxf(xm, fabsf(xn));
  }
  S.mu = (float)v[3];
  *xmax = xm;
  return 2.0f * alpha * (float)v[2];
}

// ------------------------------------------------------------ driver -------
__device__ __forceinline__ bool should_continue(const XState &S, const XProblem &P, int *reason) {
  if (P.alg == ALG_HTSD || P.alg == ALG_HTCG) {
    // HT_SD_S_gen (algorithms.cu:846): err > tol, iter < maxiter, diff > 0.1 tol;
    // HT_CG_S_gen (algorithms.cu:1913): squared errors, tol^2 and 10 tol^2
    const float tcg = P.tol * P.tol;
    const float lim = P.alg == ALG_HTCG ? tcg : P.tol;
    const float dlim = P.alg == ALG_HTCG ? 10.0f * tcg : (float)(0.1 * (double)P.tol);
    if (!(S.err > lim)) { *reason = 0; return false; }
    if (!(S.iter < P.maxiter)) { *reason = 1; return false; }
    if (!(S.diff > dlim)) { *reason = 3; return false; }
    return true;
  }
  if (!(S.err > P.tol)) { *reason = 0; return false; }
  if (!(S.iter < P.maxiter)) { *reason = 1; return false; }
  if (!(S.err < 100.0f * S.err_start)) { *reason = 2; return false; }
  if (!((double)S.diff > .01 * (double)P.tol)) { *reason = 3; return false; }
  if (S.fail != 0) { *reason = 4; return false; }
  if (!S.cycle) { *reason = 5; return false; }
  return true;
}

// residNorm_evolution / cycle / stagnation bookkeeping (algorithms.cu:1398-1421).
// IHT has no cycle test (algorithms.cu:422-480): cycle_test = false.
__device__ void stop_update(XState &S, int fail_after, bool cycle_test = true) {
#pragma unroll
  for (int j = 0; j < 15; j++) S.evo[j] = S.evo[j + 1];
  S.evo[15] = S.prev[14] - S.prev[15];
  S.diff = max16(S.evo);
  if (cycle_test)
    for (int j = 0; j < 15; j++)
      if ((S.prev[15] == S.prev[j]) && (S.iter > 4)) S.cycle = 0;
  if (S.iter > fail_after) {
    const float root = 1 / 15.0f;
    float rate = S.prev[15] / S.prev[0];
    rate = powf(rate, root);
    if (rate > 0.999f) S.fail = 1;
  }
}

// The timing variants' bookkeeping (algorithms_timings.cu:607-619, 1525-1539): no
// cycle test, the stagnation rate with root 1/16.
__device__ void stop_update_timing(XState &S, int fail_after) {
#pragma unroll
  for (int j = 0; j < 15; j++) S.evo[j] = S.evo[j + 1];
  S.evo[15] = S.prev[14] - S.prev[15];
  S.diff = max16(S.evo);
  if (S.iter > fail_after) {
    const float root = 1 / 16.0f;
    float rate = S.prev[15] / S.prev[0];
    rate = powf(rate, root);
    if (rate > 0.999f) S.fail = 1;
  }
}

// The k-th largest |v| over the team (the value a sort of the magnitudes puts
// at n - k, functions.cu:451-452): bitwise search over the bit patterns of the
// non-negative floats, one exact team count per bit.  k >= 1.
__device__ float team_kth_largest_abs(Team &t, const XProblem &P, XG(const float) v, int k) {
  uint32_t thr = 0;
  for (int bit = 30; bit >= 0; bit--) {
    const uint32_t cand = thr | (1u << bit);
    int c = 0;
    for (int i = t.gtid(); i < P.n; i += t.gsize()) c += (__float_as_uint(fabsf(v[i])) >= cand) ? 1 : 0;
    double w[1] = {(double)c};
    const int op[1] = {0};
    team_reduce<double, 1>(t, w, op);
    if ((long)w[0] >= (long)k) thr = cand;
  }
  return __uint_as_float(thr);
}

__device__ void trace_write(const Team &t, const XProblem &P, int idx, int kb, float e) {
  if (t.rank == 0 && threadIdx.x == 0) {
    if (P.trace_kbin) P.trace_kbin[idx] = kb;
    if (P.trace_err) P.trace_err[idx] = e;
  }
}

// Threshold x by the current bins (kernels.cu:74-81); strided.
__device__ void threshold_x(Team &t, const XProblem &P, int kb) {
  for (int i = t.gtid(); i < P.n; i += t.gsize())
    if (P.bins[i] > kb) P.x[i] = 0.f;
}

// Rebin x with a fresh max (the `minVal <= maxChange` branch shared by NIHT,
// HTP and CGIHT).  xmax_partial: thread partial of max|x|.
__device__ void rebin_x(Team &t, Lds &L, const XProblem &P, XState &S, float xmax_partial,
                        bool save_prev) {
  {
    double v[1] = {xmax_partial};
    const int op[1] = {1};
    zero_counters(t, P);
    if (save_prev)
      for (int i = t.gtid(); i < P.n; i += t.gsize()) P.bins2[i] = P.bins[i];
    reduce(t, v, op);  // barrier: counters zeroed everywhere
    S.max_value = (float)v[0];
    S.slope = (float)(P.num_bins - 1) / S.max_value;
  }
  find_support_bin(t, L, P, P.x, P.bins, S, S.slope, S.max_value, &S.k_bin);
}

// No yielding: the solve runs until its budget or its stopping rule.
struct NoYield {
  __device__ bool operator()(const XState &) const { return false; }
};

// Solve (or continue) the instance for at most `budget` outer iterations.
// yield(S) is asked after every iteration, by every thread of the team (it must
// answer uniformly); true ends the solve there with the state saved, to be
// continued later as any other budget-limited solve.
template <class Yield = NoYield>
__device__ void solve_instance(Team &t, Lds &L, const XProblem &P, int budget,
                               Yield yield = Yield()) {
  XState S = *P.st;
  const int n = P.n, m = P.m;
  if (S.done) return;
  if (!S.initialized) {
    // common initialisation (algorithms.cu:1284-1358 and equivalents)
    S.iter = 0;
    S.k_bin = 0;
    S.k_bin_grad = 0;
    S.sum = 0;
    // alpha = 0 (MaxBin = num_bins) for the one-shot thresholds (algorithms.cu:795, 1836)
    S.alpha_bin = (P.alg == ALG_HTSD || P.alg == ALG_HTCG) ? 0.0f : P.timing ? P.alpha0 : 0.25f;
    S.thr = 0.f;
    S.max_bin = (int)((float)P.num_bins * (1.0f - S.alpha_bin));
    S.min_val = 0.f;
    S.max_change = (P.alg == ALG_NIHT || P.alg == ALG_CGIHT) ? 1.0f : 0.0f;
    S.mu = 0.f;
    S.diff = 1.f;
    S.fail = 0;
    S.cycle = 1;
    S.beta_to_zero = 1;
    S.supp_change = 1;
    S.stop_reason = 0;
    for (int j = 0; j < 16; j++) {
      S.prev[j] = 0.f;
      S.evo[j] = 1.f;
    }
    double e2 = 0.0;
    for (int i = t.gtid(); i < m; i += t.gsize()) {
      const float r = P.y[i];
      P.resid[i] = r;
      e2 += (double)r * (double)r;
    }
    zero_counters(t, P);
    t.sync();
    float xm = 0.f;
    opAT(t, L, P, S, P.y, [&](int j, float g) {
      P.x[j] = g;
      xm = fmaxf(xm, fabsf(g));
    });
    double v[2] = {e2, xm};
    const int op[2] = {0, 1};
    reduce(t, v, op);
    S.err = (float)sqrt(v[0]);
    S.err_start = S.err;
    S.max_value = (float)v[1];
    if (S.max_value == 0.f) {  // A^T y == 0: x = 0 is returned
      S.initialized = 1;
      S.done = 1;
      S.supp_count = 0;
      if (t.rank == 0 && threadIdx.x == 0) *P.st = S;
      return;
    }
    if (P.warm && P.alg == ALG_CGIHT) {
      // Warm start (no counterpart in the reference): x = least squares on the
      // given support by the restricted CG projection, then the usual start
      // from that x instead of A^T y.
      for (int j = t.gtid(); j < n; j += t.gsize()) {
        const int in = P.warm[j];
        if (!in) P.x[j] = 0.f;
        P.bins[j] = in ? 0 : P.num_bins;
      }
      t.sync();
      S.k_bin = 0;
      S.supp_count = build_support(t, P, 0);
      (void)cg_projection(t, L, P, S, false, P.warm_cg);
      S.mu = 0.f;
      float xw = 0.f;
      for (int j = t.gtid(); j < n; j += t.gsize()) xw = fmaxf(xw, fabsf(P.x[j]));
      double w[1] = {xw};
      const int o1[1] = {1};
      reduce(t, w, o1);
      if (w[0] > 0.0) S.max_value = (float)w[0];
    }
    S.slope = (float)(P.num_bins - 1) / S.max_value;
    if (P.alg == ALG_IHT) {
      // IHT_S_gen (algorithms.cu:397-402): the bins' slope and intercept come from
      // A^T y and stay fixed; x starts at 0 and is first binned inside the loop.
      for (int j = t.gtid(); j < n; j += t.gsize()) P.x[j] = 0.f;
      S.supp_count = 0;
    } else {
      // FindSupportSet with maxChange 1 (NIHT/CGIHT/one-shot thresholds) or max_value
      // (HTP/CSMPSP): minVal = 0 is never greater, so this always bins.
      find_support_bin(t, L, P, P.x, P.bins, S, S.slope, S.max_value, &S.k_bin);
      threshold_x(t, P, S.k_bin);
      S.supp_count = build_support(t, P, S.k_bin);
      trace_write(t, P, 0, S.k_bin, S.err);
    }
    if (P.alg == ALG_CSMPSP) {
      // the initial projection counts as iteration 1 (algorithms.cu:3486-3490)
      const float errCG = cg_projection(t, L, P, S, false);
      S.err = sqrtf(errCG);
      S.prev[15] = S.err;
      S.iter = 1;
      trace_write(t, P, 1, S.k_bin, S.err);
    } else if (P.alg == ALG_HTCG) {
      // HT_CG_S_gen (algorithms.cu:1875-1898): r = y - A x, s = (A^T r)_S as the
      // first direction and CG residual, mu = |s|^2, err = |r|^2 into the ring
      double e = residual(t, L, P, S, P.resid, P.resid_update);
      t.sync();
      float g2 = 0.f;
      opAT(t, L, P, S, P.resid, [&](int j, float g) {
        const float th = (P.bins[j] <= S.k_bin) ? g : 0.f;
        P.grad[j] = th;
        P.gprev[j] = th;
        g2 = fmaf(th, th, g2);
      });
      double w[2] = {g2, e};
      const int o2[2] = {0, 0};
      reduce(t, w, o2);
      S.mu = (float)w[0];
      S.err = (float)w[1];
      S.prev[15] = S.err;
    } else if (P.alg == ALG_FIHT || P.alg == ALG_ALPS) {
      // FIHT_S_gen's (and ALPS_S_gen's) extra first iteration (algorithms.cu:5513-5559): x_prev = x,
      // x += A^T (y - A x), the threshold, A x_prev kept in resid2.
      double e = residual(t, L, P, S, P.resid, P.resid_update);
      {
        double w[1] = {e};
        const int o1[1] = {0};
        reduce(t, w, o1);
        S.err = (float)sqrt(w[0]);
        S.prev[15] = S.err;
      }
      opAT(t, L, P, S, P.resid, [&](int j, float g) { P.grad[j] = g; });
      t.sync();
      float xm = 0.f;
      for (int i = t.gtid(); i < n; i += t.gsize()) {
        const float xi = P.x[i];
        P.gprev[i] = xi;
        const float xn = __fadd_rn(xi, P.grad[i]);
        P.x[i] = xn;
        xm = fmaxf(xm, fabsf(xn));
      }
      for (int i = t.gtid(); i < m; i += t.gsize()) P.resid2[i] = P.resid_update[i];
      S.min_val = 0.f;
      rebin_x(t, L, P, S, xm, false);
      threshold_x(t, P, S.k_bin);
      t.sync();
      S.supp_count = build_support(t, P, S.k_bin);
      e = residual(t, L, P, S, P.resid, P.resid_update);
      {
        double w[1] = {e};
        const int o1[1] = {0};
        reduce(t, w, o1);
        S.err = (float)sqrt(w[0]);
      }
      push16(S.prev, S.err);
#pragma unroll
      for (int j = 0; j < 15; j++) S.evo[j] = S.evo[j + 1];
      S.evo[15] = S.prev[14] - S.prev[15];
      S.diff = max16(S.evo);
    } else if (P.alg == ALG_CGIHT) {
      // r^0 and its restriction (algorithms.cu:3762-3808)
      double e = residual(t, L, P, S, P.resid, P.resid_update);
      double w[1] = {e};
      const int o1[1] = {0};
      reduce(t, w, o1);
      S.err = (float)sqrt(w[0]);
      S.prev[15] = S.err;
      opAT(t, L, P, S, P.resid, [&](int j, float g) {
        P.gprev[j] = g;
        P.gprev_thres[j] = (P.bins[j] <= S.k_bin) ? g : 0.f;
      });
      for (int j = 0; j < 15; j++) S.evo[j] = S.evo[j + 1];
      S.evo[15] = S.prev[14] - S.prev[15];
      S.beta_to_zero = 1;
      S.supp_change = 1;
    } else if (P.alg == ALG_CGIHTP) {
      // CGIHTprojected_S_gen initialisation (algorithms.cu:4560-4590): r = y - A x,
      // g = A^T r, g_S = g on the support (thres), A g_S (resid_update), with the
      // norms |g_S|^2 and |A g_S|^2 kept for the first step length
      double e = residual(t, L, P, S, P.resid, P.resid_update);
      t.sync();
      double g2 = 0.0;
      const int kb = S.k_bin;
      opAT(t, L, P, S, P.resid, [&](int j, float g) {
        P.grad[j] = g;
        const float th = (P.bins[j] <= kb) ? g : 0.f;
        P.thres[j] = th;
        g2 += (double)th * (double)th;
      });
      t.sync();
      opA(t, L, P, S, P.thres, P.resid_update);
      double a2 = 0.0;
      for (int i = t.gtid(); i < m; i += t.gsize()) a2 += (double)P.resid_update[i] * (double)P.resid_update[i];
      double w[3] = {e, g2, a2};
      const int o3[3] = {0, 0, 0};
      reduce(t, w, o3);
      S.err = (float)sqrt(w[0]);
      S.prev[15] = S.err;
      S.vt2 = (float)w[1];
      S.ru2 = (float)w[2];
      S.ap2 = 0.f;
#pragma unroll
      for (int j = 0; j < 15; j++) S.evo[j] = S.evo[j + 1];
      S.evo[15] = S.prev[14] - S.prev[15];
      S.supp_change = 1;
    }
    S.initialized = 1;
    t.sync();
  }

  int reason = 0;
  if (t.aborted) {  // a team barrier timed out: the instance is abandoned
    S.done = 1;
    S.stop_reason = STOP_ABORTED;
    if (t.rank == 0 && threadIdx.x == 0) *P.st = S;
    return;
  }
#ifdef XCS_PHASE_TIMING
  unsigned long long loop_t0 = wall_clock64();
#endif
  while (budget > 0 && should_continue(S, P, &reason)) {
    if (t.aborted) {
      S.done = 1;
      S.stop_reason = STOP_ABORTED;
      if (t.rank == 0 && threadIdx.x == 0) *P.st = S;
      return;
    }
    budget--;
    if (P.alg == ALG_IHT) {
      // IHT_S_gen loop (algorithms.cu:422-480), mu = 0.65 (gaga_gen.cu:654)
      const float mu = 0.65f;
      float gm = 0.f;
      opAT(t, L, P, S, P.resid, [&](int j, float g) {
        P.grad[j] = g;
        gm = fmaxf(gm, fabsf(g));
      });
      {
        double v[1] = {gm};
        const int op[1] = {1};
        reduce(t, v, op);
        S.max_change = 2.0f * mu * (float)v[0];
      }
      for (int i = t.gtid(); i < n; i += t.gsize()) P.x[i] = fmaf(mu, P.grad[i], P.x[i]);
      if (S.min_val <= S.max_change) {
        zero_counters(t, P);
        t.sync();
        find_support_bin(t, L, P, P.x, P.bins, S, S.slope, S.max_value, &S.k_bin);
      } else {
        S.min_val = S.min_val - S.max_change;
      }
      threshold_x(t, P, S.k_bin);
      t.sync();
      S.supp_count = build_support(t, P, S.k_bin);
      double e2 = residual(t, L, P, S, P.resid, P.resid_update);
      double v[1] = {e2};
      const int op[1] = {0};
      reduce(t, v, op);
      S.err = (float)sqrt(v[0]);
      push16(S.prev, S.err);
      stop_update(S, 749, false);
    } else if (P.alg == ALG_HTSD) {
      // HT_SD_S_gen loop (algorithms.cu:846-870): restricted steepest descent on the
      // fixed support, then the threshold again
      float xm;
      (void)step_restricted_sd(t, L, P, S, &xm);
      threshold_x(t, P, S.k_bin);
      t.sync();
      S.err = S.prev[15];
#pragma unroll
      for (int j = 0; j < 15; j++) S.evo[j] = S.evo[j + 1];
      S.evo[15] = S.prev[14] - S.prev[15];
      S.diff = max16(S.evo);
    } else if (P.alg == ALG_HTCG) {
      // HT_CG_S_gen loop (algorithms.cu:1913-1940): one restricted CG step, squared
      // residuals in the ring
      step_restricted_cg(t, L, P, S, S.prev);
      S.err = S.prev[15];
#pragma unroll
      for (int j = 0; j < 15; j++) S.evo[j] = S.evo[j + 1];
      S.evo[15] = S.prev[14] - S.prev[15];
      S.diff = max16(S.evo);
    } else if (P.alg == ALG_FIHT || P.alg == ALG_ALPS) {
      // RestrictedFIHT_S_gen (functions.cu:1668-1746) and RestrictedALPS_S_gen
      // (functions.cu:1748-1851).  Names: x_prev in gprev, the extrapolated point e in
      // gprev_thres, A x_prev in resid2, A e (then A of the step direction) in resid3,
      // A x in resid_update.
      float tau, tmp;
      {
        double tn = 0.0, td = 0.0;
        for (int i = t.gtid(); i < m; i += t.gsize()) {
          const float a = __fsub_rn(P.resid2[i], P.resid_update[i]);
          P.resid2[i] = a;
          tn += (double)P.resid[i] * (double)a;
          td += (double)a * (double)a;
        }
        double v[2] = {tn, td};
        const int op[2] = {0, 0};
        reduce(t, v, op);
        tau = (float)v[0];
        tmp = (float)v[1];
      }
      tau = (fabsf(tau) < 400.0f * fabsf(tmp)) ? tau / tmp : 0.f;
      for (int i = t.gtid(); i < n; i += t.gsize()) {
        const float xi = P.x[i];
        P.gprev_thres[i] = fmaf(tau, __fsub_rn(P.gprev[i], xi), xi);
      }
      for (int i = t.gtid(); i < m; i += t.gsize()) {
        const float ae = fmaf(tau, P.resid2[i], P.resid_update[i]);
        P.resid3[i] = ae;
        P.resid[i] = __fsub_rn(P.y[i], ae);
      }
      t.sync();
      opAT(t, L, P, S, P.resid, [&](int j, float g) { P.grad[j] = g; });
      t.sync();
      double th2 = 0.0;
      if (P.alg == ALG_ALPS) {
        // threshold_three: the gradient off e's support, binned with the current
        // alpha and MaxBin left unchanged (RestrictedALPS takes them by value), cut to
        // its k largest; threshold_four adds the gradient on e's support back
        float tm = 0.f;
        for (int i = t.gtid(); i < n; i += t.gsize()) {
          P.gprev[i] = P.x[i];
          const float th = (P.gprev_thres[i] == 0.f) ? P.grad[i] : 0.f;
          P.thres[i] = th;
          tm = fmaxf(tm, fabsf(th));
        }
        for (int i = t.gtid(); i < m; i += t.gsize()) P.resid2[i] = P.resid_update[i];
        zero_counters(t, P);
        float mv;
        {
          double v[1] = {tm};
          const int op[1] = {1};
          reduce(t, v, op);  // barrier: counters zeroed, thres visible
          mv = (float)v[0];
        }
        const float sa = S.alpha_bin;
        const int smb = S.max_bin;
        int kbi;
        find_support_bin(t, L, P, P.thres, P.bins, S, (float)(P.num_bins - 1) / mv, mv, &kbi);
        S.alpha_bin = sa;
        S.max_bin = smb;
        for (int i = t.gtid(); i < n; i += t.gsize()) {
          float th = (P.bins[i] <= kbi) ? P.thres[i] : 0.f;
          if (P.gprev_thres[i] != 0.f) th = P.grad[i];
          P.thres[i] = th;
          th2 += (double)th * (double)th;
        }
        t.sync();
        S.supp_count = build_support_if(t, P, [&](int i) { return P.thres[i] != 0.f; });
      } else {
        for (int i = t.gtid(); i < n; i += t.gsize()) {
          P.gprev[i] = P.x[i];
          const float th = (P.gprev_thres[i] == 0.f) ? 0.f : P.grad[i];  // threshold_two
          P.thres[i] = th;
          th2 += (double)th * (double)th;
        }
        for (int i = t.gtid(); i < m; i += t.gsize()) P.resid2[i] = P.resid_update[i];
        t.sync();
        S.supp_count = build_support_if(t, P, [&](int i) { return P.gprev_thres[i] != 0.f; });
      }
      opA(t, L, P, S, P.thres, P.resid3);
      float mu;
      {
        double a2 = 0.0;
        for (int i = t.gtid(); i < m; i += t.gsize()) a2 += (double)P.resid3[i] * (double)P.resid3[i];
        double v[2] = {th2, a2};
        const int op[2] = {0, 0};
        reduce(t, v, op);
        mu = (float)v[0];
        const float den = (float)v[1];
        mu = (mu < 400.0f * den) ? mu / den : 1.0f;
      }
      float xm = 0.f;
      for (int i = t.gtid(); i < n; i += t.gsize()) {
        const float xn = fmaf(mu, P.grad[i], P.gprev_thres[i]);
        P.x[i] = xn;
        xm = fmaxf(xm, fabsf(xn));
      }
      // the hard threshold (algorithms.cu:5571-5580)
      S.min_val = 0.f;
      rebin_x(t, L, P, S, xm, false);
      threshold_x(t, P, S.k_bin);
      t.sync();
      S.supp_count = build_support(t, P, S.k_bin);
      (void)residual(t, L, P, S, P.resid, P.resid_update);
      t.sync();
      // steepest descent on the restricted support (algorithms.cu:5581-5602)
      const int kb = S.k_bin;
      double s2 = 0.0;
      opAT(t, L, P, S, P.resid, [&](int j, float g) {
        P.grad[j] = g;
        const float th = (P.bins[j] <= kb) ? g : 0.f;
        P.thres[j] = th;
        s2 += (double)th * (double)th;
      });
      t.sync();
      opA(t, L, P, S, P.thres, P.resid3);
      {
        double a2 = 0.0;
        for (int i = t.gtid(); i < m; i += t.gsize()) a2 += (double)P.resid3[i] * (double)P.resid3[i];
        double v[2] = {s2, a2};
        const int op[2] = {0, 0};
        reduce(t, v, op);
        mu = (float)v[0];
        const float den = (float)v[1];
        mu = (mu < 400.0f * den) ? mu / den : 1.0f;
      }
      for (int i = t.gtid(); i < n; i += t.gsize()) P.x[i] = fmaf(mu, P.thres[i], P.x[i]);
      double e2 = 0.0;
      for (int i = t.gtid(); i < m; i += t.gsize()) {
        const float ru = fmaf(mu, P.resid3[i], P.resid_update[i]);
        P.resid_update[i] = ru;
        const float r = __fsub_rn(P.y[i], ru);
        P.resid[i] = r;
        e2 += (double)r * (double)r;
      }
      {
        double v[1] = {e2};
        const int op[1] = {0};
        reduce(t, v, op);
        S.err = (float)sqrt(v[0]);
      }
      push16(S.prev, S.err);
      stop_update(S, 749);
    } else if (P.alg == ALG_CGIHTP) {
      // CGIHTprojected_S_gen loop (algorithms.cu:4602-4785).  Names: g_S in thres,
      // the CG direction p in gprev, A p in resid2, A g_S in resid_update once the
      // iteration ends.  A steepest-descent step with a fresh threshold while the
      // gradient's part off the current support is large against its part on it
      // (|g - p| / |g_S| > projFracTol), else a CG step on the current support.
      const int kb0 = S.k_bin;
      double e2, vt2, dd, ru2, ap2;
      if (S.supp_change) {
        float mu = (S.vt2 < 400.0f * S.ru2) ? S.vt2 / S.ru2 : 1.0f;
        float xm = 0.f;
        for (int i = t.gtid(); i < n; i += t.gsize()) {
          const float xn = fmaf(mu, P.grad[i], P.x[i]);
          P.x[i] = xn;
          xm = fmaxf(xm, fabsf(xn));
        }
        S.min_val = 0.f;
        S.max_change = 1.0f;
        rebin_x(t, L, P, S, xm, false);
        threshold_x(t, P, S.k_bin);
        t.sync();
        S.supp_count = build_support(t, P, S.k_bin);
        e2 = residual(t, L, P, S, P.resid, P.resid_update);
        t.sync();
        const int kb = S.k_bin;
        double g2 = 0.0, d2 = 0.0;
        opAT(t, L, P, S, P.resid, [&](int j, float g) {
          P.grad[j] = g;
          const bool in = P.bins[j] <= kb;
          const float th = in ? g : 0.f;
          P.thres[j] = th;
          P.gprev[j] = th;  // p = g_S
          g2 += (double)th * (double)th;
          if (!in) d2 += (double)g * (double)g;  // g - p is g off the support
        });
        t.sync();
        opA(t, L, P, S, P.thres, P.resid_update);
        double a2 = 0.0;
        for (int i = t.gtid(); i < m; i += t.gsize()) {
          const float ru = P.resid_update[i];
          P.resid2[i] = ru;  // A p = A g_S
          a2 += (double)ru * (double)ru;
        }
        double v[4] = {e2, g2, d2, a2};
        const int op[4] = {0, 0, 0, 0};
        reduce(t, v, op);
        e2 = v[0];
        vt2 = v[1];
        dd = v[2];
        ru2 = v[3];
        ap2 = v[3];
      } else {
        float mu = (S.vt2 < 400.0f * S.ap2) ? S.vt2 / S.ap2 : 1.0f;
        // p lies on the current support, so x stays on it
        for (int i = t.gtid(); i < n; i += t.gsize()) P.x[i] = fmaf(mu, P.gprev[i], P.x[i]);
        t.sync();
        e2 = residual(t, L, P, S, P.resid, P.resid_update);
        t.sync();
        double g2 = 0.0;
        opAT(t, L, P, S, P.resid, [&](int j, float g) {
          P.grad[j] = g;
          const float th = (P.bins[j] <= kb0) ? g : 0.f;
          P.thres[j] = th;
          g2 += (double)th * (double)th;
        });
        t.sync();
        opA(t, L, P, S, P.thres, P.resid_update);
        double v[2] = {e2, g2};
        const int op2[2] = {0, 0};
        reduce(t, v, op2);
        e2 = v[0];
        vt2 = v[1];
        float beta = (float)vt2;
        beta = (beta < 400.0f * S.vt2) ? beta / S.vt2 : 0.f;
        double d2 = 0.0;
        for (int i = t.gtid(); i < n; i += t.gsize()) {
          const float pn = __fadd_rn(__fmul_rn(beta, P.gprev[i]), P.thres[i]);
          P.gprev[i] = pn;
          const float d = __fsub_rn(P.grad[i], pn);
          d2 += (double)d * (double)d;
        }
        double r2 = 0.0, q2 = 0.0;
        for (int i = t.gtid(); i < m; i += t.gsize()) {
          const float ru = P.resid_update[i];
          const float ap = __fadd_rn(__fmul_rn(beta, P.resid2[i]), ru);
          P.resid2[i] = ap;
          r2 += (double)ru * (double)ru;
          q2 += (double)ap * (double)ap;
        }
        double w[3] = {d2, r2, q2};
        const int op3[3] = {0, 0, 0};
        reduce(t, w, op3);
        dd = w[0];
        ru2 = w[1];
        ap2 = w[2];
      }
      S.vt2 = (float)vt2;
      S.ru2 = (float)ru2;
      S.ap2 = (float)ap2;
      const float pf = (float)sqrt(dd), tn = (float)sqrt(vt2);
      S.supp_change = (pf < 1000.0f * tn) ? ((pf / tn > P.proj_frac_tol) ? 1 : 0) : 1;
      S.err = (float)sqrt(e2);
      push16(S.prev, S.err);
      stop_update(S, 749);
    } else if ((P.alg == ALG_NIHT || P.alg == ALG_HTP) && P.timing) {
      // NIHT_S_timings_gen / HTP_S_timings_gen (algorithms_timings.cu:546-640,
      // 1359-1545): the support by supportFlag 0 (the skip rule), 1 (FindSupportSet
      // asked to bin at every step; slope and intercept refreshed only when the skip
      // rule allows), 2 (the sort-based threshold T, lowered by maxChange between
      // sorts) or 3 (a sort at every step)
      const unsigned long long c0 = wall_clock64();
      float xm;
      S.max_change = step_restricted_sd(t, L, P, S, &xm);
      const unsigned long long c1 = wall_clock64();
      const int sf = P.supp_flag;
      if (sf < 2) {
        if (S.min_val <= S.max_change) {
          double v[1] = {xm};
          const int op[1] = {1};
          reduce(t, v, op);
          S.max_value = (float)v[0];
          S.slope = (float)(P.num_bins - 1) / S.max_value;
        }
        const float mc = sf == 0 ? S.max_change : S.max_value;
        if (S.min_val > mc) {
          S.min_val = S.min_val - mc;
        } else {
          zero_counters(t, P);
          t.sync();
          find_support_bin(t, L, P, P.x, P.bins, S, S.slope, S.max_value, &S.k_bin);
        }
        threshold_x(t, P, S.k_bin);
        t.sync();
        S.supp_count = build_support(t, P, S.k_bin);
      } else {
        // FindSupportSet_sort (functions.cu:438-458) with threshold_and_support
        // (kernels.cu:85-95): entries below T are cut and their bins set to 2; the
        // sort branch first sets every bin to 1.  A kept entry may keep bin 2, so the
        // operator's support list also takes the nonzeros of x.
        S.k_bin = 1;
        const float mcT = sf == 2 ? S.max_change : S.thr;
        t.sync();  // x complete before it is counted
        const bool sort = !(S.thr > mcT);
        if (sort)
          S.thr = team_kth_largest_abs(t, P, P.x, P.k);
        else
          S.thr = __fsub_rn(S.thr, mcT);
        const float T = S.thr;
        for (int i = t.gtid(); i < n; i += t.gsize()) {
          if (sort) P.bins[i] = 1;
          if (fabsf(P.x[i]) < T) {
            P.x[i] = 0.f;
            P.bins[i] = 2;
          }
        }
        t.sync();
        S.supp_count = build_support_if(t, P, [&](int i) { return P.bins[i] <= 1 || P.x[i] != 0.f; });
      }
      const unsigned long long c2 = wall_clock64();
      int icg = 0;
      if (P.alg == ALG_NIHT) {
        S.err = S.prev[15];
        stop_update_timing(S, 749);
      } else {
        const float errCG = cg_projection(t, L, P, S, false, 15, &icg);
        S.err = sqrtf(errCG);
        push16(S.prev, S.err);
        stop_update_timing(S, 125);
      }
      const unsigned long long c3 = wall_clock64();
      if (P.trace_ticks && t.rank == 0 && threadIdx.x == 0) {
        XG(unsigned long long) tt = P.trace_ticks + 4 * (size_t)S.iter;
        tt[0] = c3 - c0;
        tt[1] = c2 - c1;
        tt[2] = (unsigned long long)icg;
        tt[3] = P.alg == ALG_HTP ? c3 - c2 : 0ull;
      }
    } else if (P.alg == ALG_NIHT || P.alg == ALG_HTP) {
      float xm;
      S.max_change = step_restricted_sd(t, L, P, S, &xm);
      if (S.min_val <= S.max_change) {
        rebin_x(t, L, P, S, xm, false);
      } else {
        S.min_val = S.min_val - S.max_change;
      }
      threshold_x(t, P, S.k_bin);
      t.sync();
      S.supp_count = build_support(t, P, S.k_bin);
      if (P.alg == ALG_NIHT) {
        S.err = S.prev[15];
        stop_update(S, 749);
      } else {
        const float errCG = cg_projection(t, L, P, S, false);
        S.err = sqrtf(errCG);
        push16(S.prev, S.err);
        stop_update(S, 125);
      }
    } else if (P.alg == ALG_CSMPSP) {
      // gradient support, joined with the current one (algorithms.cu:3524-3542)
      float gm = 0.f;
      zero_counters(t, P);
      opAT(t, L, P, S, P.resid, [&](int j, float g) {
        P.grad[j] = g;
        gm = fmaxf(gm, fabsf(g));
      });
      {
        double v[1] = {gm};
        const int op[1] = {1};
        reduce(t, v, op);
        S.max_value = (float)v[0];
      }
      S.min_val = 0.f;
      S.slope = (float)(P.num_bins - 1) / S.max_value;
      find_support_bin(t, L, P, P.grad, P.bins2, S, S.slope, S.max_value, &S.k_bin_grad);
      for (int i = t.gtid(); i < n; i += t.gsize())
        if (P.bins2[i] <= S.k_bin_grad && P.bins[i] > S.k_bin) P.bins[i] = S.k_bin;
      t.sync();
      S.supp_count = build_support(t, P, S.k_bin);
      cg_projection(t, L, P, S, true);
      // forced rebin of x (algorithms.cu:3607-3620)
      float xm = 0.f;
      for (int i = t.gtid(); i < n; i += t.gsize()) xm = fmaxf(xm, fabsf(P.x[i]));
      S.min_val = 0.f;
      rebin_x(t, L, P, S, xm, false);
      threshold_x(t, P, S.k_bin);
      t.sync();
      S.supp_count = build_support(t, P, S.k_bin);
      double e2 = residual(t, L, P, S, P.resid, P.resid_update);
      double v[1] = {e2};
      const int op[1] = {0};
      reduce(t, v, op);
      S.err = (float)sqrt(v[0]);
      push16(S.prev, S.err);
      stop_update(S, 125);
    } else {  // CGIHT
      float xm;
      if (P.restart || !S.supp_change) {
        S.max_change = step_cg_restricted(t, L, P, S, &xm);
#ifdef XCS_PHASE_TIMING
        if (P.phase_ticks && t.rank == 0 && threadIdx.x == 0) atomicAdd(&P.phase_ticks[16], 1ull);
#endif
      } else {
        PHASE_BEGIN();
        S.max_change = step_cg_unrestricted(t, L, P, S, &xm);
        PHASE(P, t, 11);
#ifdef XCS_PHASE_TIMING
        if (P.phase_ticks && t.rank == 0 && threadIdx.x == 0) atomicAdd(&P.phase_ticks[17], 1ull);
#endif
      }
      S.beta_to_zero = 0;
      PHASE_BEGIN();
      if (S.min_val <= S.max_change) {
        const int kb_prev = S.k_bin;
        rebin_x(t, L, P, S, xm, true);
        PHASE(P, t, 12);
        // checkSupportEvolution (kernels.cu:178-193), evaluated race-free
        float ch = 0.f;
        for (int i = t.gtid(); i < n; i += t.gsize())
          if (P.bins2[i] <= kb_prev && P.bins[i] > S.k_bin) ch = 1.f;
        double v[1] = {ch};
        const int op[1] = {1};
        reduce(t, v, op);
        S.supp_change = v[0] > 0.0 ? 1 : 0;
        if (S.supp_change) {
          if (P.restart) {
            S.beta_to_zero = 1;
          } else {
            for (int i = t.gtid(); i < n; i += t.gsize())
              P.gprev_thres[i] = (P.bins[i] <= S.k_bin) ? P.gprev[i] : 0.f;
          }
        }
        threshold_x(t, P, S.k_bin);
        t.sync();
        S.supp_count = build_support(t, P, S.k_bin);
        PHASE(P, t, 12);
      } else {
        S.supp_change = 0;
        S.min_val = S.min_val - S.max_change;
        threshold_x(t, P, S.k_bin);
        t.sync();
        PHASE(P, t, 12);
      }
      S.err = S.prev[15];
      stop_update(S, 749);
    }
    S.iter++;
    trace_write(t, P, S.iter, S.k_bin, S.prev[15]);
    if (yield(S)) break;
  }
#ifdef XCS_PHASE_TIMING
  if (P.phase_ticks && t.rank == 0 && threadIdx.x == 0) {
    atomicAdd(&P.phase_ticks[13], wall_clock64() - loop_t0);
    atomicAdd(&P.phase_ticks[14], (unsigned long long)S.iter);
  }
#endif
  if (t.aborted) {
    S.done = 1;
    S.stop_reason = STOP_ABORTED;
  } else if (!should_continue(S, P, &reason)) {
    S.done = 1;
    S.stop_reason = reason;
  }
  if (t.rank == 0 && threadIdx.x == 0) *P.st = S;
}

}  // namespace xcs
