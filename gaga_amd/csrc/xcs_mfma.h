// Matrix-core (MFMA) products for many right-hand sides, gfx950.
//
// C = A_op * B_op with both operands K-contiguous ("TN"):
//   A_op: M x K, row r at A + r * lda_bytes
//   B_op: K x N, column c at B + col(c) * ldb_bytes
//   C:    C[col(c) * ldc + r] or, by position, C[c * ldc + r] (fp32), optionally
//         one slice per K split
// col(c) = col_map ? col_map[c] : c for c < *ncols, so a product can run over
// the active signals only.  Formats: BF16 (v_mfma_f32_32x32x16_bf16) and OCP
// FP8 e4m3 (v_mfma_f32_32x32x64_f8f6f4, format code 0 for both operands);
// accumulation in FP32.
//
// Tiling: GM x GN waves (64 GM GN threads), each wave WM x WN MFMA 32 x 32
// blocks, so the block tile is (32 WM GM) x (32 WN GN): 2 x 2 waves of 2 x 2
// blocks -> 128 x 128; 4 x 2 waves of 2 x 4 blocks -> 256 x 256 (8 waves, each
// wave's 6 LDS reads per K step feed 8 MFMAs); 128 bytes of K per stage (64 bf16
// or 128 fp8), two LDS stages with the next stage prefetched into registers
// while the current one is multiplied.  Products that fill the chip with 256 x
// 128 tiles take gemm_tn8_kernel below instead.
//
// MFMA operand placement used here: lane l holds row (l % 32) of the A block
// and column (l % 32) of the B block, with the same run of K values (bytes
// [16 * (l / 32), +16) of each 32-byte K slice for bf16, [32 * (l / 32), +32)
// of each 64-byte slice for fp8) in both, so every product pairs equal K.
// Result: accumulator v of lane l is C[8 (v / 4) + 4 (l / 32) + v % 4][l % 32].
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

namespace xcs {

typedef __bf16 bf16x8_t __attribute__((ext_vector_type(8)));
typedef float f32x16_t __attribute__((ext_vector_type(16)));
typedef int i32x8_t __attribute__((ext_vector_type(8)));
typedef int i32x4_t __attribute__((ext_vector_type(4)));

enum GemmFmt { FMT_BF16 = 0, FMT_FP8 = 1 };

constexpr int GT_M = 128, GT_N = 128;  // block tile
constexpr int GT_KB = 128;             // K bytes per stage
constexpr int GT_ROW = GT_KB + 16;     // padded LDS row, bytes (conflict-free b128 reads)
constexpr int GT_THREADS = 256;
constexpr float FP8_MAX = 448.0f;      // largest finite OCP e4m3 value

struct GemmArgs {
  const uint8_t *A;
  long lda_bytes;
  const uint8_t *B;
  long ldb_bytes;
  float *C;
  long ldc;           // floats
  long split_stride;  // floats between K-split slices of C
  int M, K, N;        // K in elements; N = columns the grid covers
  int ksplit;
  const int *ncols;      // device, nullable (then N)
  const int *col_map;    // device, nullable (identity)
  int c_by_pos;          // C's columns by position c instead of col(c)
  const float *row_scale;  // per output row, nullable
  const float *col_scale;  // per physical column, nullable
};

__device__ __forceinline__ int gemm_esize(int fmt) { return fmt == FMT_BF16 ? 2 : 1; }

// WM x WN MFMA 32 x 32 blocks per wave, GM x GN waves.  LDS: two stages of
// (BM + BN) rows of 128 K bytes (padded).
template <int FMT, int WM, int WN, int GM = 2, int GN = 2>
__global__ void __launch_bounds__(64 * GM * GN) gemm_tn_kernel(GemmArgs g) {
  constexpr int NT = 64 * GM * GN;                  // threads
  constexpr int BM = 32 * WM * GM, BN = 32 * WN * GN;
  constexpr int RP = NT / 8;                        // rows one pass of 16-byte chunks covers
  constexpr int CA = BM * 8 / NT, CB = BN * 8 / NT;  // 16-byte chunks per thread
  static_assert(BM % RP == 0 && BN % RP == 0, "whole row passes");
  __shared__ __attribute__((aligned(16))) uint8_t lds[2][(BM + BN) * GT_ROW];
  const int ncols = g.ncols ? *g.ncols : g.N;
  // XCD-aware tile order: workgroups are dealt to the 8 XCDs round-robin in
  // linear id order (x fastest), so the gy column tiles of one row slice of A
  // get linear ids 8 apart and run together on one XCD, whose L2 then fetches
  // that slice of A once for all of them.  A bijection on the tiles of each K
  // slice; the identity unless gx is a multiple of 8 and gy > 1.
  int bx = blockIdx.x, by = blockIdx.y;
  {
    const int gx = gridDim.x, gy = gridDim.y;
    if (gy > 1 && gx % 8 == 0) {
      const int l = blockIdx.x + gx * blockIdx.y;
      bx = ((l >> 3) / gy) * 8 + (l & 7);
      by = (l >> 3) % gy;
    }
  }
  const int m0 = bx * BM, n0 = by * BN;
  if (n0 >= ncols) return;
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const long kbytes = (long)g.K * (FMT == FMT_BF16 ? 2 : 1);
  const long kb_split = kbytes / g.ksplit;
  const long kb0 = (long)blockIdx.z * kb_split;
  const int nsteps = (int)(kb_split / GT_KB);

  // global -> register assignment: chunks of 16 bytes, 8 per 128-byte row
  const uint8_t *pa[CA], *pb[CB];
  bool okb[CB];
#pragma unroll
  for (int i = 0; i < CA; i++) {
    const int row = (tid >> 3) + RP * i;
    pa[i] = g.A + (long)(m0 + row) * g.lda_bytes + kb0 + (tid & 7) * 16;
  }
#pragma unroll
  for (int i = 0; i < CB; i++) {
    const int row = (tid >> 3) + RP * i;
    const int c = n0 + row;
    okb[i] = c < ncols;
    const int phys = okb[i] ? (g.col_map ? g.col_map[c] : c) : 0;
    pb[i] = g.B + (long)phys * g.ldb_bytes + kb0 + (tid & 7) * 16;
  }
  i32x4_t ra[CA], rb[CB];
  auto gload = [&](long off) {
#pragma unroll
    for (int i = 0; i < CA; i++) ra[i] = *(const i32x4_t *)(pa[i] + off);
#pragma unroll
    for (int i = 0; i < CB; i++)
      rb[i] = okb[i] ? *(const i32x4_t *)(pb[i] + off) : i32x4_t{0, 0, 0, 0};
  };
  auto lstore = [&](int buf) {
#pragma unroll
    for (int i = 0; i < CA; i++)
      *(i32x4_t *)(&lds[buf][((tid >> 3) + RP * i) * GT_ROW + (tid & 7) * 16]) = ra[i];
#pragma unroll
    for (int i = 0; i < CB; i++)
      *(i32x4_t *)(&lds[buf][(BM + (tid >> 3) + RP * i) * GT_ROW + (tid & 7) * 16]) = rb[i];
  };

  f32x16_t acc[WM][WN];
#pragma unroll
  for (int a = 0; a < WM; a++)
#pragma unroll
    for (int b = 0; b < WN; b++)
#pragma unroll
      for (int v = 0; v < 16; v++) acc[a][b][v] = 0.f;

  const int wm = wave / GN, wn = wave % GN, r32 = lane & 31, h = lane >> 5;
  gload(0);
  lstore(0);
  __syncthreads();
  for (int s = 0; s < nsteps; s++) {
    const int buf = s & 1;
    if (s + 1 < nsteps) gload((long)(s + 1) * GT_KB);
    const uint8_t *LA = lds[buf], *LB = lds[buf] + BM * GT_ROW;
    // a wave in its MFMA section gets issue priority over waves that are
    // loading or storing (measured 5-10 % faster for BF16 A^T R 16384 x 512 x 4096)
    __builtin_amdgcn_s_setprio(1);
    if (FMT == FMT_BF16) {
#pragma unroll
      for (int kk = 0; kk < 4; kk++) {
        bf16x8_t fa[WM], fb[WN];
#pragma unroll
        for (int i = 0; i < WM; i++)
          fa[i] = *(const bf16x8_t *)(LA + (wm * 32 * WM + i * 32 + r32) * GT_ROW + kk * 32 + h * 16);
#pragma unroll
        for (int i = 0; i < WN; i++)
          fb[i] = *(const bf16x8_t *)(LB + (wn * 32 * WN + i * 32 + r32) * GT_ROW + kk * 32 + h * 16);
#pragma unroll
        for (int a = 0; a < WM; a++)
#pragma unroll
          for (int b = 0; b < WN; b++)
            acc[a][b] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(fa[a], fb[b], acc[a][b], 0, 0, 0);
      }
    } else {
#pragma unroll
      for (int kk = 0; kk < 2; kk++) {
        i32x8_t fa[WM], fb[WN];
#pragma unroll
        for (int i = 0; i < WM; i++) {
          const uint8_t *q = LA + (wm * 32 * WM + i * 32 + r32) * GT_ROW + kk * 64 + h * 32;
          const i32x4_t x0 = *(const i32x4_t *)q, x1 = *(const i32x4_t *)(q + 16);
          fa[i] = i32x8_t{x0[0], x0[1], x0[2], x0[3], x1[0], x1[1], x1[2], x1[3]};
        }
#pragma unroll
        for (int i = 0; i < WN; i++) {
          const uint8_t *q = LB + (wn * 32 * WN + i * 32 + r32) * GT_ROW + kk * 64 + h * 32;
          const i32x4_t x0 = *(const i32x4_t *)q, x1 = *(const i32x4_t *)(q + 16);
          fb[i] = i32x8_t{x0[0], x0[1], x0[2], x0[3], x1[0], x1[1], x1[2], x1[3]};
        }
#pragma unroll
        for (int a = 0; a < WM; a++)
#pragma unroll
          for (int b = 0; b < WN; b++)
            acc[a][b] = __builtin_amdgcn_mfma_scale_f32_32x32x64_f8f6f4(fa[a], fb[b], acc[a][b], 0,
                                                                        0, 0, 0, 0, 0);
      }
    }
    __builtin_amdgcn_s_setprio(0);
    if (s + 1 < nsteps) lstore(buf ^ 1);
    __syncthreads();
  }

  float *C = g.C + (long)blockIdx.z * g.split_stride;
#pragma unroll
  for (int b = 0; b < WN; b++) {
    const int c = n0 + wn * 32 * WN + b * 32 + r32;
    if (c >= ncols) continue;
    const int phys = g.col_map ? g.col_map[c] : c;
    const float cs = g.col_scale ? g.col_scale[phys] : 1.0f;
#pragma unroll
    for (int a = 0; a < WM; a++)
#pragma unroll
      for (int q = 0; q < 4; q++) {
        const int r = m0 + wm * 32 * WM + a * 32 + q * 8 + h * 4;
        float4 v = make_float4(acc[a][b][4 * q], acc[a][b][4 * q + 1], acc[a][b][4 * q + 2],
                               acc[a][b][4 * q + 3]);
        if (g.row_scale) {
          v.x *= g.row_scale[r];
          v.y *= g.row_scale[r + 1];
          v.z *= g.row_scale[r + 2];
          v.w *= g.row_scale[r + 3];
        }
        v.x *= cs;
        v.y *= cs;
        v.z *= cs;
        v.w *= cs;
        *(float4 *)(C + (long)(g.c_by_pos ? c : phys) * g.ldc + r) = v;
      }
  }
}

// 256 x 128 block tile by 8 waves (4 x 2, each 64 x 64), global loads straight
// into LDS.  What bounded the register-staged kernel above was the path from
// global memory through registers into LDS (its MFMA section alone runs in half
// the time): here each wave issues 16-byte global -> LDS loads two stages ahead
// of the MFMAs, three stages of 48 KB in LDS, and waits with a counted vmcnt, so
// a stage's loads stay in flight over a whole stage of MFMAs and one barrier.
// The loads write LDS in lane order (8 rows of 128 bytes per instruction, no
// padding); bank conflicts are avoided by the order of the chunks within a row
// instead: row r keeps its 16-byte chunk c at position c ^ (r & 7), so the eight
// lanes of a read phase (eight rows, one chunk) touch all banks.  Columns past
// ncols load column 0 and are not stored.  Each MFMA chain adds K in the order
// of the kernel above, so the products are the same bits.  Measured: BF16
// 16384 x 512 x 4096 77 -> 59 us (1154 TFLOP/s; without the loads 55, without the
// products 41, and the matrix cores alone do 1.8 PFLOP/s on random operands).
typedef const __attribute__((address_space(1))) uint8_t *gptr_t;
typedef __attribute__((address_space(3))) uint8_t *lptr_t;
constexpr int G8_BM = 256, G8_BN = 128, G8_NT = 512;
constexpr int G8_STAGE = (G8_BM + G8_BN) * GT_KB;
template <int FMT>
__global__ void __launch_bounds__(G8_NT) gemm_tn8_kernel(GemmArgs g) {
  __shared__ __attribute__((aligned(128))) uint8_t lds0[G8_STAGE];
  __shared__ __attribute__((aligned(128))) uint8_t lds1[G8_STAGE];
  __shared__ __attribute__((aligned(128))) uint8_t lds2[G8_STAGE];
  const int ncols = g.ncols ? *g.ncols : g.N;
  int bx = blockIdx.x, by = blockIdx.y;
  {  // XCD-aware tile order, as in gemm_tn_kernel
    const int gx = gridDim.x, gy = gridDim.y;
    if (gy > 1 && gx % 8 == 0) {
      const int l = blockIdx.x + gx * blockIdx.y;
      bx = ((l >> 3) / gy) * 8 + (l & 7);
      by = (l >> 3) % gy;
    }
  }
  const int m0 = bx * G8_BM, n0 = by * G8_BN;
  if (n0 >= ncols) return;
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const long kbytes = (long)g.K * (FMT == FMT_BF16 ? 2 : 1);
  const long kb_split = kbytes / g.ksplit;
  const long kb0 = (long)blockIdx.z * kb_split;
  const int nsteps = (int)(kb_split / GT_KB);
  // load i of this wave fills rows 8 (wave + 8 i) .. + 7 of the stage (A rows
  // first, then B columns); lane l: row l / 8, LDS position l % 8
  constexpr int NL = (G8_BM + G8_BN) / 64;  // 6 loads per wave and stage
  const uint8_t *src[NL];
  const int lr = lane >> 3, lc = ((lane & 7) ^ lr) * 16;
#pragma unroll
  for (int i = 0; i < NL; i++) {
    const int row = 8 * (wave + 8 * i) + lr;
    if (i < G8_BM / 64) {
      src[i] = g.A + (long)(m0 + row) * g.lda_bytes + kb0 + lc;
    } else {
      const int c = n0 + row - G8_BM;
      const int phys = c < ncols ? (g.col_map ? g.col_map[c] : c) : (g.col_map ? g.col_map[0] : 0);
      src[i] = g.B + (long)phys * g.ldb_bytes + kb0 + lc;
    }
  }
  // In assembly (it has no output register; LDS is its destination): the
  // compiler would make every later LDS read wait for all such loads in flight.
  auto issue = [&](uint8_t *buf, int s) {
    const unsigned l0 = (unsigned)(uintptr_t)(lptr_t)buf + 1024 * wave;
#pragma unroll
    for (int i = 0; i < NL; i++)
      asm volatile("s_mov_b32 m0, %1\n\t"
                   "s_nop 0\n\t"
                   "global_load_lds_dwordx4 %0, off"
                   :
                   : "v"((gptr_t)(src[i] + (long)s * GT_KB)),
                     "s"(__builtin_amdgcn_readfirstlane(l0 + 8192 * i))
                   : "memory", "m0");
  };
  f32x16_t acc[2][2];
#pragma unroll
  for (int a = 0; a < 2; a++)
#pragma unroll
    for (int b = 0; b < 2; b++)
#pragma unroll
      for (int v = 0; v < 16; v++) acc[a][b][v] = 0.f;
  const int wm = wave >> 1, wn = wave & 1, r32 = lane & 31, h = lane >> 5;
  const int arow = (wm * 64 + r32) * GT_KB, brow = (G8_BM + wn * 64 + r32) * GT_KB, sw = r32 & 7;
  auto compute = [&](const uint8_t *L) {
    __builtin_amdgcn_s_setprio(1);
    if (FMT == FMT_BF16) {
      bf16x8_t fa[4][2], fb[4][2];
      auto read = [&](int kk) {
        const int at = ((kk * 2 + h) ^ sw) * 16;
#pragma unroll
        for (int i = 0; i < 2; i++) {
          fa[kk][i] = *(const bf16x8_t *)(L + arow + i * 32 * GT_KB + at);
          fb[kk][i] = *(const bf16x8_t *)(L + brow + i * 32 * GT_KB + at);
        }
      };
      read(0);
#pragma unroll
      for (int kk = 0; kk < 4; kk++) {
        if (kk < 3) read(kk + 1);
#pragma unroll
        for (int a = 0; a < 2; a++)
#pragma unroll
          for (int b = 0; b < 2; b++)
            acc[a][b] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(fa[kk][a], fb[kk][b],
                                                                acc[a][b], 0, 0, 0);
      }
      // LDS reads stay two operand sets ahead of the MFMAs
      __builtin_amdgcn_sched_group_barrier(0x100, 8, 0);
#pragma unroll
      for (int q = 0; q < 8; q++) {
        __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
        __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);
      }
      __builtin_amdgcn_sched_group_barrier(0x008, 8, 0);
    } else {
#pragma unroll
      for (int kk = 0; kk < 2; kk++) {
        const int c0 = ((kk * 4 + h * 2) ^ sw) * 16, c1 = ((kk * 4 + h * 2 + 1) ^ sw) * 16;
        i32x8_t fa[2], fb[2];
#pragma unroll
        for (int i = 0; i < 2; i++) {
          const uint8_t *q = L + arow + i * 32 * GT_KB;
          const i32x4_t x0 = *(const i32x4_t *)(q + c0), x1 = *(const i32x4_t *)(q + c1);
          fa[i] = i32x8_t{x0[0], x0[1], x0[2], x0[3], x1[0], x1[1], x1[2], x1[3]};
          const uint8_t *w = L + brow + i * 32 * GT_KB;
          const i32x4_t y0 = *(const i32x4_t *)(w + c0), y1 = *(const i32x4_t *)(w + c1);
          fb[i] = i32x8_t{y0[0], y0[1], y0[2], y0[3], y1[0], y1[1], y1[2], y1[3]};
        }
#pragma unroll
        for (int a = 0; a < 2; a++)
#pragma unroll
          for (int b = 0; b < 2; b++)
            acc[a][b] = __builtin_amdgcn_mfma_scale_f32_32x32x64_f8f6f4(fa[a], fb[b], acc[a][b], 0,
                                                                        0, 0, 0, 0, 0);
      }
    }
    __builtin_amdgcn_s_setprio(0);
  };
  // stage s: its loads have landed once at most the next stage's are in flight;
  // after the barrier every wave has also finished reading stage s - 1 (lgkmcnt: its
  // LDS reads have returned, wherever their products are scheduled), whose buffer
  // stage s + 2 takes
  auto step = [&](uint8_t *cur, uint8_t *nxt2, int s) {
    if (s + 1 < nsteps)
      asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)" ::"n"(NL) : "memory");
    else
      asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)" ::: "memory");
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
    if (s + 2 < nsteps) issue(nxt2, s + 2);
    compute(cur);
  };
  issue(lds0, 0);
  if (nsteps > 1) issue(lds1, 1);
  for (int s = 0; s < nsteps; s += 3) {
    step(lds0, lds2, s);
    if (s + 1 < nsteps) step(lds1, lds0, s + 1);
    if (s + 2 < nsteps) step(lds2, lds1, s + 2);
  }

  float *C = g.C + (long)blockIdx.z * g.split_stride;
#pragma unroll
  for (int b = 0; b < 2; b++) {
    const int c = n0 + wn * 64 + b * 32 + r32;
    if (c >= ncols) continue;
    const int phys = g.col_map ? g.col_map[c] : c;
    const float cs = g.col_scale ? g.col_scale[phys] : 1.0f;
#pragma unroll
    for (int a = 0; a < 2; a++)
#pragma unroll
      for (int q = 0; q < 4; q++) {
        const int r = m0 + wm * 64 + a * 32 + q * 8 + h * 4;
        float4 v = make_float4(acc[a][b][4 * q], acc[a][b][4 * q + 1], acc[a][b][4 * q + 2],
                               acc[a][b][4 * q + 3]);
        if (g.row_scale) {
          v.x *= g.row_scale[r];
          v.y *= g.row_scale[r + 1];
          v.z *= g.row_scale[r + 2];
          v.w *= g.row_scale[r + 3];
        }
        v.x *= cs;
        v.y *= cs;
        v.z *= cs;
        v.w *= cs;
        *(float4 *)(C + (long)(g.c_by_pos ? c : phys) * g.ldc + r) = v;
      }
  }
}

// Block tile of a product whose M is a multiple of 256: the 256 x 128 tile where
// its workgroups (one per CU) about fill the chip, else the 128 x 128 one, of
// which there are twice as many.  Measured on MI355X, us, 128 x 128 against
// 256 x 128: BF16 16384 x 512 x 4096 (256 large tiles) 77 / 59, its transpose with
// K split 4 85 / 68, FP8 41 / 36 and 44 / 44; BF16 8192 x 300 x 2048 (96 large
// tiles) 29 / 32, FP8 18 / 21; BF16 4096 x 200 x 1024 (32) 16 / 19.
inline int gemm_tile(int M, int N, int ksplit) {
  return (long)(M / G8_BM) * ((N + G8_BN - 1) / G8_BN) * ksplit >= 192 ? 1 : 0;
}

// Launch of the TN GEMM with block tile `tile`: 0 128 x 128 (4 waves), 1
// 256 x 128 (8 waves), 2 256 x 256 (8 waves).  M must be a multiple of the
// tile's rows (128 or 256); the grid covers N (masked beyond ncols) and ksplit
// slices of K.
template <int FMT>
static hipError_t gemm_tn_launch(int tile, const GemmArgs &g, hipStream_t st) {
  const int bm = tile == 0 ? 128 : 256, bn = tile == 2 ? 256 : 128;
  const dim3 grid(g.M / bm, (g.N + bn - 1) / bn, g.ksplit);
  if (tile == 2)
    hipLaunchKernelGGL((gemm_tn_kernel<FMT, 2, 4, 4, 2>), grid, dim3(512), 0, st, g);
  else if (tile == 1)
    hipLaunchKernelGGL((gemm_tn8_kernel<FMT>), grid, dim3(G8_NT), 0, st, g);
  else
    hipLaunchKernelGGL((gemm_tn_kernel<FMT, 2, 2>), grid, dim3(GT_THREADS), 0, st, g);
  return hipGetLastError();
}

// Sum of the K-split slices in split order (deterministic), active columns.
__global__ void gemm_split_sum_kernel(float *C, long ldc, long split_stride, int ksplit, int M,
                                      int N, const int *ncols, const int *col_map) {
  const int nc = ncols ? *ncols : N;
  const long total = (long)nc * M;
  for (long e = (long)blockIdx.x * blockDim.x + threadIdx.x; e < total;
       e += (long)gridDim.x * blockDim.x) {
    const int c = (int)(e / M), r = (int)(e - (long)c * M);
    const long o = (long)(col_map ? col_map[c] : c) * ldc + r;
    float s = C[o];
    for (int z = 1; z < ksplit; z++) s += C[o + z * split_stride];
    C[o] = s;
  }
}

// ------------------------------------------------------------ quantizers ----
// float -> bf16, round to nearest even (finite inputs).
__host__ __device__ __forceinline__ uint16_t f2bf16_rne(float f) {
  uint32_t u;
  __builtin_memcpy(&u, &f, 4);
  u += 0x7FFFu + ((u >> 16) & 1u);
  return (uint16_t)(u >> 16);
}

// float -> OCP e4m3 (round to nearest even in hardware); inputs are clamped
// to +-448 first so nothing overflows.
__device__ __forceinline__ uint32_t f2fp8x4(float a, float b, float c, float d) {
  a = fminf(fmaxf(a, -FP8_MAX), FP8_MAX);
  b = fminf(fmaxf(b, -FP8_MAX), FP8_MAX);
  c = fminf(fmaxf(c, -FP8_MAX), FP8_MAX);
  d = fminf(fmaxf(d, -FP8_MAX), FP8_MAX);
  int w = __builtin_amdgcn_cvt_pk_fp8_f32(a, b, 0, false);
  w = __builtin_amdgcn_cvt_pk_fp8_f32(c, d, w, true);
  return (uint32_t)w;
}

}  // namespace xcs
