/*
 * gaga_amd: MI355X-native greedy sparse recovery (NIHT, HTP, CSMPSP, CGIHT, and the
 * reference's IHT, ThresholdSD, ThresholdCG, FIHT, ALPS, CGIHTprojected over
 * the 'gen', 'smv' and 'dct' ensembles).  C ABI; plain pointers and sizes.
 *
 * The entry points mirror the reference's MATLAB/MEX call surface
 *   gaga_cs(alg, ens, k, m, n[, p], options)          GAGA/gaga/gaga_cs.m:7-64
 * whose drivers are the MEX functions in GAGA/gaga/gaga_gen.cu:41,
 * GAGA/gaga/gaga_smv.cu:38 and GAGA/gaga/gaga_dct.cu.  The reference's licence
 * (GAGA/GAGA_license:5) reserves the names gaga_cs / gaga_gen / gaga_smv /
 * gaga_dct, so this library exports the same surface under the xcs_ prefix.
 *
 * Conventions (all entry points):
 *   - return 0 on success, a negative XCS_E* code on error; xcs_last_error()
 *     gives a message (thread-local).  Nothing calls exit().
 *   - host buffers are caller-owned; device memory is owned by the library
 *     unless an entry point says it takes device pointers.
 *   - index arrays of the user-problem forms are 1-based, as MATLAB passes
 *     them (the reference shifts them with indexShiftDown, kernels.cu:155-159).
 *   - calls are synchronous and thread-safe (one HIP stream per call).
 */
#ifndef GAGA_AMD_H
#define GAGA_AMD_H
#include <stddef.h>
#ifdef __cplusplus
extern "C" {
#endif

enum {
  XCS_OK = 0,
  XCS_EINVAL = -1,   /* bad argument (algorithm, ensemble, size, option) */
  XCS_EHIP = -2,     /* HIP runtime error */
  XCS_ENOMEM = -3,   /* device allocation failed */
  XCS_ENODEV = -4,   /* no usable GPU */
  XCS_EUNSUP = -5    /* valid request this build does not implement */
};

/* Options: the reference's gagaOptions list (GAGA/gaga/gagaOptions.m:8-58,
 * parsed at GAGA/gaga/gaga_gen.cu:205-320) plus this build's execution knobs.
 * Always initialise with xcs_options_default(). */
typedef struct xcs_options {
  float tol;                 /* stop when ||y - A x||_2 <= tol (reference 'tol') */
  int tol_reference_default; /* 1: use the reference GPU default tol = 10^(-4) in C,
                                which evaluates to -10 (gaga_gen.cu:183); never stops */
  int maxiter;               /* 'maxiter'; default 300 for HTP/CSMPSP, 5000 otherwise */
  int num_bins;              /* 'numBins'; default max(n/20, 1000) */
  int restart;               /* 'restartFlag' for CGIHT (0 off, 1 on) */
  unsigned int seed;         /* 'seed' (generator key word 0) */
  unsigned int instance;     /* generator key word 1 (instance id) */
  int vec_distribution;      /* 'vecDistribution': 0 uniform, 1 binary (default), 2 gaussian */
  int matrix_ensemble;       /* 'matrixEnsemble': gen 1 gaussian; smv 1 ones/sqrt(p),
                                2 binary +-1/sqrt(p), 3 ones (reference smv default) */
  int gpu_number;            /* 'gpuNumber' */
  int mode;                  /* 0 device-resident solve (one launch); 1 plain form:
                                one outer iteration per launch, host-side stop test */
  int team_size;             /* workgroups cooperating on one instance; 0 = auto */
  int block_size;            /* threads per workgroup; 0 = auto */
  float proj_frac_tol;       /* 'projFracTol' of CGIHTprojected (default 3.0,
                                gaga_gen.cu:190); <= 0 selects the default */
  int timing;                /* 'timing' on (1): NIHT and HTP run their timing variants
                                (algorithms_timings.cu), with per-iteration times */
  int supp_flag;             /* 'supportFlag' of the timing variants: 0 adaptive binning,
                                1 binning at every step, 2 sort-based threshold with
                                dynamic detection, 3 a sort at every step (gaga_gen.cu:168) */
  float alpha;               /* 'alpha' (alpha_start) of the timing variants, in [0, 1);
                                xcs_options_default sets 0.25 */
  long barrier_spin_limit;   /* bound of every wait of a multi-workgroup team, in polls of
                                about a microsecond (0: the default, 2^26); a wait that
                                exceeds it abandons the solve with XCS_EHIP ("team barrier
                                timed out") instead of hanging */
} xcs_options;

/* Fill *opts with the reference defaults for (alg, ens, n). */
int xcs_options_default(const char *alg, const char *ens, int n, xcs_options *opts);

/* Generate-and-solve form: [norms times iterations support convRate xout] =
 * gaga_cs(alg, ens, k, m, n[, p], options)  (gaga_gen.cu:90-114, gaga_smv.cu:131-158).
 *   norms[3]   relative l1, l2, linf error of x_out vs the planted x (results.cu:444-487)
 *   times[3]   solve ms, ms per iteration, total ms including generation
 *   support[4] TP, FP, TN, FN (results.cu:400-430)
 *   x_out[n]   recovered vector (may be NULL); x_true[n] planted vector (may be NULL)
 * p is the smv nonzeros per column (ignored for gen/dct). */
int xcs_cs_generate(const char *alg, const char *ens, int k, int m, int n, int p,
                    const xcs_options *opts, float norms[3], float times[3], int *iterations,
                    int support[4], float *conv_rate, float *x_out, float *x_true);

/* The results line the reference appends after every generated solve:
 * File_output / File_output_smv / File_output_gen (GAGA/gaga/functions.cu:34-80), called
 * from results / results_smv / results_gen (GAGA/gaga/results.cu:166-182, 336-352,
 * 509-525).  Same keys, order and number formats ("CGIHT_S_gen output: k 20, m 256, ...
 * seed 7 \n"); matrix_ensemble is printed for gen and smv, p for smv.  Writes the line
 * and its NUL into buf; returns the line length, or XCS_EINVAL if buf_len is too small. */
int xcs_results_line(char *buf, size_t buf_len, const char *alg, const char *ens, int k, int m,
                     int n, int p, int matrix_ensemble, int vec_distribution, const float norms[3],
                     const float times[3], int iterations, float conv_rate, const int support[4],
                     unsigned int seed);

/* Appends that line to <dir>/gpu_data_<ens>YYYYMMDD.txt (local date; dir NULL or "": the
 * working directory), the file the reference opens with "a+" (results.cu:509-525). */
int xcs_results_append(const char *dir, const char *alg, const char *ens, int k, int m, int n,
                       int p, int matrix_ensemble, int vec_distribution, const float norms[3],
                       const float times[3], int iterations, float conv_rate,
                       const int support[4], unsigned int seed);

/* The timing variants' results text (File_output_timings*, functions.cu:82-212): the line
 * with alpha and supp_flag, then one line per iteration (HTP: with its CG steps and CG
 * time; cg_per_iteration and time_for_cg may be NULL for NIHT).  Returns its length. */
int xcs_results_timing_text(char *buf, size_t buf_len, const char *alg, const char *ens, int k,
                            int m, int n, int p, int matrix_ensemble, int vec_distribution,
                            const float norms[3], const float times[3], int iterations,
                            float conv_rate, const int support[4], unsigned int seed, float alpha,
                            int supp_flag, const float *time_iteration, const float *time_supp_set,
                            const int *cg_per_iteration, const float *time_for_cg);
/* Appends that text to <dir>/gpu_timings_data_<ens>YYYYMMDD.txt (results.cu:1540-1560). */
int xcs_results_timing_append(const char *dir, const char *alg, const char *ens, int k, int m,
                              int n, int p, int matrix_ensemble, int vec_distribution,
                              const float norms[3], const float times[3], int iterations,
                              float conv_rate, const int support[4], unsigned int seed,
                              float alpha, int supp_flag, const float *time_iteration,
                              const float *time_supp_set, const int *cg_per_iteration,
                              const float *time_for_cg);

/* Solve-given-problem forms ([outputVector iterations convRate] = gaga_cs(alg,
 * 'gen', y, A, k, options), gaga_gen.cu:115-134).  A is column-major m x n. */
int xcs_cs_gen(const char *alg, const float *y, const float *A, int m, int n, int k,
               const xcs_options *opts, float *x_out, int *iterations, float *conv_rate);
/* Allocation-free variant of xcs_cs_gen.  No counterpart in the reference: it is for
 * callers that cannot allocate device memory (code under HIP graph capture, tight
 * serving loops, harnesses that forbid hipMalloc).  It calls no hipMalloc/hipFree
 * and no allocating library routine: the solver's workspace lives in a fixed
 * 4 MiB device array of the library (one per GPU, held until the process ends).
 *   d_y[m], d_A (column-major, leading dimension lda: a multiple of 64, >= m; rows
 *   m..lda-1 must be finite, zero recommended) and d_x_out[n] are caller-owned
 *   device pointers (16-byte aligned); stream is a hipStream_t or NULL.
 * Limits: n <= XCS_NOALLOC_MAX_N, lda <= XCS_NOALLOC_MAX_LDA, numBins <=
 * XCS_NOALLOC_MAX_BINS; larger requests fail with XCS_EINVAL before any launch.
 * One workgroup solves the instance (opts->block_size threads, default 256), so the
 * result equals xcs_cs_gen's with team_size 1 and the same block size, bit for bit.
 * With iterations and conv_rate NULL the call only enqueues work on the stream (and
 * can be captured); otherwise it waits for the stream and reports them.  Every call on
 * one GPU shares its workspace: calls that overlap on one GPU (other streams, other
 * host threads) race and must be serialised by the caller. */
#define XCS_NOALLOC_MAX_N 16384
#define XCS_NOALLOC_MAX_LDA 4096
#define XCS_NOALLOC_MAX_BINS 16384
int xcs_cs_gen_noalloc(const char *alg, const float *d_y, const float *d_A, int lda, int m, int n,
                       int k, const xcs_options *opts, float *d_x_out, int *iterations,
                       float *conv_rate, void *stream);
/* smv: (rows, cols, vals) triplets, nz entries, 1-based (gaga_smv.cu:159-195). */
int xcs_cs_smv(const char *alg, const float *y, const int *rows, const int *cols,
               const float *vals, int nz, int m, int n, int k, const xcs_options *opts,
               float *x_out, int *iterations, float *conv_rate);
/* dct: m sampled rows of the orthonormal n-point DCT-II, 1-based (gaga_dct.cu:112-117);
 * n must be a power of two. */
int xcs_cs_dct(const char *alg, const float *y, const int *rows, int k, int m, int n,
               const xcs_options *opts, float *x_out, int *iterations, float *conv_rate);

/* ---- resident plans: inputs generated into / kept in HBM, solves timed on device ---- */
typedef struct xcs_plan xcs_plan;
/* Per-iteration timings of the last solve of a plan run with timing on (NIHT, HTP):
 * iteration time and support-set time in ms, HTP's CG iterations and CG time in ms
 * (time_per_iteration, time_supp_set, cg_per_iteration, time_for_cg of
 * algorithms_timings.cu:1540-1543), for the first len iterations; any may be NULL. */
int xcs_plan_timings(xcs_plan *plan, float *iter_ms, float *supp_ms, int *cg_iters, float *cg_ms,
                     int len);
/* The times of the plan's last solve as xcs_cs_generate reports them (ms): solve, solve
 * per iteration, solve + generation (the reference's timeALG, timeIter, timeTotal). */
int xcs_plan_times(xcs_plan *plan, float times[3]);
/* Generate one instance on the device (seed/instance from opts) and keep it. */
int xcs_plan_create(const char *alg, const char *ens, int k, int m, int n, int p,
                    const xcs_options *opts, xcs_plan **plan);
/* Solve from x = 0 with the inputs already resident; *ms = device time. */
int xcs_plan_solve(xcs_plan *plan, float *ms);
/* Results of the last solve (any pointer may be NULL). */
int xcs_plan_results(xcs_plan *plan, float norms[3], int *iterations, int support[4],
                     float *conv_rate, int *stop_reason, float *x_out, float *x_true);
/* Per-iteration trace of the last solve: k_bin and residual norm, length iterations+1. */
int xcs_plan_trace(xcs_plan *plan, int *k_bin, float *resid_norm, int len);
/* Time `reps` back-to-back applications of A^T (transpose = 1, on the planted y) or A_S
 * (transpose = 0, on the planted x) on the resident instance with the plan's team;
 * *ms_per = device ms per application, *bytes = its algorithmic bytes. */
int xcs_plan_apply_timed(xcs_plan *plan, int transpose, int reps, float *ms_per, double *bytes);
/* Algorithmic bytes moved by the operator applications of the last solve
 * (gen A_S x_S: 4m|S|+8|S|+4m; gen A^T r: 4mn+4m+4n, or 4m|S|+4m+4|S| where a CG step forms it
 * on the support only; smv: 8nz+4m+4n; dct: 4n+8m). */
int xcs_plan_bytes(xcs_plan *plan, double *bytes);
/* The team geometry the plan runs with once defaults are applied (no counterpart in the
 * reference): team_size workgroups of block_size threads per cooperative launch. */
int xcs_plan_geometry(xcs_plan *plan, int *team_size, int *block_size);
/* The form its solves run in: 0 the general one, 1 resident (gen: the vectors in every
 * workgroup's LDS), 2 split (smv, dct: slices of them).  smv in the split form: whether the
 * support bits are in LDS too, and in how many workgroups the own rows' and the own columns'
 * matrix entries are (0 otherwise).  Any pointer may be NULL. */
int xcs_plan_form(xcs_plan *plan, int *form, int *support_bits, int *rows_staged, int *columns_staged);
void xcs_plan_destroy(xcs_plan *plan);

/* ---- batched persistent form: many independent instances in one launch ---- */
/* Ensemble codes for the per-instance arrays below. */
enum { XCS_ENS_GEN = 0, XCS_ENS_SMV = 1, XCS_ENS_DCT = 2 };
typedef struct xcs_batch xcs_batch;
/* Generate `count` instances on the device (instance i: ensemble ens[i], sizes k[i], m[i],
 * n[i], smv p[i]; generator key (opts->seed, instance ? instance[i] : i)).  One algorithm
 * for all.  opts->team_size workgroups cooperate per instance (default 1); instances are
 * taken largest first from a device queue (the phase-transition sweep driver,
 * GAGA/CGIHTcode/shared/tests_delta_fixed.m:48-137, issues them one call at a time). */
int xcs_batch_create(const char *alg, int count, const int *ens, const int *k, const int *m,
                     const int *n, const int *p, const unsigned int *instance,
                     const xcs_options *opts, xcs_batch **batch);
/* Solve every instance from x = 0 in one persistent launch; *ms = device time.
 * With one workgroup per instance the reset and the launch are a captured HIP graph,
 * replayed on every call. */
int xcs_batch_solve(xcs_batch *batch, float *ms);
/* Change the team geometry: team_size workgroups of block_size threads per instance for the
 * big_count largest instances (big_count < 0: all of them); the rest run one per workgroup
 * once those are taken.  Without a tail schedule a solve takes teams of twice, four times, ...
 * team_size where the chip has room for all of them at once (unless xcs_batch_exact says
 * otherwise).  Recovery does not depend on the geometry (reduction order does). */
int xcs_batch_configure(xcs_batch *batch, int team_size, int block_size, int big_count);
/* exact != 0: solves run teams of exactly the configured size; 0 (the default): larger ones
 * where the chip has room. */
int xcs_batch_exact(xcs_batch *batch, int exact);
/* The teams of the last solve (its first launch, where a tail schedule made several);
 * xcs_batch_info reports the configured geometry. */
int xcs_batch_ran(xcs_batch *batch, int *teams, int *team_size);
/* Tail schedule (no counterpart in the reference, whose sweep driver runs one problem per
 * call): phase 0 solves every instance on the configured geometry for at most budgets[0]
 * iterations; phase p = 1 .. phases-1 gives the instances still running teams of
 * team_sizes[p] workgroups for budgets[p] more iterations (the last phase runs them to
 * their stopping rule; team_sizes[0] and budgets[phases-1] are ignored).  The few slow
 * instances of a batch then finish on many workgroups instead of one.  phases = 0 returns
 * to one launch; otherwise phases >= 2.  Results do not depend on the schedule beyond the
 * reduction order of the team sizes used. */
int xcs_batch_schedule(xcs_batch *batch, int phases, const int *team_sizes, const int *budgets);
/* How the tail schedule runs (no counterpart in the reference).  adaptive = 1 (the default):
 * one persistent cooperative launch of every resident workgroup; an instance that outlives
 * phase p's budget is queued for phase p + 1 at once, and workgroups that find no fresh
 * instance form that phase's teams on the device, so phases overlap and no workgroup waits
 * for a phase to end.  split_team >= 2 (default 4): once no fresh instance is left, a
 * phase-0 solve with idle workgroups around stops at an iteration boundary and a team of
 * split_team workgroups finishes its phase-0 iterations (0 or 1: no splitting).  Needs team
 * size 1 for phase 0, at most 15 phases with splitting, and the later team sizes (and
 * split_team) minus one adding up to fewer than the resident workgroups.  adaptive = 0: one
 * launch per phase, each after the last has ended.  Results do not depend on the mode beyond
 * the reduction order of the team sizes used. */
int xcs_batch_schedule_mode(xcs_batch *batch, int adaptive, int split_team);
/* Instances each phase of the last solve took (phases entries; 0 past the last phase run).
 * Adaptive form: the entry one past the last phase counts the phase-0 solves that split
 * teams finished. */
int xcs_batch_phase_counts(xcs_batch *batch, int *counts, int phases);
/* Autotuner: time every candidate geometry (team 1/2/4/8 x block 256/512/1024 x teams for all,
 * or for the largest 1/16, 1/8, 1/4 of the instances) on this batch with each instance capped
 * at probe_iters iterations (0: whole solves), keep the fastest; candidates that come to the
 * same launch (larger teams where the chip has room) are timed once.  cache_path (may be NULL) is
 * a text file of "<signature> <team> <block> <big_count> <ms>" lines: a hit skips the probes,
 * a miss appends the result.  verbose != 0 prints each candidate's time to stderr. */
int xcs_batch_tune(xcs_batch *batch, int probe_iters, const char *cache_path, int verbose,
                   int *team_size, int *block_size, int *big_count, float *probe_ms);
/* Per-instance results, caller indexing: norms[3*i..3*i+2] relative l1/l2/linf. */
int xcs_batch_results(xcs_batch *batch, float *norms, int *iterations, int *stop_reason,
                      float *conv_rate);
int xcs_batch_x(xcs_batch *batch, int index, float *x_out, float *x_true);
int xcs_batch_info(xcs_batch *batch, int *teams, int *team_size, int *block_size, float *gen_ms);
/* Time `reps` launches that apply A^T y to every instance (one workgroup per instance,
 * the batched solver's streaming product in isolation); *ms_per per launch, *bytes
 * its algorithmic bytes summed over instances. */
int xcs_batch_apply_timed(xcs_batch *batch, int reps, float *ms_per, double *bytes);
/* Algorithmic operator bytes of the last batch solve, summed over instances. */
int xcs_batch_bytes(xcs_batch *batch, double *bytes);
void xcs_batch_destroy(xcs_batch *batch);
/* Phase tick counters (10 ns; 32 entries) of builds made with -DXCS_PHASE_TIMING; zeros otherwise. */
int xcs_batch_phase_ticks(xcs_batch *batch, unsigned long long *ticks32);

/* ---- many right-hand sides: one gen A shared by many signals ---- */
/* The reference's gaga_cs('CGIHT', 'gen', k, m, n, options) solves one signal per call
 * (GAGA/gaga/gaga_gen.cu:41, CGIHT_S_gen at GAGA/gaga/algorithms.cu:3689-3942); this form
 * solves `count` signals against one A in lock step, the products as MFMA GEMMs.
 * A ~ N(0, 1/m) from key (opts->seed, opts->instance); signal s is k-sparse with key
 * (opts->seed, opts->instance + 1 + s) and values by opts->vec_distribution; y = A x (FP32 A,
 * FP64 sums).  precision: "bf16" (A in BF16) or "fp8" (A in OCP e4m3 with per-column scales,
 * then BF16); both end with a least-squares refinement on the k largest entries (FP32 CG,
 * BF16 products, FP64 residual from the FP32 A) and, for signals still above tol, hard
 * thresholding pursuit corrections on the exact residual.  Needs m % 128 == 0,
 * n % 512 == 0, m <= 8192. */
typedef struct xcs_mrhs xcs_mrhs;
int xcs_mrhs_create(int m, int n, int k, int count, const char *precision,
                    const xcs_options *opts, xcs_mrhs **handle);
/* *ms = device time of the whole solve; lp_iterations[3] = lock-step iterations issued in the
 * FP8 (or BF16) phase and in the BF16 continuation (0 for "bf16"), and the support-correction
 * steps taken for signals still above tol after the refinement. */
int xcs_mrhs_solve(xcs_mrhs *handle, float *ms, int *lp_iterations);
/* norms[3*s..]: relative l1/l2/linf error against the planted signal; iterations[s]: CGIHT
 * iterations; resid_rel[s] = ||y - A x|| / ||y|| in FP64 with the FP32 A. */
int xcs_mrhs_results(xcs_mrhs *handle, float *norms, int *iterations, double *resid_rel);
int xcs_mrhs_x(xcs_mrhs *handle, int signal, float *x_out, float *x_true, float *y);
/* Time `reps` of one product over all signals: transpose = 1 for A^T R (M = n, K = m), 0 for
 * A V (M = m, K = n, K split in 4); fmt "bf16" or "fp8"; *flops = 2 m n count. */
int xcs_mrhs_gemm_timed(xcs_mrhs *handle, int transpose, const char *fmt, int reps,
                        float *ms_per, double *flops);
/* The same signals [first, first + cnt) solved one at a time by the FP32 single-instance
 * engine on the resident A and y (mode 0: one cooperative launch per solve; 1: one outer
 * iteration per launch, host-side stop test): *ms_total = summed device time,
 * norms[3*q..] and iterations[q] per signal. */
int xcs_mrhs_fp32_solve(xcs_mrhs *handle, int first, int cnt, int mode, float *ms_total,
                        float *norms, int *iterations);
/* Solver knobs: low-precision stopping tolerance c * ||y|| for the BF16 and FP8 phases
 * (defaults 2^-7, 2^-3), cap on support-correction steps (6), refinement outer and inner
 * (CG) steps (2, 4). */
int xcs_mrhs_configure(xcs_mrhs *handle, float c_bf16, float c_fp8, int corrections,
                       int ref_outer, int ref_inner);
/* GEMM block tile of the products where the row count allows (no counterpart in the
 * reference): 0 128 x 128 with 4 waves, 1 256 x 128 with 8 waves, 2 256 x 256 with 8 waves,
 * -1 (the default) each product's by its sizes.  Results do not depend on it.  They do depend, in
 * the rounding of the products only, on the number of signals that are still active: it decides
 * in how many slices a product sums. */
int xcs_mrhs_gemm_tile(xcs_mrhs *handle, int tile);
/* keep = 0 gives back the copy of A that the exact residual reads by blocks of rows (4 m n
 * bytes; it then reads A as it is, for the same bits in about twice the time); otherwise the copy
 * is made if it is not there (XCS_ENOMEM where it does not fit).  A handle is created with it
 * where there is memory left. */
int xcs_mrhs_row_blocks(xcs_mrhs *handle, int keep);
/* Device ms of the last solve's phases: start, low-precision phase, BF16 continuation,
 * refinement, support corrections (with their refinements), 0. */
int xcs_mrhs_phase_ms(xcs_mrhs *handle, float *ms6);
void xcs_mrhs_destroy(xcs_mrhs *handle);

/* ---- learned warm start for CGIHT (no counterpart in the reference) ---- */
/* A per-coordinate MLP (8 features of g = A^T y -> 512 -> 512 -> 1, ReLU; FP32 weights with
 * BF16 copies for the MFMA layer) scores support membership; trained on the GPU by the
 * library's own forward/backward kernels with Adam. */
typedef struct xcs_mlp xcs_mlp;
int xcs_mlp_create(unsigned int seed, xcs_mlp **net);
void xcs_mlp_destroy(xcs_mlp *net);
/* Number of parameters; layout W1[512][8], b1[512], W2[512][512] (out x in), b2[512],
 * W3[512], b3. */
int xcs_mlp_param_count(void);
int xcs_mlp_get_params(xcs_mlp *net, float *params);
int xcs_mlp_set_params(xcs_mlp *net, const float *params);
/* Forward + backward on a host batch (X: B x 8, labels 0/1): gradients of the mean weighted
 * binary cross-entropy (positives weighted pos_w) and the mean loss. */
int xcs_mlp_grad(xcs_mlp *net, const float *X, const float *labels, int B, float pos_w,
                 float *grad, float *loss);
int xcs_mlp_scores(xcs_mlp *net, const float *X, int N, float *logits);
/* Resident training set and `steps` Adam steps over consecutive batches of it. */
int xcs_mlp_set_data(xcs_mlp *net, const float *X, const float *labels, long N);
int xcs_mlp_train(xcs_mlp *net, int steps, int batch, float lr, float pos_w, float *mean_loss,
                  float *ms);
/* Training samples from a solved many-RHS handle: `per` coordinates per signal (half among the
 * 2k largest |A^T y|, half uniform) with their features and label = in the recovered support. */
int xcs_mrhs_samples(xcs_mrhs *handle, int per, unsigned int seed, float *X, float *labels);
/* CGIHT on a plan started from the network's k best-scored coordinates: x = A^T y on them,
 * improved by cg_steps (0..15) steps of least-squares CG on that support, then CGIHT; plain
 * CGIHT from x = 0 is the fallback when that stops above tol and above 1e-5 ||y|| (the FP32
 * floor of the residual).  net = NULL starts from the k
 * largest |A^T y| instead (the same start without the network). */
int xcs_plan_solve_warm(xcs_plan *plan, xcs_mlp *net, int cg_steps, float *ms, float *warm_ms,
                        int *fallback);

/* ---- kernel-level entry points (host buffers; used by parity tests) ---- */
/* One FindSupportSet call (functions.cu:397-436) on the device:
 * in/out state: *min_val, *alpha, *max_bin, *k_bin; out: bins[n], *sum
 * (*sum = -1 when the skip branch is taken). */
int xcs_find_support_set(const float *v, int n, int k, int num_bins, float slope,
                         float intercept, float max_change, float *min_val, float *alpha,
                         int *max_bin, int *k_bin, int *bins, int *sum);
/* y = A x (transpose = 0, x length n) or g = A^T r (transpose = 1, r length m) for one
 * ensemble; gen: A column-major m x n; smv: 0-based CSC (col_ptr[n+1], rows, vals);
 * dct: 0-based rows[m]. Unused pointers may be NULL. */
int xcs_apply(const char *ens, int transpose, int m, int n, const float *A, const int *col_ptr,
              const int *rows, const float *vals, const int *dct_rows, const float *in,
              float *out);
/* Device generator (Philox4x32-10): gen A column-major m x n with N(0, 1/m) entries. */
/* C[c*M + r] = sum_k q(A)[r, k] q(B)[c, k] on the MFMA GEMM (A: M x K row-major, B: N x K
 * row-major, host FP32).  fmt "bf16": q = RNE to bf16; "fp8": q = e4m3(v / s) * s with s the
 * row's max |v| / 448.  A_q, B_q (nullable) receive the dequantized operands.  Needs
 * M % 128 == 0 and K * element bytes % 128 == 0. */
/* The warm-start features of one instance from g = A^T y (host buffers): X (n x 8). */
int xcs_mlp_features(const float *g, int n, int m, int k, float *X);
/* Calibration: `reps` launches of a plain streaming copy of `bytes` (reads and writes `bytes`
 * each); *ms_per = average launch time.  Reference point for HBM traffic counters. */
int xcs_stream_copy(long bytes, int reps, float *ms_per);
/* `reps` launches of a streaming read of `bytes` (non-temporal float4 loads summed per
 * workgroup, as the solver streams A); *ms_per = average launch time: the read bandwidth
 * the chip delivers to a streaming kernel, the practical ceiling beside the nominal 8 TB/s. */
int xcs_stream_read(long bytes, int reps, float *ms_per);
int xcs_gemm_tn(const char *fmt, int M, int N, int K, const float *A, const float *B, float *C,
                float *A_q, float *B_q);
int xcs_generate_gen(int m, int n, unsigned int seed, unsigned int instance, float *A);
/* The smv generator alone (createProblem_smv.cu:31-167, createMeasurements_smv.cu:129-427,
 * zero-row repair :263-383): p distinct rows per column (p <= 64) drawn on the device,
 * ensemble 1 ones/sqrt(p), 2 random signs/sqrt(p), 3 ones.  rows, vals: CSC with p per
 * column (n*p); row_ptr (m+1), cols, rvals: the CSR copy, columns ascending in a row (each
 * may be NULL); *empty (may be NULL): empty rows the repair filled. */
int xcs_generate_smv(int m, int n, int p, int ens, unsigned int seed, unsigned int instance,
                     int *rows, float *vals, int *row_ptr, int *cols, float *rvals, int *empty);

const char *xcs_last_error(void);
const char *xcs_version(void);

#ifdef __cplusplus
}
#endif
#endif
