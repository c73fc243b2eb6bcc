/*
 * jax_finufft_amd: MI355X (gfx950) NUFFT backend, C ABI.
 *
 * Two layers, both plain C with pointers and sizes:
 *
 * 1. The plan interface (jfa_makeplan / jfa_setpts / jfa_execute /
 *    jfa_destroy).  It replaces the cuFINUFFT guru calls that the reference's
 *    host driver makes through its wrapper:
 *      makeplan  lib/cufinufft_wrapper.cc:48-61   (called at lib/kernels.cc.cu:51)
 *      setpts    lib/cufinufft_wrapper.cc:63-73   (called at lib/kernels.cc.cu:63-68)
 *      execute   lib/cufinufft_wrapper.cc:75-89   (called at lib/kernels.cc.cu:75)
 *      destroy   lib/cufinufft_wrapper.cc:91-99   (called at lib/kernels.cc.cu:84)
 *      default_opts / update_opts  lib/cufinufft_wrapper.cc:11-46
 *
 * 2. Eighteen transform entry points, one per XLA FFI handler of the
 *    reference (lib/jax_finufft_gpu.cc:363-384), with the same attribute list
 *    in the same order (lib/jax_finufft_gpu.cc:28-60) and the same operand
 *    order (source, points..., [targets...], output; points and n_k already
 *    reversed into x-fastest order by the lowering,
 *    src/jax_finufft/lowering.py:96-105).  Each replaces one
 *    nufft{d}d{t}{f}_impl of lib/kernels.cc.cu:117-215 + run_nufft
 *    (lib/kernels.cc.cu:25-92).  Unlike the reference they take plans from a
 *    per-device cache and queue all work on `stream` without blocking the
 *    host, with one exception: type 3 sizes its grids from the points, so its
 *    setpts waits for two small device-to-host copies (the point and target
 *    extents, then the targets per box).  Elsewhere the library waits on the
 *    host only where noted: jfa_ragged_run (the previous run's pointer-table
 *    copy), debug = 1 stage printing, jfa_autotune, and plan destruction.
 *
 * All device pointers are HIP device memory.  Complex arrays are interleaved
 * (re, im) in the transform's precision.  Single precision entry points end in
 * "f" and take float points and complex64 data; the others take double.
 *
 * Return codes: 0 success, 1 the eps-too-small warning (not an error, as in
 * lib/kernels.cc.cu:52-55), >= 2 an error; jfa_last_error() describes the
 * last error raised on the calling thread.
 */
#ifndef JAX_FINUFFT_AMD_H_
#define JAX_FINUFFT_AMD_H_

#include <stdint.h>

#ifdef __cplusplus
extern "C" {
#endif

/* A hipStream_t, passed as an opaque pointer (NULL = the null stream). */
typedef void *jfa_stream_t;

typedef struct jfa_plan_s *jfa_plan;

enum {
    JFA_OK = 0,
    JFA_WARN_EPS_TOO_SMALL = 1,
    JFA_ERR_BAD_ARG = 2,
    JFA_ERR_ALLOC = 3,
    JFA_ERR_HIP = 4,
    JFA_ERR_FFT = 5,
    JFA_ERR_NOT_SUPPORTED = 6,
    JFA_ERR_TOO_LARGE = 7,
    JFA_ERR_INTERNAL = 8  /* a consistency check of the library's own tables failed */
};

/* Spread/interp method (gpu_method): 0 auto, 1 global-memory atomics in
 * sorted order, 2 LDS subproblem tiles, 3 register strips (2D and 3D
 * spreading, atomic-free; a 3D grid is spread as a stack of 2D slices;
 * interpolation then uses the LDS tiles).  3 needs a grid of at least 64 x 2w
 * (x 2w) cells.  Auto picks it for spreading there, and on narrower grids of up
 * to 2^20 rows, else 2 when the tile fits in LDS, else 1. */
enum { JFA_METHOD_AUTO = 0, JFA_METHOD_GM_SORT = 1, JFA_METHOD_SM = 2, JFA_METHOD_STRIP = 3 };

/* Options.  The first seven fields are the ones the reference forwards to the
 * GPU (src/jax_finufft/options.py:105-119, lowering.py:157-174); the rest are
 * the GPU fields it declares (options.py:66-79) plus stream/device and two
 * additions of this backend. */
typedef struct {
    int modeord;           /* 0: CMCL order -N/2..(N-1)/2; 1: FFT order */
    double upsampfac;      /* sigma; 2.0 default (gpu_upsampfac) */
    int gpu_method;        /* JFA_METHOD_* */
    int gpu_sort;          /* 1: sort points into bins (always used by SM) */
    int gpu_kerevalmeth;   /* 1: Horner piecewise polynomial (0: exp/sqrt) */
    int gpu_maxbatchsize;  /* transforms per spread/FFT batch; 0 = all */
    int debug;             /* 1: print per-stage timings to stderr */
    int gpu_binsizex, gpu_binsizey, gpu_binsizez; /* LDS-tile bins; for the strip
                              method gpu_binsizey asks for the unit height in rows,
                              of which a unit has w to 33 - w (to 128 where w > 8);
                              0 = default (or the autotuner's choice) */
    int gpu_maxsubprobsize;  /* points per LDS subproblem / strip piece; 0 = default */
    int gpu_spreadinterponly; /* 1: execute spreads/interpolates only; the mode
                                 array is then the fine grid (nf = nmodes) */
    int gpu_device_id;     /* -1: current device */
    jfa_stream_t gpu_stream;
    int width_rule;        /* 0: width reaches eps (w = ceil(log10(20/eps)));
                              1: FINUFFT's published rule w = ceil(log10(10/eps)) */
    int kernel_width;      /* >0: force this width (2..16) */
    int64_t t3_max_cells;  /* type 3: most cells of one spread or inner grid before the
                              targets are split into boxes (0: 2^32) */
} jfa_opts;

void jfa_default_opts(jfa_opts *opts);

/* type 1, 2 or 3; dim 1..3; nmodes[3] in x-fastest order (ignored for type 3);
 * iflag sign of the exponent; ntransf stacked transforms sharing the points. */
int jfa_makeplan(int type, int dim, const int64_t *nmodes, int iflag, int ntransf, double eps,
                 int is_double, const jfa_opts *opts, jfa_plan *plan_out);

/* M points (x, y, z device arrays of length M; unused ones may be NULL).
 * Type 3 also takes N target frequencies s, t, u.  Points may be any real
 * value (they are folded periodically). */
int jfa_setpts(jfa_plan plan, int64_t M, const void *x, const void *y, const void *z, int64_t N,
               const void *s, const void *t, const void *u);

/* Type 1: c (ntransf x M) -> fk (ntransf x modes); type 2: fk -> c;
 * type 3: c (ntransf x M) -> fk (ntransf x N). */
int jfa_execute(jfa_plan plan, void *c, void *fk);

/* Fused adjoint pass of a type-2 plan (no reference counterpart; it replaces
 * the D extra stacked transforms of the reference's differentiation rule,
 * src/jax_finufft/ops.py:214-236 and :295-312).  From the mode array fk
 * (ntransf x modes) it computes, in one interpolation pass sharing one
 * amplify + FFT:
 *   val[t][j]   = sum_k fk[t][k] e^{i iflag k.x_j}            (if val != NULL)
 *   grad[d][j]  = sum_t Re(conj(w[t][j]) d val[t][j] / d x_dj)  (if grad != NULL)
 * with d in the plan's x-fastest order and grad laid out d-major (dim x M).
 * fk == NULL reuses the fine grid of the plan's last type-2 execute, skipping
 * amplify + FFT: the reverse pass of a type-2 evaluation then costs one
 * interpolation pass.  That grid exists only when the execute ran all
 * transforms in one batch and had points; otherwise the call returns
 * JFA_ERR_NOT_SUPPORTED and the caller passes fk or uses the stacked
 * transforms.  Plans of the LDS-tile method interpolate from tiles, plans of
 * the global-memory method (gpu_method 1) read the taps from the fine grid. */
int jfa_interp_grad(jfa_plan plan, const void *fk, const void *w, void *val, void *grad);

/* Queue subsequent work of this plan on `stream`, ordered after the plan's
 * previous work on whatever stream it used before. */
int jfa_set_stream(jfa_plan plan, jfa_stream_t stream);

int jfa_destroy(jfa_plan plan);

/* Kernel parameters the plan chose: width, beta, fine grid (x-fastest). */
int jfa_plan_info(jfa_plan plan, int *ns, double *beta, int64_t *nf /* [3] */);

/* Stage timing of a plan made with opts.debug == 2, which records HIP events
 * around every stage on the plan's stream without synchronising.  Returns the
 * accumulated milliseconds and launch count of `stage` ("setpts", "zero",
 * "spread", "fft", "deconv", "amplify", "interp"); waits for the recorded
 * events.  reset != 0 clears the accumulators afterwards.  (No reference
 * counterpart: the reference's GPU debug attribute, lowering.py:173, only
 * turns on cuFINUFFT's own prints.) */
int jfa_plan_timing(jfa_plan plan, const char *stage, int reset, double *total_ms,
                    int64_t *count);

/* Diagnostics of setpts (no reference counterpart; they expose the integer
 * outputs of the point sort cuFINUFFT runs inside setpts, called at
 * lib/kernels.cc.cu:63-68, so that they can be checked bit for bit).
 * jfa_setpts_info fills info[24] (host only):
 *   [0] sorted entries n (M; M * ns for the 3D strip spreader, whose entries
 *       are slice points; 0 when the plan does not sort)
 *   [1] bins nb_total; [2] key shift: bin = key >> shift; [3] lowest key bit
 *       the sort orders by (bits below it keep input order within equal keys)
 *   [4] method; [5] layout: 0 bin keys with gathered points, 1 keys carrying
 *       the first taps' offsets within the bin, 2 strip keys
 *   [6..8] bin size, [9..11] bins, [12..14] fine grid (x fastest), [15] ns,
 *   [16] bins ordered y fastest, [17] strips per slice, [18..20] offset bits
 *       per dimension (layout 1), [21] strip width, [22] type 3: target boxes
 * jfa_setpts_copy queues copies on the plan's stream of the sorted keys
 * (uint32[n]), the permutation (int32[n]: sorted position -> input entry) and
 * the bin starts (int32[nb_total + 1]) into caller device buffers (any may be
 * NULL). */
int jfa_setpts_info(jfa_plan plan, int64_t *info);
int jfa_setpts_copy(jfa_plan plan, void *keys, void *perm, void *bin_start);

const char *jfa_last_error(void);

/* ------------------------------------------------------------------------
 * Ragged batches (no reference counterpart; the reference's equivalent is a
 * Python loop of nufft1 calls, each a run_nufft with its own plan,
 * lib/kernels.cc.cu:25-92).  nprob independent 2D type-1 problems with their
 * own point counts, mode grids and numbers of stacked strength vectors, all
 * with one eps and iflag, run as one sequence of launches: one point sort over
 * every problem, one strip-spreading launch over every problem's units, one
 * merge, one batched FFT per fine-grid size, one deconvolution.  With
 * use_graph != 0 the launches after the sort are captured once into a HIP
 * graph and replayed on later runs.
 *   nmodes:   nprob x dim mode counts, x fastest (the backend's axis order)
 *   ntransf:  nprob stacked strength vectors per problem
 *   npoints:  nprob point counts
 * opts: modeord, upsampfac, width_rule, kernel_width, gpu_kerevalmeth,
 * gpu_maxsubprobsize, gpu_stream and gpu_device_id are honoured.  dim must be
 * 2 and every fine grid at least 64 x 2*ns (JFA_ERR_NOT_SUPPORTED otherwise).
 * ------------------------------------------------------------------------ */
typedef struct jfa_ragged_s *jfa_ragged;
int jfa_ragged_makeplan(int dim, int nprob, const int64_t *nmodes, const int64_t *ntransf,
                        const int64_t *npoints, int iflag, double eps, int is_double,
                        const jfa_opts *opts, int use_graph, jfa_ragged *plan_out);
/* points: dim x nprob device pointers (x of every problem, then y); c, f:
 * nprob device pointers each, c[i] holding ntransf[i] x npoints[i] complex
 * strengths and f[i] receiving ntransf[i] x modes complex outputs.  Queues
 * setpts + execute of every problem on the plan's stream.  The one host wait:
 * before refilling the pinned pointer table it waits until the previous run's
 * copy of that table has left it (normally long done). */
int jfa_ragged_run(jfa_ragged plan, const void *const *points, const void *const *c,
                   void *const *f);
/* 1 if runs replay a captured graph; 0 if they launch eagerly (no graph
 * requested, or no run yet); -1 if the capture failed, after which the plan
 * launches eagerly for good (the run that found it sets jfa_last_error). */
int jfa_ragged_uses_graph(jfa_ragged plan);
int jfa_ragged_set_stream(jfa_ragged plan, jfa_stream_t stream);
int jfa_ragged_destroy(jfa_ragged plan);
/* Host-only check (no device memory, no reference counterpart): builds the
 * tables jfa_ragged_makeplan would build for these arguments and checks every
 * offset and range against the buffer sizes it would allocate; makeplan runs
 * the same check.  info (optional, 8 values): total points, sort bins,
 * spreading units, virtual problems (problem, transform), fine-grid cells,
 * pruned-FFT cells, scratch-tile cells, pieces at most.  Returns JFA_OK or
 * JFA_ERR_INTERNAL with the failed check in jfa_last_error(). */
int jfa_ragged_check_layout(int dim, int nprob, const int64_t *nmodes, const int64_t *ntransf,
                            const int64_t *npoints, double eps, int is_double,
                            const jfa_opts *opts, int64_t *info);

/* ------------------------------------------------------------------------
 * Autotuner (no reference counterpart: the reference declares the knobs,
 * src/jax_finufft/options.py:66-79, but forwards no bin size to the GPU).
 * jfa_autotune times candidate choices of gpu_method, bin sizes (for the
 * strip method gpu_binsizey = unit height) and gpu_maxsubprobsize for one
 * type-1 or type-2 transform on the caller's device data (setpts + execute,
 * best of three runs each on opts->gpu_stream; host waits), records the
 * fastest under the workload's key (type, dim, precision, modes, width,
 * upsampfac, ntransf, half-octave of M) and leaves its result in fk.  The
 * default choice is always a candidate, so the recorded one is never slower
 * than it on the measured data.  opts must leave those knobs at 0.
 * chosen / best_ms / default_ms may be NULL.
 * jfa_tuned_opts fills the knobs of *opts from a record (returns 1), unless
 * the caller set any of them (returns 0); the transform entry points call it
 * before taking a plan.  Records persist in the JSON file named by the
 * environment variable JFA_TUNE_CACHE, when set.  jfa_tune_clear forgets
 * the in-memory records.
 * ------------------------------------------------------------------------ */
int jfa_autotune(int type, int dim, const int64_t *nmodes, int iflag, int ntransf, double eps,
                 int is_double, const jfa_opts *opts, int64_t M, const void *x, const void *y,
                 const void *z, void *c, void *fk, jfa_opts *chosen, double *best_ms,
                 double *default_ms);
int jfa_tuned_opts(int type, int dim, const int64_t *nmodes, int ntransf, double eps,
                   int is_double, int64_t M, jfa_opts *opts);
void jfa_tune_clear(void);

/* Number of plans held by the per-device plan cache, and a way to drop them. */
int jfa_cache_size(void);
void jfa_cache_clear(void);

/* Host-only plan-time mathematics (no device work; usable without a GPU).
 * They expose what makeplan computes inside cuFINUFFT in the reference
 * (called at lib/kernels.cc.cu:51), so it can be checked on its own.
 *   jfa_kernel_params: width ns, shape beta and Horner coefficient count nc for
 *     eps at upsampling factor upsampfac; returns 1 if eps was clamped.
 *   jfa_fine_grid_size: fine grid for n modes (next even 2,3,5-smooth >=
 *     max(upsampfac n, 2 ns)).
 *   jfa_horner_table: nc x ns monomial coefficients, power-major.
 *   jfa_kernel_fourier: psi_hat(2 pi k / nf) for k = kmin .. kmin+n-1. */
int jfa_kernel_params(double eps, double upsampfac, int width_rule, int is_double, int *ns,
                      double *beta, int *nc);
int64_t jfa_fine_grid_size(int64_t n, double upsampfac, int ns);
int jfa_horner_table(int ns, int nc, double beta, double *coef);
int jfa_kernel_fourier(int ns, double beta, int64_t nf, int64_t kmin, int64_t n, double *out);

/* ------------------------------------------------------------------------
 * Transform entry points, one per XLA FFI handler of the reference
 * (lib/jax_finufft_gpu.cc:363-384).  Attribute order matches
 * NUFFT_COMMON_ATTRS_{FLOAT,DOUBLE} (lib/jax_finufft_gpu.cc:28-60).
 * n_tot independent problems, each with n_transf stacked transforms over n_j
 * points; problem `idx` reads points at idx*n_j, strengths at
 * idx*n_j*n_transf and writes modes at idx*n_k_total*n_transf
 * (lib/kernels.cc.cu:57-60).  Type 3 reads n_k_1 targets per problem at
 * idx*n_k_1 (lib/kernels.cc.cu:66).
 * ------------------------------------------------------------------------ */
#define JFA_ATTRS_F                                                                      \
    jfa_stream_t stream, float eps, int64_t iflag, int64_t n_tot, int64_t n_transf,      \
        int64_t n_j, int64_t n_k_1, int64_t n_k_2, int64_t n_k_3, int64_t modeord,       \
        double upsampfac, int64_t gpu_method, int64_t gpu_sort, int64_t gpu_kerevalmeth, \
        int64_t gpu_maxbatchsize, int64_t debug
#define JFA_ATTRS_D                                                                      \
    jfa_stream_t stream, double eps, int64_t iflag, int64_t n_tot, int64_t n_transf,     \
        int64_t n_j, int64_t n_k_1, int64_t n_k_2, int64_t n_k_3, int64_t modeord,       \
        double upsampfac, int64_t gpu_method, int64_t gpu_sort, int64_t gpu_kerevalmeth, \
        int64_t gpu_maxbatchsize, int64_t debug

/* type 1: source (n_tot, n_transf, n_j) -> output (n_tot, n_transf, modes) */
int jfa_nufft1d1f(JFA_ATTRS_F, const void *source, const void *points_x, void *output);
int jfa_nufft1d1(JFA_ATTRS_D, const void *source, const void *points_x, void *output);
int jfa_nufft2d1f(JFA_ATTRS_F, const void *source, const void *points_x, const void *points_y,
                  void *output);
int jfa_nufft2d1(JFA_ATTRS_D, const void *source, const void *points_x, const void *points_y,
                 void *output);
int jfa_nufft3d1f(JFA_ATTRS_F, const void *source, const void *points_x, const void *points_y,
                  const void *points_z, void *output);
int jfa_nufft3d1(JFA_ATTRS_D, const void *source, const void *points_x, const void *points_y,
                 const void *points_z, void *output);

/* type 2: source (n_tot, n_transf, modes) -> output (n_tot, n_transf, n_j) */
int jfa_nufft1d2f(JFA_ATTRS_F, const void *source, const void *points_x, void *output);
int jfa_nufft1d2(JFA_ATTRS_D, const void *source, const void *points_x, void *output);
int jfa_nufft2d2f(JFA_ATTRS_F, const void *source, const void *points_x, const void *points_y,
                  void *output);
int jfa_nufft2d2(JFA_ATTRS_D, const void *source, const void *points_x, const void *points_y,
                 void *output);
int jfa_nufft3d2f(JFA_ATTRS_F, const void *source, const void *points_x, const void *points_y,
                  const void *points_z, void *output);
int jfa_nufft3d2(JFA_ATTRS_D, const void *source, const void *points_x, const void *points_y,
                 const void *points_z, void *output);

/* type 3: source (n_tot, n_transf, n_j) -> output (n_tot, n_transf, n_k_1) */
int jfa_nufft1d3f(JFA_ATTRS_F, const void *source, const void *points_x, const void *target_x,
                  void *output);
int jfa_nufft1d3(JFA_ATTRS_D, const void *source, const void *points_x, const void *target_x,
                 void *output);
int jfa_nufft2d3f(JFA_ATTRS_F, const void *source, const void *points_x, const void *points_y,
                  const void *target_x, const void *target_y, void *output);
int jfa_nufft2d3(JFA_ATTRS_D, const void *source, const void *points_x, const void *points_y,
                 const void *target_x, const void *target_y, void *output);
int jfa_nufft3d3f(JFA_ATTRS_F, const void *source, const void *points_x, const void *points_y,
                  const void *points_z, const void *target_x, const void *target_y,
                  const void *target_z, void *output);
int jfa_nufft3d3(JFA_ATTRS_D, const void *source, const void *points_x, const void *points_y,
                 const void *points_z, const void *target_x, const void *target_y,
                 const void *target_z, void *output);

/* Fused type-2 adjoint entry points (no reference counterpart): the same
 * attributes and plan cache as jfa_nufft{d}d2{f}, then jfa_interp_grad per
 * problem.  weights and value_out are (n_tot, n_transf, n_j) complex,
 * grad_out is (n_tot, dim, n_j) real in x-fastest dimension order; value_out
 * or grad_out (with weights) may be NULL. */
int jfa_nufft1d2f_grad(JFA_ATTRS_F, const void *source, const void *points_x,
                       const void *weights, void *value_out, void *grad_out);
int jfa_nufft1d2_grad(JFA_ATTRS_D, const void *source, const void *points_x,
                      const void *weights, void *value_out, void *grad_out);
int jfa_nufft2d2f_grad(JFA_ATTRS_F, const void *source, const void *points_x,
                       const void *points_y, const void *weights, void *value_out,
                       void *grad_out);
int jfa_nufft2d2_grad(JFA_ATTRS_D, const void *source, const void *points_x,
                      const void *points_y, const void *weights, void *value_out,
                      void *grad_out);
int jfa_nufft3d2f_grad(JFA_ATTRS_F, const void *source, const void *points_x,
                       const void *points_y, const void *points_z, const void *weights,
                       void *value_out, void *grad_out);
int jfa_nufft3d2_grad(JFA_ATTRS_D, const void *source, const void *points_x,
                      const void *points_y, const void *points_z, const void *weights,
                      void *value_out, void *grad_out);

/* Allocation-free variant of jfa_nufft2d1f (no counterpart in the reference),
 * for callers that cannot allocate device memory: code under HIP graph
 * capture, tight serving loops, harnesses that forbid hipMalloc.  Same
 * attributes, operands and result as jfa_nufft2d1f; it queues kernels only (no
 * hipMalloc / hipFree / memset / copies) and keeps everything beyond the
 * caller's buffers in one 192 MiB device array per GPU, held until the process
 * ends.  Limits: fine grids of at most 4096 cells per axis (2,3,5-smooth) and
 * at least 64 x 2*width, gpu_method 0 or 3 (strip spreading), and sizes whose
 * scratch fits the array (about 49 bytes per point plus the grid-sized
 * buffers); beyond them it returns JFA_ERR_TOO_LARGE / JFA_ERR_NOT_SUPPORTED
 * before queueing anything.  Every call on a GPU shares that GPU's array:
 * calls that overlap on one GPU (other streams or host threads) race, so
 * order them.  gpu_sort, gpu_maxbatchsize and debug are ignored (one transform
 * at a time). */
int jfa_nufft2d1f_noalloc(JFA_ATTRS_F, const void *source, const void *points_x,
                          const void *points_y, void *output);

#ifdef __cplusplus
}
#endif

#endif /* JAX_FINUFFT_AMD_H_ */
