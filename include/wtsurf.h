/*
 * wtsurf -- MI355X (gfx950) surface Green's function library: C ABI.
 *
 * Drop-in boundary for the WannierTools surface-state hot path.  Every entry
 * point takes plain pointers and sizes, returns 0 on success and a negative
 * code on failure (wtsurf_last_error gives the reason), and is synchronous
 * unless its name says otherwise.  One context per host thread.
 *
 * Array conventions are the reference's (Fortran): complex matrices are
 * column-major interleaved (re, im) doubles with leading dimension = order;
 * orbital lists are 1-based; grid outputs are laid out like the reference's
 * dos_l(knv2, omeganum), k index fastest.  Energies are in whatever unit H(R)
 * is given in (the reference works in Hartree).
 */
#ifndef WTSURF_H
#define WTSURF_H

#ifdef __cplusplus
extern "C" {
#endif

typedef struct wtsurf_ctx wtsurf_ctx;

/* Precision of the decimation. */
enum {
    WTSURF_FP64 = 0,  /* all arithmetic in FP64, as the reference */
    WTSURF_FP32 = 1,  /* FP32 working precision: FP32 MFMA inverse and GEMMs in every
                         iteration, FP64 eps accumulators, convergence sum, final
                         inverses and traces; no refinement step.  A speed/accuracy
                         measurement mode: the doubling recursion amplifies FP32
                         rounding, measured on the 512 x 512 Ndim 72 grid at a median
                         relative error of 4.7e-4 on A(k, omega) and a maximum of 87.
                         Beyond Ndim 80 it diverges on some instances, so runs with
                         Ndim > 80 fail with an error in this mode. */
    WTSURF_MIXED = 2  /* Within 1e-6 of FP64 on A(k, omega), Ndim <= 80, for callers that
                         allow it.  Runs as WTSURF_FP64 on the automatic schedule, whatever
                         wtsurf_set_schedule says, with the same results: the FP32 working
                         precision holds that bound in the last sixth of an instance's
                         iterations at most, and the kernels that switched there took 1.5
                         times as long as the FP64 rounds. */
};

/* Per-instance status bits (wtsurf_grid_download / wtsurf_spectral_grid). */
enum {
    WTSURF_STATUS_SINGULAR = 1,      /* an exactly singular solve (identity used, as
                                        src/inverse.f90:51-55 leaves it) */
    WTSURF_STATUS_NOT_CONVERGED = 2  /* itermax reached (src/surfgreen.f90:86) */
};

/* Context on HIP device `device` with its own streams (default priority).
 * No reference counterpart (the reference has no device state). */
int wtsurf_ctx_create(int device, wtsurf_ctx **ctx);
void wtsurf_ctx_destroy(wtsurf_ctx *ctx);
/* Message of the last failed call on ctx ("" if none; never NULL). */
const char *wtsurf_last_error(const wtsurf_ctx *ctx);

/* Model upload: the module-`para` state that get_hmnr_cell leaves for
 * ham_qlayer2qlayer (src/readHmnR.f90:578-766, src/module.f90:957-968):
 * Num_wann = nw, Np = np, nrpts_surfacecell = nr, ijmax, irvec_surfacecell
 * as [nr][3] ints, HmnR_surfacecell as [nr] column-major nw x nw complex
 * blocks already divided by ndegen.  Resets the orbital lists to their
 * defaults (wtsurf_set_orbitals applies to the current model). */
int wtsurf_set_model(wtsurf_ctx *ctx, int nw, int np, int nr, int ijmax,
                     const int *irvec, const double *hr);

/* Decimation stop rule: the reference hard-codes itermax = 100 and
 * accuracy = 1e-16 (a single-precision literal) on sum_ij |alpha_ij|
 * (src/surfgreen.f90:39,42,120-122); those are the defaults. */
int wtsurf_set_stop_rule(wtsurf_ctx *ctx, int itermax, double accuracy);

/* Schedule of the decimation kernels for orders up to 80 (larger orders always
 * run as rounds).  The rounds' device workspace is kept by the context: up to
 * 3.1 GB at Ndim 72 and 7.4 GB at Ndim 112, at most a quarter of the free memory
 * where that is less, and fewer slots where an allocation fails.  No reference counterpart (the reference solves one
 * instance at a time, src/surfstat.f90:123-146).
 *   WTSURF_SCHEDULE_ROUNDS      every iteration is two launches (inverse, GEMMs)
 *                               over a set of instance slots, two sets on two
 *                               streams; slots refill from a device queue.
 *   WTSURF_SCHEDULE_PERSISTENT  one launch of one workgroup per CU; each
 *                               workgroup runs whole instances (all iterations,
 *                               final inverses, traces) and takes the next one
 *                               from a device queue.
 *   WTSURF_SCHEDULE_SMALL       Ndim <= 32, FP64: whole instances, in the
 *                               registers of one wave up to Ndim 16 (up to 8
 *                               four to a wave), beyond that in one workgroup
 *                               on the vector ALUs; larger orders and other
 *                               precisions run as ROUNDS.
 *   WTSURF_SCHEDULE_AUTO        SMALL where it applies, else ROUNDS. */
enum {
    WTSURF_SCHEDULE_ROUNDS = 0,
    WTSURF_SCHEDULE_PERSISTENT = 1,
    WTSURF_SCHEDULE_SMALL = 2,
    WTSURF_SCHEDULE_AUTO = 3
};
int wtsurf_set_schedule(wtsurf_ctx *ctx, int schedule);

/* TopOrbitals / BottomOrbitals (src/readinput.f90:2851-2962): top indices in
 * 1..Ndim, bottom indices in 1..Num_wann (offset by Ndim - Num_wann as
 * src/surfstat.f90:155).  Defaults: 1..Num_wann for both. */
int wtsurf_set_orbitals(wtsurf_ctx *ctx, int ntop, const int *top, int nbot,
                        const int *bot);

/* ham_qlayer2qlayer(k, H00, H01) (src/ham_qlayer2qlayer.f90:1-102) for nk
 * k points at once: kpts is [nk][2] (fractional, surface reciprocal
 * basis); h00 and h01 receive [nk] column-major Ndim x Ndim blocks. */
int wtsurf_ham_qlayer2qlayer(wtsurf_ctx *ctx, int nk, const double *kpts,
                             double *h00, double *h01);

/* surfgreen_1985(omega, GLL, GRR, GB, H00, H01, ones, eta)
 * (src/surfgreen.f90:7-137) for one instance of order n: full GLL, GRR, GB
 * out.  iters (may be NULL) receives the decimation iteration count.  Does
 * not need a model. */
int wtsurf_surfgreen_1985(wtsurf_ctx *ctx, int n, double omega, double eta,
                          const double *h00, const double *h01, double *gll,
                          double *grr, double *gb, int *iters);

/* wtsurf_surfgreen_1985 for callers that cannot allocate device memory (code
 * under HIP graph capture, tight serving loops, harnesses that forbid
 * hipMalloc): no reference counterpart.  Device pointers in and out (d_h00,
 * d_h01, d_gll, d_grr, d_gb: column-major n x n complex double, leading
 * dimension n; d_iters may be NULL); n <= 80.  The call allocates nothing: its
 * working memory is a fixed 2 MiB device array of the library (one per device,
 * held until the process ends), so calls that overlap on one device race.
 * Returns once the outputs are written.  ctx must be on the device of the
 * pointers. */
int wtsurf_surfgreen_1985_noalloc(wtsurf_ctx *ctx, int n, double omega, double eta,
                                  const double *d_h00, const double *d_h01, double *d_gll,
                                  double *d_grr, double *d_gb, int *d_iters);

/* The (k, omega) loops of surfstat (src/surfstat.f90:123-160; divisor = 1)
 * and SurfaceDOSkk (src/fermiarc.f90:206-248; divisor = pi): for every k
 * in kpts and every omega, decimate and take the traces
 *   dos_l    = -sum_{io in top} Im GLL(io,io) / divisor
 *   dos_r    = -sum_{b in bot}  Im GRR(Ndim-Num_wann+b, same) / divisor
 *   dos_bulk = -sum_{i=1..Ndim} Im GB(i,i) / divisor
 * Outputs are [nomega][nk] (k fastest).  iters and status may be NULL. */
int wtsurf_spectral_grid(wtsurf_ctx *ctx, int nk, const double *kpts,
                         int nomega, const double *omega, double eta,
                         double divisor, int precision, double *dos_l,
                         double *dos_r, double *dos_bulk, int *iters,
                         int *status);

/* Per-instance batch (the mixed workload: any set of (k, omega, eta)):
 * instance i is k = kpts[k_index[i]] (k_index 0-based, < nk), omega[i] and
 * eta[i]; H00/H01 are formed once per k point.  Traces as
 * wtsurf_spectral_grid, in instance order ([ninst]); iters and status may be
 * NULL.  The reference drives the same solves from its (k, omega) loops
 * (src/surfstat.f90:123-160, src/fermiarc.f90:193-248); this entry point has no
 * single counterpart there. */
int wtsurf_spectral_batch(wtsurf_ctx *ctx, int nk, const double *kpts, int ninst,
                          const int *k_index, const double *omega, const double *eta,
                          double divisor, int precision, double *dos_l,
                          double *dos_r, double *dos_bulk, int *iters, int *status);

/* The same computation split so inputs can stay resident in device memory:
 * upload the grid once, run, wait, fetch.  The run enqueues its work on the
 * context streams in rounds and watches a device counter of finished
 * instances to know when to stop; it returns once the last rounds are
 * queued, shortly before the work completes.  wtsurf_grid_timing reports
 * the device time of the Fourier and decimation stages of the last grid run
 * or wtsurf_spectral_batch call (HIP events on the context's first stream).
 * No reference counterpart. */
int wtsurf_grid_upload(wtsurf_ctx *ctx, int nk, const double *kpts, int nomega,
                       const double *omega);
int wtsurf_grid_run_async(wtsurf_ctx *ctx, double eta, double divisor,
                          int precision);
int wtsurf_sync(wtsurf_ctx *ctx);
int wtsurf_grid_timing(wtsurf_ctx *ctx, float *ms_fourier, float *ms_decimate);
int wtsurf_grid_download(wtsurf_ctx *ctx, double *dos_l, double *dos_r,
                         double *dos_bulk, int *iters, int *status);

/* Spin-resolved traces, taken by the runs that follow (wtsurf_spectral_grid,
 * wtsurf_grid_run_async, wtsurf_spectral_batch) from the same GLL and GRR:
 *   s_c = -sum_{io} Im (G sigma_c)(io, io) / divisor,   c = x, y, z,
 * with the spin operators of src/surfstat.f90:102-115 (orbitals 1..Num_wann/2
 * of every principal layer spin up, the next Num_wann/2 their spin-down
 * partners).  The left sums run over the top orbitals on GLL.  The right sums
 * run on GRR over
 *   WTSURF_SPIN_SURFSTAT: the top orbital indices, as surfstat does
 *                         (src/surfstat.f90:178-191);
 *   WTSURF_SPIN_ARC:      the bottom orbitals of the last principal layer, as
 *                         SurfaceDOSkk does (src/fermiarc.f90:298-327).
 * The reference forms each sum from a full ZGEMM G*sigma (src/mat_mul.f90:3-27);
 * here each term is one element of G, the same number. */
enum {
    WTSURF_SPIN_OFF = 0,
    WTSURF_SPIN_SURFSTAT = 1,
    WTSURF_SPIN_ARC = 2
};
int wtsurf_set_spin_traces(wtsurf_ctx *ctx, int mode);
/* The last run's spin traces (fails if it took none): spin_l and spin_r are
 * [3][ninst] each (sx, sy, sz blocks), every block in the order of that run's
 * dos_l.  Either pointer may be NULL. */
int wtsurf_spin_download(wtsurf_ctx *ctx, double *spin_l, double *spin_r);

/* The QPI autocorrelation of SurfaceDOSkk over a k-plane
 * (src/fermiarc.f90:496-560): for every q = (iq1, iq2),
 *   out(iq1, iq2) = sum_{ik1, ik2} sum_{f < nfield} a_f(ik1, ik2) a_f(ik1q, ik2q),
 *   ik1q = mod(ik1 + iq1 - 2, m1) + 1,   ik2q = mod(ik2 + iq2 - 2, m2) + 1
 * (1-based).  The reference takes m1 = nkx - 1, m2 = nky - 1 with nfield = 1
 * (dos_*_only) for jdos, and m1 = Nk1 - 1, m2 = Nk2 - 1 with nfield = 4
 * (dos_*_only, sx, sy, sz) for jsdos.  fields is [nfield][nky][nkx] and out
 * [nky][nkx], ik1 fastest (the reference's (nkx, nky) arrays).  Requires
 * 1 <= m1 <= nkx, 1 <= m2 <= nky, m1 <= 2048.  The sum is taken in a
 * different order than the reference's loops. */
int wtsurf_kplane_autocorrelation(wtsurf_ctx *ctx, int nkx, int nky, int m1, int m2,
                                  int nfield, const double *fields, double *out);

/* The k-path joint density of states of surfstat_jdos
 * (src/surfstat.f90:891-907), each field and energy on its own: with
 * h = (nk - 1)/2 and iq1 = iq - h,
 *   out_f(iq, j) = sum_{ik1 = max(1, 1 - iq1)}^{min(2h + 1, 2h + 1 - iq1)} a_f(ik1, j) a_f(ik1 + iq1, j)
 * (1-based; the reference's imin1 / imax1).  fields and out are
 * [nfield][nomega][nk], k fastest (the reference's dos_l(knv2, omeganum)).
 * Each sum is taken in the reference's order. */
int wtsurf_kpath_jdos(wtsurf_ctx *ctx, int nk, int nomega, int nfield,
                      const double *fields, double *out);
/* The same sums for arrays with the energy fastest, [nfield][nk][nomega]. */
int wtsurf_kpath_jdos_energy_fastest(wtsurf_ctx *ctx, int nk, int nomega, int nfield,
                                     const double *fields, double *out);

/* Largest Ndim the FP64 decimation kernels are built for. */
int wtsurf_max_ndim(void);

#ifdef __cplusplus
}
#endif
#endif /* WTSURF_H */
