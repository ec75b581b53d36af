/*
 * fasteddy_amd.h -- C-ABI of the MI355X (gfx950) FastEddy time-step library.
 *
 * The entry points below replace the reference's CUDA layer one for one.
 * They keep the reference's names, signatures, argument meanings and return
 * convention (0 = success); inputs are the host modules' process globals and
 * host arrays (halo-inclusive, z fastest), exactly as the reference's CUDA
 * layer reads them.  Differences: errors are returned as non-zero codes
 * instead of exit(), and only a single rank (numProcsX = numProcsY = 1) is
 * accepted, with lateral periodicity applied on the device.
 */
#ifndef FASTEDDY_AMD_H
#define FASTEDDY_AMD_H

#ifdef __cplusplus
extern "C" {
#endif

/* Error codes (non-zero returns). */
#define FE_OK                 0
#define FE_ERR_NO_DEVICE      101
#define FE_ERR_HIP            102
#define FE_ERR_ALLOC          103
#define FE_ERR_UNSUPPORTED    104   /* a selector combination this build does not implement */
#define FE_ERR_TERRAIN        105   /* J31/J32 != 0, or terrain not periodic at the lateral boundaries */
#define FE_ERR_STATE          106   /* call order violated (e.g. Commence before Init) */
#define FE_ERR_RANKS          107   /* numProcsX*numProcsY != 1 */

/* SRC/FECUDA/fecuda.h:35-64 (fecuda.c:38-118): parameters, device selection and launch geometry.
 * fecuda_GetParams queries the mandatory tBx/tBy/tBz keys (defined in the device layer with the
 * other FECUDA globals) through the host parameter module's queryIntegerParameter. */
int fecuda_GetParams(void);
int fecuda_Init(void);
int fecuda_Cleanup(void);
int fecuda_SetBlocksPerGrid(int Nx, int Ny, int Nz);        /* halo-inclusive extents, recorded */
int fecuda_AllocateHaloBuffers(int Nxp, int Nyp, int Nzp, int Nh); /* single rank: no-op */
int fecuda_DeallocateHaloBuffers(void);

/* SRC/GRID/CUDA/cuda_grid.c:24,36: upload of the vertical coordinate and metric profiles. */
int cuda_gridInit(void);
int cuda_gridCleanup(void);

/* SRC/HYDRO_CORE/CUDA/cuda_hydroCore.h:30,35: physics constants, base state, device fields. */
int cuda_hydroCoreInit(void);
int cuda_hydroCoreCleanup(void);

/* SRC/TIME_INTEGRATION/CUDA/cuda_timeInt.h:30,35,40:
 * Init allocates the RK stage buffers and copies the initial state to the device;
 * Commence(it) runs NtBatch RK3 steps (uploading the host state again when
 * it == simTime_itRestart), advances simTime/simTime_it, and copies the state,
 * perturbation pressure and surface fields back to the host arrays. */
int cuda_timeIntInit(void);
int cuda_timeIntCommence(int it);
int cuda_timeIntCleanup(void);

/* ---- Build-only additions (no counterpart in the reference) ------------------ */

/* Tendency of one RK stage from the current device state, written into the host
 * arrays hydroFldsFrhs / sgstkeScalarsFrhs / moistScalarsFrhs (interior cells,
 * halos zero).  The fused kernels never store F in normal operation; this is the
 * parity hook.  'stage' is the 0-based RK stage; simTime/simTime_it as in
 * cuda_hydroCoreDeviceBuildFrhs (SRC/HYDRO_CORE/CUDA/cuda_hydroCoreDevice.cu:246). */
int fe_debug_build_frhs(int stage);
/* Copy host state arrays to the device (same as the first-batch upload). */
int fe_upload_state(void);
/* Copy the device state back into the host arrays without stepping. */
int fe_download_state(void);
/* Device step time of the last Commence, in ms per step (HIP events). */
float fe_last_ms_per_step(void);
/* Run nsteps RK3 steps on the device without any host transfer (benchmarking). */
int fe_device_steps(int nsteps);
/* Per-kernel HIP-event timing on the launch stream (classes: 0 column pass,
 * 1 stage kernel without SGS physics, 2 stage kernel with SGS physics, 3 lateral
 * halo fill).  fe_timing_enable(npairs) arms a pool for the next npairs launches,
 * which carry their events (0 disarms); fe_timing_read synchronises and returns
 * summed ms and launch counts. */
int fe_timing_enable(int npairs);
int fe_timing_read(double *ms, int *count, int ncls);
/* Streaming float4 copy of nfloats floats, reps times; returns GB/s (read+write). */
double fe_copy_probe(long nfloats, int reps);
/* Name of the kernel variant selected for the stage-1/2 and stage-3 tendencies. */
const char *fe_kernel_info(void);
/* Horizontal-mean profile statistics of the current device state, computed on the
 * device in FP64: out[Nz][nstat] with nstat = 17 columns <u>, <v>, <w>, <theta>,
 * <u'u'>, <u'w'>, <v'v'>, <v'w'>, <w'w'>, resolved TKE, <theta'w'>, <e>, <q_v>, <q_l>,
 * and, from the SGS stresses emitted by the last batch (hydroSubGridWrite), the
 * cell-centred |<tau13>, <tau23>|, <tau33>, <tau_theta3> (0 otherwise).
 * No counterpart in the reference's C code; it restates the reference's
 * post-processing (tutorials/notebooks/fetutorialfunctions.py:55-83,344-431). */
int fe_profiles(double *out, int nstat);
/* fe_profiles without any device allocation (no hipMalloc, hipFree or allocating library
 * routine), for callers that cannot allocate: code under HIP graph capture, tight serving
 * loops, harnesses that forbid it.  No counterpart in the reference.  The per-level rows go
 * to a static device array of the library (one per GPU, held until the process ends) that
 * holds at most 2048 levels: a grid with more returns FE_ERR_UNSUPPORTED.  Every call on a
 * GPU shares that GPU's array; calls that overlap on one GPU race. */
int fe_profiles_noalloc(double *out, int nstat);
/* Per-field state summary of the current device state (the on-device counterpart
 * of hydro_coreStateLogDump / hydro_coreFldStateLogEntry, SRC/HYDRO_CORE/hydro_core.c:1282-1525),
 * out[nrow][12] with nrow = 6 + TKE fields + moisture species, rows rho, u, v, w,
 * theta, p', TKE, q_v, q_l (rho-weighted fields per unit mass): max, its (i,j,k),
 * min, its (i,j,k) (halo-inclusive indices, first occurrence in i-j-k loop order),
 * mean over all interior cells of the finite values, NaN count, Inf count, and the
 * volume integral of the raw field (sum of field * D_Jac * dX dY dZ: the mass,
 * rho*theta, ... budgets).  FP64 sums on the device; returns FE_ERR_UNSUPPORTED
 * for a wrong nrow. */
int fe_state_summary(double *out, int nrow);

/* ---- Batched ensemble (no counterpart in the reference: the reference advances one model
 * per process, SRC/TIME_INTEGRATION/CUDA/cuda_timeIntDevice.cu:105-157).  Members of
 * uneven size advance together: one persistent member x tile launch per RK stage,
 * one hipGraph replay per step.  A member is set up by the entry points above
 * (through cuda_timeIntInit, state uploaded), then moved into the ensemble. ------ */
/* Move the current model's device state into the ensemble; returns the member index,
 * or -FE_ERR_* (variant without ensemble kernels, large-scale forcing, a physics-stage
 * schedule other than the ensemble's).  The model's device entry points then return
 * FE_ERR_STATE until it is set up again. */
int fe_ens_add_member(void);
int fe_ens_count(void);
/* info[0..8] = Nx, Ny, Nz, row pitch P, fields NF, z segments, segment length, step index,
 * simulation time in ms; n >= 9. */
int fe_ens_member_info(int m, int *info, int n);
/* Member state ([field][z][y][x], row pitch P), n = NF*Nz*Ny*P floats. */
int fe_ens_member_state(int m, float *out, long n);
/* Member friction velocity ([y][x], pitch P), n = Ny*P floats. */
int fe_ens_member_ustar(int m, float *out, long n);
/* z segments of member m (work tile 64 x 8 x ceil(Nz/nseg) levels).  Members that are given none, by this
 * or by amd_zSegments, share a segment length chosen for all members together, again whenever one is added. */
int fe_ens_set_segments(int m, int nseg);
/* nsteps RK3 steps of every member (graph replays, one synchronisation). */
int fe_ens_steps(int nsteps);
/* nsteps RK3 steps of each member in turn through the plain (one model per launch) kernels. */
int fe_ens_steps_sequential(int nsteps);
/* Device ms of each step: ensemble steps, or (sequential = 1) member plain steps in turn, each
 * member launched with the z segments the plain path chooses for its grid. */
int fe_ens_step_times(int nsteps, int sequential, float *ms);
/* Choose each member shape's z segments by timing trial_steps graph replays per candidate;
 * state and step rows are restored afterwards; a text report goes to report[len]. */
int fe_ens_autotune(int trial_steps, char *report, int len);
/* Free every member and table. */
int fe_ens_clear(void);

/* ---- Bitwise checkpoint (no counterpart in the reference, whose restart goes through the
 * per-unit-mass netCDF output, SRC/FEMAIN/FastEddy.c:202-243, and re-derives the surface
 * exchange coefficients on the first step after it). ---------------------------------- */
/* Write the device state (rho-weighted fields as the device holds them), every 2-D surface
 * plane, simTime, simTime_it and simTime_itRestart to path. */
int fe_checkpoint_write(const char *path);
/* Restore them (after cuda_timeIntInit of the same model) and copy the state into the host
 * arrays; N steps equal k steps + checkpoint + resume + N-k steps bit for bit.  Another
 * model's file, a truncated file or a hash mismatch returns FE_ERR_UNSUPPORTED. */
int fe_checkpoint_read(const char *path);

/* ---- Learned SGS closure (no counterpart in the reference; it stands beside the TKE
 * closure of SRC/HYDRO_CORE/CUDA/cuda_sgsTurbDevice.cu:202-367 and
 * cuda_sgstkeDevice.cu:68-397, which stays the fallback).  Network 256 -> 64 -> 64 -> 64
 * (GELU) -> 16 (first 9 outputs used), BF16 MFMA GEMMs with FP32 accumulation, FP32 master
 * weights; features and outputs as described in fe_sgs_kernels.hip. ------------------- */
/* Box-filter the current device state by fac (and the SGS stresses the last batch emitted,
 * hydroSubGridWrite = 1) and append its features and Favre-filtered SGS targets to the
 * training set; returns the set's row count or -FE_ERR_*. */
int fe_sgs_collect(int fac);
/* The same filter without touching the training set (an evaluation run's filtered fields);
 * returns the filtered cell count or -FE_ERR_*. */
int fe_sgs_filter(int fac);
/* Last filtered state [5][zc][yc][xc] and its target rows [cells][16]; either may be null. */
int fe_sgs_filtered(float *state, long nstate, float *targets, long ntarget);
/* Feature and target normalisation of the set (FP64 statistics), applied in place. */
int fe_sgs_prepare(void);
/* Glorot-uniform weights, zero biases, from a seeded generator; Adam moments cleared. */
int fe_sgs_init_params(unsigned seed);
/* Adam over epochs passes of mini-batches of batch rows; mean loss per epoch to loss. */
int fe_sgs_train(int epochs, int batch, float lr, unsigned seed, double *loss, int nloss);
/* Parameter vector (fe_sgs_nparam floats) out (get = 1) or in (get = 0). */
int fe_sgs_params(float *buf, long n, int get);
long fe_sgs_nparam(void);
/* Normalisation [4][256] (feature means, feature 1/std, target means, target std) out or in. */
int fe_sgs_norm(float *buf, long n, int get);
/* Network forward of M feature rows [M][256] into Y [M][16] (host buffers). */
int fe_mlp_forward(const float *X, long M, float *Y);
/* Loss (mean squared error over the 9 outputs) and its gradient for the parameter vector. */
int fe_mlp_gradient(const float *X, const float *T, long M, float *grad, double *loss);
/* Learned closure in the physics stage on/off; cells pass where every |normalised feature|
 * <= gate and the predicted stress tensor is realizable; elsewhere the TKE closure stays. */
int fe_sgs_enable(int on, float gate);
/* out[0] cells evaluated since enabling, out[1] cells that passed (n >= 2). */
int fe_sgs_stats(double *out, int n);
/* Learned cell stresses [9][cells] and pass masks of the last physics stage. */
int fe_sgs_last(float *tau, unsigned char *mask, long n);
/* The TKE closure's stresses the last physics stage emitted, [9][Nz][Ny][P]. */
int fe_sgs_emitted(float *tau, long n);
/* Inference through the fused kernels (on = 1, the default: a gradient pass and one persistent
 * BF16-MFMA network kernel) or the unfused feature / GEMM / activation kernels (on = 0); the
 * same bits either way. */
int fe_sgs_set_fused(int on);
/* Free the training set, network and inference buffers. */
int fe_sgs_clear(void);

#ifdef __cplusplus
}
#endif
#endif
