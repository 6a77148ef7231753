/*
 * leap_hip.h — C ABI of the MI355X (gfx950) LEAP calibrator.
 *
 * The drop-in boundary: plain pointers, sizes and status codes, no C++ or
 * framework types.  The C++ class icrar::hip::HipLeapCalibrator (see
 * icrar-leap-accelerate_amd/cpp/) implements the reference's ILeapCalibrator
 * over these entry points, and the Python test harness binds them with ctypes.
 *
 * Reference interfaces replaced (paths relative to src/icrar/leap-accelerate/
 * of ska-telescope/icrar-leap-accelerate v0.8.0):
 *   leap_hip_calibrate              ILeapCalibrator::Calibrate
 *                                   (algorithm/ILeapCalibrator.h:62-68), as done by
 *                                   cuda::CudaLeapCalibrator::Calibrate
 *                                   (algorithm/cuda/CudaLeapCalibrator.cu:94-233)
 *   leap_hip_create/destroy         CudaLeapCalibrator ctor/dtor (CudaLeapCalibrator.cu:73-92)
 *   leap_hip_metadata_create        cpu::MetaData::MetaData (model/cpu/MetaData.cc:42-137)
 *                                   + cuda::DeviceMetaData upload (model/cuda/DeviceMetaData.cu)
 *   leap_hip_rotate_visibilities    CudaLeapCalibrator::RotateVisibilities
 *                                   (CudaLeapCalibrator.cu:355-400; CPU form
 *                                   CpuLeapCalibrator.cc:181-217)
 *   leap_hip_apply_inversion        the inversion half of CudaLeapCalibrator::PhaseRotate
 *                                   (CudaLeapCalibrator.cu:248-261; CPU form
 *                                   CpuLeapCalibrator.cc:159-178)
 *   leap_hip_dd_matrix              cpu::MetaData::GenerateDDMatrix (MetaData.cc:166-203)
 *   leap_ms_view                    the accessors of icrar::MeasurementSet used on the
 *                                   path (ms/MeasurementSet.h:54-224, MetaData.cc:46-89,
 *                                   Integration.cc:54-55)
 *
 * Errors: every entry point returns LEAP_OK (0) or a negative leap_status; the
 * message is available from leap_hip_last_error().  No entry point exits the
 * process (the reference's CUDA path calls exit() on CUDA errors,
 * cuda/helper_cuda.cuh:613-624).  Argument errors the reference raises as
 * icrar::invalid_argument_exception / icrar::exception carry the reference's
 * message text.
 *
 * Threading: a leap_ctx owns one HIP stream on one device and its device
 * workspace; use one context per host thread.  Calls are synchronous: on
 * return all device work of the call has completed.  Device pointers passed in
 * a leap_ms_view must be fully written (the caller synchronised) before the call.
 */
#ifndef LEAP_HIP_H
#define LEAP_HIP_H

#include <stdint.h>

#ifdef __cplusplus
extern "C" {
#endif

typedef enum leap_status {
    LEAP_OK = 0,
    LEAP_ERR_INVALID_ARGUMENT = -1, /* icrar::invalid_argument_exception */
    LEAP_ERR_RANGE = -2,            /* icrar::exception (ranges, slices, ms layout) */
    LEAP_ERR_HIP = -3,              /* a HIP runtime call failed */
    LEAP_ERR_OUT_OF_MEMORY = -4,
    LEAP_ERR_NOT_IMPLEMENTED = -5,
    LEAP_ERR_CALLBACK = -6,         /* the output callback returned non-zero */
    LEAP_ERR_INTERNAL = -7
} leap_status;

typedef enum leap_vis_dtype {
    LEAP_VIS_C128 = 0, /* complex<double> */
    LEAP_VIS_C64 = 1   /* complex<float>, the DATA column's own type */
} leap_vis_dtype;

/* In-memory measurement set: the accessor contract of icrar::MeasurementSet.
 * antenna1/antenna2/time/flag/uvw are host memory.  vis is host memory, or
 * device memory of the context's device when vis_on_device is 1.  uvw_device
 * optionally gives a device copy of uvw (saves the upload).  The field order up
 * to vis_on_device is shared with the CPU oracle's view. */
typedef struct leap_ms_view {
    uint32_t num_stations;          /* GetNumStations (MeasurementSet.cc:132-135) */
    uint32_t total_antennas;        /* GetTotalAntennas: ANTENNA table rows (:110-113) */
    uint32_t num_baselines;         /* GetNumBaselines (:154-167) */
    uint32_t num_rows;              /* GetNumRows (:105-108) */
    uint32_t num_channels;          /* SPECTRAL_WINDOW NUM_CHAN[0] (:169-179) */
    uint32_t num_pols;              /* POLARIZATION NUM_CORR[0] (:137-147) */
    double freq_start_hz;           /* SPECTRAL_WINDOW REF_FREQUENCY[0] (MetaData.cc:59) */
    double freq_inc_hz;             /* SPECTRAL_WINDOW CHAN_WIDTH[0][0] (MetaData.cc:60) */
    double phase_centre_ra_rad;     /* FIELD PHASE_DIR[0] (MetaData.cc:67-79) */
    double phase_centre_dec_rad;
    const int32_t* antenna1;        /* ANTENNA1 of rows [0, num_baselines) */
    const int32_t* antenna2;        /* ANTENNA2 of rows [0, num_baselines) */
    const double* time;             /* TIME of all rows (epochs, MeasurementSet.cc:120-130) */
    const uint8_t* flag;            /* FLAG[row][0][0] for rows [0, num_baselines) (:181-197) */
    const double* uvw;              /* UVW, num_rows x 3 */
    const void* vis;                /* DATA, [num_rows][num_channels][num_pols] complex */
    int32_t vis_dtype;              /* leap_vis_dtype */
    int32_t vis_on_device;          /* 1: vis is a device pointer */
    const double* uvw_device;       /* optional device copy of uvw, or NULL */
} leap_ms_view;

typedef enum leap_precision {
    /* FP64 phase, FP64 sincos, FP64 sums: the reference's arithmetic.  Batched pol-0
     * calls with 96..512 channels and at least 16 directions sum the channels with the
     * width-16 NUFFT by default (LEAP_CHANNEL_SUM_AUTO; see LEAP_CHANNEL_SUM_NUFFT_W16),
     * other calls with the FP64 Horner chains. */
    LEAP_PRECISION_FP64 = 0,
    /* Visibilities stored as complex64 (or converted on load), the phase
     * argument and its reduction in FP64, Ad * dphi as split-3 x BF16 MFMA
     * with FP32 accumulation.  The channel sums of pol 0 follow channel_sum:
     * by default (LEAP_CHANNEL_SUM_AUTO) the NUFFT for 96..512 channels and at
     * least 16 directions, else a full-row FP64 Horner evaluation (FP64 FMA
     * issues at the rate of non-packed FP32 on gfx950).  The fp32_blocks
     * option selects FP32 sincos / Horner / Kahan sums instead of the FP64
     * Horner.  Needs the batched strategy. */
    LEAP_PRECISION_MIXED = 1
} leap_precision;

typedef enum leap_strategy {
    /* Every sample rotated by its own phase, as the reference; up to eight directions per
     * pass over the visibilities. */
    LEAP_STRATEGY_PER_DIRECTION = 0,
    /* One pass over the visibilities for a block of directions. */
    LEAP_STRATEGY_BATCHED = 1
} leap_strategy;

typedef enum leap_channel_sum {
    /* Pol 0, 96..512 channels and at least 16 directions: the NUFFT in mixed precision,
     * the width-16 NUFFT in FP64 precision; otherwise Horner.  FP64 calls on a device cube that
     * name no tile take Horner up to 32 directions on 2,048 rows or more and up to 48 on 16,384,
     * where its folded kernel is the faster. */
    LEAP_CHANNEL_SUM_AUTO = 0,
    /* FP64 Horner sums (rounding error at most n eps of sum |v|): on a device cube with no tile
     * named by folded blocks of eight channels, 2.5 FMAs per channel and direction; else four. */
    LEAP_CHANNEL_SUM_HORNER = 1,
    /* Type-2 non-uniform FFT per row (one inverse FFT of 256..1024 points, then W = 10 or 12
     * grid points per direction); mixed precision, pol 0, 1..512 channels.  A device-resident
     * complex64 cube with 1, 2 or 4 pols (16-byte aligned for 2 or 4) is read by the NUFFT kernel
     * itself; other sources (host-resident or complex128 cubes, 3 pols) are first packed to
     * pol-0 rows.  Error of a
     * row's channel sum: about 1e-11 of sum |v| (the tests bound avgData by 5e-10 of the sum
     * of |v| over the interval's rows and channels). */
    LEAP_CHANNEL_SUM_NUFFT = 2,
    /* The same NUFFT with the transform, the grid and the interpolation in FP32 (W = 8 or
     * 10; the shift factor, grid coordinate, phasor and the sums over rows stay FP64):
     * about a third less time at 384 channels, 2e-8 to 7e-8 of sum |v| per row (tests:
     * avgData within 2e-7 of the sum of |v|).  Outside the 1e-5 rad budget of the mixed
     * precision: a baseline whose sum nearly cancels takes a phase error of that order,
     * which the inversion spreads over the calibration (measured 4e-5 rad on 48 stations,
     * 2.5e-2 rad on the 256-station, 128-timestep set). */
    LEAP_CHANNEL_SUM_NUFFT_FP32 = 3,
    /* The NUFFT with an FP64 transform and a kernel of width 16 (16 grid points per
     * direction), for either precision; pol 0, 1..512 channels.  The kernel's truncation
     * (exp(-beta), 2e-18 to 1.3e-16) lies below FP64 rounding, so a row's channel sum is
     * within about 1e-15 of sum |v| of the exact sum at the same FP64 phase step, closer than
     * the FP64 Horner chains (n eps, about 2e-14 at 384 channels).  A device-resident
     * complex64 or complex128 cube with 1, 2 or 4 pols (16-byte aligned, except one complex64
     * pol) is read by the kernel itself; other sources are packed to pol-0 rows first. */
    LEAP_CHANNEL_SUM_NUFFT_W16 = 4
} leap_channel_sum;

typedef struct leap_options {
    int32_t precision;        /* leap_precision */
    int32_t strategy;         /* leap_strategy */
    int32_t direction_block;  /* batched: directions per workgroup (32, 64, 128, 256); 0 = tuned */
    int32_t all_pols;         /* batched: also accumulate polarisations 1..P-1 of avgData */
    int32_t fp32_blocks;      /* mixed: FP32 Horner blocks of 32 channels re-anchored by FP32
                                 sincos, Kahan sums (faster; outside the 1e-5 rad budget on
                                 decorrelated baselines); 0 = full-row FP64 Horner */
    int32_t lane_directions;  /* batched FP64 Horner: directions per lane (1, 2, 4); 0 = tuned */
    int32_t workgroups_per_cu; /* multi-set launch: persistent workgroups per CU (1..64);
                                  -1 = one work item per workgroup; 0 = tuned */
    int32_t graph;            /* 1: capture the call's device work (every solution interval's
                                 rotate/average and inversion) as a HIP graph, kept in the
                                 context and replayed by later calls with the same shapes,
                                 options and device addresses; results reach the callback
                                 after the whole graph.  Needs vis_on_device and uvw_device. */
    int32_t direct_cube;      /* batched pol 0: 1 = run the Horner kernel straight from the cube;
                                 0 = automatic: a tuned call on a device cube packs
                                 pol 0 first (FP64, non-finite (row, channel)s zeroed; 16 B per
                                 row and channel of device memory; the Horner kernel then reads
                                 it with scalar loads) only above a number of directions set by
                                 measured rates (with 4 pols about 600 of 384 channels, 440
                                 of 48); host cubes and packed tiles always pack */
    int32_t pack_timesteps;   /* packed path: timesteps per pack chunk; chunks are packed on a
                                 second stream while the Horner kernel runs the previous one.
                                 0 = automatic; >= the interval's timesteps = one chunk */
    int32_t channel_sum;      /* leap_channel_sum: how the batched pol-0 path sums channels */
    int32_t reserved[1];
} leap_options;

/* One solution interval's result: cpu::Calibration (model/cpu/calibration/Calibration.h:42-111)
 * holding one cpu::BeamCalibration per direction (BeamCalibration.h:45-124). */
typedef struct leap_solution {
    uint32_t index;               /* solution number */
    double start_epoch;           /* epochs[s * interval] (CpuLeapCalibrator.cc:107-109) */
    double end_epoch;             /* epochs[(s + 1) * interval - 1] */
    uint32_t n_directions;
    const double* directions;     /* [n_directions][2] (ra, dec) */
    uint32_t n_antennas;          /* A.cols() = max(antenna1, antenna2) + 1 */
    const double* calibrations;   /* [n_directions][n_antennas], valid during the callback */
} leap_solution;

/* Called once per solution interval, in order.  Return 0 to continue. */
typedef int (*leap_solution_cb)(void* user, const leap_solution* solution);

typedef struct leap_ctx leap_ctx;
typedef struct leap_metadata leap_metadata;

/* Diagnostics the reference writes to its log (Boost LOG(warning)). */
typedef enum leap_log_level { LEAP_LOG_INFO = 0, LEAP_LOG_WARNING = 1 } leap_log_level;
typedef void (*leap_log_cb)(void* user, int32_t level, const char* message);

/* ---- context -------------------------------------------------------------- */
int leap_hip_create(leap_ctx** out, int32_t device);
void leap_hip_destroy(leap_ctx* ctx);
/* Message of the last failure of ctx on this thread (ctx may be NULL). */
const char* leap_hip_last_error(const leap_ctx* ctx);
/* Library version string. */
const char* leap_hip_version(void);

/* ---- calibration (drop-in for ILeapCalibrator::Calibrate) ----------------- */
/* slice_* follow icrar::Slice(start, interval, end) with -1 wildcards
 * (common/Slice.cc:36-63); reference_antenna < 0 means none; use_cache keeps
 * the pseudo-inverse of A in the context keyed by a hash of A (the reference
 * caches it in files A.hash / Ad.cache, MetaData.cc:112-120).  opts may be NULL
 * (FP64, per direction). */
int leap_hip_calibrate(leap_ctx* ctx, const leap_ms_view* ms, const double* directions,
                       uint32_t n_directions, int32_t slice_start, int32_t slice_interval,
                       int32_t slice_end, double min_baseline_threshold,
                       int32_t reference_antenna, int32_t use_cache, const leap_options* opts,
                       leap_solution_cb callback, void* user);

/* Same, with metadata built beforehand by leap_hip_metadata_create for this ms. */
int leap_hip_calibrate_md(leap_ctx* ctx, const leap_metadata* md, const leap_ms_view* ms,
                          const double* directions, uint32_t n_directions, int32_t slice_start,
                          int32_t slice_interval, int32_t slice_end, const leap_options* opts,
                          leap_solution_cb callback, void* user);

/* Bytes of the device scratch array behind leap_hip_calibrate_md_noalloc (one
 * per GPU, held until the process ends). */
#define LEAP_NOALLOC_SCRATCH_BYTES (16u << 20)

/* No counterpart in the reference.  For callers that cannot allocate device
 * memory (code under HIP graph capture, tight serving loops, harnesses that
 * forbid hipMalloc): leap_hip_calibrate_md on its FP64 per-direction route,
 * allocating nothing.  The direction table, dd matrices, one direction's
 * avgData and the inversion's cal1 and antenna sums live in
 * a fixed device array of LEAP_NOALLOC_SCRATCH_BYTES per GPU; the results are
 * bit-identical to leap_hip_calibrate_md with opts NULL.
 *   ms         visibilities and uvw device-resident (vis_on_device = 1,
 *              uvw_device set)
 *   cal_out    device memory, [n_solutions][n_directions][n_antennas] doubles;
 *              NULL only reports n_solutions_out and computes nothing
 *   epochs_out host memory, [n_solutions][2] (start, end), or NULL
 * Returns LEAP_ERR_RANGE when one solution's working set (16 B per direction
 * and 72 B of dd, 16 B per baseline and pol, 8 B per row of A and A1 and per
 * antenna, plus 8 B per antenna and 64 of those rows) exceeds the scratch (more than the
 * sums above take; the bound is part of the interface).  Every call on a GPU
 * shares that GPU's scratch: calls that overlap on one GPU (other threads,
 * other contexts on the device) race.  Synchronous on return. */
int leap_hip_calibrate_md_noalloc(leap_ctx* ctx, const leap_metadata* md, const leap_ms_view* ms,
                                  const double* directions, uint32_t n_directions, int32_t slice_start,
                                  int32_t slice_interval, int32_t slice_end, double* cal_out,
                                  double* epochs_out, int32_t* n_solutions_out);

/* ---- several measurement sets in one launch -------------------------------- */
/* One measurement set of leap_hip_calibrate_batch: the metadata built for it by
 * leap_hip_metadata_create, its directions and its Slice (as leap_hip_calibrate). */
typedef struct leap_batch_set {
    const leap_metadata* metadata;
    const leap_ms_view* ms;
    const double* directions;  /* [n_directions][2] (ra, dec) */
    uint32_t n_directions;
    int32_t slice_start, slice_interval, slice_end;
} leap_batch_set;

/* Called once per (set, solution interval): interval s of every set that has
 * one, in set order, before interval s + 1.  Return 0 to continue. */
typedef int (*leap_batch_cb)(void* user, uint32_t set, const leap_solution* solution);

/* Calibrate of several measurement sets with uneven antenna, baseline, channel
 * and timestep counts: each set gets the solutions leap_hip_calibrate_md would
 * give it with the same options.  Solution interval s of all sets, all
 * directions, is rotated and averaged in ONE persistent launch where a tile is named, and
 * for the sets that do not fill the GPU by themselves (fewer than 8,192 rows, and not given the
 * folded kernel by the automatic rule; the others take the launch of a single-set call): a device
 * descriptor per set and (set, baseline, direction block) work items
 * statically load-balanced over the grid on the host (longest processing time
 * first), so the result does not depend on scheduling.  In mixed precision the
 * sets that qualify for the NUFFT channel sums (channel_sum automatic: 96..512
 * channels, 16 or more directions; or channel_sum = LEAP_CHANNEL_SUM_NUFFT)
 * and hold complex64 cubes with 1, 2 or 4 pols take them instead, one launch
 * per group of sets that share a grid and kernel width, with their
 * (set, baseline, direction block) items in decreasing rows per item (the single-set launch
 * for a group of one set); each
 * item's sums are those of the single-set NUFFT kernel.  Needs the batched
 * strategy, all_pols = 0, fp32_blocks = 0 and channel_sum other than
 * LEAP_CHANNEL_SUM_NUFFT_FP32.  No reference counterpart: the
 * reference calibrates one measurement set per ILeapCalibrator::Calibrate call
 * (algorithm/ILeapCalibrator.h:62-68). */
int leap_hip_calibrate_batch(leap_ctx* ctx, const leap_batch_set* sets, uint32_t n_sets,
                             const leap_options* opts, leap_batch_cb callback, void* user);

/* The static schedule leap_hip_calibrate_batch uses, on the host (no GPU):
 * the work items of sets with the given shapes for the persistent kernel tile
 * (directions per workgroup * 10 + directions per lane) over n_blocks
 * workgroups.  Workgroup g runs items [offsets[g], offsets[g + 1]);
 * item_set / item_local give the set and baseline + nbl * direction block of
 * each.  offsets holds n_blocks + 1 entries; item arrays hold
 * sum_s nbl_s * ceil(D_s / (tile / 10)) entries; *makespan_out (may be NULL)
 * gets the largest per-workgroup cost in the cost model's units. */
int leap_multi_schedule(const uint32_t* nbl, const uint32_t* timesteps, const uint32_t* channels,
                        const uint32_t* n_directions, uint32_t n_sets, int32_t tile, uint32_t n_blocks,
                        uint32_t* offsets, uint32_t* item_set, uint32_t* item_local, double* makespan_out);
/* Cost-model units of one work item of a set with the given shape (the weights the
 * schedule balances). */
double leap_multi_item_cost(uint32_t timesteps, uint32_t channels, int32_t tile);

/* ---- metadata (A, I, A1, I1 and their pseudo-inverses, on the device) ------ */
int leap_hip_metadata_create(leap_ctx* ctx, const leap_ms_view* ms, int32_t reference_antenna,
                             double min_baseline_threshold, int32_t use_cache,
                             leap_metadata** out);
void leap_hip_metadata_destroy(leap_metadata* md);
/* Receives the context's diagnostics (NULL drops them): the warnings "Ad is
 * degenerate" / "Ad1 is degenerate" of MetaData::MetaData (model/cpu/MetaData.cc:129-136),
 * raised when (Ad A).isApprox(I, 0.001) fails, i.e. when the baseline graph has
 * a component without the constraint antenna (an unused antenna column included). */
int leap_hip_set_log_callback(leap_ctx* ctx, leap_log_cb callback, void* user);
/* Those two conditions of a built metadata (1 = degenerate). */
int leap_hip_metadata_diagnostics(const leap_metadata* md, int32_t* ad_degenerate, int32_t* ad1_degenerate);
/* dims = {K = A.rows, N = A.cols, K1 = A1.rows, nbaselines, referenceAntenna} */
void leap_hip_metadata_dims(const leap_metadata* md, int32_t* dims);
/* Host copies, column-major like Eigen; any pointer may be NULL.
 * A: K x N, I: K-1, Ad: N x K, A1: K1 x N, I1: K1-1, Ad1: N x K1. */
int leap_hip_metadata_copy(const leap_metadata* md, double* A, int32_t* I, double* Ad,
                           double* A1, int32_t* I1, double* Ad1);

/* ---- the two halves of PhaseRotate ---------------------------------------- */
/* avgData for rows [row_start, row_start + n_rows) and n_directions
 * directions; avg_out is host [n_directions][nbaselines][num_pols] complex128
 * (interleaved re, im).  With opts->all_pols == 0 under the batched strategy
 * only polarisation 0 is written (the others are left 0). */
int leap_hip_rotate_visibilities(leap_ctx* ctx, const leap_metadata* md, const leap_ms_view* ms,
                                 uint32_t row_start, uint32_t n_rows, const double* directions,
                                 uint32_t n_directions, const leap_options* opts, double* avg_out);

/* cal = Ad * dphi + Ad1 * phi1 from host avgData [n_directions][nbaselines][num_pols]
 * complex128; cal_out is host [n_directions][N]. */
int leap_hip_apply_inversion(leap_ctx* ctx, const leap_metadata* md, const double* avg,
                             uint32_t n_directions, const leap_options* opts, double* cal_out);

/* The direction-dependent rotation matrices, computed by the device kernel;
 * dd_out is host [n_directions][3][3] row-major. */
int leap_hip_dd_matrix(leap_ctx* ctx, double phase_centre_ra, double phase_centre_dec,
                       const double* directions, uint32_t n_directions, double* dd_out);

/* ---- differentiation ------------------------------------------------------ */
/* Calibration-residual loss of one solution interval over all rows and its
 * gradient with respect to direction offsets and antenna positions.  No
 * reference counterpart: it differentiates the reference's calibration
 * (CpuLeapCalibrator.cc:147-217) for direction and array refinement.
 *   uvw(row)  = uvw(row) + M_t (dp[antenna2] - dp[antenna1]),  M_t = enu_to_uvw[t] (3x3 row-major)
 *   direction = directions[d] + offsets[d]                      (ra, dec radians)
 *   loss      = sum_d sum_{n < K-1} wrap((A cal_d)(n) - arg avgData_d(I(n)))^2
 * with avgData and cal computed in FP64 as leap_hip_calibrate does (pol 0).
 * Everything runs on the device: the forward rotate/average and inversion,
 * the loss, the adjoint of arg and of the pseudo-inverse products, and the
 * adjoint of rotate/average as leap_hip_set_adjoint_mode selects; one
 * synchronisation per call.  offsets (D x 2),
 * antenna_delta (N x 3, metres east/north/up) may be NULL (zero); grad_offsets
 * (D x 2) and grad_antenna (N x 3) may be NULL.  1 <= D <= 256. */
/* How leap_hip_residual_loss_grad forms the adjoint of rotate/average:
 *   LEAP_ADJOINT_AUTO (the default): as ROW_SUMS when the row sums take no more
 *     memory than the visibility cube (32 D <= channels x pols x element bytes),
 *     else as RECOMPUTE;
 *   LEAP_ADJOINT_RECOMPUTE: the forward pass keeps nothing; the adjoint reads
 *     the cube again and recomputes the phasors, the channel sum P(z) and its
 *     derivative by Horner's rule;
 *   LEAP_ADJOINT_ROW_SUMS: the forward pass also keeps each row's channel sums
 *     e0 P(z) and e0 z P'(z) (32 bytes per row and direction, no phasors) and
 *     the adjoint reads them instead of the cube.
 * The result is the same to rounding.  Applies to later calls on ctx. */
enum { LEAP_ADJOINT_AUTO = 0, LEAP_ADJOINT_RECOMPUTE = 1, LEAP_ADJOINT_ROW_SUMS = 2 };
int leap_hip_set_adjoint_mode(leap_ctx* ctx, int32_t mode);
int leap_hip_residual_loss_grad(leap_ctx* ctx, const leap_metadata* md, const leap_ms_view* ms,
                                const double* directions, const double* offsets, uint32_t n_directions,
                                const double* antenna_delta, const double* enu_to_uvw, double* loss,
                                double* grad_offsets, double* grad_antenna);

/* ---- host model (no GPU needed) ------------------------------------------- */
/* cpu::PhaseMatrixFunction (algorithm/cpu/PhaseMatrixFunction.cc:35-93).
 * ref_ant < 0 means none.  A_out holds (n + 1) x (max(a1, a2) + 1) doubles,
 * column-major with leading dimension n + 1, of which the first *K rows are
 * set; I_out holds n ints, of which *K - 1 are set. */
int leap_phase_matrix(const int32_t* a1, const int32_t* a2, const uint8_t* fg, int32_t n,
                      int32_t ref_ant, double* A_out, int32_t* I_out, int32_t* K, int32_t* N);
/* cpu::PseudoInverse (math/cpu/matrix_invert.h:70-74) of the phase matrix that
 * leap_phase_matrix builds from the same arguments, computed on the host the
 * way the device metadata computes it; Ad_out is N x K column-major. */
int leap_phase_matrix_pinv(const int32_t* a1, const int32_t* a2, const uint8_t* fg, int32_t n,
                           int32_t ref_ant, double* Ad_out);

/* exp(i theta) as the batched Horner kernels compute it (Cody-Waite reduction
 * by pi/2, Taylor series), on the host: cos_out[i], sin_out[i] of theta[i].
 * No reference counterpart (the reference calls std::exp on a complex,
 * CpuLeapCalibrator.cc:198); exported so the routine can be checked without a GPU. */
int leap_phasor64(const double* theta, uint32_t n, double* cos_out, double* sin_out);

/* The NUFFT plan of LEAP_CHANNEL_SUM_NUFFT for C channels (1..512): grid size
 * N, kernel width W, frequency offset h (channel c is frequency c - h), the
 * kernel's beta, the weight polynomials coef[j * 12 + m] (coefficient of s^m of
 * tap j < W / 2; 6 x 12 doubles) and the C precorrection factors scale[c].
 * Any output may be null.  No reference counterpart (the reference sums the
 * channels directly, CpuLeapCalibrator.cc:181-217); exported so the plan can be
 * checked without a GPU. */
int leap_nufft_plan(uint32_t C, uint32_t* N, uint32_t* W, uint32_t* h, double* beta, double* coef, double* scale);
/* The same for the FP32 transform of LEAP_CHANNEL_SUM_NUFFT_FP32 (narrower kernel). */
int leap_nufft_plan32(uint32_t C, uint32_t* N, uint32_t* W, uint32_t* h, double* beta, double* coef,
                      double* scale);
/* The same for LEAP_CHANNEL_SUM_NUFFT_W16 (W = 16): coef[j * 16 + m], 8 x 16 doubles. */
int leap_nufft_plan_w16(uint32_t C, uint32_t* N, uint32_t* W, uint32_t* h, double* beta, double* coef,
                        double* scale);

/* ---- synthetic measurement sets ------------------------------------------- */
typedef struct leap_synth_config {
    uint32_t n_antennas;
    int32_t layout;             /* 0: uniform disk, 1: three-arm log spiral */
    double array_radius_m;      /* disk radius, or outer radius of the spiral */
    int32_t autocorrelations;   /* include (a, a) baselines */
    uint32_t n_timesteps;
    double integration_s;
    uint32_t n_channels;
    double freq_start_hz;
    double freq_inc_hz;
    uint32_t n_pols;            /* 1..4 */
    double phase_centre_ra_rad;
    double phase_centre_dec_rad;
    double latitude_rad;
    uint32_t n_sources;
    double source_flux_min, source_flux_max;   /* Jy, uniform */
    double source_offset_max_rad;              /* |d ra|, |d dec| uniform in [-x, x] */
    double noise_sigma;                        /* per real / imaginary part */
    double flag_fraction;                      /* fraction of baselines flagged */
    double nan_fraction;                       /* fraction of (row, chan, pol) set to NaN */
    uint64_t seed;
} leap_synth_config;

typedef struct leap_synth_ms leap_synth_ms;

/* Builds the host-side columns (antennas, uvw, time, flags) and the sky model;
 * no visibilities yet.  Works without a GPU. */
int leap_synth_create(const leap_synth_config* cfg, leap_synth_ms** out);
void leap_synth_destroy(leap_synth_ms* ms);
/* Fills view with the host columns; vis is NULL until a fill call. */
void leap_synth_view(const leap_synth_ms* ms, leap_ms_view* view);
/* Per-timestep 3x3 matrices M_t (row-major, [T][3][3]) with uvw = M_t * (enu_a2 - enu_a1). */
void leap_synth_enu_to_uvw(const leap_synth_ms* ms, double* out);
/* Sky model for tests: n_sources x {ra, dec, flux}, and per-antenna phases. */
void leap_synth_sky(const leap_synth_ms* ms, double* sources, double* antenna_phase);
/* Host visibilities for rows [row_start, row_start + n_rows) into out
 * ([n_rows][C][P] of vis_dtype).  Works without a GPU. */
int leap_synth_fill_vis_host(const leap_synth_ms* ms, uint32_t row_start, uint32_t n_rows,
                             int32_t vis_dtype, void* out);
/* Device visibilities for all rows into the device buffer out (vis_dtype),
 * generated by a kernel; also uploads uvw.  The view's vis / uvw_device then
 * point at device memory.  out must hold num_rows * C * P complex values. */
int leap_hip_synth_fill_vis_device(leap_ctx* ctx, const leap_synth_ms* ms, int32_t vis_dtype,
                                   void* out_device, double* uvw_device_out);

/* ---- device memory helpers (for harnesses without their own allocator) ---- */
int leap_hip_malloc(leap_ctx* ctx, uint64_t bytes, void** out);
int leap_hip_free(leap_ctx* ctx, void* ptr);
int leap_hip_memcpy_d2h(leap_ctx* ctx, void* dst, const void* src, uint64_t bytes);
int leap_hip_memcpy_h2d(leap_ctx* ctx, void* dst, const void* src, uint64_t bytes);

/* ---- timing of the last calibrate / rotate call --------------------------- */
/* Average device time per launch (ms) of the rotate/average kernel and number of
 * launches in the last call: from the kernel's first workgroup to the start of the
 * inversion on the device's clock where a calibration takes one plain or folded Horner
 * kernel, else by HIP events on the context's stream.  total_ms: HIP events from the
 * start of the call to the end of its last device work. */
int leap_hip_last_kernel_times(const leap_ctx* ctx, double* rotate_ms_avg, int32_t* rotate_launches,
                               double* total_ms);
/* Tile the batched kernel used in the last call: directions per workgroup * 10
 * + directions per lane (0 if none). */
int leap_hip_last_direction_block(const leap_ctx* ctx);
/* Route of the last batched calibrate / rotate call: the channel sums used
 * (LEAP_CHANNEL_SUM_HORNER or _NUFFT) and whether the kernel read the cube
 * directly (1) or packed pol-0 rows (0).  Any output may be null. */
int leap_hip_last_route(const leap_ctx* ctx, int32_t* channel_sum, int32_t* direct_cube);
/* Workgroups per CU of the last multi-set launch (-1: one work item per
 * workgroup; 0 if none). */
int leap_hip_last_workgroups_per_cu(const leap_ctx* ctx);
/* Device times (on the device's clock, from the kernel's first workgroup to the start of
 * the kernel after it) of the last leap_hip_residual_loss_grad's forward rotate/average
 * kernel and adjoint kernel (0 when no gradient was asked for). */
int leap_hip_last_loss_grad_times(const leap_ctx* ctx, double* forward_ms, double* adjoint_ms);
/* Graph use of the last calibrate call: 0 none, 1 captured a new graph,
 * 2 replayed the context's graph. */
int leap_hip_last_graph(const leap_ctx* ctx);
/* Average device time (ms) of the pol-0 pack launches of the last call and
 * their number (0 when the call packed nothing). */
int leap_hip_last_pack_times(const leap_ctx* ctx, double* pack_ms_avg, int32_t* pack_launches);
/* ---- autotuner cache ------------------------------------------------------ */
/* The tiles (and multi-set grid depths) the context's autotuners chose, as a
 * JSON document {"format": "leap-hip-tuning", "version": 1, "batched": [...],
 * "multi": [...]}.  Writes at most cap bytes, NUL-terminated, into buf (may be
 * NULL) and the document's length + 1 into *needed. */
int leap_hip_tuning_save(const leap_ctx* ctx, char* buf, uint64_t cap, uint64_t* needed);
/* Adds the choices of a document written by leap_hip_tuning_save; later calls
 * of those shapes use them without timing candidates.  The document is checked
 * whole before anything is added. */
int leap_hip_tuning_load(leap_ctx* ctx, const char* json);

/* Bytes the last call sent host -> device through the pinned staging buffers
 * (host-resident visibilities; pol 0 only on the packed path). */
uint64_t leap_hip_last_staged_bytes(const leap_ctx* ctx);

#ifdef __cplusplus
}
#endif

#endif /* LEAP_HIP_H */
