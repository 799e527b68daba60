/*
 * fmdbzp.h — C ABI of the MI355X FM-DBZP acquisition engine (libfmdbzp.so).
 *
 * The engine replaces the inner search of Acquisition.jl's `acquire!`: the
 * PRN-independent prologue (`_downconvert!` + `_precompute_signal_block_ffts!`,
 * src/acquire.jl:92-104, src/coherent_integration.jl:12-56) and the per-PRN
 * search (`_acquire_prn_streamed!`, src/acquire.jl:242-327, or
 * `_accumulate_prn_step_tiled!`, src/noncoherent_integration.jl:760-812,
 * followed by `est_signal_noise_power`, src/est_signal_noise_power.jl:211-243).
 * Argument validation, Doppler / code-phase label arithmetic, CN0, the
 * parabolic interpolation formulas, the secondary-code phase gate and CFAR stay
 * in the host language above this boundary (src/acquire.jl:544-781).
 *
 * Conventions
 *  - Plain C types only; every pointer is a host pointer unless a flag says
 *    otherwise. The library never keeps a caller pointer after a call returns.
 *  - All indices are 0-based (a Julia caller adds 1).
 *  - Every call returns an int status (FMDBZP_OK == 0, negative on error);
 *    fmdbzp_last_error() returns a thread-local message for the last failure.
 *  - A plan handle serialises its own calls (one acquire per plan at a time,
 *    the reference's contract, src/plan.jl:186-190) and runs on its own HIP
 *    stream on the device that was current when the plan was created.
 */
#ifndef FMDBZP_H
#define FMDBZP_H

#include <stddef.h>
#include <stdint.h>

#ifdef __cplusplus
extern "C" {
#endif

#define FMDBZP_ABI_VERSION 1

enum fmdbzp_status {
    FMDBZP_OK = 0,
    FMDBZP_EINVAL = -1,  /* bad argument or descriptor */
    FMDBZP_ENOMEM = -2,  /* device or host allocation failed */
    FMDBZP_EHIP = -3,    /* HIP runtime error */
    FMDBZP_ENODEV = -4,  /* no usable gfx950 device */
    FMDBZP_EHANDLE = -5  /* null or destroyed plan handle */
};

/* Sample formats accepted by fmdbzp_acquire. `ComplexF32(x)` of each sample
 * is what enters the search (src/acquire.jl:94, :101). */
enum fmdbzp_eltype {
    FMDBZP_CF32 = 0,     /* interleaved float re,im (Julia ComplexF32) */
    FMDBZP_CF64 = 1,     /* interleaved double re,im (Julia ComplexF64) */
    FMDBZP_I16 = 2,      /* real int16 (Julia Int16 IF samples) */
    FMDBZP_CI8 = 3,      /* interleaved int8 re,im (Julia Complex{Int8}) */
    FMDBZP_CI16 = 4,     /* interleaved int16 re,im (Julia Complex{Int16}) */
    FMDBZP_F32 = 5,      /* real float (Julia Float32) */
    FMDBZP_F64 = 6,      /* real double (Julia Float64) */
    FMDBZP_C2BIT = 7     /* packed 2-bit complex SDR samples: byte i holds samples
                            2i (low nibble) and 2i+1 (high nibble); a nibble is
                            I in bits 0-1 and Q in bits 2-3, each code c mapping to
                            (c & 1 ? 3 : 1) * (c & 2 ? -1 : +1), i.e. {+1, +3, -1, -3}.
                            The reference sees the same values as Complex{Int8}. */
};

/* Search path, as selected by the reference (src/acquire.jl:250-253,
 * src/noncoherent_integration.jl:769-772). */
enum fmdbzp_path {
    FMDBZP_PATH_SIMPLE = 0,    /* N_db == 1, E == 1, no rotation search   */
    FMDBZP_PATH_SIGN = 1,      /* data-bit / bit-edge sign search          */
    FMDBZP_PATH_ROTATION = 2   /* secondary-code rotation search           */
};

enum fmdbzp_noise_estimator {
    FMDBZP_NOISE_OPPOSITE_ROW = 0,  /* src/est_signal_noise_power.jl:70  */
    FMDBZP_NOISE_GLOBAL_MEAN = 1    /* src/est_signal_noise_power.jl:100 */
};

enum fmdbzp_precision {
    FMDBZP_PREC_FP32 = 0,     /* plain FP32 path */
    /* Mixed: the coherent tile (block-correlation output, column-FFT input)
     * is stored in FP16, scaled by an exact power of two chosen from the
     * integer sample type's bound so that no tile value can overflow; all
     * arithmetic stays FP32. Half the tile traffic between the two stages.
     * Ndop-160 simple-path plans (the L1 C/A 10 ms searches) and integer
     * samples (I16, CI8, CI16, C2BIT) only; other plans are rejected at
     * creation and float samples at the search call (FMDBZP_EINVAL). */
    FMDBZP_PREC_TILE_FP16 = 1,
    /* Per call: FP32 where the full-period correlation runs (the faster form),
     * else FMDBZP_PREC_TILE_FP16 when the plan admits it and the samples are
     * integers, FMDBZP_PREC_MFMA on the plans that admit it with n1 = 10 or 20,
     * else FP32; never rejected. For batches of requests whose plans and sample
     * types differ. At n1 = 10 and 20 the choice is fixed, not the faster one:
     * the matrix-core kernel takes 48.4 and 109 ms per PRN-step at 25 MHz, FP32
     * (k_column_rot25) 34.5 and 79 (two steps); take FMDBZP_PREC_FP32 for speed. */
    FMDBZP_PREC_AUTO = 2,
    /* Mixed, on matrix cores: the column Doppler transforms of the secondary-
     * code rotation search run as complex DFT-matrix products on
     * v_mfma_f32_32x32x{16,8}_f16 (FP16 operands, FP32 accumulation), the
     * column scaled by an exact power of two into [0.5, 1) before the FP16
     * conversion; the last radix stage, powers and accumulation stay FP32.
     * Plans on the direct rotation path with 25 coherent periods and
     * ndop = 625 n1, n1 in {2, 4, 10, 20} (the E1-like searches at +-5 to
     * +-50 kHz) only; other plans are rejected at creation (FMDBZP_EINVAL). */
    FMDBZP_PREC_MFMA = 3
};

/* Plan options (fmdbzp_plan_desc.options). With N_db == 1 the bit-edge
 * offsets of the sign search only rotate each column circularly, so every
 * edge has the same |FFT|^2 (shift theorem) and the engine evaluates one edge;
 * FMDBZP_OPT_LITERAL_EDGES evaluates every edge offset as the reference's loop
 * does (src/noncoherent_integration.jl:670-684). Results agree to FP32 rounding. */
#define FMDBZP_OPT_LITERAL_EDGES 0x1
/* Capture each call's launch sequence in a hipGraph and replay it while calls
 * repeat the previous call's signal pointer, sample type, IF, flags and PRN
 * list (a serving loop over a ring of device buffers). Calls that store
 * surfaces or run with kernel timing launch directly. No counterpart in the
 * reference. */
#define FMDBZP_OPT_GRAPH 0x2
/* At plan creation, time the admissible launch configurations of the block
 * correlation (buffering, transforms per pass, pass split) and of the generic
 * simple column kernel (columns per workgroup) on the plan's workspace and
 * keep the fastest, for the calls that run on the tile (the full-period
 * correlation has none); choices are cached per geometry for the process. The
 * reference plans its FFTs by measurement (FFTW MEASURE, src/plan.jl:468-483).
 * The environment variable FMDBZP_AUTOTUNE=1 turns it on for every plan. */
#define FMDBZP_OPT_AUTOTUNE 0x4
/* Downconvert with the FP64 carrier phase -2 pi IF n / fs of absolute sample
 * n instead of the reference's Float32 argument (src/acquire.jl:96-101),
 * whose error grows with the sample index: at IF 4.092 MHz and 16.368 MHz
 * samples up to about 0.1 rad at the end of 80 ms and 0.75 rad at 400 ms (the
 * Float32 step's representation error times the index, plus half an ulp of
 * the phase). The Float32 form stays the default, for parity with the
 * reference. No effect at IF = 0. No counterpart in the reference. */
#define FMDBZP_OPT_FP64_PHASE 0x8
/* Run every call of a simple-path plan on the coherent tile (block correlation,
 * then the column stage). By default calls that return statistics only run the
 * full-period correlation where the plan admits it (one circular correlation
 * of the code period per Doppler row, no tile); calls with surfaces, and calls
 * of few Doppler rows over all their PRNs at long code periods, run on the
 * tile either way (fmdbzp_plan_call_kernels tells). For measuring the tile
 * kernels. Results agree to FP32 rounding. No counterpart in the reference. */
#define FMDBZP_OPT_TILE_PATH 0x10
/* Largest size of the code spectra of the full-period correlation, plan data
 * of 8 bytes x samples_per_code x num_doppler_bins per PRN held beside the
 * workspace (the L1 C/A search at 16.368 MHz, 160 bins, 32 PRNs: 0.67 GB).
 * Plans that would exceed it run on the tile. The limit depends neither on the
 * workspace budget nor on the memory in use. */
#define FMDBZP_FULL_SPECTRA_MAX_BYTES (4ull << 30)

/* fmdbzp_acquire flags */
#define FMDBZP_FLAG_STORE_SURFACES 0x1u  /* copy (ndop, spc_eff) power surfaces out */
#define FMDBZP_FLAG_DEVICE_SIGNAL  0x2u  /* `signal` is a device pointer           */
#define FMDBZP_FLAG_DEVICE_OUTPUT  0x4u  /* surface pointers are device pointers   */

/*
 * Plan descriptor: every scalar the reference derives in `plan_acquire`
 * (src/plan.jl:385-528). The host computes these with the reference's exact
 * arithmetic; the engine only consumes them.
 */
typedef struct fmdbzp_plan_desc {
    int32_t abi_version;             /* FMDBZP_ABI_VERSION                          */
    int32_t samples_per_code;        /* spc, src/plan.jl:386                        */
    int32_t num_blocks;              /* nb,  src/plan.jl:418-426                    */
    int32_t block_size;              /* bs = spc / nb, src/plan.jl:448              */
    int32_t fft_size;                /* F = nextprod((2,3,5,7), 2 bs), :460         */
    int32_t num_coh;                 /* N_coh                                       */
    int32_t num_data_bits;           /* N_db, src/plan.jl:464                       */
    int32_t bit_edge_search_steps;   /* E                                           */
    int32_t num_noncoherent;         /* N_nc                                        */
    int32_t num_secondary_rotations; /* R, src/plan.jl:511-515                      */
    int32_t num_doppler_bins;        /* ndop = N_coh * nb, src/plan.jl:465          */
    int32_t samples_per_code_eff;    /* spc * R (rotation) or spc, :524-525         */
    int32_t num_patterns;            /* Q columns of the sign-pattern matrix        */
    int32_t path;                    /* enum fmdbzp_path                            */
    int32_t noise_estimator;         /* enum fmdbzp_noise_estimator                 */
    int32_t samples_per_chip;        /* floor(fs / f_code), GlobalMean exclusion    */
    int32_t precision;               /* enum fmdbzp_precision                       */
    int32_t options;                 /* FMDBZP_OPT_* bits, 0 = defaults             */
    int32_t reserved[6];
    double sampling_freq_hz;
} fmdbzp_plan_desc;

/*
 * Per-PRN search statistics returned by fmdbzp_acquire: what the reference's
 * per-PRN search hands to result extraction (src/acquire.jl:202-209 and
 * :549-555), plus the four neighbour cells that parabolic interpolation reads
 * (src/acquire.jl:597-618, :718-737), so no surface has to cross the bus.
 */
typedef struct fmdbzp_prn_stats {
    float peak_power;      /* max of the (ndop, spc_eff) power surface            */
    int32_t peak_row;      /* 0-based sorted-Doppler row of the peak              */
    int32_t peak_col;      /* 0-based effective column (rotation * spc + col)     */
    float noise_power;     /* estimator output (OppositeRow or GlobalMean)         */
    float code_left;       /* (peak_row, scrambled col - 1 mod spc, same rotation) */
    float code_right;      /* (peak_row, scrambled col + 1 mod spc, same rotation) */
    float dop_left;        /* (peak_row - 1 wrapping, peak_col)                    */
    float dop_right;       /* (peak_row + 1 wrapping, peak_col)                    */
    double noise_sum;      /* FP64 sum of the cells averaged into noise_power      */
    int64_t noise_cells;   /* number of those cells                                */
} fmdbzp_prn_stats;

typedef struct fmdbzp_plan fmdbzp_plan;  /* opaque, device-resident plan */

/*
 * Create a device-resident plan. Replaces plan.jl's device-independent tables:
 * the conjugated PRN sub-block FFTs (`_precompute_prn_ffts!`,
 * src/plan.jl:230-251, computed on the device from the code samples given
 * here), the sign patterns (src/plan.jl:627-672) and the per-step code-drift
 * shifts (`_fill_code_drift_shifts!`, src/noncoherent_integration.jl:600-619,
 * evaluated by the host in FP64).
 *
 *  code_samples   nprn x spc int8 (+1/-1): gen_code(spc, system, prn, fs, f_code, 0)
 *  patterns       npattern_sets x (N_coh x Q) float, column-major like the
 *                 reference's Matrix{Float32} (row = coherent period)
 *  pattern_set    nprn int32: which pattern set each PRN uses (may be NULL
 *                 when npattern_sets <= 1)
 *  drift_shifts   N_nc x ndop int32 in [0, spc), indexed [step][sorted row]
 */
int fmdbzp_plan_create(const fmdbzp_plan_desc* desc,
                       int32_t nprn,
                       const int8_t* code_samples,
                       int32_t npattern_sets,
                       const float* patterns,
                       const int32_t* pattern_set,
                       const int32_t* drift_shifts,
                       fmdbzp_plan** out_plan);

/*
 * Run the search for `nreq` PRNs of the plan (indices into the plan's PRN
 * list) over `signal` (n_samples samples of `eltype`, at least N_nc segments
 * of N_coh * spc samples, src/acquire.jl:65-72). Replaces the body of
 * `acquire!` from `_downconvert!` to the per-PRN statistics
 * (src/acquire.jl:114-215).
 *
 *  out_stats      nreq entries
 *  out_surfaces   NULL, or nreq pointers to (ndop, spc_eff) float surfaces in
 *                 Julia column-major order (row fastest), written when
 *                 FMDBZP_FLAG_STORE_SURFACES is set (store_power_bins).
 */
int fmdbzp_acquire(fmdbzp_plan* plan,
                   const void* signal,
                   int32_t eltype,
                   int64_t n_samples,
                   double interm_freq_hz,
                   const int32_t* prn_index,
                   int32_t nreq,
                   uint32_t flags,
                   fmdbzp_prn_stats* out_stats,
                   float* const* out_surfaces);

/*
 * Result formulas of one PRN (src/acquire.jl:9-13, :544-671): Float32 power
 * ratios, code phase and Doppler in Float64.
 */
typedef struct fmdbzp_prn_result {
    double cn0_dbhz;        /* 10 log10(signal / noise / coherent time); -inf, NaN as the ratio is 0, below */
    double code_phase;      /* chips, in [0, code length)                             */
    double doppler_offset;  /* Hz from the peak row's bin (0 without interpolation)   */
    float peak_to_noise;
    int32_t reserved;
} fmdbzp_prn_result;

/*
 * Evaluate the result formulas over the statistics of a call, on the host.
 * `interpolate` != 0: a parabola through the code (Doppler) neighbours where
 * the larger one exceeds sqrt(noise). FMDBZP_EINVAL on a null pointer or
 * non-positive sizes.
 */
int fmdbzp_prn_results(const fmdbzp_prn_stats* stats, int32_t n, int32_t samples_per_code, int32_t num_blocks,
                       int32_t block_size, double sampling_freq_hz, double code_freq_hz, double code_length,
                       double coherent_time_s, double doppler_spacing_hz, int32_t interpolate,
                       fmdbzp_prn_result* out);

/*
 * One request of a batch: the arguments of fmdbzp_acquire. `nprn` PRN
 * indices of `plan` searched over `signal`.
 */
typedef struct fmdbzp_request {
    fmdbzp_plan* plan;
    const void* signal;
    int32_t eltype;
    int32_t nprn;
    int64_t n_samples;
    double interm_freq_hz;
    const int32_t* prn_index;
    uint32_t flags;
    uint32_t reserved;
    fmdbzp_prn_stats* out_stats;
    float* const* out_surfaces;
} fmdbzp_request;

/*
 * Run `nreqs` searches of possibly different plans (geometry, system, sample
 * rate, Doppler span, PRN count, N_nc) as one submission: every request is
 * enqueued on its plan's stream with no host synchronisation in between, so
 * requests on different plans run concurrently on the device, and the call
 * returns when all have finished. No counterpart in the reference, which runs
 * one `acquire!` per plan (the batched uneven mix is a sequence of `acquire!`
 * calls there). A plan listed twice runs its requests in order.
 */
int fmdbzp_acquire_batch(const fmdbzp_request* reqs, int32_t nreqs);

/*
 * fmdbzp_acquire without any allocation. No counterpart in the reference: for
 * callers that cannot allocate device or host memory during a search (code
 * under HIP graph capture, tight serving loops, harnesses that forbid
 * hipMalloc). The search and its results are those of fmdbzp_acquire on the
 * same plan and samples. Differences:
 *  - `signal` must be device memory (no host staging), and no surfaces are
 *    returned;
 *  - every buffer beyond the inputs and outputs (signal FFT cache, PRN list,
 *    tile, accumulator, reductions, statistics) lives in one file-scope
 *    device array of FMDBZP_NOALLOC_SCRATCH_BYTES per device, held until the
 *    process ends; PRNs run in batches that fit it, and a search whose
 *    signal FFTs plus one PRN's tile and accumulator exceed it is rejected
 *    with FMDBZP_EINVAL (the message gives the bytes it needs);
 *  - calls on one device share that array and are serialised by a lock held
 *    until each call has synchronised (overlapping calls would race on it);
 *  - no kernel timing is recorded. Synchronous.
 */
#define FMDBZP_NOALLOC_SCRATCH_BYTES (128u << 20)
int fmdbzp_acquire_noalloc(fmdbzp_plan* plan,
                           const void* signal,
                           int32_t eltype,
                           int64_t n_samples,
                           double interm_freq_hz,
                           const int32_t* prn_index,
                           int32_t nreq,
                           fmdbzp_prn_stats* out_stats);

/* Release every device allocation of the plan. NULL is accepted. */
int fmdbzp_plan_destroy(fmdbzp_plan* plan);

/* Thread-local text of the last error ("" when none). */
const char* fmdbzp_last_error(void);

/* Device and build facts: writes a NUL-terminated string into buf. */
int fmdbzp_query(char* buf, size_t buflen);

/*
 * Optional per-kernel timing for measurement: when enabled, the plan records
 * HIP events around every kernel launch on its own stream and accumulates the
 * elapsed time per kernel class. fmdbzp_plan_kernel_times fills up to `n`
 * entries of total milliseconds and launch counts, in the order of
 * enum fmdbzp_kernel_class, and returns the number of classes.
 */
enum fmdbzp_kernel_class {
    FMDBZP_K_CODE_FFT = 0,    /* plan-time conj code FFTs                 */
    FMDBZP_K_SIGNAL_FFT = 1,  /* downconvert + signal double-block FFTs   */
    FMDBZP_K_CORR_TILE = 2,   /* block correlation: multiply + inverse FFT */
    FMDBZP_K_COLUMN = 3,      /* column Doppler FFT / sign search + accumulate, or
                                 the whole full-period correlation of a call   */
    FMDBZP_K_REDUCE = 4,      /* per-row sums and peak candidates          */
    FMDBZP_K_FINALIZE = 5,    /* per-PRN peak, noise, neighbours           */
    FMDBZP_K_EXPORT = 6,      /* surface transpose for store_power_bins    */
    FMDBZP_K_NUM_CLASSES = 7
};
int fmdbzp_plan_set_timing(fmdbzp_plan* plan, int32_t enable);
/* The autotuner's record for the plan (choice and measured candidates; ""
 * when it did not run). */
int fmdbzp_plan_tuning(fmdbzp_plan* plan, char* buf, size_t buflen);
/* Graphs captured and replayed by a FMDBZP_OPT_GRAPH plan so far. */
int fmdbzp_plan_graph_counts(fmdbzp_plan* plan, int64_t* captures, int64_t* replays);
/* Form of the column stage that the plan selects on the coherent tile (the
 * column Doppler transforms, sign or rotation search and accumulation), by the
 * name of a kernel, e.g. "k_column_rotmma<8,3,20>". A form keeps its name where
 * a later kernel serves part of its geometries: k_column_rot2000 and
 * k_column_rotbig are also the forms of the searches that k_column_rot25 runs.
 * fmdbzp_plan_call_kernels names the kernels themselves. No counterpart in the
 * reference (which has one CPU implementation); for tests and reports. */
int fmdbzp_plan_column_kernel(fmdbzp_plan* plan, char* buf, size_t buflen);
/* Kernels that a call of fmdbzp_acquire with these samples, PRN count and flags
 * launches for the search: the full-period correlation ("k_full31_corr<512>"),
 * or the block correlation and the column kernel, separated by a space
 * ("k_corr_tile<1,true,2500> k_column_rot25<80>"; ",fp16" with an FP16 tile).
 * No counterpart in the reference; for tests and reports. */
int fmdbzp_plan_call_kernels(fmdbzp_plan* plan, int32_t eltype, int32_t nreq, uint32_t flags, char* buf,
                             size_t buflen);
/* Form of the full-period correlation that a statistics-only FP32 call over
 * nprn PRNs runs, on a simple-path plan of those PRNs; host only, for cost models.
 * FMDBZP_FULL_NONE: the tile. It depends on the factors of the code period, not
 * on the FFT size. 31-axis: 31 a b samples, a and b coprime radices of its
 * stages, up to 16384 samples: of the multiples of 1023 the 2, 3, 4, 5, 6, 8, 10
 * and 16 fold. Radices: no prime factor above 13, up to 20480 samples.
 * FMDBZP_EINVAL on a non-positive size. */
enum fmdbzp_full_form {
    FMDBZP_FULL_NONE = 0,
    FMDBZP_FULL_RADIX = 1,
    FMDBZP_FULL_AXIS31 = 2
};
int fmdbzp_full_period_form(int32_t samples_per_code, int32_t num_blocks, int32_t num_coh, int32_t num_noncoherent,
                            int32_t nprn);
int fmdbzp_plan_kernel_times(fmdbzp_plan* plan, double* total_ms, int64_t* launches, int32_t n);

/*
 * Layout of the surfaces that FMDBZP_FLAG_STORE_SURFACES returns (the plot
 * recipe's input, src/plot.jl:35-57; src/acquire.jl:221-228 stores them).
 * nbins = 0 (default): the reference's (ndop, spc_eff) surface, rows in
 * sorted-Doppler order, columns in scrambled FM-DBZP order. nbins in [1, spc]:
 * a chip-ordered (ndop, nbins) surface, reduced on the device. chip_order
 * holds the spc code columns in ascending code phase
 * (mod(-tau f_code / fs, spc f_code / fs) of `_fmdbzp_sort_by_chip`, a stable
 * order), and bin b is the maximum over columns chip_order[b spc / nbins ..
 * (b + 1) spc / nbins) and over the R rotation slices of each. With nbins =
 * spc and R = 1 it is the reference's chip-sorted surface itself. A 25 MHz
 * E1-like surface is 20 GB; 8184 bins (two per chip) are 65 MB.
 */
int fmdbzp_plan_set_surface_layout(fmdbzp_plan* plan, int32_t nbins, const int32_t* chip_order);

/*
 * Secondary-code phase of detected PRNs on the device: the replacement for
 * `_estimate_secondary_code_phase` (src/acquire.jl:503-538), called by the
 * result extraction for each PRN whose peak-to-noise ratio passes
 * cfar_threshold(0.01, ndop spc R) (src/acquire.jl:646-652). Each request
 * despreads the first L code periods of `signal` at its estimated Doppler
 * (carrier interm_freq_hz + doppler_hz at the plan's sampling rate) with
 * `code` (spc samples of gen_code at the estimated code phase), in the
 * reference's order of operations, and returns the rotation r in [0, L) whose
 * sum over periods of secondary[(k + r) mod L] z_k has the largest |.|^2
 * (first one on ties). The signal is in device memory with
 * FMDBZP_FLAG_DEVICE_SIGNAL, else on the host (its first L spc samples are
 * copied). Synchronous.
 */
typedef struct fmdbzp_secondary_request {
    const int8_t* code;       /* spc samples, +-1 (host) */
    const int8_t* secondary;  /* num_rotations secondary chips, +-1 (host) */
    double doppler_hz;
    int32_t num_rotations;    /* L, 1..64 */
    int32_t reserved;
} fmdbzp_secondary_request;
int fmdbzp_secondary_phase(fmdbzp_plan* plan, const void* signal, int32_t eltype, int64_t n_samples,
                           double interm_freq_hz, uint32_t flags, const fmdbzp_secondary_request* reqs,
                           int32_t nreq, int32_t* out_phase);

/* --------------------------------------------------------------------------
 * Seeded synthetic signals generated on the device: the analogue of
 * `generate_test_signal` (src/generate_test_signal.jl:32-82) for benchmark
 * scenes of many emitters. Samples are noise plus the emitters' terms, added
 * in emitter order, each evaluated in FP64:
 *   pos   = code_phase_chips + (n * code_freq_hz) / sampling_freq_hz,  c = floor(pos)
 *   chip  = chips[c mod code_length]
 *           (* -1 where pos - c >= 1/2, when boc != 0)
 *           (* secondary[(floor(c / code_length) + secondary_phase) mod secondary_length])
 *           (* bits[min((floor(n * 1000 / sampling_freq_hz) + bit_edge_ms) / bit_ms,
 *                       num_bits - 1)], bit_edge_ms >= 0)
 *   angle = (2 pi carrier_hz) * n / sampling_freq_hz + carrier_phase
 *   real scenes:    x += (amplitude * chip) * cos(angle)
 *   complex scenes: x += (amplitude * chip) * (cos(angle) + i sin(angle))
 * Noise is Philox4x32-10 (key = seed, counter = (block, noise_stream, 0)) with
 * Box-Muller in FP64, one counter block per complex sample or per pair of
 * real samples, times noise_scale. Output: FMDBZP_CF32 (complex scenes),
 * FMDBZP_I16 (real; round half to even, saturated) or FMDBZP_F32 (real).
 * The same samples, up to the last bit of log / sqrt / cos / sin, come from
 * the host generator in acquisition.signals (render_host).
 * fmdbzp_synthesize rejects (FMDBZP_EINVAL, before any device work) null pointers, non-positive
 * sizes, an output type that does not fit the scene, and tables holding
 * values other than +-1.
 * -------------------------------------------------------------------------- */
typedef struct fmdbzp_emitter {
    const int8_t* chips;      /* primary code, +-1, code_length entries (host) */
    int32_t code_length;
    int32_t boc;              /* 1: BOC(1,1) square subcarrier */
    const int8_t* secondary;  /* +-1 per primary period, or NULL */
    int32_t secondary_length;
    int32_t secondary_phase;
    const int8_t* bits;       /* +-1 data bits, or NULL */
    int32_t num_bits;
    int32_t bit_ms;           /* data bit length in whole ms */
    int32_t bit_edge_ms;
    int32_t reserved;
    double amplitude;
    double code_freq_hz;      /* including code Doppler */
    double code_phase_chips;
    double carrier_hz;        /* IF + Doppler */
    double carrier_phase;
} fmdbzp_emitter;

typedef struct fmdbzp_scene {
    int64_t n_samples;
    double sampling_freq_hz;
    int32_t complex_samples;  /* 0: real IF samples, 1: complex baseband */
    int32_t out_eltype;       /* FMDBZP_CF32 (complex); FMDBZP_I16 or FMDBZP_F32 (real) */
    double noise_scale;
    uint64_t seed;
    uint32_t noise_stream;
    int32_t reserved;
} fmdbzp_scene;

/* Write scene->n_samples samples into `out` (device memory of the current
 * device, sized for out_eltype). Synchronous. */
int fmdbzp_synthesize(const fmdbzp_scene* scene, const fmdbzp_emitter* emitters, int32_t n_emitters,
                      void* out);

#ifdef __cplusplus
}
#endif

#endif /* FMDBZP_H */
