// fmdbzp.hip — C ABI of the MI355X FM-DBZP acquisition engine.
//
// One device-resident plan per `plan_acquire` (src/plan.jl:312-697) and one
// `fmdbzp_acquire` per `acquire!` (src/acquire.jl:54-215). A call runs, on
// the plan's own HIP stream:
//   1. k_signal_fft     downconvert + double-block FFTs for all N_nc segments
//   2. per PRN batch, per step: k_corr_tile -> k_column_{simple,sign,rotation}
//   3. per PRN batch: k_reduce_rows -> k_finalize (-> k_export when surfaces
//      are requested)
// and copies the per-PRN statistics back. PRN batches bound the workspace
// (tile + accumulator) to a budget; the reference bounds its CPU footprint
// the same way with a scratch slot per thread (src/plan.jl:574-608).
#include <hip/hip_runtime.h>
#include <stdarg.h>
#include <stdint.h>
#include <stdio.h>
#include <stdlib.h>
#include <string.h>
#include <math.h>
#include <cmath>
#include <algorithm>
#include <mutex>
#include <string>
#include <vector>

#include "../../include/fmdbzp.h"
#include "kernels.hpp"
#include "full_corr.hpp"
#include "synth.hpp"

namespace {

thread_local std::string g_err;

int set_err(int code, const char* fmt, ...) __attribute__((format(printf, 2, 3)));
int set_err(int code, const char* fmt, ...)
{
    char buf[1024];
    va_list ap;
    va_start(ap, fmt);
    vsnprintf(buf, sizeof(buf), fmt, ap);
    va_end(ap);
    g_err = buf;
    return code;
}

#define HIP_TRY(expr)                                                                     \
    do {                                                                                  \
        hipError_t e_ = (expr);                                                           \
        if (e_ != hipSuccess)                                                             \
            return set_err(e_ == hipErrorOutOfMemory ? FMDBZP_ENOMEM : FMDBZP_EHIP,       \
                           "%s failed: %s (%s:%d)", #expr, hipGetErrorString(e_),         \
                           __FILE__, __LINE__);                                           \
    } while (0)

// exp(-2 pi i m / n) in FP64 with exact values at multiples of pi/2.
void sincospi_d(double x, double* s, double* c)
{
    double r = x - 2.0 * nearbyint(x * 0.5);
    double sgn_c = 1.0;
    if (r > 0.5) { r = 1.0 - r; sgn_c = -1.0; }
    else if (r < -0.5) { r = -1.0 - r; sgn_c = -1.0; }
    double ar = fabs(r), ss, cc;
    if (ar <= 0.25) { ss = sin(M_PI * ar); cc = cos(M_PI * ar); }
    else { double t = 0.5 - ar; ss = cos(M_PI * t); cc = sin(M_PI * t); }
    if (r < 0) ss = -ss;
    *s = ss;
    *c = sgn_c * cc;
}

std::vector<float2> twiddles(int n)
{
    std::vector<float2> tw((size_t)n);
    for (int m = 0; m < n; m++) {
        double s, c;
        sincospi_d(2.0 * (double)m / (double)n, &s, &c);
        tw[(size_t)m] = make_float2((float)c, (float)(-s));
    }
    return tw;
}

// Radix sequence of an n-point transform: 16s (when allowed), then 8, 4, 2,
// 5, 3, then any larger prime.
int make_fft_plan(int n, FftPlanDev* p, bool radix16)
{
    p->n = n;
    p->nst = 0;
    int m = n;
    auto push = [&](int r) {
        if (p->nst >= FFT_MAX_STAGES) return false;
        p->radix[p->nst++] = r;
        return true;
    };
    if (radix16)
        while (m % 16 == 0) { if (!push(16)) return -1; m /= 16; }
    while (m % 8 == 0) { if (!push(8)) return -1; m /= 8; }
    while (m % 4 == 0) { if (!push(4)) return -1; m /= 4; }
    while (m % 2 == 0) { if (!push(2)) return -1; m /= 2; }
    while (m % 5 == 0) { if (!push(5)) return -1; m /= 5; }
    while (m % 3 == 0) { if (!push(3)) return -1; m /= 3; }
    for (int f = 7; m > 1; f += 2)
        while (m % f == 0) { if (!push(f)) return -1; m /= f; }
    return 0;
}

// Radices 10, then 5 (the row transforms of the four-step rotation kernel);
// -1 when another factor remains.
int make_row_plan(int n, FftPlanDev* p)
{
    p->n = n;
    p->nst = 0;
    int m = n;
    for (int r : {10, 5})
        while (m % r == 0) {
            if (p->nst >= FFT_MAX_STAGES) return -1;
            p->radix[p->nst++] = r;
            m /= r;
        }
    return m == 1 ? 0 : -1;
}

constexpr size_t kLdsMax = 160 * 1024;   // gfx950 LDS per workgroup

// Radix sequence of the full-period transform (full_corr.hpp) of n points: the
// cheapest ordered product of its radices under a per-point cost of the
// butterflies and of each further pass (twiddle, addresses, LDS, barrier),
// with a stage's cost scaled up to whole waves on the four SIMDs. The first
// radix is odd unless n is a power of two (bank spread); with one noncoherent
// step 25 may run first and 20 and 22 in the middle, else at most 16. false: n has a
// prime factor above 13, more than FC_MAX_STAGES stages, or fewer than two.
bool make_full_plan(int n, int nthr, bool multi, FullPlanDev* f)
{
    struct Radix {
        int r;
        double cost;
    };
    static const Radix kRadix[] = {{2, 2},     {3, 5.3},   {4, 4},     {5, 6.4},   {6, 7.3},   {7, 9},
                                   {8, 6.5},   {9, 12.4},  {10, 8.4},  {11, 14},   {12, 9.3},  {13, 16},
                                   {15, 11.7}, {16, 10.5}, {20, 10.4}, {22, 16},   {25, 15.4}};
    if (n < 64) return false;
    const bool pow2 = (n & (n - 1)) == 0;
    auto admitted = [&](const Radix& x, int left, int depth) {
        if (left % x.r != 0) return false;
        if (x.r > 16 && (multi || (depth == 0 ? x.r != 25 : x.r > 22))) return false;
        if (depth == 0 && !pow2 && x.r % 2 == 0) return false;
        // the last stage: at most FC_CELLS outputs per thread
        return left != x.r || (depth > 0 && x.r <= 16 && n / x.r <= FC_CELLS / x.r * nthr);
    };
    auto cost = [&](const Radix& x) {
        const int waves = (n / x.r + 63) / 64;
        const double fill = (double)((waves + 3) / 4 * 4 * 64) * x.r / n;
        return (x.cost + 16.0) * std::min(fill, 4.0);
    };
    // Least cost of the stages from `depth` on, once per divisor, then the first
    // sequence of that cost. Trying every sequence took 0.84 ms at 20160 points
    // and 55 us at 16384, this 35 and 4 us.
    std::vector<std::pair<int, double>> memo[FC_MAX_STAGES];
    auto rest = [&](auto&& self, int left, int depth) -> double {
        if (left == 1) return 0.0;
        if (depth == FC_MAX_STAGES) return 1e30;
        for (const auto& m : memo[depth])
            if (m.first == left) return m.second;
        double least = 1e30;
        for (const Radix& x : kRadix)
            if (admitted(x, left, depth)) least = std::min(least, cost(x) + self(self, left / x.r, depth + 1));
        memo[depth].push_back({left, least});
        return least;
    };
    const double least = rest(rest, n, 0) + 1e-9;
    if (least > 1e29) return false;
    std::vector<int> best, cur;
    double best_cost = 1e30;
    auto search = [&](auto&& self, int left, double sum) -> void {
        if (left == 1) {
            if (sum < best_cost) {
                best = cur;
                best_cost = sum;
            }
            return;
        }
        if ((int)cur.size() == FC_MAX_STAGES) return;
        for (const Radix& x : kRadix) {
            if (!admitted(x, left, (int)cur.size())) continue;
            const double c = sum + cost(x);
            cur.push_back(x.r);
            if (c + rest(rest, left / x.r, (int)cur.size()) <= least) self(self, left / x.r, c);
            cur.pop_back();
        }
    };
    search(search, n, 0.0);
    if (best.empty()) return false;
    *f = FullPlanDev{};
    f->n = n;
    f->nst = (int)best.size();
    f->pad_shift = 31;
    if (best[0] % 2 == 0) f->pad_shift = __builtin_ctz((unsigned)best[0]);
    int ns = 1, at = 0;
    for (int t = 0; t < f->nst; t++) {
        const int R = best[(size_t)t];
        f->radix[t] = R;
        f->ns[t] = ns;
        f->inv_ns[t] = 1.0f / (float)ns;
        f->twoff[t] = at;
        if (t > 0) at += (R - 1) * ns;
        ns *= R;
    }
    return true;
}

// k_corr_tile variants: transforms per pass and LDS transform buffers
static int corr_nt(int v)
{
    switch (v) {
    case 2: case 3: case 5: case 8: return 2;
    case 6: return 10;
    case 7: return 5;
    default: return 1;
    }
}
static int corr_nbuf(int v)
{
    switch (v) {
    case 1: case 4: case 9: return 1;
    case 6: return 10;
    case 7: return 5;
    default: return 2;  // two transforms per pass, or the ping-pong pair
    }
}

// Axes of the 31 x rb x rc transform of n points (full_corr.hpp): pairwise
// coprime, radices of its switches, the widest c axis (the fewest last-stage
// butterflies). rc is odd but for 22 = 2 mod 4, which spreads its stride over
// the banks; pk = 4 mod 8 does so for the four row groups that a
// wave stores from the matrix products.
bool make_full31_plan(int n, Full31Dev* f)
{
    if (n % 31 != 0 || (n / 31) % 31 == 0) return false;
    const int m = n / 31;
    bool found = false;
    for (int rb = 2; rb <= 24; rb++) {
        if (m % rb != 0 || !fc31_b_ok(rb) || !fc31_c_ok(m / rb)) continue;
        const int rc = m / rb;
        int a = rb, b = rc;
        while (b) {
            const int t = a % b;
            a = b;
            b = t;
        }
        if (a != 1) continue;
        if (found && rc <= f->rc) continue;
        *f = Full31Dev{n, m, rb, rc, rc, 0, 1.0f / (float)rb, 1.0f / (float)rc};
        f->pk = m + 1 + ((4 - (m + 1) % 8) + 8) % 8;  // at least one spare slot per row
        found = true;
    }
    return found;
}

constexpr size_t kLdsDefault = 64 * 1024;
// bytes of one row's partial of a column-major reduction chunk (FP64 sum, key, value)
constexpr size_t kRedPart = sizeof(double) + sizeof(uint64_t) + sizeof(float);

struct TimedEvent {
    int cls;
    hipEvent_t start, stop;
};

}  // namespace

// PRN lanes: a batch of PRNs can be split over up to kLanes streams, so the
// block correlation of one lane overlaps the column stage of the other.
// FMDBZP_LANES sets the count (default 1): on the 32-PRN L1 C/A workload two
// lanes gain under 1%, as each kernel runs about half as fast while they
// overlap (they compete for the same CU slots), and per-launch timings then
// include the other lane's work.
constexpr int kLanes = 2;

static int lanes_requested()
{
    const char* s = getenv("FMDBZP_LANES");
    const int n = s ? atoi(s) : 1;
    return n < 1 ? 1 : (n > kLanes ? kLanes : n);
}

struct fmdbzp_plan {
    std::mutex mu;
    int device = 0;
    hipStream_t stream = nullptr;
    hipStream_t lane[kLanes] = {};
    hipEvent_t ev_fork = nullptr;
    hipEvent_t ev_join[kLanes] = {};
    int nlanes = 1;
    fmdbzp_plan_desc d{};
    int nprn = 0;
    int nsets = 0;
    FftPlanDev pf{}, pd{};
    FftPlanDev pf8{};  // F-point plan without radix 16 (forward signal / code FFTs: fewer live inputs per thread)
    float2* d_twF = nullptr;
    float2* d_twD = nullptr;
    char* d_arena = nullptr;     // one allocation: code FFTs, signal FFTs, tiles, accumulator, code spectra
    float2* d_prnconj = nullptr;
    float* d_patterns = nullptr;
    int32_t* d_pset = nullptr;
    int32_t* d_shifts = nullptr;
    // workspace
    void* d_signal = nullptr;
    size_t signal_cap = 0;
    int8_t* d_codes = nullptr;   // code samples, during creation
    float2* d_sigfft = nullptr;
    float2* d_tile = nullptr;
    float2* d_tile2 = nullptr;   // second step's tile of a two-step column launch (col_pair)
    float* d_acc = nullptr;
    double* d_rowsum = nullptr;
    float* d_rowbest_v = nullptr;
    uint64_t* d_rowbest_k = nullptr;
    // column-major accumulator (few columns per column-stage workgroup): the
    // row reduction runs over column chunks of red_cw, partials per chunk in
    // the consumed tile
    bool acc_cm = false;
    int apc = 0;             // column pitch (ndop rounded up to 32)
    size_t acc_ps = 0;       // accumulator elements per PRN
    int red_cw = 0, red_nchunk = 0;
    double* d_psum = nullptr;
    float* d_pbest_v = nullptr;
    uint64_t* d_pbest_k = nullptr;
    int32_t* d_req = nullptr;
    size_t req_cap = 0;
    int req_n = 0;           // entries of d_req that hold the last uploaded request list (h_req)
    fmdbzp_prn_stats* d_stats = nullptr;
    // pinned host staging, so copies stay asynchronous to the host
    int32_t* h_req = nullptr;
    fmdbzp_prn_stats* h_stats = nullptr;
    void* h_signal = nullptr;
    size_t h_signal_cap = 0;
    // the request whose statistics are staged in h_stats, not yet returned
    fmdbzp_prn_stats* pending_out = nullptr;
    int32_t pending_n = 0;
    float* d_export = nullptr;  // one staging surface per lane (ndop x surface columns)
    int surf_bins = 0;          // 0: scrambled (ndop, spc_eff) surfaces; > 0: chip-ordered (ndop, surf_bins)
    int32_t* d_chip_order = nullptr;  // [spc] code columns in ascending code phase
    char* d_sec = nullptr;            // secondary-phase requests: codes, chips, descriptors, results
    size_t sec_cap = 0;
    int batch = 1;
    int LB = 1, bstride = 1, sst = 1;
    bool simple_kernel = false;  // column stage runs k_column_simple
    int tp = 0, ap = 0;          // tile / accumulator row pitches (multiples of 32 elements)
    bool col_onebuf = false;     // simple column kernel runs its FFT stages in place
    bool col_static = false;     // simple column kernel uses the compile-time ndop = 160 transform
    // k_column_c160_pair: steps s and s + 1 in one launch where no row's drift
    // shift changes by more than one column between them (pair_ok[s])
    bool col_pair = false;
    std::vector<uint8_t> pair_ok;
    size_t col_lds2 = 0;
    // block correlation on the in-place transforms of full_corr.hpp (corr_variant 10)
    FullPlanDev fc{};
    int fc_nthr = 0;
    size_t fc_lds = 0;
    float2* d_fc_tw = nullptr;
    // full-period correlation (full_corr.hpp): statistics-only calls of simple plans
    bool full = false;
    FullPlanDev fp{};
    Full31Dev fp31{};                // the chip-rate multiples' form (fp31.n != 0)
    int full_nthr = 0;
    size_t full_lds = 0;
    float2* d_full_tw = nullptr;
    float2* d_full_code = nullptr;   // [nprn][ndop][spc] code spectra
    uint16_t* d_full_map = nullptr;  // [spc] column of delay tau
    bool tile_half = false;      // FMDBZP_PREC_TILE_FP16: FP16 coherent tile
    bool tile_auto = false;      // FMDBZP_PREC_AUTO on a plan that admits the FP16 tile: per call, by sample type
    bool rot_direct = false;     // rotation kernel writes transform outputs straight to the accumulator
    bool col_reg = false;        // simple path, few Doppler rows: k_column_reg
    bool bitsplit = false;       // data-bit search of two 20-period bits: k_column_bitsplit
    int rotsplit = 0;            // direct rotation, few Doppler rows: columns per workgroup of k_column_rotsplit
    // accumulator layout and size that fmdbzp_acquire_noalloc's limit counts
    bool lim_cm = false;
    size_t lim_acc_ps = 0;
    bool rot25 = false;          // 25 periods of 50, 80, 100, 250 or 500 rows: k_column_rot25
    bool rot2000 = false;        // direct rotation at ndop 2000: compile-time kernel, one column per workgroup
    // Direct rotation at large ndop (k_column_rotbig), accumulated in code-column
    // chunks: every chunk owns chunk_cols scrambled code columns (the last one
    // fewer) and holds a window of them plus one halo column on each side (no
    // halo when one chunk covers the code period); per step the tile holds the
    // column blocks whose drifted cells reach the window.
    int rotbig = 0;              // 0: off; else k_column_rotbig's thread count
    FftPlanDev prow{};           // its nb-point row transform
    float2* d_twR = nullptr;     // its row twiddles W_nb^j, j < nb
    int rgrp = 1;                // rows a wave transforms together
    int rotbig_nt = 256;
    int rotmma = 0;              // FMDBZP_PREC_MFMA: k_column_rotmma's n1 (nb = 25 n1) in place of k_column_rotbig
    int chunk_cols = 0, nchunks = 0, halo = 0, win_max = 0;
    int nrb_max = 0;             // tile blocks per PRN
    int nsub = 0, nparts = 0;    // reduction parts per (chunk, slice) and per PRN
    std::vector<int> smin, smax; // signed drift range per step
    float4* d_pnbr = nullptr;    // chunk partials: best cell's neighbours
    float4* d_rownbr = nullptr;
    double* d_colsum = nullptr;  // GlobalMean: FP64 sum over rows per effective column
    int corr_variant = 0;        // 10 = k_corr_fc; k_corr_tile: 6-9 = compile-time F = 400, 800, 2000, 4000,
                                 // 5 = compile-time F = 500, 4 = compile-time F = 2500,
                                 // 3 = compile-time F = 2048, 2 = two in-place transforms per
                                 // pass, 1 = one, 0 = ping-pong
    size_t col_lds = 0;
    int split_wgs = 2048;        // correlation grids below this many workgroups split their passes
    std::string tuning;          // autotuner record (FMDBZP_OPT_AUTOTUNE)
    size_t fft_lds = 0;
    size_t corr_lds = 0;
    float inv_f = 0.f;
    float pscale = 1.f;          // factor in the conj code spectra (1/F when F is a power of two)
    float tile_scale = 0.f;      // factor the block correlation applies (1/F otherwise)
    // hipGraph of the last call's launch sequence (FMDBZP_OPT_GRAPH): replayed
    // while calls repeat its signal pointer, sample type, IF, flags and PRN list
    bool use_graph = false;
    hipGraph_t graph = nullptr;
    hipGraphExec_t graph_exec = nullptr;
    const void* g_sig = nullptr;
    const int32_t* g_req = nullptr;
    const fmdbzp_prn_stats* g_stats = nullptr;
    int32_t g_eltype = -1, g_nreq = 0;
    uint32_t g_flags = 0;
    double g_if = 0.0;
    std::vector<int32_t> g_prns;
    int64_t graph_captures = 0, graph_replays = 0;
    // timing
    bool timing = false;
    std::vector<TimedEvent> pending;
    std::vector<hipEvent_t> pool;
    double tot_ms[FMDBZP_K_NUM_CLASSES] = {};
    int64_t launches[FMDBZP_K_NUM_CLASSES] = {};
};

namespace {

// LDS of the block-correlation variant v.
size_t corr_lds_of(const fmdbzp_plan* P, int v)
{
    if (v == 10) return P->fc_lds;
    return ((size_t)P->d.fft_size + (size_t)corr_nbuf(v) * fft_lds_span(P->d.fft_size)) * sizeof(float2);
}

int acquire_finish(fmdbzp_plan* P);
int autotune(fmdbzp_plan* P);
size_t workspace_budget();

size_t elsize(int eltype)
{
    switch (eltype) {
    case FMDBZP_CF32: return 8;
    case FMDBZP_CF64: return 16;
    case FMDBZP_I16: return 2;
    case FMDBZP_CI8: return 2;
    case FMDBZP_CI16: return 4;
    case FMDBZP_F32: return 4;
    case FMDBZP_F64: return 8;
    default: return 0;  // FMDBZP_C2BIT is sized in signal_bytes()
    }
}

hipEvent_t get_event(fmdbzp_plan* P)
{
    if (!P->pool.empty()) {
        hipEvent_t e = P->pool.back();
        P->pool.pop_back();
        return e;
    }
    hipEvent_t e = nullptr;
    if (hipEventCreate(&e) != hipSuccess) return nullptr;
    return e;
}

// Launch bracket: records HIP events on the launch's stream when timing is on.
// When two lanes run at once, a launch's interval also covers the other
// lane's work that overlaps it.
struct Timed {
    fmdbzp_plan* P;
    hipStream_t st;
    TimedEvent ev{};
    bool on;
    Timed(fmdbzp_plan* p, int cls, hipStream_t stream, bool enable = true)
        : P(p), st(stream), on(enable && p->timing)
    {
        if (on) {
            ev.cls = cls;
            ev.start = get_event(P);
            ev.stop = get_event(P);
            if (!ev.start || !ev.stop) on = false;
            else hipEventRecord(ev.start, st);
        }
    }
    ~Timed()
    {
        if (on) {
            hipEventRecord(ev.stop, st);
            P->pending.push_back(ev);
        }
    }
};

void collect_timing(fmdbzp_plan* P)
{
    for (auto& e : P->pending) {
        float ms = 0.f;
        if (hipEventElapsedTime(&ms, e.start, e.stop) == hipSuccess) {
            P->tot_ms[e.cls] += ms;
            P->launches[e.cls] += 1;
        }
        P->pool.push_back(e.start);
        P->pool.push_back(e.stop);
    }
    P->pending.clear();
}

int validate_desc(const fmdbzp_plan_desc* d)
{
    if (d->abi_version != FMDBZP_ABI_VERSION)
        return set_err(FMDBZP_EINVAL, "abi_version %d != %d", d->abi_version, FMDBZP_ABI_VERSION);
    if (d->samples_per_code <= 0 || d->num_blocks <= 0 || d->block_size <= 0 || d->fft_size <= 0 ||
        d->num_coh <= 0 || d->num_data_bits <= 0 || d->bit_edge_search_steps <= 0 ||
        d->num_noncoherent <= 0 || d->num_secondary_rotations <= 0 || d->num_doppler_bins <= 0 ||
        d->num_patterns <= 0)
        return set_err(FMDBZP_EINVAL, "descriptor has a non-positive size");
    if ((int64_t)d->num_blocks * d->block_size != d->samples_per_code)
        return set_err(FMDBZP_EINVAL, "num_blocks * block_size != samples_per_code");
    if ((int64_t)d->num_coh * d->num_blocks != d->num_doppler_bins)
        return set_err(FMDBZP_EINVAL, "num_doppler_bins != num_coh * num_blocks");
    if (d->fft_size < 2 * d->block_size)
        return set_err(FMDBZP_EINVAL, "fft_size %d < 2 * block_size %d", d->fft_size, d->block_size);
    if ((int64_t)d->samples_per_code * d->num_secondary_rotations != d->samples_per_code_eff)
        return set_err(FMDBZP_EINVAL, "samples_per_code_eff != samples_per_code * rotations");
    if (d->num_coh % d->num_data_bits != 0)
        return set_err(FMDBZP_EINVAL, "num_coh %% num_data_bits != 0");
    if (d->num_data_bits > 30) return set_err(FMDBZP_EINVAL, "num_data_bits too large");
    if (d->path < 0 || d->path > 2) return set_err(FMDBZP_EINVAL, "bad path %d", d->path);
    if (d->path == FMDBZP_PATH_ROTATION &&
        d->num_patterns != (1 << (d->num_data_bits - 1)) * d->num_secondary_rotations)
        return set_err(FMDBZP_EINVAL, "rotation path needs Q = 2^(N_db-1) * R patterns");
    if (d->path == FMDBZP_PATH_ROTATION && d->num_coh > 256)
        return set_err(FMDBZP_EINVAL, "rotation path supports num_coh <= 256");
    if (d->path == FMDBZP_PATH_SIGN && d->num_patterns != (1 << (d->num_data_bits - 1)))
        return set_err(FMDBZP_EINVAL, "sign path needs Q = 2^(N_db-1) patterns");
    if (d->path != FMDBZP_PATH_ROTATION && d->num_secondary_rotations != 1)
        return set_err(FMDBZP_EINVAL, "rotations > 1 only on the rotation path");
    if (d->noise_estimator != FMDBZP_NOISE_OPPOSITE_ROW && d->noise_estimator != FMDBZP_NOISE_GLOBAL_MEAN)
        return set_err(FMDBZP_EINVAL, "bad noise estimator %d", d->noise_estimator);
    if (d->precision != FMDBZP_PREC_FP32 && d->precision != FMDBZP_PREC_TILE_FP16 && d->precision != FMDBZP_PREC_AUTO &&
        d->precision != FMDBZP_PREC_MFMA)
        return set_err(FMDBZP_EINVAL, "unsupported precision %d", d->precision);
    if (d->sampling_freq_hz <= 0) return set_err(FMDBZP_EINVAL, "sampling_freq_hz <= 0");
    // LDS: the F-point transforms need two F-entry buffers in one workgroup
    if (((size_t)2 * fft_lds_span(d->fft_size) + d->fft_size) * sizeof(float2) > kLdsMax)
        return set_err(FMDBZP_EINVAL, "fft_size %d exceeds the LDS transform limit", d->fft_size);
    // the column stage needs three ndop-entry complex buffers + two float rows,
    // except the direct rotation search, whose large-ndop kernel needs one
    // buffer (checked with its radix plan at plan creation)
    const bool direct_rot = d->path == FMDBZP_PATH_ROTATION && d->num_data_bits == 1 &&
                            d->bit_edge_search_steps == 1 && d->num_doppler_bins % 2 == 0;
    if (!direct_rot &&
        (size_t)(fft_lds_span(d->num_doppler_bins) | 1) * 24 + (size_t)(d->num_doppler_bins | 1) * 12 > kLdsMax)
        return set_err(FMDBZP_EINVAL, "num_doppler_bins %d exceeds the LDS column limit", d->num_doppler_bins);
    if (direct_rot && (size_t)fft_lds_span(d->num_doppler_bins) * 8 + 256 > kLdsMax)
        return set_err(FMDBZP_EINVAL, "num_doppler_bins %d exceeds the LDS column limit", d->num_doppler_bins);
    int64_t seglen = (int64_t)d->num_coh * d->samples_per_code;
    if (seglen * d->num_noncoherent > ((int64_t)1 << 40)) return set_err(FMDBZP_EINVAL, "signal too long");
    return FMDBZP_OK;
}

// The dynamic-LDS limit of a kernel is one process-wide attribute shared by
// every plan that launches it: it is only ever raised (to the largest size
// any plan has asked for), so a plan created later with a smaller need does
// not lower it under an existing plan.
std::mutex g_lds_mu;
std::vector<std::pair<const void*, size_t>> g_lds_max;

int set_lds_attr(const void* func, size_t bytes)
{
    if (bytes <= kLdsDefault) return FMDBZP_OK;
    std::lock_guard<std::mutex> lk(g_lds_mu);
    for (auto& f : g_lds_max)
        if (f.first == func) {
            if (f.second >= bytes) return FMDBZP_OK;
            hipError_t e = hipFuncSetAttribute(func, hipFuncAttributeMaxDynamicSharedMemorySize, (int)bytes);
            if (e != hipSuccess)
                return set_err(FMDBZP_EHIP, "hipFuncSetAttribute(%zu bytes LDS): %s", bytes, hipGetErrorString(e));
            f.second = bytes;
            return FMDBZP_OK;
        }
    hipError_t e = hipFuncSetAttribute(func, hipFuncAttributeMaxDynamicSharedMemorySize, (int)bytes);
    if (e != hipSuccess)
        return set_err(FMDBZP_EHIP, "hipFuncSetAttribute(%zu bytes LDS): %s", bytes, hipGetErrorString(e));
    g_lds_max.emplace_back(func, bytes);
    return FMDBZP_OK;
}

template <typename T>
int dev_alloc(T** p, size_t count)
{
    if (count == 0) count = 1;
    hipError_t e = hipMalloc((void**)p, count * sizeof(T));
    if (e != hipSuccess)
        return set_err(e == hipErrorOutOfMemory ? FMDBZP_ENOMEM : FMDBZP_EHIP, "hipMalloc(%zu bytes): %s",
                       count * sizeof(T), hipGetErrorString(e));
    return FMDBZP_OK;
}

void free_plan(fmdbzp_plan* P)
{
    if (!P) return;
    hipSetDevice(P->device);
    if (P->stream) hipStreamSynchronize(P->stream);
    hipFree(P->d_twF);
    hipFree(P->d_twD);
    hipFree(P->d_arena);
    hipFree(P->d_patterns);
    hipFree(P->d_pset);
    hipFree(P->d_shifts);
    hipFree(P->d_signal);
    hipFree(P->d_codes);
    hipFree(P->d_full_tw);
    hipFree(P->d_fc_tw);
    hipFree(P->d_full_map);
    hipFree(P->d_rowsum);
    hipFree(P->d_rowbest_v);
    hipFree(P->d_rowbest_k);
    hipFree(P->d_psum);
    hipFree(P->d_pbest_v);
    hipFree(P->d_pbest_k);
    hipFree(P->d_pnbr);
    hipFree(P->d_twR);
    hipFree(P->d_rownbr);
    hipFree(P->d_colsum);
    hipFree(P->d_req);
    hipFree(P->d_stats);
    hipFree(P->d_export);
    hipFree(P->d_chip_order);
    hipFree(P->d_sec);
    hipHostFree(P->h_req);
    hipHostFree(P->h_stats);
    hipHostFree(P->h_signal);
    for (auto& e : P->pending) { hipEventDestroy(e.start); hipEventDestroy(e.stop); }
    for (auto e : P->pool) hipEventDestroy(e);
    for (int l = 0; l < kLanes; l++) {
        if (P->lane[l]) hipStreamSynchronize(P->lane[l]);
        if (P->ev_join[l]) hipEventDestroy(P->ev_join[l]);
        if (P->lane[l]) hipStreamDestroy(P->lane[l]);
    }
    if (P->ev_fork) hipEventDestroy(P->ev_fork);
    if (P->graph_exec) hipGraphExecDestroy(P->graph_exec);
    if (P->graph) hipGraphDestroy(P->graph);
    if (P->stream) hipStreamDestroy(P->stream);
    delete P;
}

// Workspace budget for the per-batch tile + accumulator, bytes.
size_t workspace_budget()
{
    const char* s = getenv("FMDBZP_WORKSPACE_GB");
    double gb = s ? atof(s) : 32.0;
    if (!(gb > 0)) gb = 32.0;
    size_t free_b = 0, total_b = 0;
    size_t want = (size_t)(gb * 1024.0 * 1024.0 * 1024.0);
    if (hipMemGetInfo(&free_b, &total_b) == hipSuccess && free_b > 0) {
        size_t cap = free_b / 2;
        if (want > cap) want = cap;
    }
    return want;
}

// Most coherent periods of the full-period correlation. Its fold costs
// num_coh^2 n and adds num_coh samples one after the other in FP32, where the
// tile's column transform grows and rounds with the logarithm. At 2.048 MHz, full-
// period and tile: 4 PRNs 84 / 94 us at 40 periods, 190 / 147 at 200, 2555 /
// 304 at 2000; one PRN 61 / 67 at 30, 67 / 64 at 40, 77 / 71 at 64; the peak's
// error against 64 bits 3.2e-7 / 1.4e-7 at 1000 periods and 4.9e-7 / 1.3e-7 at 2000.
constexpr int kFullMaxCoh = 32;

// Few rows of long periods over nreq PRNs: a row is one workgroup of the full-
// period correlation, and up to 32 of them leave most of the device idle over 13
// to 18 us of transform per step, where the tile's kernels split every row. Call
// times in us, full-period and tile: at 20 MHz 16 rows 73 / 65 (one step),
// 208 / 161 (8 steps); 32 rows 74 / 70, 208 / 181; 48 rows 76 / 74, 210 / 200; at
// 16.384 MHz 16 rows 66 / 60, 156 / 145; 32 rows 67 / 63, 158 / 159; at 15 MHz 20
// rows 65 / 67, 151 / 209. The 31-axis form is the faster one from two steps on
// (16.368 MHz, 16 rows: 67 / 60, 141 / 149).
bool full_few_rows(int n, bool several, bool axis31, int64_t rows)
{
    return n > 15360 && rows < (several ? 33 : 32) && !(several && axis31);
}
bool full_few_rows(const fmdbzp_plan* P, int nreq)
{
    return full_few_rows(P->d.samples_per_code, P->d.num_noncoherent > 1, P->fp31.n != 0,
                         (int64_t)P->d.num_doppler_bins * nreq);
}

// 32 elements behind the last spectrum: k_full31_corr's groups read past a row's end
size_t full_spectra_bytes(int64_t nprn, int64_t ndop, int64_t n) { return ((size_t)(nprn * ndop * n) + 32) * sizeof(float2); }

// The full-period transform of n points: the axes of make_full31_plan
// (FMDBZP_FULL_AXIS31) or the radices of make_full_plan (FMDBZP_FULL_RADIX) in
// one LDS buffer, its threads and LDS; FMDBZP_FULL_NONE where neither fits.
int full_form(int n, bool several, FullPlanDev* fp, Full31Dev* fp31, int* nthr, size_t* lds)
{
    if (n > 65535) return FMDBZP_FULL_NONE;
    const bool axis31 = make_full31_plan(n, fp31);
    if (axis31) {
        *lds = (size_t)fc31_lds_span(*fp31) * sizeof(float2);
        // one butterfly of the last stage per thread, 24 or 32 cells per thread
        *nthr = (31 * fp31->rb > 256 || n > 6144) ? 512 : 256;
        if (31 * fp31->rb > *nthr || n > 32 * *nthr) return FMDBZP_FULL_NONE;
    } else {
        fp31->n = 0;
        *nthr = n > 10240 ? 1024 : n > 5120 ? 512 : 256;  // at most FC_CELLS cells per thread
        if (!make_full_plan(n, *nthr, several, fp)) return FMDBZP_FULL_NONE;
        *lds = (size_t)fc_lds_span(*fp) * sizeof(float2);
    }
    // the cell exchange reads whole groups of four cells per thread
    const size_t group = (size_t)4 * *nthr;
    *lds = std::max(*lds, ((size_t)n + group - 1) / group * group * sizeof(float));
    return *lds > kLdsMax ? FMDBZP_FULL_NONE : axis31 ? FMDBZP_FULL_AXIS31 : FMDBZP_FULL_RADIX;
}

// Full-period correlation of a plan, where it admits it: simple column stage
// (any E with one data bit included), a full_form, up to kFullMaxCoh periods and
// the code spectra, plan data like the code FFTs, within
// FMDBZP_FULL_SPECTRA_MAX_BYTES. That limit is a constant, so that neither the
// workspace budget nor the memory in use decides how a search rounds; only if
// the device cannot hold admitted spectra beside the plan's workspace does the
// plan keep to the tile path (fmdbzp_plan_call_kernels tells). The size of the
// spectra; 0: the plan does not admit it.
size_t full_plan(fmdbzp_plan* P)
{
    const fmdbzp_plan_desc& d = P->d;
    if (!P->simple_kernel || P->tile_half || (d.options & FMDBZP_OPT_TILE_PATH) || d.num_coh > kFullMaxCoh) return 0;
    const size_t spec = full_spectra_bytes(P->nprn, d.num_doppler_bins, d.samples_per_code);
    if (spec > FMDBZP_FULL_SPECTRA_MAX_BYTES ||
        full_form(d.samples_per_code, d.num_noncoherent > 1, &P->fp, &P->fp31, &P->full_nthr, &P->full_lds) ==
            FMDBZP_FULL_NONE ||
        full_few_rows(P, P->nprn))  // no call would use them
        return 0;
    return spec;
}

// Tables and code spectra of the full-period correlation (d_codes on the device).
int full_spectra(fmdbzp_plan* P)
{
    const fmdbzp_plan_desc& d = P->d;
    const int n = d.samples_per_code, ndop = d.num_doppler_bins, nb = d.num_blocks, bs = d.block_size;
    int rc;
    if ((rc = set_lds_attr((const void*)k_full_corr<256, true>, P->full_lds)) ||
        (rc = set_lds_attr((const void*)k_full_corr<256, false>, P->full_lds)) ||
        (rc = set_lds_attr((const void*)k_full_corr<512, true>, P->full_lds)) ||
        (rc = set_lds_attr((const void*)k_full_corr<512, false>, P->full_lds)) ||
        (rc = set_lds_attr((const void*)k_full_corr<1024, true>, P->full_lds)) ||
        (rc = set_lds_attr((const void*)k_full_corr<1024, false>, P->full_lds)) ||
        (rc = set_lds_attr((const void*)k_full31_corr<256>, P->full_lds)) ||
        (rc = set_lds_attr((const void*)k_full31_corr<512>, P->full_lds)) ||
        (rc = set_lds_attr((const void*)k_full_signal<512>, P->full_lds)) ||
        (rc = set_lds_attr((const void*)k_full31_signal<512>, P->full_lds)) ||
        (rc = set_lds_attr((const void*)k_full_code, P->full_lds)) ||
        (rc = set_lds_attr((const void*)k_full31_code, P->full_lds)))
        return rc;
    auto grid = [](int count) { return dim3((count + 255) / 256); };
    hipStream_t st = P->stream;
    const size_t nmap = P->fp31.n ? (size_t)(P->fp31.rc + 1) / 2 * 2 * 31 * P->fp31.rb : (size_t)n;
    if ((rc = dev_alloc(&P->d_full_map, nmap))) return rc;
    if (P->fp31.n) {
        k_full31_map<<<grid(n), 256, 0, st>>>(P->d_full_map, P->fp31, nb, bs);
        k_full31_code<<<dim3(ndop, P->nprn), FC_FWD_NTHR, P->full_lds, st>>>(
            P->d_codes, P->d_full_code, P->fp31, bs, d.num_coh, 1.0f / (float)n);
    } else {
        const int ntw = fc_tw_count(P->fp);
        if ((rc = dev_alloc(&P->d_full_tw, (size_t)ntw))) return rc;
        k_fc_twiddles<<<grid(ntw), 256, 0, st>>>(P->fp, P->d_full_tw, ntw);
        k_full_map<<<grid(n), 256, 0, st>>>(P->d_full_map, n, nb, bs);
        k_full_code<<<dim3(ndop, P->nprn), FC_FWD_NTHR, P->full_lds, st>>>(
            P->d_codes, P->d_full_code, P->fp, P->d_full_tw, bs, d.num_coh, 1.0f / (float)n);
    }
    HIP_TRY(hipGetLastError());
    return FMDBZP_OK;
}

bool int_samples(int32_t eltype)
{
    return eltype == FMDBZP_I16 || eltype == FMDBZP_CI8 || eltype == FMDBZP_CI16 || eltype == FMDBZP_C2BIT;
}

// Whether a call over nreq PRNs runs the full-period correlation: not with
// surfaces (their time is the copy to the caller, and the tile path's column
// kernels stay the ones that write them), nor with few rows. Under
// FMDBZP_PREC_AUTO it comes before the FP16 tile, being the faster form (2.00
// against 3.40 ms for the 16.368 MHz search of 32 PRNs and 8 steps) and FP32.
bool full_call(const fmdbzp_plan* P, int32_t nreq, bool store)
{
    return P->full && !store && !full_few_rows(P, nreq);
}

// Column-stage form of the plan on the tile (fmdbzp_plan_column_kernel).
void column_name(const fmdbzp_plan* P, char* buf, size_t buflen)
{
    static const char* const rotmma[] = {"k_column_rotmma<2,1,2>", "k_column_rotmma<4,1,4>",
                                         "k_column_rotmma<4,3,10>", "k_column_rotmma<8,3,20>"};
    char tmp[64];
    const char* name = tmp;
    if (P->rotmma) name = rotmma[P->rotmma == 2 ? 0 : P->rotmma == 4 ? 1 : P->rotmma == 10 ? 2 : 3];
    else if (P->rotbig) snprintf(tmp, sizeof tmp, "k_column_rotbig<%d,25>", P->rotbig_nt);
    else if (P->rot2000) name = "k_column_rot2000";
    else if (P->rotsplit) snprintf(tmp, sizeof tmp, "k_column_rotsplit<%d,%d>", P->d.num_coh, P->d.num_blocks);
    else if (P->col_pair) name = P->tile_half ? "k_column_c160_pair<32,512,fp16>" : "k_column_c160_pair<32,512>";
    else if (P->col_static) name = P->tile_half ? "k_column_c160<32,512,fp16>" : "k_column_c160<32,512>";
    else if (P->col_reg) snprintf(tmp, sizeof tmp, "k_column_reg<%d>", P->d.num_doppler_bins);
    else if (P->simple_kernel) name = P->col_onebuf ? "k_column_simple<onebuf>" : "k_column_simple";
    else if (P->d.path == FMDBZP_PATH_ROTATION) name = "k_column_rotation";
    else if (P->bitsplit) snprintf(tmp, sizeof tmp, "k_column_bitsplit<%d>", P->d.num_blocks);
    else name = "k_column_sign";
    snprintf(buf, buflen, "%s", name);
}

// k_secondary_phase by sample type, for requests of up to LP - 1 rotations
using SecKernel = void (*)(const void*, int, const SecReqDev*, int32_t*);
template <int LP>
SecKernel secondary_kernel(int eltype)
{
    switch (eltype) {
    case FMDBZP_CF32: return k_secondary_phase<FMDBZP_CF32, LP>;
    case FMDBZP_CF64: return k_secondary_phase<FMDBZP_CF64, LP>;
    case FMDBZP_I16: return k_secondary_phase<FMDBZP_I16, LP>;
    case FMDBZP_CI8: return k_secondary_phase<FMDBZP_CI8, LP>;
    case FMDBZP_CI16: return k_secondary_phase<FMDBZP_CI16, LP>;
    case FMDBZP_F32: return k_secondary_phase<FMDBZP_F32, LP>;
    case FMDBZP_F64: return k_secondary_phase<FMDBZP_F64, LP>;
    default: return k_secondary_phase<FMDBZP_C2BIT, LP>;
    }
}

}  // namespace

extern "C" {

const char* fmdbzp_last_error(void) { return g_err.c_str(); }

int fmdbzp_query(char* buf, size_t buflen)
{
    if (!buf || buflen == 0) return set_err(FMDBZP_EINVAL, "null buffer");
    int dev = 0, n = 0;
    hipError_t e = hipGetDeviceCount(&n);
    if (e != hipSuccess || n == 0) {
        snprintf(buf, buflen, "abi=%d devices=0", FMDBZP_ABI_VERSION);
        return set_err(FMDBZP_ENODEV, "no HIP device: %s", hipGetErrorString(e));
    }
    hipGetDevice(&dev);
    hipDeviceProp_t prop;
    HIP_TRY(hipGetDeviceProperties(&prop, dev));
    snprintf(buf, buflen, "abi=%d device=%d name=%s arch=%s cus=%d lds_per_block=%zu hbm_bytes=%zu",
             FMDBZP_ABI_VERSION, dev, prop.name, prop.gcnArchName, prop.multiProcessorCount,
             (size_t)prop.sharedMemPerBlock, (size_t)prop.totalGlobalMem);
    return FMDBZP_OK;
}

int fmdbzp_plan_create(const fmdbzp_plan_desc* desc, int32_t nprn, const int8_t* code_samples,
                       int32_t npattern_sets, const float* patterns, const int32_t* pattern_set,
                       const int32_t* drift_shifts, fmdbzp_plan** out_plan)
{
    g_err.clear();
    if (!desc || !out_plan || !code_samples || !drift_shifts)
        return set_err(FMDBZP_EINVAL, "null argument to fmdbzp_plan_create");
    *out_plan = nullptr;
    int rc = validate_desc(desc);
    if (rc) return rc;
    if (nprn <= 0) return set_err(FMDBZP_EINVAL, "nprn must be positive");
    const fmdbzp_plan_desc& d = *desc;
    if (d.path != FMDBZP_PATH_SIMPLE) {
        if (npattern_sets <= 0 || !patterns)
            return set_err(FMDBZP_EINVAL, "sign/rotation path needs sign patterns");
        if (npattern_sets > 1 && !pattern_set) return set_err(FMDBZP_EINVAL, "pattern_set is NULL");
    }
    for (int64_t i = 0; i < (int64_t)d.num_noncoherent * d.num_doppler_bins; i++)
        if (drift_shifts[i] < 0 || drift_shifts[i] >= d.samples_per_code)
            return set_err(FMDBZP_EINVAL, "drift shift %d out of [0, spc)", drift_shifts[i]);
    int ndev = 0;
    if (hipGetDeviceCount(&ndev) != hipSuccess || ndev == 0)
        return set_err(FMDBZP_ENODEV, "no HIP device visible");

    fmdbzp_plan* P = new fmdbzp_plan();
    P->d = d;
    P->nprn = nprn;
    P->nsets = d.path == FMDBZP_PATH_SIMPLE ? 0 : npattern_sets;
    hipGetDevice(&P->device);
    auto fail = [&](int code) {
        free_plan(P);
        return code;
    };
    if (hipStreamCreateWithFlags(&P->stream, hipStreamNonBlocking) != hipSuccess)
        return fail(set_err(FMDBZP_EHIP, "hipStreamCreate failed"));
    for (int l = 0; l < kLanes; l++)
        if (hipStreamCreateWithFlags(&P->lane[l], hipStreamNonBlocking) != hipSuccess ||
            hipEventCreateWithFlags(&P->ev_join[l], hipEventDisableTiming) != hipSuccess)
            return fail(set_err(FMDBZP_EHIP, "lane stream / event creation failed"));
    if (hipEventCreateWithFlags(&P->ev_fork, hipEventDisableTiming) != hipSuccess)
        return fail(set_err(FMDBZP_EHIP, "hipEventCreate failed"));
    if (make_fft_plan(d.fft_size, &P->pf, true) || make_fft_plan(d.fft_size, &P->pf8, false) ||
        make_fft_plan(d.num_doppler_bins, &P->pd, false))
        return fail(set_err(FMDBZP_EINVAL, "FFT size has too many factors"));
    const int F = d.fft_size, ndop = d.num_doppler_bins, nb = d.num_blocks, bs = d.block_size;
    const int spc = d.samples_per_code, spc_eff = d.samples_per_code_eff;
    P->inv_f = 1.0f / (float)F;
    // Power-of-two F: 1/F is exact and goes into the conj code spectra, so the
    // correlation's inverse FFT needs no scaling (same values: multiplying by a
    // power of two commutes exactly with every add and multiply of the FFT).
    const bool f_pow2 = (F & (F - 1)) == 0;
    P->pscale = f_pow2 ? P->inv_f : 1.0f;
    P->tile_scale = f_pow2 ? 1.0f : P->inv_f;
    // Row pitches rounded to 32 elements: every tile row and accumulator row
    // starts on a 256 / 128-byte boundary, so a workgroup's column segment
    // does not straddle more cache lines than its size needs.
    P->tp = (bs + 31) & ~31;
    P->ap = (spc_eff + 31) & ~31;
    // the correlation addresses one PRN's code spectra and one pass's tile
    // rows by 32-bit byte offsets
    if ((size_t)nb * F * sizeof(float2) >= (1ull << 31) || (size_t)2 * ndop * P->tp * sizeof(float2) >= (1ull << 31))
        return fail(set_err(FMDBZP_EINVAL, "geometry too large: nb*F = %lld, ndop*bs = %lld", (long long)nb * F,
                            (long long)ndop * bs));
    P->fft_lds = (size_t)2 * fft_lds_span(F) * sizeof(float2);
    // block correlation: the staged signal-FFT row plus, with in-place
    // stages, one buffer per concurrent transform (two when they fit the
    // register bound), else two ping-pong buffers
    if (F == 2048) P->corr_variant = 3;  // compile-time 16 x 16 x 8 transforms, two per pass, unscaled
    else if (F == 2500) P->corr_variant = 4;  // compile-time 10 x 10 x 5 x 5, one per pass
    else if (F == 500) P->corr_variant = 5;   // compile-time 4 x 5 x 5 x 5, two per pass
    // the E1-like sizes: one pass's transforms must stay within nb distinct
    // code blocks and within 2^31 bytes of tile
    else if (F == 400 && nb >= 10 && (size_t)10 * ndop * P->tp * sizeof(float2) < (1ull << 31)) P->corr_variant = 6;
    else if (F == 800 && nb >= 5 && (size_t)5 * ndop * P->tp * sizeof(float2) < (1ull << 31)) P->corr_variant = 7;
    else if (F == 2000 && nb >= 2) P->corr_variant = 8;
    else if (F == 4000) P->corr_variant = 9;
    else if (fft_inplace_ok(P->pf) && 2 * F <= FMDBZP_CORR_MAXV * FMDBZP_NTHR) P->corr_variant = 2;
    else if (fft_inplace_ok(P->pf) && F <= FMDBZP_CORR_MAXV * FMDBZP_NTHR) P->corr_variant = 1;
    else P->corr_variant = 0;
    if (P->corr_variant < 2) {  // one transform per pass, runtime radices: in place instead, where F factors
        P->fc_nthr = F > 5120 ? 512 : 256;
        if (make_full_plan(F, P->fc_nthr, false, &P->fc)) {
            P->corr_variant = 10;
            P->fc_lds = (size_t)fc_lds_span(P->fc) * sizeof(float2);
            P->pscale = P->inv_f;  // 1/F in the code spectra for every F
            P->tile_scale = 1.0f;
        }
    }
    P->corr_lds = corr_lds_of(P, P->corr_variant);

    // column-stage geometry: LB columns per workgroup, padded column stride
    // (odd, so lanes on consecutive columns spread over the LDS banks)
    P->bstride = ndop | 1;
    P->sst = ndop | 1;
    // The sign search with one data bit per coherent block evaluates a single
    // edge offset (every offset gives the same power spectrum) and a single
    // all-ones pattern, so it is one column FFT followed by the half-swap fold.
    // For even ndop the half-swap equals the simple path's (w + ndop/2) mod ndop
    // fold, and the simple kernel runs it.
    P->simple_kernel = d.path == FMDBZP_PATH_SIMPLE ||
                       (d.path == FMDBZP_PATH_SIGN && d.num_data_bits == 1 && ndop % 2 == 0 &&
                        !(d.options & FMDBZP_OPT_LITERAL_EDGES));
    // simple: one in-place column buffer; sign/rotation: input column, two
    // ping-pong columns, stage and raw-power rows (+ one row of pattern signs)
    // (two ping-pong columns when one column exceeds the in-place register bound)
    P->col_onebuf = P->simple_kernel && ndop <= FMDBZP_COL_MAXV * FMDBZP_COL_NTHR && fft_inplace_ok(P->pd);
    // rotation path with one pattern per rotation slice (no data-bit combos,
    // one edge offset) and even ndop: transforms write the accumulator directly
    P->rot_direct = d.path == FMDBZP_PATH_ROTATION && d.num_data_bits == 1 && d.bit_edge_search_steps == 1 &&
                    ndop % 2 == 0;
    const size_t per_col = P->simple_kernel ? (size_t)P->bstride * (P->col_onebuf ? 1 : 2) * sizeof(float2)
                           : P->rot_direct  ? (size_t)P->bstride * 3 * sizeof(float2)
                                            : (size_t)P->bstride * 3 * sizeof(float2) +
                                                  (size_t)P->sst * 2 * sizeof(float);
    const size_t fixed = d.path == FMDBZP_PATH_ROTATION && !P->rot_direct ? (size_t)ndop * sizeof(float) : 0;
    // the sign/rotation kernels add static LDS to the dynamic part
    const size_t budget = P->simple_kernel ? kLdsDefault : kLdsDefault - 1024;
    int LB = budget > fixed ? (int)((budget - fixed) / per_col) : 0;
    if (P->col_onebuf && LB > FMDBZP_COL_MAXV * FMDBZP_COL_NTHR / ndop) LB = FMDBZP_COL_MAXV * FMDBZP_COL_NTHR / ndop;
    // ndop 160: compile-time 10 x 16 transform over a fixed column count
    if (LB > 64) LB = 64;
    // whole 128-byte accumulator / 256-byte tile segments where possible
    if (LB >= 32) LB &= ~31;
    else if (LB >= 16) LB &= ~15;
    else if (LB >= 8) LB &= ~7;
    if (LB < 1) LB = 1;
    if (LB > bs) LB = bs;
    // ndop 160 (and a column block of at least 32 lags): compile-time 10 x 16
    // column kernel with a fixed column count (k_column_c160)
    // k_column_c160 addresses one PRN's accumulator and one tile block by 32-bit byte offsets
    P->col_static = P->simple_kernel && ndop == 160 && bs >= 32 &&
                    (size_t)ndop * P->ap * sizeof(float) < (1ull << 31);
    if (P->col_static) LB = 32;
    // up to 32 rows with an in-register transform (32-bit byte offsets in a PRN's
    // accumulator and a tile block): 46 -> 15.7 us (see the kernel)
    if (P->simple_kernel && !P->col_static && (size_t)ndop * P->ap * sizeof(float) < (1ull << 32) &&
        (size_t)ndop * P->tp * sizeof(float2) < (1ull << 32)) {
#define CR_OK(NN) if (ndop == NN) P->col_reg = true;
        COLREG_ALL(CR_OK)
#undef CR_OK
    }
    P->use_graph = (d.options & FMDBZP_OPT_GRAPH) != 0;
    P->tile_half = d.precision == FMDBZP_PREC_TILE_FP16;
    P->tile_auto = d.precision == FMDBZP_PREC_AUTO && P->col_static;
    if (P->tile_half && !P->col_static)
        return fail(set_err(FMDBZP_EINVAL, "FP16 tiles need a simple-path plan with 160 Doppler bins and "
                                           "block size >= 32"));
    // two steps per column launch (ndop 160): pairs of consecutive steps whose
    // shifts differ by at most one column in every row
    if (P->col_static && d.num_noncoherent >= 2) {
        const char* cp = getenv("FMDBZP_COL_PAIR");  // "0": one step per launch (measurement, tests)
        P->pair_ok.assign((size_t)d.num_noncoherent, 0);
        bool any = false;
        for (int s2 = 0; s2 + 1 < d.num_noncoherent; s2++) {
            bool ok = true;
            for (int w = 0; w < ndop && ok; w++) {
                int dd = drift_shifts[(size_t)(s2 + 1) * ndop + w] - drift_shifts[(size_t)s2 * ndop + w];
                if (dd > spc / 2) dd -= spc;
                else if (dd < -spc / 2) dd += spc;
                ok = dd >= -1 && dd <= 1;
            }
            P->pair_ok[(size_t)s2] = ok ? 1 : 0;
            any = any || ok;
        }
        P->col_pair = any && !(cp && atoi(cp) == 0);
        P->col_lds2 = (size_t)(32 + 2) * P->bstride * sizeof(float2) + 2 * 160 * sizeof(int32_t);
    }
    P->LB = LB;
    // With fewer than 16 columns per workgroup, a row-major accumulator turns
    // every scatter into isolated 4-byte updates; those plans keep the
    // accumulator column-major, with rows contiguous per code column.
    P->acc_cm = !P->simple_kernel && LB < 16;
    // k_column_rot2000 addresses a rotation slice of the accumulator by 32-bit byte offsets
    const char* r2k = getenv("FMDBZP_ROT2000");  // "0": the four-step kernel at 2000 bins too (measurement)
    P->rot2000 = P->rot_direct && ndop == 2000 && d.num_coh <= 32 && !(r2k && atoi(r2k) == 0) &&
                 (size_t)spc * ((ndop + 31) & ~31) * sizeof(float) < (1ull << 32);
    if (P->rot2000) {
        // 25 periods of 80 rows, the E1-like search: 10.5 ms per PRN-step at 25 MHz
        // against 15.1 ms of the 16 x 5 x 5 x 5 kernel, which serves other N_coh
        // (the masks of a workgroup hold at most 64 rotations)
        P->rot25 = d.num_coh == 25 && d.num_secondary_rotations <= 64;
        P->acc_cm = true;
        LB = P->LB = 1;
    }
    // direct rotation with 25 coherent periods (ndop = 25 nb, the E1-like
    // searches) other than the compile-time 2000-bin case: the four-step
    // kernel, one lag per thread (nb <= 512), at most 25 accumulator cells
    // per thread; a wave transforms rgrp = 640 / nb rows together, with at
    // most 1 and 2 butterflies per lane in its radix-10 and radix-5 stages
    // (nb = 2^a 5^b with a <= b: 50, 100, 250, 500)
    if (P->rot_direct && !P->rot2000 && d.num_coh == 25 && nb >= 8 && nb <= 512) {
        const int nt = nb <= 64 ? 64 : nb <= 128 ? 128 : nb <= 256 ? 256 : nb <= 320 ? 320 : 512;
        P->rgrp = std::max(1, 640 / nb);
        bool ok = make_row_plan(nb, &P->prow) == 0 && P->prow.nst >= 1 && (ndop + nt - 1) / nt <= 25;
        for (int st = 0; ok && st < P->prow.nst; st++) {
            const int R = P->prow.radix[st];
            const int mb = R == 10 ? 1 : 2;
            ok = (P->rgrp * (nb / R) + 63) / 64 <= mb;
        }
        const size_t lds = (size_t)(25 * fft_lds_span(nb) + nb) * sizeof(float2) +
                           ((size_t)ndop + d.num_secondary_rotations) * sizeof(uint32_t);
        if (ok && lds <= kLdsMax) {
            P->rotbig = nt;
            P->rotbig_nt = nt;
            // 25 MHz, per PRN-step against k_column_rotbig: 6.3 / 8.9 ms at 50 rows, 12.9 / 17.6 at
            // 100, 32.3 / 55.6 at 250, 72 / 132 at 500 (the masks of a workgroup hold at most 64 rotations)
            P->rot25 = (nb == 50 || nb == 100 || nb == 250 || nb == 500) && d.num_secondary_rotations <= 64;
            P->acc_cm = true;
            LB = P->LB = 1;
        }
    }
    P->lim_cm = P->acc_cm;
    // direct rotation of 10 or 20 coherent periods and a row length with an
    // in-register transform (the L5-like searches up to +-10 kHz): 32 columns
    // per workgroup where both roles fit its threads, else 16
    if (P->rot_direct && !P->rot2000 && !P->rotbig && d.num_secondary_rotations <= 64 &&
        (size_t)ndop * P->ap * sizeof(float) < (1ull << 32)) {
#define RS_OK(PP, NN) if (d.num_coh == PP && nb == NN) P->rotsplit = 32 * std::max(PP, NN) <= ROTSPLIT_NTHR ? 32 : 16;
        ROTSPLIT_ALL(RS_OK)
#undef RS_OK
        if (P->rotsplit) {
            P->acc_cm = false;
            LB = P->LB = P->rotsplit;
        }
    }
    // two bits of 20 periods, edge offsets of whole periods, a row length with an
    // in-register transform and 16 columns: 781 -> 210 us (see the kernel)
    if (d.path == FMDBZP_PATH_SIGN && d.num_data_bits == 2 && d.num_coh == 40 && 20 % d.bit_edge_search_steps == 0 &&
        bs >= BITSPLIT_C && (size_t)ndop * P->ap * sizeof(float) < (1ull << 32) &&
        (size_t)ndop * P->tp * sizeof(float2) < (1ull << 31)) {
#define BS_OK(NN) if (nb == NN) P->bitsplit = true;
        BITSPLIT_ALL(BS_OK)
#undef BS_OK
        if (P->bitsplit) {
            P->acc_cm = false;
            LB = P->LB = BITSPLIT_C;
        }
    }
    // the matrix-core form of the E1-like search (nb = 25 n1, n1 = 2, 4, 10, 20);
    // FMDBZP_PREC_AUTO takes it at n1 = 10 and 20, a fixed choice from when it
    // was the faster one (48.4 and 109 ms per PRN-step at 25 MHz over two steps,
    // k_column_rotbig 57.4 and 132); k_column_rot25 takes 34.5 and 79 in FP32
    if ((d.precision == FMDBZP_PREC_MFMA || d.precision == FMDBZP_PREC_AUTO) && P->rotbig && nb % 25 == 0 &&
        ndop == 25 * nb &&
        (nb / 25 == 2 || nb / 25 == 4 || nb / 25 == 10 || nb / 25 == 20) && d.num_secondary_rotations <= 32 &&
        (d.precision == FMDBZP_PREC_MFMA || nb / 25 >= 10))
        P->rotmma = nb / 25;
    if (d.precision == FMDBZP_PREC_MFMA && !P->rotmma)
        return fail(set_err(FMDBZP_EINVAL, "MFMA precision needs a direct rotation plan with 25 coherent periods "
                                           "and ndop = 625 n1, n1 in {2, 4, 10, 20}"));
    P->apc = (ndop + 31) & ~31;
    P->acc_ps = P->acc_cm ? (size_t)spc_eff * P->apc : (size_t)ndop * P->ap;
    P->lim_acc_ps = P->lim_cm ? (size_t)spc_eff * P->apc : (size_t)ndop * P->ap;
    if (P->rotbig) {
        const int R = d.num_secondary_rotations;
        int span = 0;
        P->smin.assign((size_t)d.num_noncoherent, 0);
        P->smax.assign((size_t)d.num_noncoherent, 0);
        for (int s2 = 0; s2 < d.num_noncoherent; s2++) {
            int lo = 0, hi = 0;
            for (int w = 0; w < ndop; w++) {
                int v = drift_shifts[(size_t)s2 * ndop + w];
                if (v > spc / 2) v -= spc;  // signed drift
                lo = std::min(lo, v);
                hi = std::max(hi, v);
            }
            P->smin[(size_t)s2] = lo;
            P->smax[(size_t)s2] = hi;
            span = std::max(span, hi - lo);
        }
        // the window of one PRN within its budget share, each rotation slice of
        // it below 2^31 bytes (32-bit offsets within a slice)
        const size_t col_bytes = (size_t)R * P->apc * sizeof(float);
        const size_t tile_col = (size_t)ndop * P->tp * sizeof(float2) / (size_t)bs + 1;
        const size_t slice_cap = ((size_t)1 << 31) / ((size_t)P->apc * sizeof(float)) - 2;
        const size_t budget = workspace_budget();
        size_t W = budget / (col_bytes + tile_col);
        const char* env = getenv("FMDBZP_CHUNK_COLS");
        if (env && atoi(env) > 0) W = (size_t)atoi(env);
        W = std::min(W, slice_cap);
        if (P->rotmma) W = std::min(W, (size_t)65532);  // 16-bit window offsets
        if (W >= (size_t)spc) W = (size_t)spc;
        if (W < 64) W = 64;
        P->chunk_cols = (int)W;
        P->nchunks = (spc + P->chunk_cols - 1) / P->chunk_cols;
        if (P->nchunks == 1) P->chunk_cols = spc;
        P->halo = P->nchunks > 1 ? 1 : 0;
        P->win_max = P->chunk_cols + 2 * P->halo;
        if ((size_t)P->win_max > slice_cap + 2 && P->nchunks > 1)
            return fail(set_err(FMDBZP_EINVAL, "code-column chunk too wide"));
        if ((size_t)P->win_max * P->apc * sizeof(float) >= ((size_t)1 << 31))
            return fail(set_err(FMDBZP_EINVAL, "rotation slice of %d columns exceeds 2^31 bytes", P->win_max));
        P->nrb_max = P->nchunks == 1 && span == 0 ? nb : std::min(nb, (P->win_max + span + bs - 1) / bs + 2);
        P->acc_ps = (size_t)R * P->win_max * P->apc;
        P->red_cw = 4096;
        P->nsub = (P->chunk_cols + P->red_cw - 1) / P->red_cw;
        P->nparts = P->nchunks * R * P->nsub;
    }
    P->col_lds = per_col * LB + fixed;
    if (P->col_static) P->col_lds = (size_t)LB * P->bstride * sizeof(float2);  // one column buffer
    if (P->rotsplit) P->col_lds = (size_t)d.num_coh * rotsplit_pitch(nb, P->rotsplit) * sizeof(float2);
    if (P->rot2000)
        P->col_lds = (size_t)(2000 + 2 * fft_lds_span(2000)) * sizeof(float2) +
                     ((size_t)d.num_secondary_rotations * 4 + 7) / 8 * 8;
    if (P->bitsplit) P->col_lds = bitsplit_lds(nb);
    if (P->rot25 && P->rot2000) P->col_lds = rot25_lds<80>();
    if (P->rotbig)
        P->col_lds = (size_t)(25 * fft_lds_span(nb) + nb) * sizeof(float2) +
                     ((size_t)ndop + d.num_secondary_rotations) * sizeof(uint32_t);
    if (P->rotmma) {  // k_column_rotmma: two buffers of FP16 group outputs, 16-bit offsets, masks, and
                      // the A operand of the groups beyond two per wave (NW = 8, 4, 4, 2 waves at n1 = 20, 10, 4, 2)
        const int n1 = P->rotmma, nw = n1 == 20 ? 8 : n1 == 2 ? 2 : 4;
        P->col_lds = (((size_t)6250 * n1 + 160 + 15) & ~(size_t)15)  // 2 n1 625 pairs + ndop = 625 n1 offsets + 160
                     + 32 * 36 * sizeof(uint32_t);                        // twiddle table
        if (n1 > 2 * nw) P->col_lds += (size_t)(n1 - 2 * nw) * 25 * 9 * 16;
    }
    if (P->col_lds > kLdsMax) return fail(set_err(FMDBZP_EINVAL, "column stage does not fit LDS"));

    if ((rc = set_lds_attr((const void*)k_code_fft, P->fft_lds)) ||
        (rc = set_lds_attr((const void*)k_signal_fft, P->fft_lds)) ||
        (rc = set_lds_attr((const void*)k_corr_tile<2, true, 2048>, P->corr_lds)) ||
        (rc = set_lds_attr((const void*)k_corr_tile<2, true>, P->corr_lds)) ||
        (rc = set_lds_attr((const void*)k_corr_tile<1, true>, P->corr_lds)) ||
        (rc = set_lds_attr((const void*)k_corr_tile<1, false>, P->corr_lds)) ||
        (rc = set_lds_attr((const void*)k_corr_tile<2, true, 2048, __half2>, P->corr_lds)) ||
        (rc = set_lds_attr((const void*)k_corr_tile<1, true, 2500>, P->corr_lds)) ||
        (rc = set_lds_attr((const void*)k_corr_tile<2, true, 500>, P->corr_lds)) ||
        (rc = set_lds_attr((const void*)k_corr_tile<10, true, 400>, P->corr_lds)) ||
        (rc = set_lds_attr((const void*)k_corr_tile<5, true, 800>, P->corr_lds)) ||
        (rc = set_lds_attr((const void*)k_corr_tile<2, true, 2000>, P->corr_lds)) ||
        (rc = set_lds_attr((const void*)k_corr_tile<1, true, 4000>, P->corr_lds)) ||
        (rc = set_lds_attr((const void*)k_corr_tile<10, true, 400, __half2>, P->corr_lds)) ||
        (rc = set_lds_attr((const void*)k_corr_tile<5, true, 800, __half2>, P->corr_lds)) ||
        (rc = set_lds_attr((const void*)k_corr_tile<2, true, 2000, __half2>, P->corr_lds)) ||
        (rc = set_lds_attr((const void*)k_corr_tile<1, true, 4000, __half2>, P->corr_lds)) ||
        (rc = set_lds_attr((const void*)k_corr_tile<2, true, 500, __half2>, P->corr_lds)) ||
        (rc = set_lds_attr((const void*)k_corr_tile<1, true, 2500, __half2>, P->corr_lds)) ||
        (rc = set_lds_attr((const void*)k_corr_tile<2, true, 0, __half2>, P->corr_lds)) ||
        (rc = set_lds_attr((const void*)k_corr_tile<1, true, 0, __half2>, P->corr_lds)) ||
        (rc = set_lds_attr((const void*)k_corr_tile<1, false, 0, __half2>, P->corr_lds)) ||
        (rc = set_lds_attr((const void*)k_column_c160<32, 512>, P->col_lds)) ||
        (rc = set_lds_attr((const void*)k_column_c160<32, 512, true>, P->col_lds)) ||
        (P->col_pair && (rc = set_lds_attr((const void*)k_column_c160_pair<32, 512>, P->col_lds2))) ||
        (P->col_pair && (rc = set_lds_attr((const void*)k_column_c160_pair<32, 512, true>, P->col_lds2))) ||
        (rc = set_lds_attr((const void*)k_column_simple<true>, P->col_lds)) ||
        (rc = set_lds_attr((const void*)k_column_simple<false>, P->col_lds)) ||
        (rc = set_lds_attr((const void*)k_column_sign, P->col_lds)) ||
        (rc = set_lds_attr((const void*)k_column_rotation, P->col_lds)) ||
        (rc = set_lds_attr((const void*)k_column_rot2000<512>, P->col_lds)) ||
        (rc = set_lds_attr((const void*)k_column_rot25<80, false>, rot25_lds<80>())) ||
        (rc = set_lds_attr((const void*)k_column_rot25<50, true>, rot25_lds<50>())) ||
        (rc = set_lds_attr((const void*)k_column_rot25<100, true>, rot25_lds<100>())) ||
        (rc = set_lds_attr((const void*)k_column_rot25<250, true>, rot25_lds<250>())) ||
        (rc = set_lds_attr((const void*)k_column_rot25<500, true>, rot25_lds<500>())) ||
#define BS_ATTR(NN) (rc = set_lds_attr((const void*)k_column_bitsplit<NN>, bitsplit_lds(NN))) ||
        BITSPLIT_ALL(BS_ATTR)
#undef BS_ATTR
        (rc = set_lds_attr((const void*)k_column_rotbig<64, 25>, P->col_lds)) ||
        (rc = set_lds_attr((const void*)k_column_rotbig<128, 25>, P->col_lds)) ||
        (rc = set_lds_attr((const void*)k_column_rotbig<256, 25>, P->col_lds)) ||
        (rc = set_lds_attr((const void*)k_column_rotbig<320, 25>, P->col_lds)) ||
        (rc = set_lds_attr((const void*)k_column_rotbig<512, 25>, P->col_lds)) ||
        (rc = set_lds_attr((const void*)k_column_rotmma<8, 3, 20>, P->col_lds)) ||
        (rc = set_lds_attr((const void*)k_column_rotmma<4, 3, 10>, P->col_lds)) ||
        (rc = set_lds_attr((const void*)k_column_rotmma<4, 1, 4>, P->col_lds)) ||
        (rc = set_lds_attr((const void*)k_column_rotmma<2, 1, 2>, P->col_lds)))
        return fail(rc);

    // tables
    {
        std::vector<float2> twF = twiddles(F), twD = twiddles(ndop);
        if ((rc = dev_alloc(&P->d_twF, (size_t)F)) || (rc = dev_alloc(&P->d_twD, (size_t)ndop)))
            return fail(rc);
        if (hipMemcpy(P->d_twF, twF.data(), sizeof(float2) * F, hipMemcpyHostToDevice) != hipSuccess ||
            hipMemcpy(P->d_twD, twD.data(), sizeof(float2) * ndop, hipMemcpyHostToDevice) != hipSuccess)
            return fail(set_err(FMDBZP_EHIP, "twiddle upload failed"));
    }
    if (P->corr_variant == 10) {
        const int count = fc_tw_count(P->fc);
        if ((rc = dev_alloc(&P->d_fc_tw, (size_t)count)) ||
            (rc = set_lds_attr((const void*)k_fc_code<256>, P->fc_lds)) ||
            (rc = set_lds_attr((const void*)k_fc_code<512>, P->fc_lds)) ||
            (rc = set_lds_attr((const void*)k_fc_signal<256>, P->fc_lds)) ||
            (rc = set_lds_attr((const void*)k_fc_signal<512>, P->fc_lds)) ||
            (rc = set_lds_attr((const void*)k_corr_fc<256, float2>, P->fc_lds)) ||
            (rc = set_lds_attr((const void*)k_corr_fc<512, float2>, P->fc_lds)) ||
            (rc = set_lds_attr((const void*)k_corr_fc<256, __half2>, P->fc_lds)) ||
            (rc = set_lds_attr((const void*)k_corr_fc<512, __half2>, P->fc_lds)))
            return fail(rc);
        k_fc_twiddles<<<dim3((count + 255) / 256), 256, 0, P->stream>>>(P->fc, P->d_fc_tw, count);
        if (hipGetLastError() != hipSuccess) return fail(set_err(FMDBZP_EHIP, "transform twiddles failed"));
    }
    if (P->rotbig) {
        std::vector<float2> twR = twiddles(nb);
        if ((rc = dev_alloc(&P->d_twR, (size_t)nb))) return fail(rc);
        if (hipMemcpy(P->d_twR, twR.data(), sizeof(float2) * nb, hipMemcpyHostToDevice) != hipSuccess)
            return fail(set_err(FMDBZP_EHIP, "row twiddle upload failed"));
    }
    if ((rc = dev_alloc(&P->d_shifts, (size_t)d.num_noncoherent * ndop))) return fail(rc);
    if (hipMemcpy(P->d_shifts, drift_shifts, sizeof(int32_t) * (size_t)d.num_noncoherent * ndop,
                  hipMemcpyHostToDevice) != hipSuccess)
        return fail(set_err(FMDBZP_EHIP, "drift shift upload failed"));
    {
        int nsets = P->nsets > 0 ? P->nsets : 1;
        size_t npat = (size_t)nsets * d.num_coh * d.num_patterns;
        if ((rc = dev_alloc(&P->d_patterns, npat)) || (rc = dev_alloc(&P->d_pset, (size_t)nprn))) return fail(rc);
        std::vector<int32_t> pset((size_t)nprn, 0);
        if (P->nsets > 1) {
            for (int i = 0; i < nprn; i++) {
                if (pattern_set[i] < 0 || pattern_set[i] >= P->nsets)
                    return fail(set_err(FMDBZP_EINVAL, "pattern_set[%d] = %d out of range", i, pattern_set[i]));
                pset[(size_t)i] = pattern_set[i];
            }
        }
        if (hipMemcpy(P->d_pset, pset.data(), sizeof(int32_t) * nprn, hipMemcpyHostToDevice) != hipSuccess)
            return fail(set_err(FMDBZP_EHIP, "pattern set upload failed"));
        if (P->nsets > 0) {
            for (size_t i = 0; i < npat; i++)
                if (patterns[i] != 1.0f && patterns[i] != -1.0f)
                    return fail(set_err(FMDBZP_EINVAL, "sign patterns must be +1/-1"));
            if (hipMemcpy(P->d_patterns, patterns, sizeof(float) * npat, hipMemcpyHostToDevice) != hipSuccess)
                return fail(set_err(FMDBZP_EHIP, "pattern upload failed"));
        }
    }
    // workspace: signal FFT cache for all segments + PRN-batch tile/accumulator
    const int tile_blocks = P->rotbig ? P->nrb_max : nb;
    {
        size_t per_prn = (size_t)tile_blocks * ndop * P->tp * sizeof(float2) * (P->col_pair ? 2 : 1) +
                         P->acc_ps * sizeof(float);
        if (P->rotbig)
            per_prn = (size_t)tile_blocks * ndop * P->tp * sizeof(float2) + P->acc_ps * sizeof(float) +
                      (size_t)P->nparts * ndop * (8 + 4 + 8 + 16) + (size_t)ndop * 16 +
                      (d.noise_estimator == FMDBZP_NOISE_GLOBAL_MEAN ? (size_t)spc_eff * 8 : 0);
        size_t budget = workspace_budget();
        size_t b = budget / per_prn;
        if (b < 1) b = 1;
        if (b > (size_t)nprn) b = (size_t)nprn;
        if (b > 65535) b = 65535;
        P->batch = (int)b;
        P->nlanes = P->batch >= lanes_requested() && !P->rotbig ? lanes_requested() : 1;
    }
    if (P->acc_cm && !P->rotbig) {
        // columns per workgroup of the column-major reduction: about 1024
        // workgroups per PRN, 32 to 4096 columns each. With 4096 columns
        // always, 8 PRNs of 4000 columns (640 Doppler rows) ran on 8
        // workgroups, 1430 us; a 2.5 M-column surface keeps 4096. Not by the
        // batch: the FP64 sums of a search round by its chunks. The partials
        // (20 bytes per row and chunk) live in the batch's tile, which is
        // consumed by then: wider chunks where they would not fit.
        const size_t rb4 = (ndop + 4 * FMDBZP_NTHR - 1) / (4 * FMDBZP_NTHR);
        const size_t cw = (size_t)spc_eff * rb4 / 1024;
        P->red_cw = (int)std::min<size_t>(4096, std::max<size_t>(32, (cw + 31) / 32 * 32));
        auto nchunk = [&]() { return (spc_eff + P->red_cw - 1) / P->red_cw; };
        while ((size_t)nchunk() * kRedPart > (size_t)nb * P->tp * sizeof(float2)) P->red_cw *= 2;
        P->red_nchunk = nchunk();
    }
    // The large buffers are one allocation: a free of each (200 to 300 us from
    // about 30 MB on) would cost more than all of a small plan's creation. The
    // code spectra come last: where they do not fit beside the rest, the plan
    // does without the full-period correlation.
    {
        const size_t tile_bytes = (size_t)P->batch * tile_blocks * ndop * P->tp * sizeof(float2);
        size_t total = 0;
        auto place = [&](size_t bytes) {  // large ones on 2 MiB pages, as an allocation of their own
            const size_t page = bytes >= (2u << 20) ? (2u << 20) : 256, at = (total + page - 1) / page * page;
            total = at + bytes;
            return at;
        };
        const size_t o_prn = place((size_t)nprn * nb * F * sizeof(float2));
        const size_t o_sig = place((size_t)d.num_noncoherent * ndop * F * sizeof(float2));
        const size_t o_tile = place(tile_bytes), o_tile2 = P->col_pair ? place(tile_bytes) : 0;
        const size_t o_acc = place((size_t)P->batch * P->acc_ps * sizeof(float));
        const size_t without = total, spec = full_plan(P), o_spec = place(spec);
        if (spec) {
            P->full = hipMalloc((void**)&P->d_arena, total) == hipSuccess;
            if (!P->full) (void)hipGetLastError();
        }
        if (!P->full && (rc = dev_alloc(&P->d_arena, without))) return fail(rc);
        P->d_prnconj = (float2*)(P->d_arena + o_prn);
        P->d_sigfft = (float2*)(P->d_arena + o_sig);
        P->d_tile = (float2*)(P->d_arena + o_tile);
        if (P->col_pair) P->d_tile2 = (float2*)(P->d_arena + o_tile2);
        P->d_acc = (float*)(P->d_arena + o_acc);
        if (P->full) P->d_full_code = (float2*)(P->d_arena + o_spec);
    }
    if ((rc = dev_alloc(&P->d_rowsum, (size_t)P->batch * ndop)) ||
        (rc = dev_alloc(&P->d_rowbest_v, (size_t)P->batch * ndop)) ||
        (rc = dev_alloc(&P->d_rowbest_k, (size_t)P->batch * ndop)))
        return fail(rc);
    if (P->rotbig) {
        const size_t np = (size_t)P->batch * P->nparts * ndop;
        if ((rc = dev_alloc(&P->d_psum, np)) || (rc = dev_alloc(&P->d_pbest_v, np)) ||
            (rc = dev_alloc(&P->d_pbest_k, np)) || (rc = dev_alloc(&P->d_pnbr, np)) ||
            (rc = dev_alloc(&P->d_rownbr, (size_t)P->batch * ndop)))
            return fail(rc);
        if (d.noise_estimator == FMDBZP_NOISE_GLOBAL_MEAN &&
            (rc = dev_alloc(&P->d_colsum, (size_t)P->batch * spc_eff)))
            return fail(rc);
    }
    // code samples -> conj sub-block FFTs on the device
    {
        for (int64_t i = 0; i < (int64_t)nprn * spc; i++)
            if (code_samples[i] != 1 && code_samples[i] != -1)
                return fail(set_err(FMDBZP_EINVAL, "code samples must be +1/-1"));
        if ((rc = dev_alloc(&P->d_codes, (size_t)nprn * spc))) return fail(rc);
        hipError_t e = hipMemcpy(P->d_codes, code_samples, (size_t)nprn * spc, hipMemcpyHostToDevice);
        if (e == hipSuccess) {
            Timed t(P, FMDBZP_K_CODE_FFT, P->stream);
            if (P->corr_variant != 10)
                k_code_fft<<<dim3(nb, nprn), FMDBZP_NTHR, P->fft_lds, P->stream>>>(
                    P->d_codes, P->d_prnconj, P->pf8, P->d_twF, spc, nb, bs, P->pscale);
            else if (P->fc_nthr == 512)
                k_fc_code<512><<<dim3(nb, nprn), 512, P->fc_lds, P->stream>>>(P->d_codes, P->d_prnconj, P->fc,
                                                                             P->d_fc_tw, spc, nb, bs, P->pscale);
            else
                k_fc_code<256><<<dim3(nb, nprn), 256, P->fc_lds, P->stream>>>(P->d_codes, P->d_prnconj, P->fc,
                                                                             P->d_fc_tw, spc, nb, bs, P->pscale);
            e = hipGetLastError();
        }
        if (e != hipSuccess) return fail(set_err(FMDBZP_EHIP, "code FFT failed: %s", hipGetErrorString(e)));
    }
    if (P->full && (rc = full_spectra(P))) return fail(rc);
    {
        const hipError_t e = hipStreamSynchronize(P->stream);
        if (e != hipSuccess) return fail(set_err(FMDBZP_EHIP, "code spectra failed: %s", hipGetErrorString(e)));
        hipFree(P->d_codes);
        P->d_codes = nullptr;
        collect_timing(P);
    }
    const char* at = getenv("FMDBZP_AUTOTUNE");
    if ((d.options & FMDBZP_OPT_AUTOTUNE) || (at && atoi(at) != 0))
        if ((rc = autotune(P))) return fail(rc);
    *out_plan = P;
    return FMDBZP_OK;
}

int fmdbzp_plan_destroy(fmdbzp_plan* plan)
{
    free_plan(plan);
    return FMDBZP_OK;
}

int fmdbzp_plan_set_timing(fmdbzp_plan* plan, int32_t enable)
{
    if (!plan) return set_err(FMDBZP_EHANDLE, "null plan");
    std::lock_guard<std::mutex> lk(plan->mu);
    plan->timing = enable != 0;
    for (int i = 0; i < FMDBZP_K_NUM_CLASSES; i++) { plan->tot_ms[i] = 0; plan->launches[i] = 0; }
    return FMDBZP_OK;
}

int fmdbzp_plan_set_surface_layout(fmdbzp_plan* plan, int32_t nbins, const int32_t* chip_order)
{
    g_err.clear();
    if (!plan) return set_err(FMDBZP_EHANDLE, "null plan");
    std::lock_guard<std::mutex> lk(plan->mu);
    const int spc = plan->d.samples_per_code;
    if (nbins < 0 || nbins > spc) return set_err(FMDBZP_EINVAL, "nbins %d outside [0, %d]", nbins, spc);
    if (nbins > 0) {
        if (!chip_order) return set_err(FMDBZP_EINVAL, "chip_order is required for nbins > 0");
        std::vector<char> seen((size_t)spc, 0);
        for (int i = 0; i < spc; i++) {
            const int c = chip_order[i];
            if (c < 0 || c >= spc || seen[(size_t)c]) return set_err(FMDBZP_EINVAL, "chip_order is not a permutation");
            seen[(size_t)c] = 1;
        }
    }
    HIP_TRY(hipSetDevice(plan->device));
    if (plan->pending_out) {
        const int rc = acquire_finish(plan);
        if (rc) return rc;
    }
    HIP_TRY(hipStreamSynchronize(plan->stream));
    if (nbins > 0) {
        if (!plan->d_chip_order) HIP_TRY(hipMalloc((void**)&plan->d_chip_order, sizeof(int32_t) * (size_t)spc));
        HIP_TRY(hipMemcpy(plan->d_chip_order, chip_order, sizeof(int32_t) * (size_t)spc, hipMemcpyHostToDevice));
    }
    if (nbins != plan->surf_bins) {  // the staging surfaces change size
        hipFree(plan->d_export);
        plan->d_export = nullptr;
    }
    plan->surf_bins = nbins;
    return FMDBZP_OK;
}

int fmdbzp_secondary_phase(fmdbzp_plan* plan, const void* signal, int32_t eltype, int64_t n_samples,
                           double interm_freq_hz, uint32_t flags, const fmdbzp_secondary_request* reqs,
                           int32_t nreq, int32_t* out_phase)
{
    g_err.clear();
    if (!plan) return set_err(FMDBZP_EHANDLE, "null plan");
    if (nreq < 0 || (nreq > 0 && (!reqs || !out_phase || !signal)))
        return set_err(FMDBZP_EINVAL, "null argument to fmdbzp_secondary_phase");
    if (nreq == 0) return FMDBZP_OK;
    if (!elsize(eltype) && eltype != FMDBZP_C2BIT) return set_err(FMDBZP_EINVAL, "unknown eltype %d", eltype);
    std::lock_guard<std::mutex> lk(plan->mu);
    const int spc = plan->d.samples_per_code;
    int Lmax = 0;
    std::vector<int8_t> codes((size_t)nreq * spc), secs((size_t)nreq * 64, 1);
    for (int i = 0; i < nreq; i++) {
        const fmdbzp_secondary_request& q = reqs[i];
        if (q.num_rotations < 1 || q.num_rotations > 64 || !q.code || !q.secondary)
            return set_err(FMDBZP_EINVAL, "request %d: 1 <= num_rotations <= 64 and code / secondary required", i);
        for (int n = 0; n < spc; n++) {
            if (q.code[n] != 1 && q.code[n] != -1) return set_err(FMDBZP_EINVAL, "request %d: code must be +-1", i);
            codes[(size_t)i * spc + n] = q.code[n];
        }
        for (int k = 0; k < q.num_rotations; k++) {
            if (q.secondary[k] != 1 && q.secondary[k] != -1)
                return set_err(FMDBZP_EINVAL, "request %d: secondary code must be +-1", i);
            secs[(size_t)i * 64 + k] = q.secondary[k];
        }
        Lmax = std::max(Lmax, q.num_rotations);
    }
    if (n_samples < (int64_t)Lmax * spc)
        return set_err(FMDBZP_EINVAL, "signal has %lld samples, fewer than %d code periods", (long long)n_samples, Lmax);
    HIP_TRY(hipSetDevice(plan->device));
    if (plan->pending_out) {
        const int rc = acquire_finish(plan);
        if (rc) return rc;
    }
    const size_t nsig = (size_t)Lmax * spc;
    const size_t sig_bytes = eltype == FMDBZP_C2BIT ? (nsig + 1) / 2 : nsig * elsize(eltype);
    const bool dev_sig = (flags & FMDBZP_FLAG_DEVICE_SIGNAL) != 0;
    if (!dev_sig && plan->signal_cap < sig_bytes) {  // host samples go through the plan's signal buffer
        hipFree(plan->d_signal);
        plan->d_signal = nullptr;
        plan->signal_cap = 0;
        HIP_TRY(hipMalloc(&plan->d_signal, sig_bytes));
        plan->signal_cap = sig_bytes;
    }
    // plan-owned request buffer: codes | secondary chips | descriptors | results
    const size_t o_sec = ((size_t)nreq * spc + 255) / 256 * 256;
    const size_t o_req = o_sec + ((size_t)nreq * 64 + 255) / 256 * 256;
    const size_t o_out = o_req + (sizeof(SecReqDev) * (size_t)nreq + 255) / 256 * 256;
    const size_t need = o_out + sizeof(int32_t) * (size_t)nreq;
    if (plan->sec_cap < need) {
        hipFree(plan->d_sec);
        plan->d_sec = nullptr;
        plan->sec_cap = 0;
        HIP_TRY(hipMalloc((void**)&plan->d_sec, need));
        plan->sec_cap = need;
    }
    int8_t* d_codes = (int8_t*)plan->d_sec;
    int8_t* d_secs = (int8_t*)(plan->d_sec + o_sec);
    SecReqDev* d_reqs = (SecReqDev*)(plan->d_sec + o_req);
    int32_t* d_out = (int32_t*)(plan->d_sec + o_out);
    std::vector<SecReqDev> rq((size_t)nreq);
    const double twopi = 6.283185307179586;  // Julia `2π`
    for (int i = 0; i < nreq; i++) {
        rq[(size_t)i].code = d_codes + (size_t)i * spc;
        rq[(size_t)i].sec = d_secs + (size_t)i * 64;
        rq[(size_t)i].phase_step = (-twopi * (interm_freq_hz + reqs[i].doppler_hz)) / plan->d.sampling_freq_hz;
        rq[(size_t)i].L = reqs[i].num_rotations;
        rq[(size_t)i].pad = 0;
    }
    const SecKernel kernel = Lmax <= 16   ? secondary_kernel<17>(eltype)
                             : Lmax <= 32 ? secondary_kernel<33>(eltype)
                                          : secondary_kernel<65>(eltype);
    const size_t lds_bytes = Lmax <= 16 ? sec_lds(17) : Lmax <= 32 ? sec_lds(33) : sec_lds(65);
    {
        const int rc = set_lds_attr((const void*)kernel, lds_bytes);
        if (rc) return rc;
    }
    hipError_t e = hipSuccess;
    if (!dev_sig) e = hipMemcpy(plan->d_signal, signal, sig_bytes, hipMemcpyHostToDevice);
    if (e == hipSuccess) e = hipMemcpy(d_codes, codes.data(), codes.size(), hipMemcpyHostToDevice);
    if (e == hipSuccess) e = hipMemcpy(d_secs, secs.data(), secs.size(), hipMemcpyHostToDevice);
    if (e == hipSuccess) e = hipMemcpy(d_reqs, rq.data(), sizeof(SecReqDev) * (size_t)nreq, hipMemcpyHostToDevice);
    if (e == hipSuccess) {
        kernel<<<nreq, FMDBZP_SEC_NTHR, lds_bytes, plan->stream>>>(
            dev_sig ? signal : plan->d_signal, spc, d_reqs, d_out);
        e = hipGetLastError();
    }
    if (e == hipSuccess) e = hipMemcpyAsync(out_phase, d_out, sizeof(int32_t) * (size_t)nreq, hipMemcpyDeviceToHost,
                                            plan->stream);
    if (e == hipSuccess) e = hipStreamSynchronize(plan->stream);
    if (e != hipSuccess) return set_err(FMDBZP_EHIP, "fmdbzp_secondary_phase: %s", hipGetErrorString(e));
    return FMDBZP_OK;
}

// Host arithmetic of the results: 44 results of four requests took 210 us in
// numpy and Python, a numpy scalar operation at a time.
int fmdbzp_prn_results(const fmdbzp_prn_stats* stats, int32_t n, int32_t samples_per_code, int32_t num_blocks,
                       int32_t block_size, double sampling_freq_hz, double code_freq_hz, double code_length,
                       double coherent_time_s, double doppler_spacing_hz, int32_t interpolate, fmdbzp_prn_result* out)
{
#pragma clang fp contract(off)
    if (n < 0 || (n > 0 && (!stats || !out))) return set_err(FMDBZP_EINVAL, "fmdbzp_prn_results: null argument");
    if (samples_per_code <= 0 || num_blocks <= 0 || block_size <= 0)
        return set_err(FMDBZP_EINVAL, "fmdbzp_prn_results: sizes must be positive");
    // Julia `mod`: fmod, shifted into the sign of y
    auto jl_mod = [](double x, double y) {
        const double r = fmod(x, y);
        if (r == 0.0) return copysign(0.0, y);
        return (r > 0) != (y > 0) ? r + y : r;
    };
    // `_parabolic_interp` in Float32; false where the denominator is zero
    auto parabola = [](float left, float peak, float right, float* frac) {
        const float denom = 2.f * ((2.f * peak - left) - right);
        if (denom == 0.f) return false;
        *frac = (right - left) / denom;
        return true;
    };
    for (int i = 0; i < n; i++) {
        const fmdbzp_prn_stats& q = stats[i];
        fmdbzp_prn_result& o = out[i];
        const float signal = q.peak_power - q.noise_power;
        o.peak_to_noise = (signal + q.noise_power) / q.noise_power;
        const double ratio = (double)(signal / q.noise_power);
        o.cn0_dbhz = ratio > 0 ? 10 * log10(ratio / coherent_time_s) : ratio == 0 ? -INFINITY : NAN;
        const int col = q.peak_col % samples_per_code, br = col / block_size;
        const int delay = ((num_blocks - br) % num_blocks) * block_size + col % block_size;
        o.code_phase = jl_mod((double)-delay * code_freq_hz / sampling_freq_hz, code_length);
        o.doppler_offset = 0.0;
        o.reserved = 0;
        if (interpolate) {
            const float sq = sqrtf(q.noise_power);
            float frac;
            if ((q.code_right > q.code_left ? q.code_right : q.code_left) > sq &&
                parabola(q.code_left, q.peak_power, q.code_right, &frac))
                o.code_phase = jl_mod((double)-((float)delay + frac) * code_freq_hz / sampling_freq_hz, code_length);
            if ((q.dop_right > q.dop_left ? q.dop_right : q.dop_left) > sq &&
                parabola(q.dop_left, q.peak_power, q.dop_right, &frac))
                o.doppler_offset = (double)frac * doppler_spacing_hz;
        }
    }
    return FMDBZP_OK;
}

int fmdbzp_plan_tuning(fmdbzp_plan* plan, char* buf, size_t buflen)
{
    if (!plan) return set_err(FMDBZP_EHANDLE, "null plan");
    if (!buf || buflen == 0) return set_err(FMDBZP_EINVAL, "null buffer");
    std::lock_guard<std::mutex> lk(plan->mu);
    snprintf(buf, buflen, "%s", plan->tuning.c_str());
    return FMDBZP_OK;
}

int fmdbzp_plan_column_kernel(fmdbzp_plan* plan, char* buf, size_t buflen)
{
    if (!plan) return set_err(FMDBZP_EHANDLE, "null plan");
    if (!buf || buflen == 0) return set_err(FMDBZP_EINVAL, "null buffer");
    column_name(plan, buf, buflen);
    return FMDBZP_OK;
}

int fmdbzp_full_period_form(int32_t samples_per_code, int32_t num_blocks, int32_t num_coh, int32_t num_noncoherent,
                            int32_t nprn)
{
    if (samples_per_code <= 0 || num_blocks <= 0 || num_coh <= 0 || num_noncoherent <= 0 || nprn <= 0)
        return set_err(FMDBZP_EINVAL, "fmdbzp_full_period_form: sizes must be positive");
    const int64_t ndop = (int64_t)num_coh * num_blocks;
    if (num_coh > kFullMaxCoh || samples_per_code > 65535 ||
        ndop * nprn > (int64_t)(FMDBZP_FULL_SPECTRA_MAX_BYTES / sizeof(float2)) ||
        full_spectra_bytes(nprn, ndop, samples_per_code) > FMDBZP_FULL_SPECTRA_MAX_BYTES)
        return FMDBZP_FULL_NONE;
    FullPlanDev fp{};
    Full31Dev fp31{};
    int nthr = 0;
    size_t lds = 0;
    const int form = full_form(samples_per_code, num_noncoherent > 1, &fp, &fp31, &nthr, &lds);
    if (full_few_rows(samples_per_code, num_noncoherent > 1, form == FMDBZP_FULL_AXIS31, ndop * nprn))
        return FMDBZP_FULL_NONE;
    return form;
}

int fmdbzp_plan_call_kernels(fmdbzp_plan* plan, int32_t eltype, int32_t nreq, uint32_t flags, char* buf, size_t buflen)
{
    g_err.clear();
    if (!plan) return set_err(FMDBZP_EHANDLE, "null plan");
    if (!buf || buflen == 0) return set_err(FMDBZP_EINVAL, "null buffer");
    if (nreq <= 0) return set_err(FMDBZP_EINVAL, "nreq must be positive");
    if (!elsize(eltype) && eltype != FMDBZP_C2BIT) return set_err(FMDBZP_EINVAL, "unknown eltype %d", eltype);
    std::lock_guard<std::mutex> lk(plan->mu);
    const fmdbzp_plan* P = plan;
    if (full_call(P, nreq, (flags & FMDBZP_FLAG_STORE_SURFACES) != 0)) {
        if (P->fp31.n) snprintf(buf, buflen, "k_full31_corr<%d>", P->full_nthr);
        else snprintf(buf, buflen, "k_full_corr<%d,%s>", P->full_nthr, P->d.num_noncoherent > 1 ? "true" : "false");
        return FMDBZP_OK;
    }
    const char* half = P->tile_half || (P->tile_auto && int_samples(eltype)) ? ",fp16" : "";
    static const char* const corr_of[] = {"1,false", "1,true", "2,true", "2,true,2048", "1,true,2500", "2,true,500",
                                          "10,true,400", "5,true,800", "2,true,2000", "1,true,4000"};
    char corr[64], col[64];
    if (P->corr_variant == 10) snprintf(corr, sizeof corr, "k_corr_fc<%d%s>", P->fc_nthr, half);
    else snprintf(corr, sizeof corr, "k_corr_tile<%s%s>", corr_of[P->corr_variant], half);
    if (P->rot25 && !P->rotmma) snprintf(col, sizeof col, "k_column_rot25<%d>", P->d.num_blocks);
    else if (P->col_static) snprintf(col, sizeof col, "k_column_c160%s<32,512%s>", P->col_pair ? "_pair" : "", half);
    else column_name(P, col, sizeof col);
    snprintf(buf, buflen, "%s %s", corr, col);
    return FMDBZP_OK;
}

int fmdbzp_plan_graph_counts(fmdbzp_plan* plan, int64_t* captures, int64_t* replays)
{
    if (!plan) return set_err(FMDBZP_EHANDLE, "null plan");
    std::lock_guard<std::mutex> lk(plan->mu);
    if (captures) *captures = plan->graph_captures;
    if (replays) *replays = plan->graph_replays;
    return FMDBZP_OK;
}

int fmdbzp_plan_kernel_times(fmdbzp_plan* plan, double* total_ms, int64_t* launches, int32_t n)
{
    if (!plan) return set_err(FMDBZP_EHANDLE, "null plan");
    std::lock_guard<std::mutex> lk(plan->mu);
    for (int i = 0; i < n && i < FMDBZP_K_NUM_CLASSES; i++) {
        if (total_ms) total_ms[i] = plan->tot_ms[i];
        if (launches) launches[i] = plan->launches[i];
    }
    return FMDBZP_K_NUM_CLASSES;
}

}  // extern "C"

namespace {

// The block-correlation kernel variant of the plan, writing an FP32 or an FP16 tile.
template <class TileT>
void launch_corr(fmdbzp_plan* P, dim3 g, hipStream_t st, const float2* sf, const int32_t* req, TileT* tile, int nb,
                 int bs, int ndop, float hscale, int rb0, int nrb)
{
    // Below split_wgs workgroups (2048 by default: under three waves of the
    // device's workgroup slots) split each row's column-block passes over g.z
    // workgroups, at most one pass each.
    const int nt = corr_nt(P->corr_variant);
    const int npass = (nrb + nt - 1) / nt;
    const int wgs = (int)(g.x * g.y);
    g.z = (P->split_wgs <= 0 || wgs >= P->split_wgs) ? 1 : std::min(npass, (P->split_wgs + wgs - 1) / wgs);
    // k_corr_fc keeps nothing between passes: one each. At 180 rows of 15 blocks (F
    // 4096, 1024 slots) 1440 workgroups of two took 49.6 us, 2700 of one 33.4.
    if (P->corr_variant == 10) g.z = std::min(npass, 65535);
    if (P->corr_variant == 10 && P->fc_nthr == 512)
        k_corr_fc<512, TileT><<<g, 512, P->fc_lds, st>>>(sf, P->d_prnconj, req, tile, P->fc, P->d_fc_tw, nb, bs, P->tp,
                                                         ndop, hscale, rb0, nrb);
    else if (P->corr_variant == 10)
        k_corr_fc<256, TileT><<<g, 256, P->fc_lds, st>>>(sf, P->d_prnconj, req, tile, P->fc, P->d_fc_tw, nb, bs, P->tp,
                                                         ndop, hscale, rb0, nrb);
    else if (P->corr_variant == 6)
        k_corr_tile<10, true, 400, TileT><<<g, FMDBZP_NTHR, P->corr_lds, st>>>(
            sf, P->d_prnconj, req, tile, P->pf, P->d_twF, nb, bs, P->tp, ndop, P->tile_scale, hscale, rb0, nrb);
    else if (P->corr_variant == 7)
        k_corr_tile<5, true, 800, TileT><<<g, FMDBZP_NTHR, P->corr_lds, st>>>(
            sf, P->d_prnconj, req, tile, P->pf, P->d_twF, nb, bs, P->tp, ndop, P->tile_scale, hscale, rb0, nrb);
    else if (P->corr_variant == 8)
        k_corr_tile<2, true, 2000, TileT><<<g, FMDBZP_NTHR, P->corr_lds, st>>>(
            sf, P->d_prnconj, req, tile, P->pf, P->d_twF, nb, bs, P->tp, ndop, P->tile_scale, hscale, rb0, nrb);
    else if (P->corr_variant == 9)
        k_corr_tile<1, true, 4000, TileT><<<g, FMDBZP_NTHR, P->corr_lds, st>>>(
            sf, P->d_prnconj, req, tile, P->pf, P->d_twF, nb, bs, P->tp, ndop, P->tile_scale, hscale, rb0, nrb);
    else if (P->corr_variant == 5)
        k_corr_tile<2, true, 500, TileT><<<g, FMDBZP_NTHR, P->corr_lds, st>>>(
            sf, P->d_prnconj, req, tile, P->pf, P->d_twF, nb, bs, P->tp, ndop, P->tile_scale, hscale, rb0, nrb);
    else if (P->corr_variant == 4)
        k_corr_tile<1, true, 2500, TileT><<<g, FMDBZP_NTHR, P->corr_lds, st>>>(
            sf, P->d_prnconj, req, tile, P->pf, P->d_twF, nb, bs, P->tp, ndop, P->tile_scale, hscale, rb0, nrb);
    else if (P->corr_variant == 3)
        k_corr_tile<2, true, 2048, TileT><<<g, FMDBZP_NTHR, P->corr_lds, st>>>(
            sf, P->d_prnconj, req, tile, P->pf, P->d_twF, nb, bs, P->tp, ndop, P->tile_scale, hscale, rb0, nrb);
    else if (P->corr_variant == 2)
        k_corr_tile<2, true, 0, TileT><<<g, FMDBZP_NTHR, P->corr_lds, st>>>(
            sf, P->d_prnconj, req, tile, P->pf, P->d_twF, nb, bs, P->tp, ndop, P->tile_scale, hscale, rb0, nrb);
    else if (P->corr_variant == 1)
        k_corr_tile<1, true, 0, TileT><<<g, FMDBZP_NTHR, P->corr_lds, st>>>(
            sf, P->d_prnconj, req, tile, P->pf, P->d_twF, nb, bs, P->tp, ndop, P->tile_scale, hscale, rb0, nrb);
    else
        k_corr_tile<1, false, 0, TileT><<<g, FMDBZP_NTHR, P->corr_lds, st>>>(
            sf, P->d_prnconj, req, tile, P->pf, P->d_twF, nb, bs, P->tp, ndop, P->tile_scale, hscale, rb0, nrb);
}

// Device buffers one search runs on: the plan's own workspace
// (fmdbzp_acquire) or the library's static scratch (fmdbzp_acquire_noalloc).
struct Work {
    float2* sigfft;
    float2* tile;
    float* acc;
    double* rowsum;
    float* rowbest_v;
    uint64_t* rowbest_k;
    double* psum;
    float* pbest_v;
    uint64_t* pbest_k;
    const int32_t* req;          // nreq PRN indices
    fmdbzp_prn_stats* stats;     // nreq statistics
    int batch;                   // PRNs per workspace pass
    int nlanes;
    bool timing;                 // record HIP events around launches (plan timing)
    float2* tile2;               // second step's tile of two-step column launches; null: one step per launch
};

int acquire_launch(fmdbzp_plan* P, const Work& W, const void* d_sig, int32_t eltype, double interm_freq_hz,
                   int32_t nreq, uint32_t flags, float* const* out_surfaces);

// Enqueue one search on the plan's stream; statistics land in the plan's
// pinned staging buffer and are returned by acquire_finish. The caller holds
// the plan's mutex.
int acquire_enqueue(fmdbzp_plan* P, const void* signal, int32_t eltype, int64_t n_samples,
                    double interm_freq_hz, const int32_t* prn_index, int32_t nreq, uint32_t flags,
                    fmdbzp_prn_stats* out_stats, float* const* out_surfaces)
{
    const fmdbzp_plan_desc& d = P->d;
    const bool store = (flags & FMDBZP_FLAG_STORE_SURFACES) != 0;
    const int ndop = d.num_doppler_bins;
    const int spc = d.samples_per_code, spc_eff = d.samples_per_code_eff, nnc = d.num_noncoherent;
    const int64_t seglen = (int64_t)d.num_coh * spc;
    if (n_samples / seglen < nnc)
        return set_err(FMDBZP_EINVAL, "signal has %lld samples, fewer than %d segments of %lld",
                       (long long)n_samples, nnc, (long long)seglen);
    HIP_TRY(hipSetDevice(P->device));

    // signal: only the N_nc segments the search reads cross the bus
    const size_t nsig = (size_t)seglen * nnc;
    const size_t sig_bytes = eltype == FMDBZP_C2BIT ? (nsig + 1) / 2 : nsig * elsize(eltype);
    const void* d_sig = signal;
    if (!(flags & FMDBZP_FLAG_DEVICE_SIGNAL)) {
        if (P->signal_cap < sig_bytes) {
            hipFree(P->d_signal);
            P->d_signal = nullptr;
            P->signal_cap = 0;
            HIP_TRY(hipMalloc(&P->d_signal, sig_bytes));
            P->signal_cap = sig_bytes;
        }
        if (P->h_signal_cap < sig_bytes) {
            hipHostFree(P->h_signal);
            P->h_signal = nullptr;
            P->h_signal_cap = 0;
            HIP_TRY(hipHostMalloc(&P->h_signal, sig_bytes, hipHostMallocDefault));
            P->h_signal_cap = sig_bytes;
        }
        memcpy(P->h_signal, signal, sig_bytes);
        HIP_TRY(hipMemcpyAsync(P->d_signal, P->h_signal, sig_bytes, hipMemcpyHostToDevice, P->stream));
        d_sig = P->d_signal;
    }
    if (P->req_cap < (size_t)nreq) {
        hipFree(P->d_req);
        hipFree(P->d_stats);
        hipHostFree(P->h_req);
        hipHostFree(P->h_stats);
        P->d_req = nullptr;
        P->d_stats = nullptr;
        P->h_req = nullptr;
        P->h_stats = nullptr;
        P->req_cap = 0;
        HIP_TRY(hipMalloc((void**)&P->d_req, sizeof(int32_t) * nreq));
        HIP_TRY(hipMalloc((void**)&P->d_stats, sizeof(fmdbzp_prn_stats) * nreq));
        HIP_TRY(hipHostMalloc((void**)&P->h_req, sizeof(int32_t) * nreq, hipHostMallocDefault));
        HIP_TRY(hipHostMalloc((void**)&P->h_stats, sizeof(fmdbzp_prn_stats) * nreq, hipHostMallocDefault));
        P->req_cap = (size_t)nreq;
        P->req_n = 0;
    }
    // A call that repeats the previous PRN list reuses the device copy: every
    // call synchronizes before it returns, so no upload is still in flight.
    if (P->req_n != nreq || memcmp(P->h_req, prn_index, sizeof(int32_t) * nreq) != 0) {
        P->req_n = 0;
        memcpy(P->h_req, prn_index, sizeof(int32_t) * nreq);
        HIP_TRY(hipMemcpyAsync(P->d_req, P->h_req, sizeof(int32_t) * nreq, hipMemcpyHostToDevice, P->stream));
        P->req_n = nreq;
    }
    const size_t surf_cols = P->surf_bins > 0 ? (size_t)P->surf_bins : (size_t)spc_eff;
    if (store && !P->d_export && !(flags & FMDBZP_FLAG_DEVICE_OUTPUT))
        HIP_TRY(hipMalloc((void**)&P->d_export, sizeof(float) * (size_t)ndop * surf_cols * kLanes));

    Work W{P->d_sigfft, P->d_tile, P->d_acc, P->d_rowsum, P->d_rowbest_v, P->d_rowbest_k, P->d_psum,
           P->d_pbest_v, P->d_pbest_k, P->d_req, P->d_stats, P->batch, P->nlanes, true,
           P->col_pair ? P->d_tile2 : nullptr};
    if (P->use_graph && !P->timing && !store && W.nlanes == 1) {
        // the same kernels with the same arguments as the last captured call:
        // replay its graph; otherwise capture this call's sequence
        const bool same = P->graph_exec && P->g_sig == d_sig && P->g_req == P->d_req && P->g_stats == P->d_stats &&
                          P->g_eltype == eltype && P->g_if == interm_freq_hz && P->g_flags == flags &&
                          P->g_nreq == nreq && memcmp(P->g_prns.data(), prn_index, sizeof(int32_t) * nreq) == 0;
        if (!same) {
            if (P->graph_exec) hipGraphExecDestroy(P->graph_exec);
            if (P->graph) hipGraphDestroy(P->graph);
            P->graph_exec = nullptr;
            P->graph = nullptr;
            HIP_TRY(hipStreamBeginCapture(P->stream, hipStreamCaptureModeThreadLocal));
            const int rc = acquire_launch(P, W, d_sig, eltype, interm_freq_hz, nreq, flags, out_surfaces);
            hipGraph_t g = nullptr;
            const hipError_t e = hipStreamEndCapture(P->stream, &g);
            if (rc) {
                if (e == hipSuccess && g) hipGraphDestroy(g);
                return rc;
            }
            if (e != hipSuccess) return set_err(FMDBZP_EHIP, "graph capture failed: %s", hipGetErrorString(e));
            P->graph = g;
            HIP_TRY(hipGraphInstantiate(&P->graph_exec, g, nullptr, nullptr, 0));
            P->g_sig = d_sig;
            P->g_req = P->d_req;
            P->g_stats = P->d_stats;
            P->g_eltype = eltype;
            P->g_if = interm_freq_hz;
            P->g_flags = flags;
            P->g_nreq = nreq;
            P->g_prns.assign(prn_index, prn_index + nreq);
            P->graph_captures++;
        } else {
            P->graph_replays++;
        }
        HIP_TRY(hipGraphLaunch(P->graph_exec, P->stream));
    } else {
        const int rc = acquire_launch(P, W, d_sig, eltype, interm_freq_hz, nreq, flags, out_surfaces);
        if (rc) return rc;
    }
    HIP_TRY(hipMemcpyAsync(P->h_stats, P->d_stats, sizeof(fmdbzp_prn_stats) * nreq, hipMemcpyDeviceToHost,
                           P->stream));
    P->pending_out = out_stats;
    P->pending_n = nreq;
    return FMDBZP_OK;
}

// Direct rotation search at large ndop (k_column_rotbig) in code-column
// chunks, on the plan's stream. For each PRN batch and chunk, every step
// builds the tile of the column blocks whose drifted cells reach the chunk's
// window and accumulates them into it (cells in step order, as the whole
// accumulator would); the chunk is then reduced to per-row partials carrying
// the best cell's neighbours (and per-column sums for GlobalMean). The
// partials of all chunks give the statistics without a whole-surface
// accumulator.
int launch_rotbig(fmdbzp_plan* P, const Work& W, ColumnArgs A, int32_t nreq, bool store, float* const* out_surfaces,
                  uint32_t flags)
{
    const fmdbzp_plan_desc& d = P->d;
    const int F = d.fft_size, ndop = d.num_doppler_bins, nb = d.num_blocks, bs = d.block_size;
    const int spc = d.samples_per_code, spc_eff = d.samples_per_code_eff, nnc = d.num_noncoherent;
    const int R = d.num_secondary_rotations;
    const int streamed_rot = nnc == 1 ? 1 : 0;
    const size_t tile_per_prn = (size_t)P->nrb_max * ndop * P->tp;
    hipStream_t st = P->stream;
    A.acc_ldr = 1;
    A.acc_ldc = P->apc;
    for (int b0 = 0; b0 < nreq; b0 += W.batch) {
        const int cnt = std::min(W.batch, nreq - b0);
        const int32_t* req = W.req + b0;
        A.req = req;
        A.tile = W.tile;
        A.acc = W.acc;
        for (int ci = 0; ci < P->nchunks; ci++) {
            const int c0 = ci * P->chunk_cols;
            const int own = std::min(P->chunk_cols, spc - c0);
            const int win0 = P->halo ? (c0 - 1 + spc) % spc : 0;
            const int winlen = own + 2 * P->halo;
            A.win0 = win0;
            A.winlen = winlen;
            A.slice_cols = P->win_max;
            for (int s = 0; s < nnc; s++) {
                // source columns [win0 - smax, win0 + winlen - smin) reach the window
                int rb0 = 0, nrb = nb;
                const int lo = win0 - P->smax[(size_t)s], hi = win0 + winlen - P->smin[(size_t)s];
                if (hi - lo < spc) {
                    const int b_lo = (int)std::floor((double)lo / bs);
                    const int b_hi = (int)std::floor((double)(hi - 1) / bs);
                    nrb = std::min(nb, b_hi - b_lo + 1);
                    rb0 = ((b_lo % nb) + nb) % nb;
                }
                if (nrb > P->nrb_max) return set_err(FMDBZP_EINVAL, "chunk tile needs %d blocks > %d", nrb, P->nrb_max);
                A.rb0 = rb0;
                A.nrb = nrb;
                {
                    Timed t(P, FMDBZP_K_CORR_TILE, st, W.timing);
                    const float2* sf = W.sigfft + (size_t)s * ndop * F;
                    launch_corr(P, dim3(ndop, cnt), st, sf, req, W.tile, nb, bs, ndop, 0.f, rb0, nrb);
                    HIP_TRY(hipGetLastError());
                }
                A.shifts = P->d_shifts + (size_t)s * ndop;
                A.first_step = s == 0;
                {
                    Timed t(P, FMDBZP_K_COLUMN, st, W.timing);
                    const dim3 g(bs, nrb, cnt);
                    const int nt = P->rotbig_nt;
                    if (P->rotmma) {
                        switch (P->rotmma) {
                        case 20: k_column_rotmma<8, 3, 20><<<g, 512, P->col_lds, st>>>(A); break;
                        case 10: k_column_rotmma<4, 3, 10><<<g, 256, P->col_lds, st>>>(A); break;
                        case 4: k_column_rotmma<4, 1, 4><<<g, 256, P->col_lds, st>>>(A); break;
                        case 2: k_column_rotmma<2, 1, 2><<<g, 128, P->col_lds, st>>>(A); break;
                        default: return set_err(FMDBZP_EINVAL, "no matrix-core rotation kernel for n1 = %d", P->rotmma);
                        }
                    } else if (P->rot25) {
                        switch (nb) {
#define R25_LAUNCH(NN)                                                                                     \
    case NN:                                                                                               \
        k_column_rot25<NN, true><<<dim3((bs + Rot25<NN>::C - 1) / Rot25<NN>::C, nrb, cnt), Rot25<NN>::NT, \
                                   rot25_lds<NN>(), st>>>(A);                                              \
        break;
                            R25_LAUNCH(50) R25_LAUNCH(100) R25_LAUNCH(250) R25_LAUNCH(500)
#undef R25_LAUNCH
                        default: return set_err(FMDBZP_EINVAL, "no rotation kernel for %d rows", nb);
                        }
                    } else {
                        switch (nt) {
                        case 64: k_column_rotbig<64, 25><<<g, 64, P->col_lds, st>>>(A, P->prow, P->d_twR, P->rgrp); break;
                        case 128: k_column_rotbig<128, 25><<<g, 128, P->col_lds, st>>>(A, P->prow, P->d_twR, P->rgrp); break;
                        case 256: k_column_rotbig<256, 25><<<g, 256, P->col_lds, st>>>(A, P->prow, P->d_twR, P->rgrp); break;
                        case 320: k_column_rotbig<320, 25><<<g, 320, P->col_lds, st>>>(A, P->prow, P->d_twR, P->rgrp); break;
                        case 512: k_column_rotbig<512, 25><<<g, 512, P->col_lds, st>>>(A, P->prow, P->d_twR, P->rgrp); break;
                        default: return set_err(FMDBZP_EINVAL, "no rotation kernel for %d threads", nt);
                        }
                    }
                    HIP_TRY(hipGetLastError());
                }
            }
            {
                Timed t(P, FMDBZP_K_REDUCE, st, W.timing);
                const int rb4 = (ndop + 4 * FMDBZP_NTHR - 1) / (4 * FMDBZP_NTHR);
                k_reduce_chunk<<<dim3(R * P->nsub, rb4, cnt), FMDBZP_NTHR, 0, st>>>(
                    W.acc, P->acc_ps, P->apc, P->win_max, ndop, spc, R, streamed_rot, win0, P->halo, own,
                    P->nchunks == 1 ? 1 : 0, P->red_cw, P->nsub, ci * R * P->nsub, P->nparts, W.psum, W.pbest_v,
                    W.pbest_k, P->d_pnbr);
                HIP_TRY(hipGetLastError());
                if (d.noise_estimator == FMDBZP_NOISE_GLOBAL_MEAN) {
                    k_colsum_chunk<<<dim3(own, R, cnt), FMDBZP_NTHR, 0, st>>>(W.acc, P->acc_ps, P->apc, P->win_max,
                                                                              ndop, spc, spc_eff, win0, P->halo,
                                                                              P->d_colsum);
                    HIP_TRY(hipGetLastError());
                }
            }
            if (store) {  // one chunk covers the code period: the window is the whole surface
                const bool dev_out = (flags & FMDBZP_FLAG_DEVICE_OUTPUT) != 0;
                const size_t surf_cols = P->surf_bins > 0 ? (size_t)P->surf_bins : (size_t)spc_eff;
                for (int p = 0; p < cnt; p++) {
                    float* dst = out_surfaces[b0 + p];
                    if (!dst) continue;
                    float* stage = dev_out ? dst : P->d_export;
                    {
                        Timed t(P, FMDBZP_K_EXPORT, st, W.timing);
                        if (P->surf_bins > 0) {
                            dim3 g(P->surf_bins, (ndop + FMDBZP_NTHR - 1) / FMDBZP_NTHR);
                            k_export_chip<<<g, FMDBZP_NTHR, 0, st>>>(W.acc + (size_t)p * P->acc_ps, stage,
                                                                     P->d_chip_order, ndop, spc, R, P->surf_bins, 1,
                                                                     P->apc);
                        } else {
                            dim3 g(spc_eff, (ndop + FMDBZP_NTHR - 1) / FMDBZP_NTHR);
                            k_export_cm<<<g, FMDBZP_NTHR, 0, st>>>(W.acc + (size_t)p * P->acc_ps, stage, ndop, P->apc);
                        }
                        HIP_TRY(hipGetLastError());
                    }
                    if (!dev_out)
                        HIP_TRY(hipMemcpyAsync(dst, stage, sizeof(float) * (size_t)ndop * surf_cols,
                                               hipMemcpyDeviceToHost, st));
                }
            }
        }
        {
            Timed t(P, FMDBZP_K_REDUCE, st, W.timing);
            k_merge_rows_nbr<<<dim3((ndop + FMDBZP_NTHR - 1) / FMDBZP_NTHR, cnt), FMDBZP_NTHR, 0, st>>>(
                W.psum, W.pbest_v, W.pbest_k, P->d_pnbr, P->nparts, ndop, W.rowsum, W.rowbest_v, W.rowbest_k,
                P->d_rownbr);
            HIP_TRY(hipGetLastError());
        }
        {
            Timed t(P, FMDBZP_K_FINALIZE, st, W.timing);
            k_finalize_chunked<<<dim3(cnt), FMDBZP_NTHR, 0, st>>>(W.rowsum, W.rowbest_v, W.rowbest_k, P->d_rownbr,
                                                                   P->d_colsum, ndop, spc, spc_eff, R, streamed_rot,
                                                                   d.noise_estimator, d.samples_per_chip,
                                                                   W.stats + b0);
            HIP_TRY(hipGetLastError());
        }
    }
    (void)tile_per_prn;
    return FMDBZP_OK;
}

// Full-period correlation search (full_corr.hpp) on the plan's stream.
int launch_full(fmdbzp_plan* P, const Work& W, const void* d_sig, int32_t eltype, double interm_freq_hz, int32_t nreq)
{
    const fmdbzp_plan_desc& d = P->d;
    const int n = d.samples_per_code, ncoh = d.num_coh, nnc = d.num_noncoherent, ndop = d.num_doppler_bins;
    const int do_if = interm_freq_hz == 0.0 ? 0 : (d.options & FMDBZP_OPT_FP64_PHASE) ? 2 : 1;
    const double dstep = (-6.283185307179586 * interm_freq_hz) / d.sampling_freq_hz;  // Julia `2π`
    hipStream_t st = P->stream;
    {
        Timed t(P, FMDBZP_K_SIGNAL_FFT, st, W.timing);
        if (ncoh > 1) {
            k_full_fold<<<dim3((n + 255) / 256, (ncoh + FC_FOLD_SB - 1) / FC_FOLD_SB, nnc), 256,
                          sizeof(float2) * (size_t)ncoh, st>>>(d_sig, eltype, W.sigfft, n, ncoh, do_if, (float)dstep,
                                                               dstep);
            HIP_TRY(hipGetLastError());
        }
        if (P->fp31.n)
            k_full31_signal<512><<<dim3(ncoh, nnc), 512, P->full_lds, st>>>(d_sig, eltype, W.sigfft, P->fp31, do_if,
                                                                            (float)dstep, dstep);
        else
            k_full_signal<512><<<dim3(ncoh, nnc), 512, P->full_lds, st>>>(d_sig, eltype, W.sigfft, P->fp,
                                                                          P->d_full_tw, do_if, (float)dstep, dstep);
        HIP_TRY(hipGetLastError());
    }
    FullArgs A{P->fp, P->d_full_tw, W.sigfft, P->d_full_code, P->d_full_map, P->d_shifts, nullptr, W.acc, W.rowsum,
               W.rowbest_v, W.rowbest_k, ncoh, ndop, nnc, 0, P->ap};
    Full31Args B{P->fp31, W.sigfft, P->d_full_code, (const uint32_t*)P->d_full_map, P->d_shifts, nullptr, W.acc, W.rowsum,
                 W.rowbest_v, W.rowbest_k, ncoh, ndop, nnc, 0, P->ap};
    for (int b0 = 0; b0 < nreq; b0 += W.batch) {
        const int cnt = std::min(W.batch, nreq - b0);
        A.cnt = B.cnt = cnt;
        A.req = B.req = W.req + b0;
        {
            Timed t(P, FMDBZP_K_COLUMN, st, W.timing);
            const dim3 g((unsigned)(ndop * cnt));
            if (P->fp31.n) {
                switch (P->full_nthr) {
                case 512: k_full31_corr<512><<<g, 512, P->full_lds, st>>>(B); break;
                default: k_full31_corr<256><<<g, 256, P->full_lds, st>>>(B); break;
                }
            } else if (nnc > 1) {
                switch (P->full_nthr) {
                case 1024: k_full_corr<1024, true><<<g, 1024, P->full_lds, st>>>(A); break;
                case 512: k_full_corr<512, true><<<g, 512, P->full_lds, st>>>(A); break;
                default: k_full_corr<256, true><<<g, 256, P->full_lds, st>>>(A); break;
                }
            } else {
                switch (P->full_nthr) {
                case 1024: k_full_corr<1024, false><<<g, 1024, P->full_lds, st>>>(A); break;
                case 512: k_full_corr<512, false><<<g, 512, P->full_lds, st>>>(A); break;
                default: k_full_corr<256, false><<<g, 256, P->full_lds, st>>>(A); break;
                }
            }
            HIP_TRY(hipGetLastError());
        }
        {
            Timed t(P, FMDBZP_K_FINALIZE, st, W.timing);
            k_finalize<<<dim3(cnt), FMDBZP_NTHR, 0, st>>>(W.acc, W.rowsum, W.rowbest_v, W.rowbest_k, ndop, n, n,
                                                          P->acc_ps, P->ap, 1, 1, 0, d.noise_estimator,
                                                          d.samples_per_chip, W.stats + b0);
            HIP_TRY(hipGetLastError());
        }
    }
    return FMDBZP_OK;
}

// Launch a search's kernels on the plan's stream (lanes joined back into it
// before returning). Reads the device signal d_sig; writes W.stats.
int acquire_launch(fmdbzp_plan* P, const Work& W, const void* d_sig, int32_t eltype, double interm_freq_hz,
                   int32_t nreq, uint32_t flags, float* const* out_surfaces)
{
    const fmdbzp_plan_desc& d = P->d;
    const bool store = (flags & FMDBZP_FLAG_STORE_SURFACES) != 0;
    const int F = d.fft_size, ndop = d.num_doppler_bins, nb = d.num_blocks, bs = d.block_size;
    const int spc = d.samples_per_code, spc_eff = d.samples_per_code_eff, nnc = d.num_noncoherent;
    const int64_t seglen = (int64_t)d.num_coh * spc;
    const size_t surf_cols = P->surf_bins > 0 ? (size_t)P->surf_bins : (size_t)spc_eff;
    if (full_call(P, nreq, store)) return launch_full(P, W, d_sig, eltype, interm_freq_hz, nreq);

    // 1. downconvert + double-block FFTs of every segment
    {
        // 1: the reference's Float32 phase argument; 2: FMDBZP_OPT_FP64_PHASE
        const int do_if = interm_freq_hz == 0.0 ? 0 : (d.options & FMDBZP_OPT_FP64_PHASE) ? 2 : 1;
        const double twopi = 6.283185307179586;  // Julia `2π`
        const double dstep = (-twopi * interm_freq_hz) / d.sampling_freq_hz;
        const float step = (float)dstep;
        Timed t(P, FMDBZP_K_SIGNAL_FFT, P->stream, W.timing);
        if (P->corr_variant != 10)
            k_signal_fft<<<dim3(ndop, nnc), FMDBZP_NTHR, P->fft_lds, P->stream>>>(
                d_sig, eltype, W.sigfft, P->pf8, P->d_twF, bs, seglen, ndop, do_if, step, dstep);
        else if (P->fc_nthr == 512)
            k_fc_signal<512><<<dim3(ndop, nnc), 512, P->fc_lds, P->stream>>>(
                d_sig, eltype, W.sigfft, P->fc, P->d_fc_tw, bs, seglen, ndop, do_if, step, dstep);
        else
            k_fc_signal<256><<<dim3(ndop, nnc), 256, P->fc_lds, P->stream>>>(
                d_sig, eltype, W.sigfft, P->fc, P->d_fc_tw, bs, seglen, ndop, do_if, step, dstep);
        HIP_TRY(hipGetLastError());
    }

    const int ndb = d.num_data_bits;
    const int ndc = 1 << (ndb - 1);
    const int bpc = d.num_coh / ndb;
    ColumnArgs A{};
    A.patterns = P->d_patterns;
    A.pset = P->d_pset;
    A.twD = P->d_twD;
    A.pd = P->pd;
    A.nb = nb; A.bs = bs; A.ndop = ndop; A.spc = spc; A.spc_eff = spc_eff;
    A.ncoh = d.num_coh; A.ndb = ndb; A.E = d.bit_edge_search_steps; A.R = d.num_secondary_rotations;
    A.Q = d.num_patterns; A.ndc = ndc; A.edge_step = (bpc * nb) / d.bit_edge_search_steps;
    A.use_max = (ndc > 1 || d.bit_edge_search_steps > 1) ? 1 : 0;
    A.LB = P->LB;
    A.bstride = P->bstride;
    A.sst = P->sst;
    A.literal_edges = (d.options & FMDBZP_OPT_LITERAL_EDGES) ? 1 : 0;
    A.tp = P->tp;
    A.ap = P->ap;
    A.acc_ps = P->acc_ps;
    A.acc_ldr = P->acc_cm ? 1 : P->ap;
    A.acc_ldc = P->acc_cm ? P->apc : 1;
    A.rot_direct = P->rot_direct ? 1 : 0;
    A.win0 = 0;
    A.winlen = spc;
    A.slice_cols = spc;
    A.rb0 = 0;
    A.nrb = nb;
    const int streamed_rot = (nnc == 1 && d.path == FMDBZP_PATH_ROTATION) ? 1 : 0;
    const int nlb = (bs + P->LB - 1) / P->LB;
    // FP16 tile: scale 2^-e with bs * max|sample| * 2^-e below the FP16 range
    // (every tile value is a sum of bs code-weighted samples of that modulus)
    float hscale = 0.f, hinv = 1.f;
    const bool tile_half = P->tile_half || (P->tile_auto && int_samples(eltype));
    if (tile_half) {
        double maxabs = 0.0;
        switch (eltype) {
            case FMDBZP_I16: maxabs = 32768.0; break;
            case FMDBZP_CI8: maxabs = 128.0 * 1.4142135623730951; break;
            case FMDBZP_CI16: maxabs = 32768.0 * 1.4142135623730951; break;
            case FMDBZP_C2BIT: maxabs = 3.0 * 1.4142135623730951; break;
            default:
                return set_err(FMDBZP_EINVAL, "FP16 tiles need integer samples (I16, CI8, CI16, C2BIT)");
        }
        int e = 0;
        while (bs * maxabs * 1.01 / std::ldexp(1.0, e) > 60000.0) e++;
        hscale = (float)std::ldexp(1.0, -e);
        hinv = (float)std::ldexp(1.0, e);
    }

    // fork the lanes off the plan's stream (signal FFT cache, request list);
    // a single lane runs on the plan's stream itself, which saves the two
    // cross-stream dependencies (about 10 us each on the device)
    const bool forked = W.nlanes > 1;
    if (forked) {
        HIP_TRY(hipEventRecord(P->ev_fork, P->stream));
        for (int l = 0; l < W.nlanes; l++) HIP_TRY(hipStreamWaitEvent(P->lane[l], P->ev_fork, 0));
    }
    if (P->rotbig) {
        const int rc = launch_rotbig(P, W, A, nreq, store, out_surfaces, flags);
        if (rc) return rc;
        return FMDBZP_OK;
    }
    const size_t tile_per_prn = (size_t)nb * ndop * P->tp;
    const size_t acc_per_prn = P->acc_ps;
    const bool dev_out = (flags & FMDBZP_FLAG_DEVICE_OUTPUT) != 0;
    for (int b0 = 0; b0 < nreq; b0 += W.batch) {
        const int nbat = nreq - b0 < W.batch ? nreq - b0 : W.batch;
        const int per_lane = (nbat + W.nlanes - 1) / W.nlanes;
        for (int l = 0; l < W.nlanes; l++) {
            // lane l: batch slots [lo, lo + cnt) on its own stream and workspace slice
            const int lo = l * per_lane;
            const int cnt = nbat - lo < per_lane ? nbat - lo : per_lane;
            if (cnt <= 0) continue;
            hipStream_t st = forked ? P->lane[l] : P->stream;
            const int32_t* req = W.req + b0 + lo;
            float2* tile = W.tile + (size_t)lo * tile_per_prn;
            float2* tile2 = W.tile2 ? W.tile2 + (size_t)lo * tile_per_prn : nullptr;
            float* acc = W.acc + (size_t)lo * acc_per_prn;
            double* rowsum = W.rowsum + (size_t)lo * ndop;
            float* rowbest_v = W.rowbest_v + (size_t)lo * ndop;
            uint64_t* rowbest_k = W.rowbest_k + (size_t)lo * ndop;
            A.tile = tile;
            A.tile2 = tile2;
            A.acc = acc;
            A.req = req;
            for (int s = 0; s < nnc; s++) {
                // steps s and s + 1 in one column launch (k_column_c160_pair)
                const bool pair = tile2 && s + 1 < nnc && P->pair_ok[(size_t)s];
                for (int k = 0; k <= (pair ? 1 : 0); k++) {
                    Timed t(P, FMDBZP_K_CORR_TILE, st, W.timing);
                    const dim3 g(ndop, cnt);
                    const float2* sf = W.sigfft + (size_t)(s + k) * ndop * F;
                    float2* tl = k ? tile2 : tile;
                    if (tile_half)
                        launch_corr(P, g, st, sf, req, (__half2*)tl, nb, bs, ndop, hscale, 0, nb);
                    else
                        launch_corr(P, g, st, sf, req, tl, nb, bs, ndop, 0.f, 0, nb);
                    HIP_TRY(hipGetLastError());
                }
                A.shifts = P->d_shifts + (size_t)s * ndop;
                A.shifts2 = pair ? P->d_shifts + (size_t)(s + 1) * ndop : nullptr;
                A.first_step = s == 0;
                {
                    Timed t(P, FMDBZP_K_COLUMN, st, W.timing);
                    const dim3 g(nlb, nb, cnt);
                    if (pair) {
                        if (tile_half)
                            k_column_c160_pair<32, 512, true><<<g, 512, P->col_lds2, st>>>(A, hinv);
                        else
                            k_column_c160_pair<32, 512><<<g, 512, P->col_lds2, st>>>(A, 1.f);
                    } else if (P->col_reg) {
                        const dim3 gr((bs + COLREG_NTHR - 1) / COLREG_NTHR, nb, cnt);
#define CR_LAUNCH(NN) if (ndop == NN) k_column_reg<NN><<<gr, COLREG_NTHR, 0, st>>>(A);
                        COLREG_ALL(CR_LAUNCH)
#undef CR_LAUNCH
                    } else if (P->simple_kernel) {
                        if (P->col_static && tile_half)
                            k_column_c160<32, 512, true><<<g, 512, P->col_lds, st>>>(A, hinv);
                        else if (P->col_static)
                            k_column_c160<32, 512><<<g, 512, P->col_lds, st>>>(A, 1.f);
                        else if (P->col_onebuf)
                            k_column_simple<true><<<g, FMDBZP_COL_NTHR, P->col_lds, st>>>(A);
                        else
                            k_column_simple<false><<<g, FMDBZP_COL_NTHR, P->col_lds, st>>>(A);
                    } else if (P->bitsplit) {
                        const int nt = (BITSPLIT_C * std::max(20, nb) + 63) & ~63;
#define BS_LAUNCH(NN) if (nb == NN) k_column_bitsplit<NN><<<g, nt, P->col_lds, st>>>(A);
                        BITSPLIT_ALL(BS_LAUNCH)
#undef BS_LAUNCH
                    } else if (d.path == FMDBZP_PATH_SIGN) {
                        k_column_sign<<<g, FMDBZP_NTHR, P->col_lds, st>>>(A);
                    } else if (P->rot25) {
                        k_column_rot25<80, false><<<dim3((bs + Rot25<80>::C - 1) / Rot25<80>::C, nb, cnt), Rot25<80>::NT, P->col_lds, st>>>(A);
                    } else if (P->rot2000) {
                        k_column_rot2000<512><<<dim3(bs, nb, cnt), 512, P->col_lds, st>>>(A);
                    } else if (P->rotsplit) {
                        const int C = P->rotsplit;
                        const int nt = (C * std::max(d.num_coh, nb) + 63) & ~63;
                        bool done = false;
#define RS_LAUNCH(PP, NN)                                                          \
    if (d.num_coh == PP && nb == NN) {                                             \
        k_column_rotsplit<PP, NN><<<g, nt, P->col_lds, st>>>(A, C);                \
        done = true;                                                               \
    }
                        ROTSPLIT_ALL(RS_LAUNCH)
#undef RS_LAUNCH
                        if (!done) return set_err(FMDBZP_EINVAL, "no rotation kernel for %d x %d", d.num_coh, nb);
                    } else {
                        k_column_rotation<<<g, FMDBZP_NTHR, P->col_lds, st>>>(A);
                    }
                    HIP_TRY(hipGetLastError());
                }
                if (pair) s++;
            }
            {
                Timed t(P, FMDBZP_K_REDUCE, st, W.timing);
                if (P->acc_cm) {
                    const size_t np = (size_t)cnt * P->red_nchunk * ndop;
                    double* psum = (double*)tile;
                    uint64_t* pbest_k = (uint64_t*)(psum + np);
                    float* pbest_v = (float*)(pbest_k + np);
                    const int rb4 = (ndop + 4 * FMDBZP_NTHR - 1) / (4 * FMDBZP_NTHR);
                    k_reduce_cols<<<dim3(P->red_nchunk, rb4, cnt), FMDBZP_NTHR, 0, st>>>(
                        acc, P->acc_ps, P->apc, ndop, spc, spc_eff, d.num_secondary_rotations, streamed_rot,
                        P->red_cw, psum, pbest_v, pbest_k);
                    HIP_TRY(hipGetLastError());
                    k_merge_rows<<<dim3((ndop + FMDBZP_MERGE_ROWS - 1) / FMDBZP_MERGE_ROWS, cnt), FMDBZP_NTHR, 0, st>>>(
                        psum, pbest_v, pbest_k, P->red_nchunk, ndop, rowsum, rowbest_v, rowbest_k);
                } else {
                    k_reduce_rows<<<dim3(ndop, cnt), FMDBZP_NTHR, 0, st>>>(acc, ndop, spc, spc_eff, P->ap,
                                                                           d.num_secondary_rotations, streamed_rot,
                                                                           rowsum, rowbest_v, rowbest_k);
                }
                HIP_TRY(hipGetLastError());
            }
            {
                Timed t(P, FMDBZP_K_FINALIZE, st, W.timing);
                k_finalize<<<dim3(cnt), FMDBZP_NTHR, 0, st>>>(acc, rowsum, rowbest_v, rowbest_k, ndop, spc, spc_eff,
                                                              P->acc_ps, A.acc_ldr, A.acc_ldc,
                                                              d.num_secondary_rotations, streamed_rot,
                                                              d.noise_estimator, d.samples_per_chip,
                                                              W.stats + b0 + lo);
                HIP_TRY(hipGetLastError());
            }
            if (store) {
                float* stage = dev_out ? nullptr : P->d_export + (size_t)l * ndop * surf_cols;
                for (int p = 0; p < cnt; p++) {
                    float* dst = out_surfaces[b0 + lo + p];
                    if (!dst) continue;
                    {
                        Timed t(P, FMDBZP_K_EXPORT, st, W.timing);
                        if (P->surf_bins > 0) {
                            dim3 g(P->surf_bins, (ndop + FMDBZP_NTHR - 1) / FMDBZP_NTHR);
                            k_export_chip<<<g, FMDBZP_NTHR, 0, st>>>(acc + (size_t)p * acc_per_prn, dev_out ? dst : stage,
                                                                     P->d_chip_order, ndop, spc,
                                                                     d.num_secondary_rotations, P->surf_bins,
                                                                     A.acc_ldr, A.acc_ldc);
                        } else if (P->acc_cm) {
                            dim3 g(spc_eff, (ndop + FMDBZP_NTHR - 1) / FMDBZP_NTHR);
                            k_export_cm<<<g, FMDBZP_NTHR, 0, st>>>(acc + (size_t)p * acc_per_prn,
                                                                   dev_out ? dst : stage, ndop, P->apc);
                        } else {
                            dim3 g((spc_eff + 31) / 32, (ndop + 31) / 32);
                            k_export<<<g, dim3(32, 8), 0, st>>>(acc + (size_t)p * acc_per_prn,
                                                                dev_out ? dst : stage, ndop, spc_eff, P->ap);
                        }
                        HIP_TRY(hipGetLastError());
                    }
                    if (!dev_out)
                        HIP_TRY(hipMemcpyAsync(dst, stage, sizeof(float) * (size_t)ndop * surf_cols,
                                               hipMemcpyDeviceToHost, st));
                }
            }
        }
    }
    // join the lanes back into the plan's stream
    for (int l = 0; forked && l < W.nlanes; l++) {
        HIP_TRY(hipEventRecord(P->ev_join[l], P->lane[l]));
        HIP_TRY(hipStreamWaitEvent(P->stream, P->ev_join[l], 0));
    }
    return FMDBZP_OK;
}

struct TuneKey {
    int F, nb, bs, ndop, batch, ncol_kind, LB;
    bool operator==(const TuneKey& o) const
    {
        return F == o.F && nb == o.nb && bs == o.bs && ndop == o.ndop && batch == o.batch && ncol_kind == o.ncol_kind &&
               LB == o.LB;
    }
};
struct TuneChoice {
    int corr_variant, split_wgs, LB;
    std::string record;
};
std::mutex g_tune_mu;
std::vector<std::pair<TuneKey, TuneChoice>> g_tune_cache;

// Launch-configuration autotuner (FMDBZP_OPT_AUTOTUNE): the reference plans
// its FFTs by measurement (FFTW MEASURE, src/plan.jl:468-483); here the
// kernels are fixed and what is measured is how they are launched. On one
// step's worth of the plan's own workspace (zeroed signal spectra; the
// timings do not depend on the values) it times every admissible block-
// correlation variant (ping-pong, in place with one or two transforms per
// pass) for each pass-split width, and for the generic simple column kernel
// the columns per workgroup, with HIP events, and keeps the fastest. Every
// candidate runs the same transforms; the variants differ only in buffering
// and work partition. Choices are cached per geometry for the process.
int autotune(fmdbzp_plan* P)
{
    const fmdbzp_plan_desc& d = P->d;
    const int F = d.fft_size, ndop = d.num_doppler_bins, nb = d.num_blocks, bs = d.block_size;
    const int cnt = std::min(P->batch, P->nprn);
    const bool col_generic = P->simple_kernel && !P->col_static && !P->col_reg;
    const TuneKey key{F, nb, bs, ndop, cnt, col_generic ? 1 : 0, P->LB};
    {
        std::lock_guard<std::mutex> g(g_tune_mu);
        for (auto& e : g_tune_cache)
            if (e.first == key) {
                P->corr_variant = e.second.corr_variant;
                P->split_wgs = e.second.split_wgs;
                P->corr_lds = corr_lds_of(P, P->corr_variant);
                if (col_generic && e.second.LB != P->LB) {
                    P->LB = e.second.LB;
                    P->col_lds = (size_t)P->bstride * (P->col_onebuf ? 1 : 2) * sizeof(float2) * P->LB;
                }
                P->tuning = e.second.record + " (cached)";
                return FMDBZP_OK;
            }
    }
    std::vector<int> variants;
    if (P->corr_variant >= 3) variants.push_back(P->corr_variant);  // compile-time transform
    else {
        if (fft_inplace_ok(P->pf) && 2 * F <= FMDBZP_CORR_MAXV * FMDBZP_NTHR) variants.push_back(2);
        if (fft_inplace_ok(P->pf) && F <= FMDBZP_CORR_MAXV * FMDBZP_NTHR) variants.push_back(1);
        variants.push_back(0);
    }
    int rc;
    for (int v : variants) {
        const size_t lds = corr_lds_of(P, v);
        if (lds > kLdsMax) continue;
        if ((rc = set_lds_attr((const void*)k_corr_tile<2, true>, lds)) ||
            (rc = set_lds_attr((const void*)k_corr_tile<1, true>, lds)) ||
            (rc = set_lds_attr((const void*)k_corr_tile<1, false>, lds)) ||
            (rc = set_lds_attr((const void*)k_corr_tile<2, true, 0, __half2>, lds)) ||
            (rc = set_lds_attr((const void*)k_corr_tile<1, true, 0, __half2>, lds)) ||
            (rc = set_lds_attr((const void*)k_corr_tile<1, false, 0, __half2>, lds)))
            return rc;
    }
    int32_t* d_req = nullptr;
    std::vector<int32_t> h_req((size_t)cnt);
    for (int i = 0; i < cnt; i++) h_req[(size_t)i] = i;
    if ((rc = dev_alloc(&d_req, (size_t)cnt))) return rc;
    hipEvent_t e0 = nullptr, e1 = nullptr;
    auto cleanup = [&]() {
        hipFree(d_req);
        if (e0) hipEventDestroy(e0);
        if (e1) hipEventDestroy(e1);
    };
    hipStream_t st = P->stream;
    if (hipEventCreate(&e0) != hipSuccess || hipEventCreate(&e1) != hipSuccess ||
        hipMemcpy(d_req, h_req.data(), sizeof(int32_t) * cnt, hipMemcpyHostToDevice) != hipSuccess ||
        hipMemsetAsync(P->d_sigfft, 0, sizeof(float2) * (size_t)ndop * F, st) != hipSuccess) {
        cleanup();
        return set_err(FMDBZP_EHIP, "autotune set-up failed");
    }
    auto time_it = [&](auto&& launch) -> float {
        launch();  // warm
        float best = 1e30f;
        for (int rep = 0; rep < 3; rep++) {
            hipEventRecord(e0, st);
            launch();
            hipEventRecord(e1, st);
            float ms = 0.f;
            if (hipEventSynchronize(e1) != hipSuccess || hipEventElapsedTime(&ms, e0, e1) != hipSuccess) return 1e30f;
            best = std::min(best, ms);
        }
        return best;
    };
    char buf[512];
    std::string rec;
    int best_v = P->corr_variant, best_split = P->split_wgs;
    float best_ms = 1e30f;
    for (int v : variants) {
        if (corr_lds_of(P, v) > kLdsMax) continue;
        for (int split : {0, 2048, 4096}) {
            P->corr_variant = v;
            P->split_wgs = split;
            P->corr_lds = corr_lds_of(P, v);
            const float ms = time_it([&]() {
                launch_corr(P, dim3(ndop, cnt), st, P->d_sigfft, d_req, P->d_tile, nb, bs, ndop, 0.f, 0, nb);
            });
            snprintf(buf, sizeof(buf), " corr v%d split %d: %.4f ms;", v, split, ms);
            rec += buf;
            if (ms < best_ms) {
                best_ms = ms;
                best_v = v;
                best_split = split;
            }
        }
    }
    P->corr_variant = best_v;
    P->split_wgs = best_split;
    P->corr_lds = corr_lds_of(P, best_v);
    int best_lb = P->LB;
    if (col_generic) {
        // columns per workgroup of k_column_simple: the plan's choice and
        // smaller ones (same transforms, more workgroups)
        ColumnArgs A{};
        A.twD = P->d_twD;
        A.pd = P->pd;
        A.nb = nb; A.bs = bs; A.ndop = ndop; A.spc = d.samples_per_code; A.spc_eff = d.samples_per_code_eff;
        A.bstride = P->bstride;
        A.tp = P->tp;
        A.ap = P->ap;
        A.acc_ps = P->acc_ps;
        A.acc_ldr = P->ap;
        A.acc_ldc = 1;
        A.tile = P->d_tile;
        A.acc = P->d_acc;
        A.req = d_req;
        A.shifts = P->d_shifts;
        A.first_step = 1;
        float best_c = 1e30f;
        const int lb0 = P->LB;
        for (int lb : {lb0, lb0 / 2, lb0 / 4}) {
            if (lb < 1 || (lb != lb0 && lb0 / lb * lb != lb0)) continue;
            A.LB = lb;
            const int nlb = (bs + lb - 1) / lb;
            const size_t lds = (size_t)P->bstride * (P->col_onebuf ? 1 : 2) * sizeof(float2) * lb;
            const float ms = time_it([&]() {
                if (P->col_onebuf)
                    k_column_simple<true><<<dim3(nlb, nb, cnt), FMDBZP_COL_NTHR, lds, st>>>(A);
                else
                    k_column_simple<false><<<dim3(nlb, nb, cnt), FMDBZP_COL_NTHR, lds, st>>>(A);
            });
            snprintf(buf, sizeof(buf), " column LB %d: %.4f ms;", lb, ms);
            rec += buf;
            if (ms < best_c) {
                best_c = ms;
                best_lb = lb;
            }
        }
        P->LB = best_lb;
        P->col_lds = (size_t)P->bstride * (P->col_onebuf ? 1 : 2) * sizeof(float2) * best_lb;
    }
    const hipError_t e = hipStreamSynchronize(st);
    cleanup();
    if (e != hipSuccess) return set_err(FMDBZP_EHIP, "autotune: %s", hipGetErrorString(e));
    snprintf(buf, sizeof(buf), "chose corr v%d split %d, column LB %d;", best_v, best_split, best_lb);
    P->tuning = std::string(buf) + rec;
    std::lock_guard<std::mutex> g(g_tune_mu);
    g_tune_cache.push_back({key, TuneChoice{best_v, best_split, best_lb, P->tuning}});
    return FMDBZP_OK;
}

// Wait for the plan's stream and return the staged statistics.
int acquire_finish(fmdbzp_plan* P)
{
    HIP_TRY(hipSetDevice(P->device));
    HIP_TRY(hipStreamSynchronize(P->stream));
    if (P->pending_out) memcpy(P->pending_out, P->h_stats, sizeof(fmdbzp_prn_stats) * P->pending_n);
    P->pending_out = nullptr;
    P->pending_n = 0;
    if (P->timing) collect_timing(P);
    return FMDBZP_OK;
}

int validate_request(fmdbzp_plan* P, const void* signal, int32_t eltype, int32_t nreq, uint32_t flags,
                     const int32_t* prn_index, fmdbzp_prn_stats* out_stats, float* const* out_surfaces)
{
    if (!signal || !prn_index || !out_stats) return set_err(FMDBZP_EINVAL, "null argument to fmdbzp_acquire");
    if (nreq <= 0) return set_err(FMDBZP_EINVAL, "nreq must be positive");
    if (!elsize(eltype) && eltype != FMDBZP_C2BIT) return set_err(FMDBZP_EINVAL, "unknown eltype %d", eltype);
    if (P->tile_half && eltype != FMDBZP_I16 && eltype != FMDBZP_CI8 && eltype != FMDBZP_CI16 &&
        eltype != FMDBZP_C2BIT)
        return set_err(FMDBZP_EINVAL, "FP16 tiles need integer samples (I16, CI8, CI16, C2BIT)");
    if ((flags & FMDBZP_FLAG_STORE_SURFACES) && !out_surfaces)
        return set_err(FMDBZP_EINVAL, "STORE_SURFACES without surface pointers");
    if ((flags & FMDBZP_FLAG_STORE_SURFACES) && P->rotbig && P->nchunks > 1)
        return set_err(FMDBZP_EINVAL, "this search accumulates in %d code-column chunks and keeps no whole surface; "
                                      "surfaces need a workspace budget (FMDBZP_WORKSPACE_GB) that holds one",
                       P->nchunks);
    for (int i = 0; i < nreq; i++)
        if (prn_index[i] < 0 || prn_index[i] >= P->nprn)
            return set_err(FMDBZP_EINVAL, "prn_index[%d] = %d out of range [0, %d)", i, prn_index[i], P->nprn);
    return FMDBZP_OK;
}

}  // namespace

extern "C" {

int fmdbzp_acquire(fmdbzp_plan* plan, const void* signal, int32_t eltype, int64_t n_samples,
                   double interm_freq_hz, const int32_t* prn_index, int32_t nreq, uint32_t flags,
                   fmdbzp_prn_stats* out_stats, float* const* out_surfaces)
{
    g_err.clear();
    if (!plan) return set_err(FMDBZP_EHANDLE, "null plan");
    std::lock_guard<std::mutex> lk(plan->mu);
    int rc = validate_request(plan, signal, eltype, nreq, flags, prn_index, out_stats, out_surfaces);
    if (rc) return rc;
    rc = acquire_enqueue(plan, signal, eltype, n_samples, interm_freq_hz, prn_index, nreq, flags, out_stats,
                         out_surfaces);
    int rc2 = acquire_finish(plan);
    return rc ? rc : rc2;
}

int fmdbzp_acquire_batch(const fmdbzp_request* reqs, int32_t nreqs)
{
    g_err.clear();
    if (!reqs || nreqs <= 0) return set_err(FMDBZP_EINVAL, "empty batch");
    std::vector<fmdbzp_plan*> plans;
    for (int i = 0; i < nreqs; i++) {
        if (!reqs[i].plan) return set_err(FMDBZP_EHANDLE, "request %d has a null plan", i);
        plans.push_back(reqs[i].plan);
    }
    std::sort(plans.begin(), plans.end());
    plans.erase(std::unique(plans.begin(), plans.end()), plans.end());
    // lock every plan of the batch in address order
    std::vector<std::unique_lock<std::mutex>> locks;
    for (auto* p : plans) locks.emplace_back(p->mu);
    int rc = FMDBZP_OK;
    for (int i = 0; i < nreqs && rc == FMDBZP_OK; i++) {
        const fmdbzp_request& q = reqs[i];
        rc = validate_request(q.plan, q.signal, q.eltype, q.nprn, q.flags, q.prn_index, q.out_stats, q.out_surfaces);
        if (rc) break;
        // a plan used twice returns its first request before the second reuses its workspace
        if (q.plan->pending_out) rc = acquire_finish(q.plan);
        if (rc) break;
        rc = acquire_enqueue(q.plan, q.signal, q.eltype, q.n_samples, q.interm_freq_hz, q.prn_index, q.nprn,
                             q.flags, q.out_stats, q.out_surfaces);
    }
    for (auto* p : plans) {
        int r2 = acquire_finish(p);
        if (rc == FMDBZP_OK) rc = r2;
    }
    return rc;
}

// ---------------------------------------------------------------------------
// fmdbzp_acquire_noalloc: the search of fmdbzp_acquire on device-resident
// samples, with every buffer beyond the caller's inputs and outputs (signal
// FFT cache, PRN list, tile, accumulator, reductions, statistics) carved out
// of one file-scope device array instead of the plan's workspace, so the call
// makes no device or host allocation. The array exists once per device and
// process; its device address comes from hipGetSymbolAddress, looked up once
// per device on the first call there (the array's name is only a host-side
// stand-in for it). Calls on one device share the array: they are serialised
// by a per-device lock, held until the call has synchronised.
// ---------------------------------------------------------------------------
static __device__ __align__(256) char scratch[FMDBZP_NOALLOC_SCRATCH_BYTES];

namespace {

constexpr int kMaxDevices = 64;
std::mutex g_scratch_mu;
char* g_scratch_ptr[kMaxDevices] = {};
std::mutex g_scratch_call_mu[kMaxDevices];

size_t align256(size_t b) { return (b + 255) & ~(size_t)255; }

// PRN indices into the scratch without a host-to-device copy: up to 64 per
// launch, passed by value.
struct ReqChunk {
    int32_t v[64];
};
__global__ void k_put_req(int32_t* __restrict__ dst, ReqChunk c, int n)
{
    if ((int)threadIdx.x < n) dst[threadIdx.x] = c.v[threadIdx.x];
}

}  // namespace

extern "C" int fmdbzp_acquire_noalloc(fmdbzp_plan* plan, const void* signal, int32_t eltype, int64_t n_samples,
                                      double interm_freq_hz, const int32_t* prn_index, int32_t nreq,
                                      fmdbzp_prn_stats* out_stats)
{
    g_err.clear();
    if (!plan) return set_err(FMDBZP_EHANDLE, "null plan");
    std::lock_guard<std::mutex> lk(plan->mu);
    fmdbzp_plan* P = plan;
    int rc = validate_request(P, signal, eltype, nreq, 0u, prn_index, out_stats, nullptr);
    if (rc) return rc;
    const fmdbzp_plan_desc& d = P->d;
    const int64_t seglen = (int64_t)d.num_coh * d.samples_per_code;
    if (n_samples / seglen < d.num_noncoherent)
        return set_err(FMDBZP_EINVAL, "signal has %lld samples, fewer than %d segments of %lld",
                       (long long)n_samples, d.num_noncoherent, (long long)seglen);
    if (P->device < 0 || P->device >= kMaxDevices) return set_err(FMDBZP_ENODEV, "device %d out of range", P->device);
    if (P->rotbig)
        return set_err(FMDBZP_EINVAL, "fmdbzp_acquire_noalloc does not run the large-ndop rotation search "
                                      "(its tile alone exceeds the scratch)");
    // scratch layout: signal FFT cache | PRN list | statistics | per-PRN batch buffers
    const int ndop = d.num_doppler_bins;
    const size_t b_sig = align256(sizeof(float2) * (size_t)d.num_noncoherent * ndop * d.fft_size);
    const size_t b_req = align256(sizeof(int32_t) * (size_t)nreq);
    const size_t b_stats = align256(sizeof(fmdbzp_prn_stats) * (size_t)nreq);
    const size_t t_prn = align256(sizeof(float2) * (size_t)d.num_blocks * ndop * P->tp);
    const size_t a_prn = align256(sizeof(float) * std::max(P->acc_ps, P->lim_acc_ps));
    // the size limit counts a reduction partial per row and 4096 columns beside
    // the tile (they are kept in the tile)
    const size_t np = P->lim_cm ? (size_t)((d.samples_per_code_eff + 4095) / 4096) * ndop : 0;
    const size_t r_prn = align256(sizeof(double) * ndop) + align256(sizeof(float) * ndop) +
                         align256(sizeof(uint64_t) * ndop) + align256(sizeof(double) * np) +
                         align256(sizeof(float) * np) + align256(sizeof(uint64_t) * np);
    const size_t per_prn = t_prn + a_prn + r_prn;
    const size_t fixed = b_sig + b_req + b_stats;
    if (fixed + per_prn > (size_t)FMDBZP_NOALLOC_SCRATCH_BYTES)
        return set_err(FMDBZP_EINVAL,
                       "search needs %zu bytes of scratch for one PRN (signal FFTs %zu, tile %zu, accumulator %zu), "
                       "more than the %zu-byte maximum of fmdbzp_acquire_noalloc",
                       fixed + per_prn, b_sig, t_prn, a_prn, (size_t)FMDBZP_NOALLOC_SCRATCH_BYTES);
    const int batch = (int)std::min<size_t>((size_t)nreq, ((size_t)FMDBZP_NOALLOC_SCRATCH_BYTES - fixed) / per_prn);
    HIP_TRY(hipSetDevice(P->device));
    char* base = nullptr;
    {
        std::lock_guard<std::mutex> g(g_scratch_mu);
        if (!g_scratch_ptr[P->device]) {
            void* ptr = nullptr;
            const hipError_t e = hipGetSymbolAddress(&ptr, HIP_SYMBOL(scratch));
            if (e != hipSuccess || !ptr)
                return set_err(FMDBZP_EHIP, "hipGetSymbolAddress(scratch) on device %d: %s", P->device,
                               hipGetErrorString(e));
            g_scratch_ptr[P->device] = (char*)ptr;
        }
        base = g_scratch_ptr[P->device];
    }
    std::lock_guard<std::mutex> call(g_scratch_call_mu[P->device]);
    if (P->pending_out) {
        rc = acquire_finish(P);
        if (rc) return rc;
    }
    // carve the batch buffers (each 256-byte aligned)
    char* q = base;
    auto take = [&](size_t bytes) {
        char* r = q;
        q += align256(bytes);
        return (void*)r;
    };
    Work W{};
    W.sigfft = (float2*)take(sizeof(float2) * (size_t)d.num_noncoherent * ndop * d.fft_size);
    int32_t* reqd = (int32_t*)take(sizeof(int32_t) * (size_t)nreq);
    W.req = reqd;
    W.stats = (fmdbzp_prn_stats*)take(sizeof(fmdbzp_prn_stats) * (size_t)nreq);
    W.tile = (float2*)q;
    q += t_prn * batch;
    W.acc = (float*)q;
    q += align256(sizeof(float) * P->acc_ps * batch);
    W.rowsum = (double*)take(sizeof(double) * ndop * batch);
    W.rowbest_v = (float*)take(sizeof(float) * ndop * batch);
    W.rowbest_k = (uint64_t*)take(sizeof(uint64_t) * ndop * batch);
    W.batch = batch;
    W.nlanes = 1;
    W.timing = false;
    if ((size_t)(q - base) > (size_t)FMDBZP_NOALLOC_SCRATCH_BYTES)
        return set_err(FMDBZP_EINVAL, "scratch layout exceeds its maximum");  // unreachable by the sizing above
    // every tile / accumulator offset the kernels form from these bases stays
    // within the per-PRN sizes checked at plan creation
    for (int i = 0; i < nreq; i += 64) {
        ReqChunk c{};
        const int n = std::min(64, nreq - i);
        for (int j = 0; j < n; j++) c.v[j] = prn_index[i + j];
        k_put_req<<<1, 64, 0, P->stream>>>(reqd + i, c, n);
        HIP_TRY(hipGetLastError());
    }
    rc = acquire_launch(P, W, signal, eltype, interm_freq_hz, nreq, 0u, nullptr);
    if (rc) {
        hipStreamSynchronize(P->stream);
        return rc;
    }
    HIP_TRY(hipMemcpyAsync(out_stats, W.stats, sizeof(fmdbzp_prn_stats) * (size_t)nreq, hipMemcpyDeviceToHost,
                           P->stream));
    HIP_TRY(hipStreamSynchronize(P->stream));
    return FMDBZP_OK;
}

}  // extern "C"

// ---------------------------------------------------------------------------
// Seeded synthetic signals on the device (fmdbzp.h).
// ---------------------------------------------------------------------------
extern "C" int fmdbzp_synthesize(const fmdbzp_scene* scene, const fmdbzp_emitter* emitters, int32_t n_emitters,
                                 void* out)
{
    if (!scene || !out || n_emitters < 0 || (n_emitters > 0 && !emitters))
        return set_err(FMDBZP_EINVAL, "null scene, emitters or output");
    const fmdbzp_scene& sc = *scene;
    if (sc.n_samples <= 0 || !(sc.sampling_freq_hz > 0.0))
        return set_err(FMDBZP_EINVAL, "n_samples and sampling_freq_hz must be positive");
    const bool cplx = sc.complex_samples != 0;
    if (cplx ? sc.out_eltype != FMDBZP_CF32 : (sc.out_eltype != FMDBZP_I16 && sc.out_eltype != FMDBZP_F32))
        return set_err(FMDBZP_EINVAL, "out_eltype must be CF32 for complex scenes, I16 or F32 for real ones");
    std::vector<int8_t> table;
    std::vector<SynthEmitter> em((size_t)n_emitters);
    auto append = [&](const int8_t* v, int64_t n, int64_t* off) -> bool {
        *off = (int64_t)table.size();
        for (int64_t i = 0; i < n; i++) {
            if (v[i] != 1 && v[i] != -1) return false;
            table.push_back(v[i]);
        }
        return true;
    };
    for (int e = 0; e < n_emitters; e++) {
        const fmdbzp_emitter& E = emitters[e];
        SynthEmitter& D = em[(size_t)e];
        if (!E.chips || E.code_length <= 0 || !(E.code_freq_hz >= 0.0))
            return set_err(FMDBZP_EINVAL, "emitter %d: chips and a positive code_length are required", e);
        if ((E.secondary && E.secondary_length <= 0) ||
            (E.bits && (E.num_bits <= 0 || E.bit_ms <= 0 || E.bit_edge_ms < 0)))
            return set_err(FMDBZP_EINVAL, "emitter %d: secondary / bit table sizes or a negative bit_edge_ms", e);
        memset(&D, 0, sizeof(D));
        if (!append(E.chips, E.code_length, &D.chips_off) ||
            (E.secondary && !append(E.secondary, E.secondary_length, &D.sec_off)) ||
            (E.bits && !append(E.bits, E.num_bits, &D.bits_off)))
            return set_err(FMDBZP_EINVAL, "emitter %d: chip, secondary and bit values must be +-1", e);
        D.code_length = E.code_length;
        D.boc = E.boc != 0;
        D.sec_len = E.secondary ? E.secondary_length : 0;
        D.sec_phase = E.secondary_phase;
        D.num_bits = E.bits ? E.num_bits : 0;
        D.bit_ms = E.bits ? E.bit_ms : 1;
        D.bit_edge_ms = E.bit_edge_ms;
        D.amplitude = E.amplitude;
        D.code_freq = E.code_freq_hz;
        D.code_phase = E.code_phase_chips;
        D.carrier_hz = E.carrier_hz;
        D.carrier_phase = E.carrier_phase;
    }
    if (table.empty()) table.push_back(1);
    int8_t* d_table = nullptr;
    SynthEmitter* d_em = nullptr;
    hipStream_t st = nullptr;
    auto cleanup = [&]() {
        if (st) hipStreamDestroy(st);
        hipFree(d_table);
        hipFree(d_em);
    };
    hipError_t e = hipStreamCreateWithFlags(&st, hipStreamNonBlocking);
    if (e == hipSuccess) e = hipMalloc((void**)&d_table, table.size());
    if (e == hipSuccess && n_emitters > 0) e = hipMalloc((void**)&d_em, sizeof(SynthEmitter) * (size_t)n_emitters);
    if (e == hipSuccess) e = hipMemcpyAsync(d_table, table.data(), table.size(), hipMemcpyHostToDevice, st);
    if (e == hipSuccess && n_emitters > 0)
        e = hipMemcpyAsync(d_em, em.data(), sizeof(SynthEmitter) * (size_t)n_emitters, hipMemcpyHostToDevice, st);
    if (e == hipSuccess) {
        const int64_t nthreads = cplx ? sc.n_samples : (sc.n_samples + 1) / 2;
        const int64_t nblk = (nthreads + 255) / 256;
        if (nblk > 0x7FFFFFFF) {
            cleanup();
            return set_err(FMDBZP_EINVAL, "n_samples too large");
        }
        k_synthesize<<<(unsigned)nblk, 256, 0, st>>>(d_em, n_emitters, d_table, sc.n_samples, sc.sampling_freq_hz,
                                                     cplx ? 1 : 0, sc.out_eltype == FMDBZP_I16 ? 1 : 0,
                                                     sc.noise_scale, (uint32_t)(sc.seed & 0xFFFFFFFFu),
                                                     (uint32_t)(sc.seed >> 32), sc.noise_stream, out);
        e = hipGetLastError();
    }
    if (e == hipSuccess) e = hipStreamSynchronize(st);
    cleanup();
    if (e != hipSuccess) return set_err(FMDBZP_EHIP, "fmdbzp_synthesize: %s", hipGetErrorString(e));
    return FMDBZP_OK;
}
