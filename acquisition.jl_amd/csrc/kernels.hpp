// kernels.hpp — FM-DBZP search kernels for gfx950 (MI355X).
//
// Data layout in HBM (all complex values are interleaved float2):
//   prnconj [prn][b][F]          conj FFT of code sub-block b      (plan.jl:230-251)
//   sigfft  [step][k][F]         FFT of signal double block k      (coherent_integration.jl:12-56)
//   tile    [p][r][k][lag]       block correlation, lag < bs       (coherent_integration.jl:136-171)
//   acc     [p][row][col_eff]    power surface, sorted-Doppler rows, scrambled FM-DBZP
//                                columns, accumulated over the N_nc steps
//                                (noncoherent_integration.jl:760-812)
// p indexes the PRNs of the current batch; the PRN is req[p].
#pragma once
#include <hip/hip_fp16.h>
#include <hip/hip_runtime.h>
#include <stdint.h>
#include "fft_lds.hpp"
#include "../../include/fmdbzp.h"

#define FMDBZP_NTHR 256
// The simple column kernel runs 512 threads, each holding at most
// FMDBZP_COL_MAXV complex values per in-place FFT stage:
// LB * ndop <= FMDBZP_COL_MAXV * FMDBZP_COL_NTHR.
#define FMDBZP_COL_NTHR 512
#define FMDBZP_COL_MAXV 16
// complex values a thread holds per in-place stage of the block-correlation
// transforms: NT * F <= FMDBZP_CORR_MAXV * FMDBZP_NTHR
#define FMDBZP_CORR_MAXV 16

// ---------------------------------------------------------------------------
// XCD-aware block order. The dispatcher hands workgroup b (linear id) to XCD
// b mod 8; each XCD has its own L2. Remapping gives every XCD one contiguous
// range of logical blocks, so neighbouring tiles (which share cache lines of
// the accumulator or the same code FFTs) meet in the same L2.
// ---------------------------------------------------------------------------
#define FMDBZP_NUM_XCD 8
__device__ __forceinline__ int xcd_logical_block()
{
    const int nblk = gridDim.x * gridDim.y * gridDim.z;
    const int bid = blockIdx.x + gridDim.x * (blockIdx.y + gridDim.y * blockIdx.z);
    const int per = nblk / FMDBZP_NUM_XCD, rem = nblk % FMDBZP_NUM_XCD;
    const int x = bid % FMDBZP_NUM_XCD, s = bid / FMDBZP_NUM_XCD;
    return x * per + min(x, rem) + s;
}

// ComplexF32(x) of one input sample (src/acquire.jl:94, :101).
__device__ __forceinline__ float2 load_sample(const void* __restrict__ sig, int eltype, int64_t i)
{
    switch (eltype) {
    case FMDBZP_CF32: return ((const float2*)sig)[i];
    case FMDBZP_CF64: {
        const double2 v = ((const double2*)sig)[i];
        return make_float2((float)v.x, (float)v.y);
    }
    case FMDBZP_I16: return make_float2((float)((const int16_t*)sig)[i], 0.f);
    case FMDBZP_CI8: {
        const char2 v = ((const char2*)sig)[i];
        return make_float2((float)v.x, (float)v.y);
    }
    case FMDBZP_CI16: {
        const short2 v = ((const short2*)sig)[i];
        return make_float2((float)v.x, (float)v.y);
    }
    case FMDBZP_F32: return make_float2(((const float*)sig)[i], 0.f);
    case FMDBZP_F64: return make_float2((float)((const double*)sig)[i], 0.f);
    case FMDBZP_C2BIT: {
        const unsigned b = ((const uint8_t*)sig)[i >> 1];
        const unsigned nib = (i & 1) ? (b >> 4) : (b & 15u);
        const unsigned ci = nib & 3u, cq = (nib >> 2) & 3u;
        const float vi = (ci & 1u ? 3.f : 1.f) * (ci & 2u ? -1.f : 1.f);
        const float vq = (cq & 1u ? 3.f : 1.f) * (cq & 2u ? -1.f : 1.f);
        return make_float2(vi, vq);
    }
    default: return make_float2(0.f, 0.f);
    }
}

// |z|^2 as Julia's abs2: re*re + im*im, never fused.
__device__ __forceinline__ float abs2_exact(float2 z)
{
#pragma clang fp contract(off)
    return z.x * z.x + z.y * z.y;
}

// ---------------------------------------------------------------------------
// Plan time: conjugated code sub-block FFTs (src/plan.jl:230-251).
// grid (nb, nprn)
// ---------------------------------------------------------------------------
struct CodeIn {
    const int8_t* code;
    int bs;
    __device__ __forceinline__ float2 operator()(int, int i) const
    {
        return make_float2(i < bs ? (float)code[i] : 0.f, 0.f);
    }
};
// conj(v) times scale: 1, or 1/F when F is a power of two (then exact, and the
// block correlation's own 1/F factor is applied here once per plan).
struct ConjOut {
    float2* out;
    float scale;
    __device__ __forceinline__ void operator()(int, int i, float2 v) const
    {
        out[i] = make_float2(v.x * scale, -v.y * scale);
    }
};

__global__ void __launch_bounds__(FMDBZP_NTHR)
k_code_fft(const int8_t* __restrict__ codes, float2* __restrict__ prnconj, FftPlanDev pf,
           const float2* __restrict__ twF, int spc, int nb, int bs, float pscale)
{
    extern __shared__ float2 lds[];
    const int F = pf.n;
    const int blk = blockIdx.x, prn = blockIdx.y;
    const int8_t* code = codes + (size_t)prn * spc + (size_t)blk * bs;
    float2* out = prnconj + ((size_t)prn * nb + blk) * F;
    const int span = fft_lds_span(F);
    fft_run<false, false, CodeIn, ConjOut, false>(lds, lds + span, pf, twF, 1, span, threadIdx.x, FMDBZP_NTHR,
                                                  CodeIn{code, bs}, ConjOut{out, pscale});
}

// ---------------------------------------------------------------------------
// Downconversion fused into the signal double-block FFTs.
// `_downconvert!` (src/acquire.jl:92-104) + `_precompute_signal_block_ffts!`
// (src/coherent_integration.jl:12-56). The IF phase argument is formed in
// Float32 with separately rounded multiply and add, as the reference does;
// sin/cos of that Float32 argument are evaluated in FP64 and rounded.
// grid (ncoh*nb, nnc)
// ---------------------------------------------------------------------------
// do_if 1: the reference's Float32 phase argument, off + Float32(j) * step
// with Float32 off = Float32(seg0) * step (src/acquire.jl:96-101); do_if 2:
// the FP64 phase dstep * (seg0 + j) of the absolute sample (an engine option
// for long signals, where the Float32 sum loses the phase).
struct DownconvIn {
    const void* sig;
    int eltype;
    int64_t seg0, seglen, blk0;
    int two_bs;
    int do_if;
    float off, step;
    double dstep;
    __device__ __forceinline__ float2 operator()(int, int i) const
    {
        float2 v = make_float2(0.f, 0.f);
        if (i < two_bs) {
            int64_t j = blk0 + i;
            if (j >= seglen) j -= seglen;  // last double block wraps (coherent_integration.jl:44-50)
            v = load_sample(sig, eltype, seg0 + j);
            if (do_if) {
#pragma clang fp contract(off)
                double dph;
                if (do_if == 2) {
                    dph = dstep * (double)(seg0 + j);
                } else {
                    const float ph = off + (float)j * step;
                    dph = (double)ph;
                }
                const float s = (float)sin(dph), c = (float)cos(dph);
                v = make_float2(v.x * c - v.y * s, v.x * s + v.y * c);
            }
        }
        return v;
    }
};
struct PlainOut {
    float2* out;
    __device__ __forceinline__ void operator()(int, int i, float2 v) const { out[i] = v; }
};

__global__ void __launch_bounds__(FMDBZP_NTHR)
k_signal_fft(const void* __restrict__ sig, int eltype, float2* __restrict__ sigfft, FftPlanDev pf,
             const float2* __restrict__ twF, int bs, int64_t seglen, int ndop, int do_if,
             float phase_step, double phase_step64)
{
    extern __shared__ float2 lds[];
    const int F = pf.n;
    const int gk = blockIdx.x, step = blockIdx.y;
    const int64_t seg0 = (int64_t)step * seglen;
    DownconvIn in{sig, eltype, seg0, seglen, (int64_t)gk * bs, 2 * bs, do_if,
                  __fmul_rn((float)seg0, phase_step) /* Float32(seg_start-1) * step */, phase_step,
                  phase_step64};
    float2* out = sigfft + ((size_t)step * ndop + gk) * F;
    const int span = fft_lds_span(F);
    fft_run<false, false, DownconvIn, PlainOut, false>(lds, lds + span, pf, twF, 1, span, threadIdx.x, FMDBZP_NTHR,
                                                       in, PlainOut{out});
}

// ---------------------------------------------------------------------------
// Block correlation: `_build_coherent_tile!` (src/coherent_integration.jl:136-171).
// Row k of column block r correlates signal double block k with code sub-block
// (k mod nb + r) mod nb: pointwise product in the frequency domain (formed in
// registers by the first FFT stage), inverse FFT (unnormalised), times
// Float32(1/F); the last stage stores only the first bs lags.
// ---------------------------------------------------------------------------
struct CorrIn {
    const float2* S;   // signal-FFT row in LDS
    const float2* P;   // conj code sub-block FFTs of this PRN, [nb][F]
    int F, nb, b0;     // transform t uses code block (b0 + t) mod nb
    __device__ __forceinline__ float2 operator()(int t, int i) const
    {
        int b = b0 + t;
        if (b >= nb) b -= nb;
        // 32-bit byte offset from the PRN's base (nb * F * 8 < 2^31, checked at
        // plan creation): the address is one vector add on a scalar base
        const uint32_t off = (uint32_t)(b * F + i) * (uint32_t)sizeof(float2);
        return cmulf(S[i], *(const float2*)((const char*)P + off));
    }
};
// TileT float2: FP32 tile. TileT __half2: FP16 tile of the values times
// hscale, a power of two (FMDBZP_PREC_TILE_FP16). SCALE: multiply by inv_f
// here; without it the 1/F factor is already in the code spectra (power-of-two
// F), which gives the same values exactly.
template <class TileT, bool SCALE = true>
struct LagOut {
    TileT* out;         // tile row of transform 0
    uint32_t tstride;   // tile distance between consecutive column blocks (elements)
    int bs;
    float inv_f;
    int nt;             // transforms of this pass that exist (the rest are padding)
    float hscale;
    __device__ __forceinline__ void operator()(int t, int i, float2 v) const
    {
        if (i < bs && t < nt) {
            const float sx = SCALE ? v.x * inv_f : v.x, sy = SCALE ? v.y * inv_f : v.y;
            // 32-bit byte offset from the pass's base (the two column blocks
            // of one pass span below 2^31 bytes, checked at plan creation)
            char* dst = (char*)out + ((uint32_t)t * tstride + (uint32_t)i) * (uint32_t)sizeof(TileT);
            // the tile is written once and read by the next kernel: nontemporal stores
            if constexpr (sizeof(TileT) == sizeof(float2)) {
                typedef float f2v __attribute__((ext_vector_type(2)));
                f2v u;
                u.x = sx;
                u.y = sy;
                __builtin_nontemporal_store(u, (f2v*)dst);
            } else {
                const __half2 h = __floats2half2_rn(sx * hscale, sy * hscale);
                __builtin_nontemporal_store(*(const uint32_t*)&h, (uint32_t*)dst);
            }
        }
    }
};

// One workgroup per (row k, PRN): the signal-FFT row is staged in LDS once and
// reused for the nrb column blocks r = (rb0 + rr) mod nb, rr < nrb (all nb
// blocks, rb0 = 0, unless the search runs in code-column chunks), NT blocks
// per pass; tile block rr of batch slot p is tile[(p nrb + rr) ndop + k]. ONEBUF: in-place
// stages, one LDS buffer per concurrent transform; else two ping-pong buffers
// (NT = 1).
// grid (ndop, batch, split)
// STATIC = 400, 800, 2000, 4000: the E1-like searches at 25 MHz and +-50,
// +-25, +-10, +-5 kHz (16 x 5 x 5, 16 x 10 x 5, 16 x 5 x 5 x 5, 16 x 10 x 5 x 5),
// with 10, 5, 2 and 1 transforms per pass, so the radix-16 stage keeps about
// 250 of the 256 threads busy;
// STATIC = 2048: compile-time 16 x 16 x 8 transform, two per pass, with the
// 1/F factor taken from the code spectra; STATIC = 2500: 10 x 10 x 5 x 5 (the
// E1-like search at 25 MHz); STATIC = 500: 4 x 5 x 5 x 5, two per pass (GPS
// L1 C/A at 5 MHz, the radix order of the runtime plan for 500). inv_f is 1
// when the code spectra carry 1/F.
template <int NT, bool ONEBUF, int STATIC = 0, class TileT = float2>
__global__ void __launch_bounds__(FMDBZP_NTHR)
// three waves per SIMD (at most 168 VGPRs), except the multi-transform
// E1-like sizes, which keep more butterflies per thread in flight
__attribute__((amdgpu_waves_per_eu(STATIC == 400 || STATIC == 800 || STATIC == 2000 || STATIC == 4000 ? 1 : 3)))
k_corr_tile(const float2* __restrict__ sigfft_step, const float2* __restrict__ prnconj,
            const int32_t* __restrict__ req, TileT* __restrict__ tile, FftPlanDev pf,
            const float2* __restrict__ twF, int nb, int bs, int tp, int ndop, float inv_f, float hscale, int rb0,
            int nrb)
{
    extern __shared__ float2 lds[];
    const int F = pf.n;
    const int span = fft_lds_span(F);
    float2* srow = lds;
    float2* a = lds + F;
    const int lbk = xcd_logical_block();
    const int k = lbk % gridDim.x, rest = lbk / gridDim.x;
    const int p = rest % gridDim.y, sp = rest / gridDim.y;
    // gridDim.z > 1 splits a row's column blocks over several workgroups (small
    // searches, where ndop x PRNs workgroups would not fill the device); this
    // workgroup takes passes [sp * chunk, (sp + 1) * chunk)
    const int npass = (nrb + NT - 1) / NT;
    const int chunk = (npass + gridDim.z - 1) / gridDim.z;
    const int r_begin = sp * chunk * NT, r_end = min(nrb, (sp + 1) * chunk * NT);
    if (r_begin >= r_end) return;  // uniform over the workgroup, before any barrier
    const int tid = threadIdx.x;
    const int prn = req[p];
    const float2* S = sigfft_step + (size_t)k * F;
    for (int i = tid; i < F; i += FMDBZP_NTHR) srow[i] = S[i];
    const float2* Pp = prnconj + (size_t)prn * nb * F;
    const int kb = k % nb;
#pragma unroll 1
    for (int r0 = r_begin; r0 < r_end; r0 += NT) {
        __syncthreads();  // srow ready / previous transforms done with the buffers
        const int nt = min(NT, nrb - r0);
        int b0 = kb + rb0 + r0;  // < 3 nb
        if (b0 >= nb) b0 -= nb;
        if (b0 >= nb) b0 -= nb;
        CorrIn in{srow, Pp, F, nb, b0};
        LagOut<TileT, STATIC != 2048> out{tile + (((size_t)p * nrb + r0) * ndop + k) * tp, (uint32_t)(ndop * tp), bs,
                                          inv_f, nt, hscale};
        if constexpr (STATIC == 2048)
            fft3_static<true, 2048, NT, FMDBZP_NTHR, 16, 16, 8>(a, twF, tid, in, out);
        else if constexpr (STATIC == 2500)
            fft4_static<true, 2500, NT, FMDBZP_NTHR, 10, 10, 5, 5>(a, twF, tid, in, out);
        else if constexpr (STATIC == 500)
            fft4_static<true, 500, NT, FMDBZP_NTHR, 4, 5, 5, 5>(a, twF, tid, in, out);
        else if constexpr (STATIC == 400)
            fft3_static<true, 400, NT, FMDBZP_NTHR, 16, 5, 5>(a, twF, tid, in, out);
        else if constexpr (STATIC == 800)
            fft3_static<true, 800, NT, FMDBZP_NTHR, 16, 10, 5>(a, twF, tid, in, out);
        else if constexpr (STATIC == 2000)
            fft4_static<true, 2000, NT, FMDBZP_NTHR, 16, 5, 5, 5>(a, twF, tid, in, out);
        else if constexpr (STATIC == 4000)
            fft4_static<true, 4000, NT, FMDBZP_NTHR, 16, 10, 5, 5>(a, twF, tid, in, out);
        else if constexpr (ONEBUF)
            fft_run_1buf<true, false, FMDBZP_CORR_MAXV>(a, pf, twF, nt, span, tid, FMDBZP_NTHR, in, out);
        else
            fft_run<true, false>(a, a + span, pf, twF, 1, span, tid, FMDBZP_NTHR, in, out);
    }
}

// ---------------------------------------------------------------------------
// Column stage. One workgroup owns LB consecutive lags (FM-DBZP columns) of
// one (PRN, column block) tile; lanes run across columns (COLFAST), so tile
// loads and accumulator read-modify-writes are coalesced along code columns.
// ---------------------------------------------------------------------------
struct ColumnArgs {
    const float2* tile;      // [batch][nb][ndop][tp], lags < bs used
    float* acc;              // [batch][ndop][ap], columns < spc_eff used
    const int32_t* shifts;   // [ndop] drift shifts of this step, sorted-row keyed, in [0, spc)
    const float* patterns;   // [nsets][Q][ncoh] (column-major (ncoh, Q) per set)
    const int32_t* pset;     // [nprn] pattern set per PRN
    const int32_t* req;      // [batch] PRN index of each batch slot
    const float2* twD;       // column FFT twiddles
    FftPlanDev pd;
    int nb, bs, ndop, spc, spc_eff, ncoh, ndb, E, R, Q, ndc, edge_step, use_max;
    int LB, bstride, sst, first_step, literal_edges;
    int tp, ap;  // tile and accumulator row pitches (elements, multiples of 32)
    // accumulator element (p, row, col) at acc + p * acc_ps + row * acc_ldr + col * acc_ldc:
    // row-major (acc_ldr = ap, acc_ldc = 1) or column-major (acc_ldr = 1, acc_ldc = column pitch)
    size_t acc_ps;
    int acc_ldr, acc_ldc;
    int rot_direct;  // rotation path with one pattern per slice and even ndop: FFT outputs go straight to acc
    // Code-column window of the accumulator (k_column_rotbig): destination
    // column dc lands at window offset (dc - win0) mod spc when that is below
    // winlen, in rotation slice q at column q * slice_cols + offset; other
    // cells are dropped. A whole-surface accumulator is win0 = 0,
    // winlen = slice_cols = spc.
    int win0, winlen, slice_cols;
    // Column blocks held in the tile: tile block rr is column block
    // (rb0 + rr) mod nb, nrb blocks per PRN.
    int rb0, nrb;
    // Second step of a two-step launch (k_column_c160_pair): its tile and
    // its drift shifts; unused elsewhere.
    const float2* tile2;
    const int32_t* shifts2;
};

// Accumulate (or store, at the first step) one power value with the drift
// shift of its sorted destination row (src/noncoherent_integration.jl:547-569,
// :728-736; issue #74 keys the shift on the destination row).
__device__ __forceinline__ void acc_cell(const ColumnArgs& A, int p, int row, int cp, int slice, float v)
{
    int dc = cp + A.shifts[row];
    if (dc >= A.spc) dc -= A.spc;
    float* dst = A.acc + (size_t)p * A.acc_ps + (size_t)row * A.acc_ldr + ((size_t)slice * A.spc + dc) * A.acc_ldc;
    if (A.first_step) *dst = v;
    else *dst = *dst + v;
}

// Tile values are read once per step. For the L1 C/A 10 ms searches (tiles of
// hundreds of MB per step) nontemporal loads keep them from displacing the
// accumulator lines in the caches; small tiles stay cached between kernels,
// and the other column kernels load them normally.
__device__ __forceinline__ float2 load_tile_nt(const float2* p)
{
    typedef float f2v __attribute__((ext_vector_type(2)));
    const f2v u = __builtin_nontemporal_load((const f2v*)p);
    return make_float2(u.x, u.y);
}

struct TileColIn {
    const float2* T;  // tile of (p, r), offset to lag0
    int bs;
    __device__ __forceinline__ float2 operator()(int t, int k) const { return T[(size_t)k * bs + t]; }
};

// Simple path output: |x|^2, fftshift fold ((raw + ndop/2) mod ndop,
// src/plan.jl:528), drift, accumulate.
struct SimpleAccOut {
    const ColumnArgs* A;
    int p, cp0, half;
    __device__ __forceinline__ void operator()(int t, int w, float2 v) const
    {
        int row = w + half;
        if (row >= A->ndop) row -= A->ndop;
        acc_cell(*A, p, row, cp0 + t, 0, abs2_exact(v));
    }
};

// `_accumulate_fftshifted_power_(drift_)pilot!` (src/noncoherent_integration.jl:482-592)
// and `_stream_power_column!` (src/acquire.jl:335-385).
template <bool ONEBUF>
__global__ void __launch_bounds__(FMDBZP_COL_NTHR, 4)
k_column_simple(ColumnArgs A)
{
    extern __shared__ float2 lds[];
    const int lbk = xcd_logical_block();
    const int lb = lbk % gridDim.x, r = (lbk / gridDim.x) % gridDim.y, p = lbk / (gridDim.x * gridDim.y);
    const int lag0 = lb * A.LB;
    const int ncol = min(A.LB, A.bs - lag0);
    const int bst = A.bstride;
    const float2* T = A.tile + (((size_t)p * A.nb + r) * A.ndop) * A.tp + lag0;
    SimpleAccOut out{&A, p, r * A.bs + lag0, A.ndop / 2};
    if constexpr (ONEBUF)
        fft_run_1buf<false, true, FMDBZP_COL_MAXV>(lds, A.pd, A.twD, ncol, bst, threadIdx.x, FMDBZP_COL_NTHR,
                                                    TileColIn{T, A.tp}, out);
    else
        fft_run<false, true>(lds, lds + (size_t)A.LB * bst, A.pd, A.twD, ncol, bst, threadIdx.x, FMDBZP_COL_NTHR,
                             TileColIn{T, A.tp}, out);
}

// Simple column stage for ndop = 160 with compile-time 10 x 16 transforms:
// LBS columns per workgroup of NT threads. Each stage-2 thread owns one
// radix-16 butterfly of one column (16 accumulator cells); it issues the loads
// of those cells before the tile loads, so both reads are in flight together
// and the accumulate needs no second memory round trip.
template <int LBS, int NT, bool HALF = false>
__global__ void __launch_bounds__(NT, 6)  // 6 waves per SIMD: three 512-thread workgroups per CU
k_column_c160(ColumnArgs A, float hinv)
{
    constexpr int N = 160, R0 = 10, M0 = N / R0, R1 = 16, M1 = N / R1;
    extern __shared__ float2 lds[];
    const int lbk = xcd_logical_block();
    const int lb = lbk % gridDim.x, r = (lbk / gridDim.x) % gridDim.y, p = lbk / (gridDim.x * gridDim.y);
    const int lag0 = lb * LBS;
    const int ncol = min(LBS, A.bs - lag0);
    const int bst = A.bstride;
    const int tid = threadIdx.x;
    const float2* T = A.tile + (((size_t)p * A.nb + r) * N) * A.tp + lag0;
    float* accp = A.acc + (size_t)p * N * A.ap;

    // stage-2 role: column t1, butterfly j1, outputs w = j1 + 10 q -> row (w + 80) mod 160
    const int t1 = tid % LBS, j1 = tid / LBS;
    const bool act1 = tid < LBS * M1 && t1 < ncol;
    const int cp = r * A.bs + lag0 + t1;
    // byte offsets of this thread's 16 accumulator cells from the PRN's base
    // (one PRN's accumulator is below 2^31 bytes, checked at plan creation)
    uint32_t aoff[R1];
#pragma unroll
    for (int q = 0; q < R1; q++) {
        int row = j1 + M1 * q + N / 2;
        if (row >= N) row -= N;
        int dc = cp + A.shifts[row];
        if (dc >= A.spc) dc -= A.spc;
        aoff[q] = (uint32_t)(row * A.ap + dc) * (uint32_t)sizeof(float);
    }
    float accv[R1];
    if (act1 && !A.first_step) {
#pragma unroll
        for (int q = 0; q < R1; q++) accv[q] = *(const float*)((const char*)accp + aoff[q]);
    }

    // stage 1: radix 10 over rows j + 16 m, straight from the tile
#pragma unroll
    for (int it = 0; it < (LBS * M0 + NT - 1) / NT; it++) {
        const int idx = tid + it * NT;
        if (idx < LBS * M0) {
            const int t = idx % LBS, j = idx / LBS;
            if (t < ncol) {
                float2 v[R0];
                if constexpr (HALF) {
                    // FP16 tile (FMDBZP_PREC_TILE_FP16): back to FP32, times 2^e exactly
                    const __half2* Th = (const __half2*)A.tile + (((size_t)p * A.nb + r) * N) * A.tp + lag0;
#pragma unroll
                    for (int m = 0; m < R0; m++) {
                        const uint32_t raw = __builtin_nontemporal_load(
                            (const uint32_t*)((const char*)Th + (uint32_t)((j + M0 * m) * A.tp + t) * (uint32_t)sizeof(__half2)));
                        const float2 u = __half22float2(*(const __half2*)&raw);
                        v[m] = make_float2(u.x * hinv, u.y * hinv);
                    }
                } else {
                    // the tile is read once: nontemporal, so it does not displace accumulator lines;
                    // 32-bit byte offsets from the block's base (a tile block is below 2^31 bytes)
#pragma unroll
                    for (int m = 0; m < R0; m++)
                        v[m] = load_tile_nt((const float2*)((const char*)T +
                                                            (uint32_t)((j + M0 * m) * A.tp + t) * (uint32_t)sizeof(float2)));
                }
                bfly10<false>(v);
#pragma unroll
                for (int m = 0; m < R0; m++) lds[t * bst + j * R0 + m] = v[m];
            }
        }
    }
    __syncthreads();
    // stage 2: twiddle W_160^(q j1), radix 16, power, fftshift fold, drift, accumulate
    if (act1) {
        float2 v[R1];
#pragma unroll
        for (int q = 0; q < R1; q++) v[q] = lds[t1 * bst + j1 + M1 * q];
#pragma unroll
        for (int q = 1; q < R1; q++) v[q] = cmulf(v[q], twid<false>(A.twD, q * j1));
        bfly16<false>(v);
#pragma unroll
        for (int q = 0; q < R1; q++) {
            const float pw = abs2_exact(v[q]);
            *(float*)((char*)accp + aoff[q]) = A.first_step ? pw : accv[q] + pw;
        }
    }
}

// Two noncoherent steps s, s + 1 of the ndop = 160 simple column stage in
// one launch (src/noncoherent_integration.jl:547-569 twice). The workgroup
// owns source columns [cp0, cp0 + ncol) of step s, whose cells land at
// destination columns cp + shift_s[row]. At step s + 1 the same destination
// cell receives source column cp - d_row, d_row = shift_{s+1}[row] -
// shift_s[row], which the host admits only in {-1, 0, 1}; so the workgroup
// also transforms the step-(s + 1) columns [cp0 - 1, cp0 + ncol + 1), one halo
// column on each side (from the neighbouring column block where the window
// crosses a block edge, circularly over spc = nb bs), and stores
// (acc + p_s) + p_{s+1}: the two roundings of two single-step launches, in
// their order. Each accumulator cell is read and written once per pair.
template <int LBS, int NT, bool HALF = false>
__global__ void __launch_bounds__(NT, 6)  // three 512-thread workgroups per CU, as k_column_c160
k_column_c160_pair(ColumnArgs A, float hinv)
{
    constexpr int N = 160, R0 = 10, M0 = N / R0, R1 = 16, M1 = N / R1;
    constexpr int NC2 = LBS + 2;  // step-(s + 1) columns with both halo columns
    constexpr int PST = N + 1;    // power stride per column (odd: columns on distinct banks)
    extern __shared__ float2 lds[];
    float* pws = (float*)lds;  // step-(s + 1) powers, over the transform buffer once it is consumed
    const int bst = A.bstride;
    int* shl = (int*)(lds + NC2 * bst);  // [2][N] drift shifts of steps s and s + 1
    const int lbk = xcd_logical_block();
    const int lb = lbk % gridDim.x, r = (lbk / gridDim.x) % gridDim.y, p = lbk / (gridDim.x * gridDim.y);
    const int lag0 = lb * LBS;
    const int ncol = min(LBS, A.bs - lag0);
    const int tid = threadIdx.x;
    float* accp = A.acc + (size_t)p * N * A.ap;
    for (int i = tid; i < 2 * N; i += NT) shl[i] = i < N ? A.shifts[i] : A.shifts2[i - N];

    // the R0 tile values of radix-10 butterfly j of lag `lag` of column block
    // rb. Step s's lines are read by this workgroup alone: nontemporal. Step
    // s + 1's edge lines are also the neighbouring workgroups' halo columns:
    // ordinary loads, so the neighbours find them in L2.
    auto load1 = [&](const float2* tile, int rb, int lag, int j, float2* v, bool temporal) {
        const size_t boff = ((size_t)p * A.nb + rb) * N * A.tp;
        if constexpr (HALF) {
            const __half2* Th = (const __half2*)tile + boff;
#pragma unroll
            for (int m = 0; m < R0; m++) {
                const uint32_t* a = (const uint32_t*)((const char*)Th + (uint32_t)((j + M0 * m) * A.tp + lag) *
                                                                            (uint32_t)sizeof(__half2));
                const uint32_t raw = temporal ? *a : __builtin_nontemporal_load(a);
                const float2 u = __half22float2(*(const __half2*)&raw);
                v[m] = make_float2(u.x * hinv, u.y * hinv);
            }
        } else {
            const float2* T = tile + boff;
#pragma unroll
            for (int m = 0; m < R0; m++) {
                const float2* a =
                    (const float2*)((const char*)T + (uint32_t)((j + M0 * m) * A.tp + lag) * (uint32_t)sizeof(float2));
                v[m] = temporal ? *a : load_tile_nt(a);
            }
        }
    };
    // radix-10 first stage into LDS column t
    auto store1 = [&](float2* v, int j, int t) {
        bfly10<false>(v);
#pragma unroll
        for (int m = 0; m < R0; m++) lds[t * bst + j * R0 + m] = v[m];
    };
    // column block and lag of step-(s + 1) window column t (global column
    // cp0 - 1 + t, circular over spc = nb bs)
    auto window = [&](int t, int* rbp, int* lagp) {
        int rb = r, lag = lag0 - 1 + t;
        if (lag < 0) {
            rb = r == 0 ? A.nb - 1 : r - 1;
            lag = A.bs - 1;
        } else if (lag >= A.bs) {
            rb = r + 1 == A.nb ? 0 : r + 1;
            lag = 0;
        }
        *rbp = rb;
        *lagp = lag;
    };
    // twiddle W_160^(q j), radix 16 and powers of LDS column t, butterfly j:
    // raw bins w = j + 10 q
    auto stage2 = [&](int t, int j, float* pw) {
        float2 v[R1];
#pragma unroll
        for (int q = 0; q < R1; q++) v[q] = lds[t * bst + j + M1 * q];
#pragma unroll
        for (int q = 1; q < R1; q++) v[q] = cmulf(v[q], twid<false>(A.twD, q * j));
        bfly16<false>(v);
#pragma unroll
        for (int q = 0; q < R1; q++) pw[q] = abs2_exact(v[q]);
    };

    // accumulate role: column t1, butterfly j1, raw bins w = j1 + 10 q -> row (w + 80) mod 160
    const int t1 = tid % LBS, j1 = tid / LBS;
    const bool act1 = tid < LBS * M1 && t1 < ncol;
    const int cp = r * A.bs + lag0 + t1;
    // byte offset of the destination cell of raw bin j1 + 10 q (row (w + 80)
    // mod 160, column cp + shift_s[row]); sh: step s's shift table
    auto cell = [&](int q, const int* sh, int* rowp) {
        int row = j1 + M1 * q + N / 2;
        if (row >= N) row -= N;
        int dc = cp + sh[row];
        if (dc >= A.spc) dc -= A.spc;
        *rowp = row;
        return (uint32_t)(row * A.ap + dc) * (uint32_t)sizeof(float);
    };
    // the accumulator loads go out first, from the global shift table; the
    // offsets are formed again for the stores from the LDS copy, so they need
    // no registers across the two transforms
    float tv[R1];
    if (act1 && !A.first_step) {
#pragma unroll
        for (int q = 0; q < R1; q++) {
            int row;
            tv[q] = *(const float*)((const char*)accp + cell(q, A.shifts, &row));
        }
    }

    // step s: the owned columns
#pragma unroll
    for (int it = 0; it < (LBS * M0 + NT - 1) / NT; it++) {
        const int idx = tid + it * NT;
        if (idx < LBS * M0) {
            const int t = idx % LBS, j = idx / LBS;
            if (t < ncol) {
                float2 v[R0];
                load1(A.tile, r, lag0 + t, j, v, false);
                store1(v, j, t);
            }
        }
    }
    __syncthreads();
    // step s's second stage: tv = acc + p_s
    auto finish_s = [&]() {
        if (act1) {
            float pw[R1];
            stage2(t1, j1, pw);
#pragma unroll
            for (int q = 0; q < R1; q++) tv[q] = A.first_step ? pw[q] : tv[q] + pw[q];
        }
    };
    // step s + 1: window columns cp0 - 1 + t, t < ncol + 2; butterfly idx is
    // column idx % NC2, position idx / NC2
    static_assert(NT <= NC2 * M0 && NC2 * M0 <= 2 * NT, "one or two step-(s + 1) butterflies per thread");
    auto load_s1 = [&](int idx, float2* v) -> bool {
        const int t = idx % NC2;
        if (t >= ncol + 2) return false;
        int rb, lag;
        window(t, &rb, &lag);
        load1(A.tile2, rb, lag, idx / NC2, v, true);
        return true;
    };
    if constexpr (HALF) {
        // FP16 tile: the NT - LBS M1 threads without a step-s second-stage
        // butterfly load two step-(s + 1) butterflies each at once, while the
        // others finish step s and then load the rest (measured: 5 % faster
        // than the form below with FP16 tiles; with FP32 tiles this form
        // spills a register and is 1 % slower)
        constexpr int S2 = LBS * M1;
        constexpr int NI = NT - S2;
        constexpr int NA = 2 * NI;
        static_assert(NI > 0 && NA <= NC2 * M0 && NC2 * M0 - NA <= S2, "step-(s + 1) butterfly split");
        float2 va[R0], vb[R0];
        bool ha = false, hb = false;
        int ia = 0, ib = 0;
        if (tid >= S2) {
            ia = tid - S2;
            ib = ia + NI;
            ha = load_s1(ia, va);
            hb = load_s1(ib, vb);
        } else {
            finish_s();
            ia = NA + tid;
            ha = ia < NC2 * M0 && load_s1(ia, va);
        }
        __syncthreads();
        if (ha) store1(va, ia / NC2, ia % NC2);
        if (hb) store1(vb, ib / NC2, ib % NC2);
    } else {
        // each thread's first butterfly (tid < NT) is loaded before the
        // barrier, while other waves finish step s; the rest (NC2 M0 - NT of
        // them) after it
        if (act1) {
            float pw[R1];
            stage2(t1, j1, pw);
#pragma unroll
            for (int q = 0; q < R1; q++) tv[q] = A.first_step ? pw[q] : tv[q] + pw[q];
        }
        {
            float2 v[R0];
            const int t = tid % NC2, j = tid / NC2;
            const bool act = t < ncol + 2;
            if (act) {
                int rb, lag;
                window(t, &rb, &lag);
                load1(A.tile2, rb, lag, j, v, true);
            }
            __syncthreads();
            if (act) store1(v, j, t);
        }
        {
            const int idx = tid + NT;
            if (idx < NC2 * M0) {
                const int t = idx % NC2, j = idx / NC2;
                if (t < ncol + 2) {
                    float2 v[R0];
                    int rb, lag;
                    window(t, &rb, &lag);
                    load1(A.tile2, rb, lag, j, v, true);
                    store1(v, j, t);
                }
            }
        }
    }
    __syncthreads();
    const int t2 = tid % NC2, j2 = tid / NC2;
    const bool act2 = tid < NC2 * M1 && t2 < ncol + 2;
    float pw2[R1];
    if (act2) stage2(t2, j2, pw2);
    __syncthreads();
    if (act2) {
#pragma unroll
        for (int q = 0; q < R1; q++) pws[t2 * PST + j2 + M1 * q] = pw2[q];
    }
    __syncthreads();
    if (act1) {
#pragma unroll
        for (int q = 0; q < R1; q++) {
            int row;
            const uint32_t off = cell(q, shl, &row);
            int d = shl[N + row] - shl[row];
            if (d > A.spc / 2) d -= A.spc;
            else if (d < -A.spc / 2) d += A.spc;
            *(float*)((char*)accp + off) = tv[q] + pws[(t1 + 1 - d) * PST + j1 + M1 * q];
        }
    }
}

// Power of each raw bin into an LDS float array (stride sst per column).
template <bool ROT>
struct PowerOut {
    float* pw;
    int sst;
    __device__ __forceinline__ void operator()(int t, int w, float2 z) const
    {
        pw[t * sst + w] = ROT ? fmaf(z.x, z.x, __fmul_rn(z.y, z.y)) : abs2_exact(z);
    }
};

// Fold raw-bin powers into the sorted stage rows the way the sign-search
// kernels do (src/noncoherent_integration.jl:92-112, :238-294): raw w < half
// goes to w + half, raw w >= half to w - half, first loop then second. For odd
// ndop both raw 0 and raw ndop-1 land on row `half` and row ndop-1 is never
// written; iterating destinations reproduces that exactly.
__device__ __forceinline__ void fold_into_stage(float* stage, const float* pw, int ncol, int ndop, int sst,
                                                int use_max, int tid)
{
    const int half = ndop / 2;
    const float inv = 1.0f / (float)ndop;
    for (int idx = tid; idx < ncol * ndop; idx += FMDBZP_NTHR) {
        int dst;
        const int c = fdivmod(idx, ndop, inv, &dst);
        float cur = stage[c * sst + dst];
        if (dst >= half && dst < 2 * half) {  // first loop: raw dst - half
            const float v = pw[c * sst + dst - half];
            if (!use_max) cur = v;
            else if (v > cur) cur = v;
        }
        if (dst < ndop - half) {  // second loop: raw dst + half
            const float v = pw[c * sst + dst + half];
            if (!use_max) cur = v;
            else if (v > cur) cur = v;
        }
        stage[c * sst + dst] = cur;
    }
}

// Scatter a stage (sorted rows) into the accumulator with drift
// (`_accumulate_sign_tile!` src/noncoherent_integration.jl:695-746).
// Lanes run along columns for a row-major accumulator and along rows for a
// column-major one, so each store instruction covers contiguous cells.
__device__ __forceinline__ void scatter_stage(const ColumnArgs& A, const float* stage, int p, int r,
                                              int lag0, int ncol, int slice, int tid)
{
    if (A.acc_ldr == 1) {
        const float inv = 1.0f / (float)A.ndop;
        for (int idx = tid; idx < ncol * A.ndop; idx += FMDBZP_NTHR) {
            int row;
            const int c = fdivmod(idx, A.ndop, inv, &row);
            acc_cell(A, p, row, r * A.bs + lag0 + c, slice, stage[c * A.sst + row]);
        }
        return;
    }
    const float inv = 1.0f / (float)ncol;
    for (int idx = tid; idx < ncol * A.ndop; idx += FMDBZP_NTHR) {
        int c;
        const int row = fdivmod(idx, ncol, inv, &c);
        acc_cell(A, p, row, r * A.bs + lag0 + c, slice, stage[c * A.sst + row]);
    }
}

// Load the LB columns of the tile into LDS (x[c][k], stride bst), coalesced.
__device__ __forceinline__ void load_columns(float2* x, const float2* T, int bs, int ndop, int ncol, int bst,
                                             int tid)
{
    const float inv = 1.0f / (float)ncol;
    for (int idx = tid; idx < ncol * ndop; idx += FMDBZP_NTHR) {
        int c;
        const int k = fdivmod(idx, ncol, inv, &c);
        x[c * bst + k] = T[(size_t)k * bs + c];
    }
}

// Data-bit / bit-edge sign search input: the pattern-signed fold of the N_db
// sub-blocks (rows ro + b*sub_len + n, circular) onto [0, sub_len), zero-padded.
struct SignFoldIn {
    const float2* x;
    const float* sg;  // sign of each data bit for this pattern
    int bst, ndop, ndb, sub_len, ro;
    __device__ __forceinline__ float2 operator()(int t, int n) const
    {
        float2 v = make_float2(0.f, 0.f);
        if (n < sub_len) {
            for (int b = 0; b < ndb; b++) {
                int src = ro + b * sub_len + n;  // < 2 ndop
                if (src >= ndop) src -= ndop;
                const float2 u = x[t * bst + src];
                v.x += sg[b] * u.x;
                v.y += sg[b] * u.y;
            }
        }
        return v;
    }
};

// Data-bit / bit-edge sign search (`_sign_search_column!`,
// src/noncoherent_integration.jl:60-115, driven by `_fill_sign_stage_column!`
// :654-686). For each edge offset and data-bit pattern d the reference sums
// the pattern-signed FFTs of the N_db zero-padded sub-blocks; by linearity
// that is the FFT of the signed fold of the sub-blocks onto [0, ndop/N_db),
// zero-padded, which is what is transformed here (one FFT per pattern).
// With N_db == 1 the edge offsets only rotate the column circularly, which
// multiplies its FFT by a unit phase ramp (shift theorem), so every edge gives
// the same |FFT|^2 and one edge is evaluated unless literal_edges is set.
__global__ void __launch_bounds__(FMDBZP_NTHR)
k_column_sign(ColumnArgs A)
{
    extern __shared__ float2 lds[];
    __shared__ float sgn[32];
    const int tid = threadIdx.x;
    const int lbk = xcd_logical_block();
    const int lb = lbk % gridDim.x, r = (lbk / gridDim.x) % gridDim.y, p = lbk / (gridDim.x * gridDim.y);
    const int lag0 = lb * A.LB;
    const int ncol = min(A.LB, A.bs - lag0);
    const int ndop = A.ndop, bst = A.bstride, sst = A.sst;
    float2* x = lds;
    float2* ya = x + (size_t)A.LB * bst;
    float2* yb = ya + (size_t)A.LB * bst;
    float* stage = (float*)(yb + (size_t)A.LB * bst);
    float* pw = stage + (size_t)A.LB * sst;
    load_columns(x, A.tile + (((size_t)p * A.nb + r) * ndop) * A.tp + lag0, A.tp, ndop, ncol, bst, tid);
    for (int idx = tid; idx < A.LB * sst; idx += FMDBZP_NTHR) stage[idx] = 0.f;
    const float* pat = A.patterns + (size_t)A.pset[A.req[p]] * A.ncoh * A.Q;
    const int sub_len = ndop / A.ndb;
    const int cpb = A.ncoh / A.ndb;
    const int E = (A.ndb == 1 && !A.literal_edges) ? 1 : A.E;
    for (int e = 0; e < E; e++) {
        for (int d = 0; d < A.Q; d++) {
            __syncthreads();
            if (tid < A.ndb) sgn[tid] = pat[(size_t)d * A.ncoh + tid * cpb];
            __syncthreads();
            SignFoldIn in{x, sgn, bst, ndop, A.ndb, sub_len, e * A.edge_step};
            fft_run<false, true>(ya, yb, A.pd, A.twD, ncol, bst, tid, FMDBZP_NTHR, in, PowerOut<false>{pw, sst});
            __syncthreads();
            fold_into_stage(stage, pw, ncol, ndop, sst, 1, tid);
        }
    }
    __syncthreads();
    scatter_stage(A, stage, p, r, lag0, ncol, 0, tid);
}

// Rotation search input: the column rotated by the per-column offset, times
// the +-1 pattern of coherent period n / nb (expanded per row in LDS).
struct RotIn {
    const float2* x;
    const float* sgn_row;  // pattern sign of each row n
    const int* eff;        // per-column row offset
    int bst, ndop;
    __device__ __forceinline__ float2 operator()(int t, int n) const
    {
        int src = eff[t] + n;
        if (src >= ndop) src -= ndop;
        const float sg = sgn_row[n];
        const float2 u = x[t * bst + src];
        return make_float2(sg * u.x, sg * u.y);
    }
};

// Rotation input with the pattern sign looked up per row: +-1 of coherent
// period n / nb of pattern q.
struct RotPatIn {
    const float2* x;
    const float* pq;  // pattern q, one sign per coherent period
    const int* eff;
    int bst, ndop, nb;
    float inv_nb;
    __device__ __forceinline__ float2 operator()(int t, int n) const
    {
        int src = eff[t] + n;
        if (src >= ndop) src -= ndop;
        int rem;
        const float sg = pq[fdivmod(n, nb, inv_nb, &rem)];
        const float2 u = x[t * bst + src];
        return make_float2(sg * u.x, sg * u.y);
    }
};

// Power (fma form, as the reference's muladd) of raw bin w straight into the
// accumulator row (w + ndop/2) mod ndop of rotation slice `slice`: the
// sign-path fold for even ndop, with nothing to max-reduce.
struct RotAccOut {
    const ColumnArgs* A;
    int p, cp0, slice, half;
    __device__ __forceinline__ void operator()(int t, int w, float2 z) const
    {
        int row = w + half;
        if (row >= A->ndop) row -= A->ndop;
        acc_cell(*A, p, row, cp0 + t, slice, fmaf(z.x, z.x, __fmul_rn(z.y, z.y)));
    }
};

// Secondary-code rotation search (`_rotation_column!`,
// src/noncoherent_integration.jl:183-297). The reference combines N_coh
// zero-padded sub-block FFTs with the phasors patterns[p,q]
// exp(-2 pi i p s / N_coh) (src/sign_patterns.jl:80-93); that combination is
// exactly the length-ndop FFT of the column, rotated by the per-column
// alignment offset and multiplied by the +-1 pattern of coherent period
// n / nb. That FFT is what is computed here (one FFT per pattern); the +-1
// multiply is exact in Float32. Patterns sharing a rotation (data-bit combos)
// and bit-edge offsets max-reduce into that rotation's stage slice.
__global__ void __launch_bounds__(FMDBZP_NTHR)
k_column_rotation(ColumnArgs A)
{
    extern __shared__ float2 lds[];
    __shared__ int seff[64];
    const int tid = threadIdx.x;
    const int lbk = xcd_logical_block();
    const int lb = lbk % gridDim.x, r = (lbk / gridDim.x) % gridDim.y, p = lbk / (gridDim.x * gridDim.y);
    const int lag0 = lb * A.LB;
    const int ncol = min(A.LB, A.bs - lag0);
    const int ndop = A.ndop, bst = A.bstride, sst = A.sst;
    float2* x = lds;
    float2* ya = x + (size_t)A.LB * bst;
    float2* yb = ya + (size_t)A.LB * bst;
    float* stage = (float*)(yb + (size_t)A.LB * bst);
    float* pw = stage + (size_t)A.LB * sst;
    float* sgn_row = pw + (size_t)A.LB * sst;
    load_columns(x, A.tile + (((size_t)p * A.nb + r) * ndop) * A.tp + lag0, A.tp, ndop, ncol, bst, tid);
    const float* pat = A.patterns + (size_t)A.pset[A.req[p]] * A.ncoh * A.Q;
    const int half_block = A.bs >> 1;
    const float inv_nb = 1.0f / (float)A.nb;
    if (A.rot_direct) {
        // one pattern per rotation slice (no data-bit combos, one edge offset)
        for (int c = tid; c < ncol; c += FMDBZP_NTHR) {
            const int pc = r * A.bs + lag0 + c;
            const int wrap = ((A.nb - pc / A.bs) % A.nb) * A.bs + (pc % A.bs);
            seff[c] = ((wrap + half_block) / A.bs) % A.nb;
        }
        for (int rot = 0; rot < A.R; rot++) {
            __syncthreads();  // seff / x ready; the previous transform is done with ya, yb
            RotPatIn in{x, pat + (size_t)rot * A.ncoh, seff, bst, ndop, A.nb, inv_nb};
            fft_run<false, true>(ya, yb, A.pd, A.twD, ncol, bst, tid, FMDBZP_NTHR, in,
                                 RotAccOut{&A, p, r * A.bs + lag0, rot, ndop / 2});
        }
        return;
    }
    for (int rot = 0; rot < A.R; rot++) {
        for (int idx = tid; idx < A.LB * sst; idx += FMDBZP_NTHR) stage[idx] = 0.f;
        for (int e = 0; e < A.E; e++) {
            __syncthreads();
            // per-column alignment to the primary-code wrap (:212-215)
            for (int c = tid; c < ncol; c += FMDBZP_NTHR) {
                const int pc = r * A.bs + lag0 + c;
                const int wrap = ((A.nb - pc / A.bs) % A.nb) * A.bs + (pc % A.bs);
                const int cro = ((wrap + half_block) / A.bs) % A.nb;
                seff[c] = (e * A.edge_step + cro) % ndop;
            }
            for (int d = 0; d < A.ndc; d++) {
                const int q = rot * A.ndc + d;
                __syncthreads();
                for (int n = tid; n < ndop; n += FMDBZP_NTHR) {
                    int rem;
                    sgn_row[n] = pat[(size_t)q * A.ncoh + fdivmod(n, A.nb, inv_nb, &rem)];
                }
                __syncthreads();
                RotIn in{x, sgn_row, seff, bst, ndop};
                fft_run<false, true>(ya, yb, A.pd, A.twD, ncol, bst, tid, FMDBZP_NTHR, in, PowerOut<true>{pw, sst});
                __syncthreads();
                fold_into_stage(stage, pw, ncol, ndop, sst, A.use_max, tid);
            }
        }
        __syncthreads();
        scatter_stage(A, stage, p, r, lag0, ncol, rot, tid);
        __syncthreads();  // the next rotation zeroes the stage this scatter reads
    }
}

// Direct rotation path at ndop = 2000 (2000 = 16 x 5 x 5 x 5, compile-time):
// one column per workgroup, two rotation slices per pass.
//
// Input of rotation q at row n: the column rotated by its alignment offset
// (held rotated in LDS) times pattern[q][n / nb]. The pattern signs are
// bitmasks (bit p set: period p negated) and the sign is applied by flipping
// the float sign bit, which equals the multiplication by -1. The period of
// row n is umulhi(n, ceil(2^32 / nb)), exact for n, nb < 2^11.
struct RotSignIn {
    const float2* xr;
    uint32_t m0, m1, magic;
    __device__ __forceinline__ float2 operator()(int t, int n) const
    {
        const uint32_t per = __umulhi((uint32_t)n, magic);
        const uint32_t s = (((t ? m1 : m0) >> per) & 1u) << 31;
        const float2 u = xr[n];
        return make_float2(__uint_as_float(__float_as_uint(u.x) ^ s), __uint_as_float(__float_as_uint(u.y) ^ s));
    }
};
// grid (bs, nb, batch); dynamic LDS: the rotated column (2000 complex), two
// padded transform buffers and the R pattern masks. Column-major accumulator.
//
// The last radix-5 stage is written out here: each thread's output cells
// (rows of its butterflies, moved by the drift of their destination rows)
// are fixed for the column, so their offsets are computed once, and the
// accumulator reads of a pass are all issued before the pass's transforms,
// instead of one dependent read-add-write per output.
// NTH threads: 512 gives the three workgroups that fit a CU's LDS six waves
// per SIMD (against three with 256) to hide the six barriers of a pass; the
// radix-16 stage then has 250 active threads and the radix-5 stages 400.
template <int NTH>
__global__ void __launch_bounds__(NTH)
k_column_rot2000(ColumnArgs A)
{
    constexpr int N = 2000;
    constexpr int BST = N + (N >> 4) + 1;
    constexpr int M3 = N / 5;                                // last stage: radix 5, stride 400
    constexpr int IT3 = (M3 + NTH - 1) / NTH;  // butterfly positions per thread
    extern __shared__ float2 lds[];
    const int tid = threadIdx.x;
    const int lbk = xcd_logical_block();
    const int lag = lbk % gridDim.x, r = (lbk / gridDim.x) % gridDim.y, p = lbk / (gridDim.x * gridDim.y);
    float2* xr = lds;
    float2* a = lds + N;
    uint32_t* smask = (uint32_t*)(lds + N + 2 * BST);
    const int pc = r * A.bs + lag;
    // per-column alignment to the primary-code wrap (src/noncoherent_integration.jl:212-215)
    const int wrap = ((A.nb - pc / A.bs) % A.nb) * A.bs + (pc % A.bs);
    const int eff = ((wrap + (A.bs >> 1)) / A.bs) % A.nb;
    const float2* T = A.tile + (((size_t)p * A.nb + r) * N) * A.tp + lag;
    for (int k = tid; k < N; k += NTH) {
        int src = k + eff;
        if (src >= N) src -= N;
        // neighbouring workgroups (the next lags) read the same tile lines: a plain, cached load
        xr[k] = T[(size_t)src * A.tp];
    }
    if (tid < A.R) {
        const float* pat = A.patterns + ((size_t)A.pset[A.req[p]] * A.Q + tid) * A.ncoh;
        uint32_t m = 0;
        for (int q = 0; q < A.ncoh; q++)
            if (pat[q] < 0.f) m |= 1u << q;
        smask[tid] = m;
    }
    // output cell offsets within a slice: raw bin w = j + 400 i goes to sorted
    // row (w + 1000) mod 2000, column cp + drift of that row (mod spc)
    uint32_t off[IT3][5];
#pragma unroll
    for (int it = 0; it < IT3; it++) {
        const int j = min(tid + it * NTH, M3 - 1);
#pragma unroll
        for (int i = 0; i < 5; i++) {
            int row = j + M3 * i + N / 2;
            if (row >= N) row -= N;
            int dc = pc + A.shifts[row];
            if (dc >= A.spc) dc -= A.spc;
            // byte offset within a rotation slice (below 2^32, checked at plan creation)
            off[it][i] = (uint32_t)(row + dc * A.acc_ldc) * (uint32_t)sizeof(float);
        }
    }
    const uint32_t magic = (uint32_t)((0x100000000ull + (uint64_t)A.nb - 1) / (uint64_t)A.nb);
    float* accp = A.acc + (size_t)p * A.acc_ps;
    const size_t slice_stride = (size_t)A.spc * A.acc_ldc;
    const bool first = A.first_step != 0;
#pragma unroll 1
    for (int q0 = 0; q0 < A.R; q0 += 2) {
        const int nq = min(2, A.R - q0);
        float* base0 = accp + (size_t)q0 * slice_stride;
        float* base1 = base0 + slice_stride;
        // Opaque per-pass copies of the byte offsets: the loads and stores then
        // see scalar base + 32-bit offset and take the scalar-base address
        // form, instead of 64-bit adds on offsets widened once outside the loop.
        uint32_t po[IT3][5];
#pragma unroll
        for (int it = 0; it < IT3; it++)
#pragma unroll
            for (int i = 0; i < 5; i++) {
                po[it][i] = off[it][i];
                asm volatile("" : "+v"(po[it][i]));
            }
        float prev[IT3][2][5];
        if (!first) {
#pragma unroll
            for (int it = 0; it < IT3; it++) {
                if (tid + it * NTH < M3) {
#pragma unroll
                    for (int i = 0; i < 5; i++) prev[it][0][i] = *(const float*)((const char*)base0 + po[it][i]);
                    if (nq > 1) {
#pragma unroll
                        for (int i = 0; i < 5; i++) prev[it][1][i] = *(const float*)((const char*)base1 + po[it][i]);
                    }
                }
            }
        }
        __syncthreads();  // column and masks ready; the previous pass is done with the buffers
        // An opaque copy of the thread index keeps the transform's index
        // arithmetic and twiddle loads inside the loop: hoisted out of it,
        // they would all stay live in registers across passes.
        int tid_pass;
        asm volatile("v_mov_b32 %0, %1" : "=v"(tid_pass) : "v"(tid));
        const uint32_t m0 = smask[q0], m1 = smask[nq > 1 ? q0 + 1 : q0];
        stage_static<16, false, N, 1, 2, NTH>(RotSignIn{xr, m0, m1, magic}, LdsOut<true>{a, BST}, A.twD,
                                                      tid_pass);
        __syncthreads();
        // last-stage twiddles, loaded ahead of the two in-place stages
        float2 w3[IT3][5];
#pragma unroll
        for (int it = 0; it < IT3; it++) {
            const int j = min(tid_pass + it * NTH, M3 - 1);
#pragma unroll
            for (int i = 1; i < 5; i++) w3[it][i] = twid<false>(A.twD, i * j);
        }
        stage_static_inplace_pair<5, false, N, 16, NTH, BST>(a, A.twD, tid_pass);
        stage_static_inplace_pair<5, false, N, 80, NTH, BST>(a, A.twD, tid_pass);
#pragma unroll
        for (int it = 0; it < IT3; it++) {
            const int j = tid_pass + it * NTH;
            if (j < M3) {
                float2 v[2][5];
                const float2* src = a + lds_pad(j);
#pragma unroll
                for (int u = 0; u < 2; u++)
#pragma unroll
                    for (int i = 0; i < 5; i++) v[u][i] = src[u * BST + i * lds_group_step<true, M3>()];
#pragma unroll
                for (int i = 1; i < 5; i++) {
                    v[0][i] = cmulf(v[0][i], w3[it][i]);
                    v[1][i] = cmulf(v[1][i], w3[it][i]);
                }
#pragma unroll
                for (int u = 0; u < 2; u++) {
                    if (u < nq) {
                        bfly<5, false>(v[u]);
                        char* b = (char*)(u ? base1 : base0);
#pragma unroll
                        for (int i = 0; i < 5; i++) {
                            // muladd(re, re, im * im), the reference's rotation power
                            const float pw = fmaf(v[u][i].x, v[u][i].x, __fmul_rn(v[u][i].y, v[u][i].y));
                            *(float*)(b + po[it][i]) = first ? pw : prev[it][u][i] + pw;
                        }
                    }
                }
            }
        }
    }
}

// W_25^k = exp(-2 pi i k / 25), k = 0..16 (the in-register 5 x 5 DFT's twiddles)
__constant__ float2 kW25[17] = {
    {1.0f, -0.0f}, {0.9685831611286311f, -0.2486898871648548f}, {0.8763066800438636f, -0.4817536741017153f},
    {0.7289686274214116f, -0.6845471059286886f}, {0.5358267949789965f, -0.8443279255020151f},
    {0.30901699437494745f, -0.9510565162951535f}, {0.06279051952931353f, -0.9980267284282716f},
    {-0.1873813145857246f, -0.9822872507286887f}, {-0.4257792915650727f, -0.9048270524660195f},
    {-0.6374239897486897f, -0.7705132427757893f}, {-0.8090169943749473f, -0.5877852522924732f},
    {-0.9297764858882513f, -0.36812455268467814f}, {-0.9921147013144778f, -0.12533323356430454f},
    {-0.9921147013144779f, 0.12533323356430429f}, {-0.9297764858882515f, 0.3681245526846779f},
    {-0.8090169943749478f, 0.5877852522924727f}, {-0.6374239897486895f, 0.7705132427757894f}};

// ---------------------------------------------------------------------------
// Reductions: peak with the reference's tie-break order, FP64 row sums.
// ---------------------------------------------------------------------------
// Visiting-order key of cell (row, col_eff). The multistep path and every
// non-rotation streamed path pick the lowest column, then the lowest row
// (src/est_signal_noise_power.jl:109-135, src/acquire.jl:352-384); the
// streamed rotation path visits (code column, rotation slice, row)
// (src/acquire.jl:311-322, :405-423).
__device__ __forceinline__ uint64_t cell_key(int row, int col, int ndop, int spc, int R, int streamed_rot)
{
    if (streamed_rot) {
        const int slice = col / spc, cp = col - slice * spc;
        return ((uint64_t)cp * R + slice) * ndop + row;
    }
    return (uint64_t)col * ndop + row;
}

__device__ __forceinline__ bool better(float v, uint64_t k, float bv, uint64_t bk)
{
    return v > bv || (v == bv && k < bk);
}

// grid (ndop, batch): one workgroup per (row, PRN).
__global__ void __launch_bounds__(FMDBZP_NTHR)
k_reduce_rows(const float* __restrict__ acc, int ndop, int spc, int spc_eff, int ap, int R, int streamed_rot,
              double* __restrict__ rowsum, float* __restrict__ rowbest_v, uint64_t* __restrict__ rowbest_k)
{
    __shared__ double ssum[FMDBZP_NTHR];
    __shared__ float sv[FMDBZP_NTHR];
    __shared__ uint64_t sk[FMDBZP_NTHR];
    const int row = blockIdx.x, p = blockIdx.y, tid = threadIdx.x;
    const float* a = acc + ((size_t)p * ndop + row) * ap;  // 128-byte aligned (ap is a multiple of 32)
    double s = 0.0;
    float bv = -INFINITY;
    uint64_t bk = ~0ull;
    // the key is only needed when the value can win (v >= bv)
    auto visit = [&](float v, int c) {
        s += (double)v;
        if (v >= bv) {
            const uint64_t k = cell_key(row, c, ndop, spc, R, streamed_rot);
            if (better(v, k, bv, bk)) { bv = v; bk = k; }
        }
    };
    // 16-byte loads, four in flight per thread
    const int n4 = spc_eff >> 2;
    const float4* a4 = (const float4*)a;
#pragma unroll 4
    for (int g = tid; g < n4; g += FMDBZP_NTHR) {
        const float4 v = a4[g];
        visit(v.x, 4 * g);
        visit(v.y, 4 * g + 1);
        visit(v.z, 4 * g + 2);
        visit(v.w, 4 * g + 3);
    }
    for (int c = 4 * n4 + tid; c < spc_eff; c += FMDBZP_NTHR) visit(a[c], c);
    ssum[tid] = s;
    sv[tid] = bv;
    sk[tid] = bk;
    __syncthreads();
    for (int w = FMDBZP_NTHR / 2; w > 0; w >>= 1) {
        if (tid < w) {
            ssum[tid] += ssum[tid + w];
            if (better(sv[tid + w], sk[tid + w], sv[tid], sk[tid])) {
                sv[tid] = sv[tid + w];
                sk[tid] = sk[tid + w];
            }
        }
        __syncthreads();
    }
    if (tid == 0) {
        rowsum[(size_t)p * ndop + row] = ssum[0];
        rowbest_v[(size_t)p * ndop + row] = sv[0];
        rowbest_k[(size_t)p * ndop + row] = sk[0];
    }
}

// Column-major accumulator, pass 1. grid (column chunks, ceil(ndop / (4 NTHR)),
// batch): each thread owns 4 consecutive rows (one 16-byte load per column;
// the column pitch is a multiple of 32 rows, so the load stays in the padded
// column) and walks the chunk's `cw` columns in order, producing the chunk's
// FP64 row sums and best (value, visit-order key) per row. A cell's key is
// formed only when its value reaches the row's best so far.
__global__ void __launch_bounds__(FMDBZP_NTHR)
k_reduce_cols(const float* __restrict__ acc, size_t acc_ps, int ldc, int ndop, int spc, int spc_eff, int R,
              int streamed_rot, int cw, double* __restrict__ psum, float* __restrict__ pbest_v,
              uint64_t* __restrict__ pbest_k)
{
    const int chunk = blockIdx.x, row0 = 4 * (blockIdx.y * FMDBZP_NTHR + threadIdx.x), p = blockIdx.z;
    if (row0 >= ndop) return;
    const float* a = acc + (size_t)p * acc_ps + row0;
    const int c0 = chunk * cw, c1 = min(spc_eff, c0 + cw);
    double s[4] = {0.0, 0.0, 0.0, 0.0};
    float bv[4] = {-INFINITY, -INFINITY, -INFINITY, -INFINITY};
    uint64_t bk[4] = {~0ull, ~0ull, ~0ull, ~0ull};
#pragma unroll 4
    for (int c = c0; c < c1; c++) {
        const float4 v4 = *(const float4*)(a + (size_t)c * ldc);
        const float v[4] = {v4.x, v4.y, v4.z, v4.w};
#pragma unroll
        for (int u = 0; u < 4; u++) {
            s[u] += (double)v[u];
            if (v[u] >= bv[u]) {
                const uint64_t k = cell_key(row0 + u, c, ndop, spc, R, streamed_rot);
                if (better(v[u], k, bv[u], bk[u])) { bv[u] = v[u]; bk[u] = k; }
            }
        }
    }
#pragma unroll
    for (int u = 0; u < 4; u++) {
        if (row0 + u < ndop) {
            const size_t o = ((size_t)p * gridDim.x + chunk) * ndop + row0 + u;
            psum[o] = s[u];
            pbest_v[o] = bv[u];
            pbest_k[o] = bk[u];
        }
    }
}

// Column-major accumulator, pass 2. grid (ceil(ndop / MERGE_ROWS), batch): 32
// rows per workgroup, eight threads per row, each over a contiguous eighth of
// the chunks in order; the eighths are combined in order. One thread per row
// walked 611 dependent chunks in 290 us (2000 rows, 2.5 M columns).
#define FMDBZP_MERGE_ROWS 32
__global__ void __launch_bounds__(FMDBZP_NTHR)
k_merge_rows(const double* __restrict__ psum, const float* __restrict__ pbest_v,
             const uint64_t* __restrict__ pbest_k, int nchunk, int ndop, double* __restrict__ rowsum,
             float* __restrict__ rowbest_v, uint64_t* __restrict__ rowbest_k)
{
    constexpr int G = FMDBZP_NTHR / FMDBZP_MERGE_ROWS;
    __shared__ double ss[G][FMDBZP_MERGE_ROWS];
    __shared__ float sv[G][FMDBZP_MERGE_ROWS];
    __shared__ uint64_t sk[G][FMDBZP_MERGE_ROWS];
    const int lr = threadIdx.x % FMDBZP_MERGE_ROWS, g = threadIdx.x / FMDBZP_MERGE_ROWS;
    const int row = blockIdx.x * FMDBZP_MERGE_ROWS + lr, p = blockIdx.y;
    const int per = (nchunk + G - 1) / G;
    double s = 0.0;
    float bv = -INFINITY;
    uint64_t bk = ~0ull;
    if (row < ndop) {
#pragma unroll 4
        for (int c = g * per; c < min(nchunk, (g + 1) * per); c++) {
            const size_t o = ((size_t)p * nchunk + c) * ndop + row;
            s += psum[o];
            if (better(pbest_v[o], pbest_k[o], bv, bk)) { bv = pbest_v[o]; bk = pbest_k[o]; }
        }
    }
    ss[g][lr] = s;
    sv[g][lr] = bv;
    sk[g][lr] = bk;
    __syncthreads();
    if (g == 0 && row < ndop) {
        for (int h = 1; h < G; h++) {
            s += ss[h][lr];
            if (better(sv[h][lr], sk[h][lr], bv, bk)) { bv = sv[h][lr]; bk = sk[h][lr]; }
        }
        rowsum[(size_t)p * ndop + row] = s;
        rowbest_v[(size_t)p * ndop + row] = bv;
        rowbest_k[(size_t)p * ndop + row] = bk;
    }
}

// grid (batch): peak, noise estimate (src/acquire.jl:687-697,
// src/est_signal_noise_power.jl:211-243) and interpolation neighbours.
__global__ void __launch_bounds__(FMDBZP_NTHR)
k_finalize(const float* __restrict__ acc, const double* __restrict__ rowsum,
           const float* __restrict__ rowbest_v, const uint64_t* __restrict__ rowbest_k, int ndop,
           int spc, int spc_eff, size_t acc_ps, int ldr, int ldc, int R, int streamed_rot, int noise_est,
           int spchip, fmdbzp_prn_stats* __restrict__ stats)
{
    __shared__ double ssum[FMDBZP_NTHR];
    __shared__ float sv[FMDBZP_NTHR];
    __shared__ uint64_t sk[FMDBZP_NTHR];
    __shared__ int s_row, s_col;
    const int p = blockIdx.x, tid = threadIdx.x;
    float bv = -INFINITY;
    uint64_t bk = ~0ull;
    double tot = 0.0;
    for (int r = tid; r < ndop; r += FMDBZP_NTHR) {
        const float v = rowbest_v[(size_t)p * ndop + r];
        const uint64_t k = rowbest_k[(size_t)p * ndop + r];
        if (better(v, k, bv, bk)) { bv = v; bk = k; }
        tot += rowsum[(size_t)p * ndop + r];
    }
    sv[tid] = bv;
    sk[tid] = bk;
    ssum[tid] = tot;
    __syncthreads();
    for (int w = FMDBZP_NTHR / 2; w > 0; w >>= 1) {
        if (tid < w) {
            ssum[tid] += ssum[tid + w];
            if (better(sv[tid + w], sk[tid + w], sv[tid], sk[tid])) {
                sv[tid] = sv[tid + w];
                sk[tid] = sk[tid + w];
            }
        }
        __syncthreads();
    }
    const double total = ssum[0];
    const float peak = sv[0];
    const uint64_t key = sk[0];
    if (tid == 0) {
        int row, col;
        if (streamed_rot) {
            row = (int)(key % (uint64_t)ndop);
            const uint64_t rest = key / (uint64_t)ndop;
            const int slice = (int)(rest % (uint64_t)R);
            const int cp = (int)(rest / (uint64_t)R);
            col = slice * spc + cp;
        } else {
            row = (int)(key % (uint64_t)ndop);
            col = (int)(key / (uint64_t)ndop);
        }
        // no comparable cell (all NaN input): report cell (0, 0), never index out of range
        if (key == ~0ull || row < 0 || row >= ndop || col < 0 || col >= spc_eff) {
            row = 0;
            col = 0;
        }
        s_row = row;
        s_col = col;
    }
    __syncthreads();
    const int row = s_row, col = s_col;
    const float* a = acc + (size_t)p * acc_ps;
    // GlobalMean exclusion: columns [col - spchip, col + spchip] clipped, all rows
    int lo = col - spchip;
    if (lo < 0) lo = 0;
    int hi = col + spchip;
    if (hi > spc_eff - 1) hi = spc_eff - 1;
    const int nex = hi - lo + 1;
    double ex = 0.0;
    if (noise_est == FMDBZP_NOISE_GLOBAL_MEAN) {
        for (int idx = tid; idx < nex * ndop; idx += FMDBZP_NTHR) {
            const int rr = idx / nex, cc = lo + idx - rr * nex;
            ex += (double)a[(size_t)rr * ldr + (size_t)cc * ldc];
        }
    }
    __syncthreads();
    ssum[tid] = ex;
    __syncthreads();
    for (int w = FMDBZP_NTHR / 2; w > 0; w >>= 1) {
        if (tid < w) ssum[tid] += ssum[tid + w];
        __syncthreads();
    }
    if (tid == 0) {
        fmdbzp_prn_stats st;
        st.peak_power = peak;
        st.peak_row = row;
        st.peak_col = col;
        if (noise_est == FMDBZP_NOISE_GLOBAL_MEAN) {
            const double s = total - ssum[0];
            const int64_t cnt = (int64_t)(spc_eff - nex) * ndop;
            st.noise_sum = s;
            st.noise_cells = cnt;
            st.noise_power = (float)s / (float)cnt;
        } else {
            const int opp = (row + ndop / 2) % ndop;
            const double s = rowsum[(size_t)p * ndop + opp];
            st.noise_sum = s;
            st.noise_cells = spc_eff;
            st.noise_power = (float)s / (float)spc_eff;
        }
        const int rot = col / spc, scr = col - rot * spc;
        const int cl = (scr == 0 ? spc - 1 : scr - 1) + rot * spc;
        const int cr = (scr == spc - 1 ? 0 : scr + 1) + rot * spc;
        const int dl = row == 0 ? ndop - 1 : row - 1;
        const int dr = row == ndop - 1 ? 0 : row + 1;
        st.code_left = a[(size_t)row * ldr + (size_t)cl * ldc];
        st.code_right = a[(size_t)row * ldr + (size_t)cr * ldc];
        st.dop_left = a[(size_t)dl * ldr + (size_t)col * ldc];
        st.dop_right = a[(size_t)dr * ldr + (size_t)col * ldc];
        stats[p] = st;
    }
}

// ---------------------------------------------------------------------------
// Rotation search at large ndop (k_column_rotbig): the direct rotation path
// (one pattern per rotation slice, one edge offset, even ndop) for
// ndop = 25 nb, the 25 coherent periods of the E1-like searches, in a
// four-step factorisation. With rows n = p nb + m (period p, lag m within the
// period) and raw bins w = s + 25 k, the FFT of the pattern-signed column is
//   X_q[s + 25 k] = sum_m W_nb^(k m) W_N^(s m) sum_p sigma_q[p] W_25^(s p) x[p nb + m],
// so per rotation q the thread of lag m takes its 25 values (held in
// registers for the whole column) through the signs and a 25-point DFT, then
// multiplies by W_N^(s m) (as W_N^(s1 m) W_N^(5 s2 m), eight held factors);
// one LDS transpose gives the 25 rows of nb values, and each wave runs the
// nb-point transforms of its rows in place in LDS with no block barrier, the
// last stage leaving the powers in the rows. After one barrier every thread
// adds the powers of its fixed accumulator cells (consecutive sorted rows
// across the threads, so the read-modify-writes are coalesced), whose
// offsets are computed once per column and whose reads are issued ahead of
// each rotation's transform. One code column per workgroup; three block
// barriers per rotation.
// grid (bs, nrb, batch); dynamic LDS: 25 padded rows of nb float2, nb row
// twiddles, ndop cell offsets, R masks.
// ---------------------------------------------------------------------------
// LDS accesses of one wave stay in program order across this point (the
// wave's own LDS operations complete in order; this keeps the compiler from
// moving them across it).
__device__ __forceinline__ void wave_lds_sync()
{
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// One in-place radix-R Stockham stage of the n-point rows s0, s0 + sstep, ...
// (nr rows, pitch rp, padded) by one wave: the rows' butterflies are spread
// over the lanes (at most MB each), loaded, then written back. Row twiddles
// W_n^j come from the n-entry table twR. LAST: the final stage, which writes
// |X|^2 (muladd(re, re, im * im)) of output k as float k of its row.
template <int R, int MB, bool LAST>
__device__ __forceinline__ void rows_stage(float2* rows, int rp, int s0, int sstep, int nr, int n, int Ns,
                                           const float2* __restrict__ twR, int lane)
{
    const int m = n / R;
    const int tstride = n / (Ns * R);
    const int total = nr * m;
    const float inv_m = 1.0f / (float)m, inv_ns = 1.0f / (float)Ns;
    float2 v[MB][R];
    int orow[MB], obase[MB];
#pragma unroll
    for (int b = 0; b < MB; b++) {
        const int idx = lane + 64 * b;
        orow[b] = -1;
        obase[b] = 0;
        if (idx < total) {
            int j, k;
            const int i = fdivmod(idx, m, inv_m, &j);
            const int g = fdivmod(j, Ns, inv_ns, &k);
            const int rb = (s0 + sstep * i) * rp;
            const float2* a = rows + rb;
#pragma unroll
            for (int r = 0; r < R; r++) v[b][r] = a[lds_pad(j + r * m)];
            if (Ns > 1) {
#pragma unroll
                for (int r = 1; r < R; r++) v[b][r] = cmulf(v[b][r], twR[r * k * tstride]);
            }
            bfly<R, false>(v[b]);
            orow[b] = rb;
            obase[b] = g * Ns * R + k;
        }
    }
    wave_lds_sync();
#pragma unroll
    for (int b = 0; b < MB; b++) {
        if (orow[b] >= 0) {
            if constexpr (LAST) {
                float* pw = (float*)(rows + orow[b]);
#pragma unroll
                for (int r = 0; r < R; r++)
                    pw[obase[b] + r * Ns] = fmaf(v[b][r].x, v[b][r].x, __fmul_rn(v[b][r].y, v[b][r].y));
            } else {
#pragma unroll
                for (int r = 0; r < R; r++) rows[orow[b] + lds_pad(obase[b] + r * Ns)] = v[b][r];
            }
        }
    }
    wave_lds_sync();
}

// row radices 10 and 5 with 1 and 2 butterflies per lane for a group of rows
// (checked on the host)
template <bool LAST>
__device__ __forceinline__ void rows_stage_any(int R, float2* rows, int rp, int s0, int sstep, int nr, int n, int Ns,
                                               const float2* __restrict__ twR, int lane)
{
    if (R == 10) rows_stage<10, 1, LAST>(rows, rp, s0, sstep, nr, n, Ns, twR, lane);
    else rows_stage<5, 2, LAST>(rows, rp, s0, sstep, nr, n, Ns, twR, lane);
}

// CPT: accumulator cells (sorted rows) per thread, ceil(ndop / NT); rgrp:
// rows a wave transforms together (both checked on the host). Serves the row
// lengths that k_column_rot25 has no instance of (10 rows) and more than 64
// rotations.
template <int NT, int CPT>
__global__ void __launch_bounds__(NT)
k_column_rotbig(ColumnArgs A, FftPlanDev prow, const float2* __restrict__ twR, int rgrp)
{
    constexpr int NC = 25;
    extern __shared__ float2 lds[];
    const int N = A.ndop, nb = A.nb;
    const int rp = fft_lds_span(nb);  // row pitch
    float2* rows = lds;
    float2* stw = lds + (size_t)NC * rp;  // row twiddles W_nb^j
    uint32_t* soff = (uint32_t*)(stw + nb);  // cell offset of each sorted row
    uint32_t* smask = soff + N;
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    for (int j = tid; j < nb; j += NT) stw[j] = twR[j];
    const int lbk = xcd_logical_block();
    // column of this workgroup (kept in scalar registers: the divisions run on
    // the vector unit)
    const int lag = __builtin_amdgcn_readfirstlane(lbk % gridDim.x);
    const int rr = __builtin_amdgcn_readfirstlane((lbk / gridDim.x) % gridDim.y);
    const int p = __builtin_amdgcn_readfirstlane(lbk / (gridDim.x * gridDim.y));
    int r = A.rb0 + rr;
    if (r >= nb) r -= nb;
    const int pc = r * A.bs + lag;
    // per-column alignment to the primary-code wrap (src/noncoherent_integration.jl:212-215)
    const int wrap = ((nb - pc / A.bs) % nb) * A.bs + (pc % A.bs);
    const int eff = ((wrap + (A.bs >> 1)) / A.bs) % nb;
    if (tid < A.R) {
        const float* pat = A.patterns + ((size_t)A.pset[A.req[p]] * A.Q + tid) * A.ncoh;
        uint32_t msk = 0;
        for (int q = 0; q < A.ncoh; q++)
            if (pat[q] < 0.f) msk |= 1u << q;
        smask[tid] = msk;
    }
    // lag m = tid: its 25 values (the column rotated by its alignment offset)
    // and the factors of W_N^(s m) = W_N^(s1 m) W_N^(5 s2 m), s = s1 + 5 s2
    const int m = tid;
    const bool act = m < nb;
    float2 x[NC], tw1[5], tw5[5];
    {
        const float2* T = A.tile + (((size_t)p * A.nrb + rr) * N) * A.tp + lag;
#pragma unroll
        for (int pp = 0; pp < NC; pp++) {
            x[pp] = make_float2(0.f, 0.f);
            if (act) {
                int src = pp * nb + m + eff;
                if (src >= N) src -= N;
                x[pp] = T[(size_t)src * A.tp];
            }
        }
#pragma unroll
        for (int i = 0; i < 5; i++) {
            tw1[i] = act ? A.twD[i * m] : make_float2(1.f, 0.f);
            tw5[i] = act ? A.twD[5 * i * m] : make_float2(1.f, 0.f);
        }
    }
    // accumulator cell of sorted row w (this thread's cells are w = tid + NT c):
    // column pc moved by the row's drift; byte offset within a rotation slice,
    // ~0u outside the window
    for (int w = tid; w < N; w += NT) {
        int dc = pc + A.shifts[w];
        if (dc >= A.spc) dc -= A.spc;
        int o = dc - A.win0;
        if (o < 0) o += A.spc;
        soff[w] = o < A.winlen ? (uint32_t)(w + o * A.acc_ldc) * (uint32_t)sizeof(float) : ~0u;
    }
    float* accp = A.acc + (size_t)p * A.acc_ps;
    const size_t slice_stride = (size_t)A.slice_cols * A.acc_ldc;
    const bool first = A.first_step != 0;
    const int nw = NT / 64;
    const int nr = (NC - wave + nw - 1) / nw;  // rows wave, wave + nw, ... below 25
#pragma unroll 1
    for (int q = 0; q < A.R; q++) {
        char* base = (char*)(accp + (size_t)q * slice_stride);
        __syncthreads();  // tables ready; the previous rotation's powers have been read
        // this rotation's accumulator cells, read ahead of its transform; cells
        // outside the window read the slice's first cell (in bounds) instead,
        // so the loads carry no branches
        float prev[CPT];
        if (!first) {
#pragma unroll
            for (int c = 0; c < CPT; c++) {
                const int w = min(tid + NT * c, N - 1);
                const uint32_t o = soff[w];
                prev[c] = *(const float*)(base + (o != ~0u ? o : 0u));
            }
        } else {
#pragma unroll
            for (int c = 0; c < CPT; c++) prev[c] = 0.f;
        }
        const uint32_t mq = smask[q];
        if (act) {
            // signs of the periods, then the 25-point DFT over p = p2 + 5 p1 as
            // 5 x 5: inner over p1, twiddle W_25^(s1 p2), outer over p2 -> s = s1 + 5 s2
            float2 u[5][5];
#pragma unroll
            for (int p2 = 0; p2 < 5; p2++) {
#pragma unroll
                for (int p1 = 0; p1 < 5; p1++) {
                    const int pp = p2 + 5 * p1;
                    const uint32_t sg = ((mq >> pp) & 1u) << 31;
                    u[p2][p1] = make_float2(__uint_as_float(__float_as_uint(x[pp].x) ^ sg),
                                            __uint_as_float(__float_as_uint(x[pp].y) ^ sg));
                }
                bfly5<false>(u[p2]);
#pragma unroll
                for (int s1 = 1; s1 < 5; s1++)
                    if (p2) u[p2][s1] = cmulf(u[p2][s1], kW25[s1 * p2]);
            }
#pragma unroll
            for (int s1 = 0; s1 < 5; s1++) {
                float2 w5[5];
#pragma unroll
                for (int p2 = 0; p2 < 5; p2++) w5[p2] = s1 ? cmulf(u[p2][s1], tw1[s1]) : u[p2][s1];
                bfly5<false>(w5);
#pragma unroll
                for (int s2 = 0; s2 < 5; s2++) {
                    const float2 y = s2 ? cmulf(w5[s2], tw5[s2]) : w5[s2];
                    rows[(s1 + 5 * s2) * rp + lds_pad(m)] = y;
                }
            }
        }
        __syncthreads();  // the 25 rows are complete
        // nb-point transforms of this wave's rows, rgrp rows at a time; the
        // last stage leaves the powers of row s as floats 0..nb-1 of its storage
        for (int i0 = 0; i0 < nr; i0 += rgrp) {
            const int g = min(rgrp, nr - i0);
            const int s0 = wave + nw * i0;
            int Ns = 1;
            for (int st = 0; st + 1 < prow.nst; st++) {
                rows_stage_any<false>(prow.radix[st], rows, rp, s0, nw, g, nb, Ns, stw, lane);
                Ns *= prow.radix[st];
            }
            rows_stage_any<true>(prow.radix[prow.nst - 1], rows, rp, s0, nw, g, nb, Ns, stw, lane);
        }
        __syncthreads();  // every row's powers are ready
        // accumulate the powers of this thread's cells: all sums first, then
        // the stores back to back (a load between two stores would make each
        // store wait for the one before it)
        const float* pwf = (const float*)rows;
#pragma unroll
        for (int c = 0; c < CPT; c++) {
            const int w = min(tid + NT * c, N - 1);
            int raw = w + (N >> 1);
            if (raw >= N) raw -= N;
            const int k = raw / NC, sr = raw - NC * k;
            const float pw = pwf[(size_t)sr * 2 * rp + k];
            prev[c] = first ? pw : prev[c] + pw;
        }
#pragma unroll
        for (int c = 0; c < CPT; c++) {
            const int w = tid + NT * c;
            const uint32_t o = w < N ? soff[w] : ~0u;
            if (o != ~0u) *(float*)(base + o) = prev[c];
        }
    }
}

// ---------------------------------------------------------------------------
// Rotation search at large ndop on matrix cores (k_column_rotmma): the mixed-
// precision form of k_column_rotbig for ndop = 25 nb with nb = 25 n1
// (n1 = 2, 4, 10, 20: the E1-like searches at +-5 to +-50 kHz). With rows
// n = p nb + a + n1 b (period p, group a < n1, b < 25) and raw bins
// w = s + 25 k2 + 625 k1 (s, k2 < 25, k1 < n1), the FFT of the
// pattern-signed column is
//   X_q[w] = sum_a W_n1^(k1 a) W_N^(a (s + 25 k2))
//            sum_b W_25^(k2 b) W_625^(s b) sum_p sigma_q[p] W_25^(s p) x[p, a, b].
// Per group a, the sum over p is a complex [25 b x 25 p] x [25 p x 25 s]
// product and the sum over b a [25 k2 x 25 b] x [25 b x 25 s] one, each a
// real product over (re, im)-stacked operands on v_mfma_f32_32x32x16_f16 and
// v_mfma_f32_32x32x8_f16: FP16 operands, FP32 accumulation. The first
// product's accumulator holds rows b of one column s per lane in the order in
// which the second product takes its B operand, so the only work between them
// is the twiddle W_625^(s b) (FP32) and the FP16 conversion. A wave keeps its
// groups' column samples (the first product's A operand) in registers for all
// rotations; a rotation enters through the signs of the first product's B
// operand. Each group's 625 outputs go to LDS as FP16 pairs; after one
// barrier a thread takes one (k2, s), applies W_N^(a (s + 25 k2)) and the
// n1-point DFT over a in FP32, and adds the powers of its n1 cells (rows
// s + 25 k2 + 625 k1 after the fftshift fold, consecutive across threads) to
// the accumulator, whose previous values it has read one rotation ahead.
// The column is scaled by an exact power of two into [0.5, 1) before the FP16
// conversion and the powers are scaled back exactly.
// grid (bs, nrb, batch) as k_column_rotbig; dynamic LDS: 2 n1 * 625 FP16
// pairs, ndop 16-bit window offsets (host: windows below 65535 columns; the
// accumulator pitch below 2^24), 32 masks, 8 floats, and the A operand of the
// groups beyond two per wave.
// ---------------------------------------------------------------------------
typedef _Float16 rmm_h2 __attribute__((ext_vector_type(2)));
typedef _Float16 rmm_h4 __attribute__((ext_vector_type(4)));
typedef _Float16 rmm_h8 __attribute__((ext_vector_type(8)));
typedef float rmm_f16 __attribute__((ext_vector_type(16)));

// W_20^k = exp(-2 pi i k / 20), k = 0..12 (the 20-point DFT's internal twiddles)
__constant__ float2 kW20[13] = {
    {1.0f, -0.0f}, {0.95105651629515353f, -0.3090169943749474f}, {0.80901699437494745f, -0.58778525229247314f},
    {0.58778525229247314f, -0.80901699437494745f}, {0.30901699437494745f, -0.95105651629515353f},
    {0.0f, -1.0f}, {-0.30901699437494734f, -0.95105651629515364f}, {-0.58778525229247303f, -0.80901699437494745f},
    {-0.80901699437494734f, -0.58778525229247325f}, {-0.95105651629515353f, -0.30901699437494751f},
    {-1.0f, -0.0f}, {-0.95105651629515375f, 0.3090169943749469f}, {-0.80901699437494756f, 0.58778525229247303f}};

// W_25^k for 0 <= k < 25 from the 17-entry table (W_25^(25 - k) = conj W_25^k)
__device__ __forceinline__ float2 w25_any(int k)
{
    const float2 w = kW25[k <= 16 ? k : 25 - k];
    return k <= 16 ? w : make_float2(w.x, -w.y);
}

// Forward n-point DFT in registers, natural order (n = 2, 4, 10, 20).
template <int NP>
__device__ __forceinline__ void dft_small(float2* v)
{
    if constexpr (NP == 20) {
        // a = 5 a1 + a2: 4-point DFTs over a1, twiddles W_20^(k1 a2), 5-point
        // DFTs over a2; output k = k1 + 4 k2
        float2 t[5][4];
#pragma unroll
        for (int a2 = 0; a2 < 5; a2++) {
#pragma unroll
            for (int a1 = 0; a1 < 4; a1++) t[a2][a1] = v[5 * a1 + a2];
            bfly4<false>(t[a2]);
#pragma unroll
            for (int k1 = 1; k1 < 4; k1++)
                if (a2) t[a2][k1] = cmulf(t[a2][k1], kW20[k1 * a2]);
        }
#pragma unroll
        for (int k1 = 0; k1 < 4; k1++) {
            float2 u[5] = {t[0][k1], t[1][k1], t[2][k1], t[3][k1], t[4][k1]};
            bfly5<false>(u);
#pragma unroll
            for (int k2 = 0; k2 < 5; k2++) v[k1 + 4 * k2] = u[k2];
        }
    } else {
        bfly<NP, false>(v);
    }
}

__device__ __forceinline__ uint32_t rmm_pack(float re, float im)
{
    const rmm_h2 v = {(_Float16)re, (_Float16)im};
    return __builtin_bit_cast(uint32_t, v);
}

__device__ __forceinline__ float2 rmm_unpack(uint32_t u)
{
    const rmm_h2 v = __builtin_bit_cast(rmm_h2, u);
    return make_float2((float)v[0], (float)v[1]);
}

// Sign-bit mask of one FP16 pair of the first product's B operand: K indices
// k and k + 1, where K index k is period k % 32 (real parts at k < 32,
// imaginary parts at k >= 32; periods 25-31 are padding); msk bit p is set
// when the rotation's pattern is negative in period p.
__device__ __forceinline__ uint32_t rmm_sign_pair(uint32_t msk, int k)
{
    const int p0 = k & 31, p1 = (k + 1) & 31;
    const uint32_t b0 = p0 < 25 ? (msk >> p0) & 1u : 0u;
    const uint32_t b1 = p1 < 25 ? (msk >> p1) & 1u : 0u;
    return (b0 << 15) | (b1 << 31);
}

// -v for a vector of FP16 values (sign bits flipped)
template <class V>
__device__ __forceinline__ V rmm_neg(V v)
{
    typedef uint32_t U __attribute__((ext_vector_type(sizeof(V) / 4)));
    return __builtin_bit_cast(V, __builtin_bit_cast(U, v) ^ (U)0x80008000u);
}

// NW waves, two per SIMD; G groups per wave (group a = wave + NW g), n1 = N1.
// The rotations are pipelined by one: in step t every wave issues the
// accumulator reads of rotation t - 1's cells, runs its groups' products of
// rotation t into E buffer t % 2, then the last stage of rotation t - 1 from
// the other buffer (its reads have landed behind the products), and all waves
// meet once. Waves with fewer groups start their last stage while others
// still run products, so matrix-core and vector work overlap on a SIMD.
template <int NW, int G, int N1>
__global__ void __launch_bounds__(64 * NW)
__attribute__((amdgpu_waves_per_eu(2, 2))) k_column_rotmma(ColumnArgs A)
{
    constexpr int NT = 64 * NW, NC = 25, NB = 25 * N1, N = 25 * NB, NI = 625;
    constexpr int ITEMS = (NI + NT - 1) / NT;
    constexpr int NP = NW;
    static_assert(G * NW >= N1 && (G - 1) * NW < N1, "groups per wave");
    extern __shared__ float2 lds[];
    uint32_t* E = (uint32_t*)lds;                  // [2][n1][625] (re, im) FP16 pairs, index k2 * 25 + s
    uint16_t* soff = (uint16_t*)(E + 2 * N1 * NI); // [N] window column of each sorted row, 0xFFFF outside
    uint32_t* smask = (uint32_t*)(soff + N);       // [32] rotation pattern masks (N is even)
    float* sred = (float*)(smask + 32);            // [8]
    // twiddles W_625^(s b) as FP16 pairs [s][36] (b < 32 used; rows padded to
    // 144 bytes so that 16-byte reads of 32 columns s spread over the banks),
    // at the next 16-byte boundary after 6250 n1 + 160 bytes
    uint32_t* TW = (uint32_t*)((char*)lds + ((6250 * N1 + 160 + 15) & ~15));
    // A operand of the groups a >= 2 NW (the third group of the first waves):
    // [a - 2 NW][25][9] FP16 octets (8 used; the ninth spreads the rows over
    // the banks), after the twiddles
    rmm_h8* XS = (rmm_h8*)(TW + 32 * 36);
    constexpr int GR = G < 2 ? G : 2;  // groups whose A operand stays in registers
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, j32 = lane & 31, h = lane >> 5;
    const int lbk = xcd_logical_block();
    // column of this workgroup (kept in scalar registers: the divisions run on
    // the vector unit)
    const int lag = __builtin_amdgcn_readfirstlane(lbk % gridDim.x);
    const int rr = __builtin_amdgcn_readfirstlane((lbk / gridDim.x) % gridDim.y);
    const int p = __builtin_amdgcn_readfirstlane(lbk / (gridDim.x * gridDim.y));
    int r = A.rb0 + rr;
    if (r >= NB) r -= NB;
    const int pc = r * A.bs + lag;
    // per-column alignment to the primary-code wrap (src/noncoherent_integration.jl:212-215)
    const int wrap = ((NB - pc / A.bs) % NB) * A.bs + (pc % A.bs);
    const int eff = ((wrap + (A.bs >> 1)) / A.bs) % NB;
    if (tid < A.R) {
        const float* pat = A.patterns + ((size_t)A.pset[A.req[p]] * A.Q + tid) * A.ncoh;
        uint32_t msk = 0;
        for (int q = 0; q < A.ncoh; q++)
            if (pat[q] < 0.f) msk |= 1u << q;
        smask[tid] = msk;
    }
    for (int w = tid; w < N; w += NT) {
        int dc = pc + A.shifts[w];
        if (dc >= A.spc) dc -= A.spc;
        int o = dc - A.win0;
        if (o < 0) o += A.spc;
        soff[w] = o < A.winlen ? (uint16_t)o : (uint16_t)0xFFFFu;
    }
    const float2* T = A.tile + (((size_t)p * A.nrb + rr) * N) * A.tp + lag;
    // column scale 2^-ex with max(|re|, |im|) 2^-ex in [0.5, 1)
    float mx = 0.f;
    for (int i = tid; i < N; i += NT) {
        const float2 v = T[(size_t)i * A.tp];
        mx = fmaxf(mx, fmaxf(fabsf(v.x), fabsf(v.y)));
    }
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) mx = fmaxf(mx, __shfl_xor(mx, o));
    if (lane == 0) sred[wave] = mx;
    __syncthreads();
    mx = sred[0];
#pragma unroll
    for (int i = 1; i < NW; i++) mx = fmaxf(mx, sred[i]);
    int ex = 0;
    if (mx > 0.f) frexpf(mx, &ex);
    const float sc = ldexpf(1.f, -ex), unsc = ldexpf(1.f, 2 * ex);
    float* accp = A.acc + (size_t)p * A.acc_ps;
    const size_t slice_stride = (size_t)A.slice_cols * A.acc_ldc;
    const bool first = A.first_step != 0;
    const uint32_t ldc = (uint32_t)A.acc_ldc;
    // first product's A operand: group a, row b = j32, K index k = 16 t + 8 h + e:
    // real part of period k (k < 32), imaginary part of period k - 32
    rmm_h8 X[GR][4];
#pragma unroll
    for (int g = 0; g < G; g++) {
        const int a = wave + NP * g;
        const bool act = a < N1 && j32 < NC;
        const int m = a + N1 * j32;
        float2 xv[NC];
#pragma unroll
        for (int pp = 0; pp < NC; pp++) {
            xv[pp] = make_float2(0.f, 0.f);
            if (act) {
                int src = pp * NB + m + eff;
                if (src >= N) src -= N;
                xv[pp] = T[(size_t)src * A.tp];
            }
        }
#pragma unroll
        for (int t = 0; t < 4; t++) {
            rmm_h8 f;
#pragma unroll
            for (int e = 0; e < 8; e++) {
                const int k0 = 16 * t + e, k1 = k0 + 8;
                const int q0 = k0 & 31, q1 = k1 & 31;
                const float v0 = q0 >= 25 ? 0.f : k0 < 32 ? xv[q0 < 25 ? q0 : 0].x : xv[q0 < 25 ? q0 : 0].y;
                const float v1 = q1 >= 25 ? 0.f : k1 < 32 ? xv[q1 < 25 ? q1 : 0].x : xv[q1 < 25 ? q1 : 0].y;
                f[e] = (_Float16)((h ? v1 : v0) * sc);
            }
            if (g < GR) X[g < GR ? g : 0][t] = f;
            else if (act) XS[((a - 2 * NW) * NC + j32) * 9 + 2 * t + h] = f;
        }
    }
    // first product's B operand without signs, as FP16 pairs: column s = j32,
    // K index k = 16 t + 8 h + 2 v (+1); the real-part tile (re W, -im W) of
    // x W_25^(s p). The imaginary-part tile (im W, re W) is the same values
    // with its K halves swapped and the first negated: K-step t of it is
    // -B1[t + 2] (t < 2) or B1[t - 2].
    typedef uint32_t rmm_u4 __attribute__((ext_vector_type(4)));
    rmm_h8 B1[4];
#pragma unroll
    for (int t = 0; t < 4; t++) {
        rmm_u4 u0;
#pragma unroll
        for (int v = 0; v < 4; v++) {
            float c0[2];
#pragma unroll
            for (int u = 0; u < 2; u++) {
                const int k = 16 * t + 8 * h + 2 * v + u;
                const int pp = k & 31;
                float2 w = make_float2(0.f, 0.f);
                if (j32 < NC && pp < NC) w = w25_any((j32 * pp) % 25);
                c0[u] = k < 32 ? w.x : -w.y;
            }
            u0[v] = rmm_pack(c0[0], c0[1]);
        }
        B1[t] = __builtin_bit_cast(rmm_h8, u0);
    }
    // second product's A operand for the real-part tile: row k2 = j32, K index
    // kk = 8 t + 4 h + e (kk < 32: re F[k2][b = kk], else -im F[k2][kk - 32]);
    // the imaginary-part tile's K-step t is -F2[t + 4] (t < 4) or F2[t - 4]
    rmm_h4 F2[8];
#pragma unroll
    for (int t = 0; t < 8; t++) {
#pragma unroll
        for (int e = 0; e < 4; e++) {
            const int kk = 8 * t + 4 * h + e;
            const int b = kk < 32 ? kk : kk - 32;
            float2 w = make_float2(0.f, 0.f);
            if (j32 < NC && b < NC) w = w25_any((j32 * b) % 25);
            F2[t][e] = (_Float16)(kk < 32 ? w.x : -w.y);
        }
    }
    // twiddles W_625^(s b) = W_N^(s n1 b), zero outside s, b < 25
    for (int i = tid; i < 32 * 32; i += NT) {
        const int sx = i >> 5, b = i & 31;
        float2 w = make_float2(0.f, 0.f);
        if (sx < NC && b < NC) w = A.twD[sx * N1 * b];
        TW[sx * 36 + b] = rmm_pack(w.x, w.y);
    }
    __syncthreads();  // the twiddle table is complete (the A operand rows in
                      // LDS are written and read by the same wave)
    // last stage items: it = tid + NT i is (k2, s) = it / 25, it % 25
    const int ct = tid;
    // accumulator cells of rotation q for this thread's items; cells outside
    // the window read the slice's first cell instead (in bounds, unused)
    auto fetch = [&](int q, float (&pp)[ITEMS][N1], int i0, int i1) {
        const char* base = (const char*)(accp + (size_t)q * slice_stride);
#pragma unroll
        for (int i = 0; i < ITEMS; i++) {
            if (i < i0 || i >= i1) continue;
            const int it = ct + NT * i;
#pragma unroll
            for (int k1 = 0; k1 < N1; k1++) {
                pp[i][k1] = 0.f;
                if (!first && it < NI) {
                    int ws = it + NI * k1 + (N >> 1);
                    if (ws >= N) ws -= N;
                    const uint32_t o = soff[ws];
                    pp[i][k1] = *(const float*)(base + (o != 0xFFFFu ? ((uint32_t)ws + __umul24(o, ldc)) * 4u : 0u));
                }
            }
        }
    };
    // rotation q's last stage: twiddle W_N^(a it), n1-point DFT over a,
    // powers of raw bins it + 625 k1 added to the cells read ahead
    auto last = [&](int q, const float (&pp)[ITEMS][N1]) {
        char* base = (char*)(accp + (size_t)q * slice_stride);
        const uint32_t* Eb = E + (q & 1) * N1 * NI;
#pragma unroll
        for (int i = 0; i < ITEMS; i++) {
            const int it = ct + NT * i;
            if (it < NI) {
                float2 v[N1];
                const float2 om = A.twD[it];
                float2 wa = om;
                v[0] = rmm_unpack(Eb[it]);
#pragma unroll
                for (int a = 1; a < N1; a++) {
                    v[a] = cmulf(rmm_unpack(Eb[a * NI + it]), wa);
                    if (a + 1 < N1) wa = cmulf(wa, om);
                }
                dft_small<N1>(v);
#pragma unroll
                for (int k1 = 0; k1 < N1; k1++) {
                    int ws = it + NI * k1 + (N >> 1);
                    if (ws >= N) ws -= N;
                    const uint32_t o = soff[ws];
                    if (o != 0xFFFFu) {
                        const float pw = fmaf(v[k1].x, v[k1].x, __fmul_rn(v[k1].y, v[k1].y)) * unsc;
                        *(float*)(base + ((uint32_t)ws + __umul24(o, ldc)) * 4u) = first ? pw : pp[i][k1] + pw;
                    }
                }
            }
        }
    };
    uint32_t mprev = 0;  // signs currently applied to B1
    float pp[ITEMS][N1];
    // items whose cells are read before the products (the rest after them,
    // still ahead of the rotation's stores)
    constexpr int EARLY = N1 >= 20 ? 1 : ITEMS;
#pragma unroll 1
    for (int t = 0; t <= A.R; t++) {
        if (t >= 1) fetch(t - 1, pp, 0, EARLY);
        if (t < A.R) {
            const uint32_t mq = __builtin_amdgcn_readfirstlane(smask[t]);
            const uint32_t dm = mq ^ mprev;
            mprev = mq;
#pragma unroll
            for (int k = 0; k < 4; k++) {
                rmm_u4 fl;
#pragma unroll
                for (int v = 0; v < 4; v++)
                    fl[v] = h ? rmm_sign_pair(dm, 16 * k + 8 + 2 * v) : rmm_sign_pair(dm, 16 * k + 2 * v);
                B1[k] = __builtin_bit_cast(rmm_h8, __builtin_bit_cast(rmm_u4, B1[k]) ^ fl);
            }
            uint32_t* Eb = E + (t & 1) * N1 * NI;
#pragma unroll
            for (int g = 0; g < G; g++) {
                const int a = wave + NP * g;
                if (a < N1) {
                    rmm_h8 xa[4];
#pragma unroll
                    for (int k = 0; k < 4; k++) {
                        if (g < GR) xa[k] = X[g < GR ? g : 0][k];
                        else xa[k] = j32 < NC ? XS[((a - 2 * NW) * NC + j32) * 9 + 2 * k + h] : rmm_h8{};
                    }
                    rmm_f16 d0 = {}, d1 = {};
#pragma unroll
                    for (int k = 0; k < 4; k++) {
                        d0 = __builtin_amdgcn_mfma_f32_32x32x16_f16(xa[k], B1[k], d0, 0, 0, 0);
                        d1 = __builtin_amdgcn_mfma_f32_32x32x16_f16(xa[k], k < 2 ? rmm_neg(B1[k + 2]) : B1[k - 2],
                                                                    d1, 0, 0, 0);
                    }
                    // twiddle, then the second product's B operand: K index kk = 8 k + 4 h + e,
                    // real parts of rows b = kk (k < 4), imaginary parts of b = kk - 32
                    rmm_h4 B2[8];
#pragma unroll
                    for (int k = 0; k < 4; k++) {
                        // rows b = 8 k + 4 h + e, e < 4: one 16-byte read
                        typedef uint32_t rmm_u4t __attribute__((ext_vector_type(4)));
                        const rmm_u4t tq = *(const rmm_u4t*)(TW + j32 * 36 + 8 * k + 4 * h);
#pragma unroll
                        for (int e = 0; e < 4; e++) {
                            const int r2 = 4 * k + e;
                            const float2 z = cmulf(make_float2(d0[r2], d1[r2]), rmm_unpack(tq[e]));
                            B2[k][e] = (_Float16)z.x;
                            B2[k + 4][e] = (_Float16)z.y;
                        }
                    }
                    rmm_f16 e0 = {}, e1 = {};
#pragma unroll
                    for (int k = 0; k < 8; k++) {
                        e0 = __builtin_amdgcn_mfma_f32_32x32x8f16(F2[k], B2[k], e0, 0, 0, 0);
                        e1 = __builtin_amdgcn_mfma_f32_32x32x8f16(k < 4 ? rmm_neg(F2[k + 4]) : F2[k - 4], B2[k],
                                                                  e1, 0, 0, 0);
                    }
                    if (j32 < NC) {
                        uint32_t* Ea = Eb + a * NI + j32;
#pragma unroll
                        for (int r2 = 0; r2 < 16; r2++) {
                            const int k2 = 8 * (r2 >> 2) + 4 * h + (r2 & 3);
                            if (k2 < NC) Ea[k2 * NC] = rmm_pack(e0[r2], e1[r2]);
                        }
                    }
                }
            }
        }
        if (t >= 1) {
            if (EARLY < ITEMS) fetch(t - 1, pp, EARLY, ITEMS);
            last(t - 1, pp);
        }
        __syncthreads();  // rotation t in E; rotation t - 1 done, its buffer free
    }
}

// Reduction of one code-column chunk of a windowed column-major accumulator
// (k_column_rotbig's output). grid (R * nsub, ceil(ndop / (4 NTHR)), batch):
// part (q, sub) walks the owned window offsets [own0 + sub cw, ...) of
// rotation slice q, each thread 4 rows, producing per row the FP64 sum and the
// best (value, visit-order key of the global cell) with that cell's four
// interpolation neighbours: code neighbours at offsets -+1 of the same slice
// (modulo spc when the window is the whole code period) and Doppler
// neighbours at rows -+1 modulo ndop. Partials go to part index
// part_base + blockIdx.x of the PRN's nparts_total.
__global__ void __launch_bounds__(FMDBZP_NTHR)
k_reduce_chunk(const float* __restrict__ acc, size_t acc_ps, int ldc, int slice_cols, int ndop, int spc, int R,
               int streamed_rot, int win0, int own0, int nown, int whole, int cw, int nsub, int part_base,
               int nparts_total, double* __restrict__ psum, float* __restrict__ pbest_v,
               uint64_t* __restrict__ pbest_k, float4* __restrict__ pnbr)
{
    const int q = blockIdx.x / nsub, sub = blockIdx.x - q * nsub;
    const int row0 = 4 * (blockIdx.y * FMDBZP_NTHR + threadIdx.x), p = blockIdx.z;
    if (row0 >= ndop) return;
    const float* a = acc + (size_t)p * acc_ps + (size_t)q * slice_cols * ldc;
    const int o0 = own0 + sub * cw, o1 = min(own0 + nown, o0 + cw);
    double s[4] = {0.0, 0.0, 0.0, 0.0};
    float bv[4] = {-INFINITY, -INFINITY, -INFINITY, -INFINITY};
    uint64_t bk[4] = {~0ull, ~0ull, ~0ull, ~0ull};
    int bo[4] = {-1, -1, -1, -1};
#pragma unroll 4
    for (int o = o0; o < o1; o++) {
        const float4 v4 = *(const float4*)(a + (size_t)o * ldc + row0);
        const float v[4] = {v4.x, v4.y, v4.z, v4.w};
        int c = win0 + o;
        if (c >= spc) c -= spc;
#pragma unroll
        for (int u = 0; u < 4; u++) {
            s[u] += (double)v[u];
            if (v[u] >= bv[u]) {
                const uint64_t k = cell_key(row0 + u, q * spc + c, ndop, spc, R, streamed_rot);
                if (better(v[u], k, bv[u], bk[u])) { bv[u] = v[u]; bk[u] = k; bo[u] = o; }
            }
        }
    }
#pragma unroll
    for (int u = 0; u < 4; u++) {
        const int row = row0 + u;
        if (row < ndop) {
            float4 nb4 = make_float4(0.f, 0.f, 0.f, 0.f);
            if (bo[u] >= 0) {
                const int o = bo[u];
                int ol = o - 1, orr = o + 1;
                if (whole) {
                    if (ol < 0) ol += spc;
                    if (orr >= spc) orr -= spc;
                }
                const int dl = row == 0 ? ndop - 1 : row - 1;
                const int dr = row == ndop - 1 ? 0 : row + 1;
                nb4 = make_float4(a[(size_t)ol * ldc + row], a[(size_t)orr * ldc + row], a[(size_t)o * ldc + dl],
                                  a[(size_t)o * ldc + dr]);
            }
            const size_t idx = ((size_t)p * nparts_total + part_base + blockIdx.x) * ndop + row;
            psum[idx] = s[u];
            pbest_v[idx] = bv[u];
            pbest_k[idx] = bk[u];
            pnbr[idx] = nb4;
        }
    }
}

// FP64 sum over rows of each owned column of a windowed accumulator chunk,
// for the GlobalMean estimator. grid (nown, R, batch); colsum [batch][spc_eff].
__global__ void __launch_bounds__(FMDBZP_NTHR)
k_colsum_chunk(const float* __restrict__ acc, size_t acc_ps, int ldc, int slice_cols, int ndop, int spc, int spc_eff,
               int win0, int own0, double* __restrict__ colsum)
{
    __shared__ double ss[FMDBZP_NTHR];
    const int o = own0 + blockIdx.x, q = blockIdx.y, p = blockIdx.z, tid = threadIdx.x;
    const float* a = acc + (size_t)p * acc_ps + ((size_t)q * slice_cols + o) * ldc;
    double t = 0.0;
    for (int row = tid; row < ndop; row += FMDBZP_NTHR) t += (double)a[row];
    ss[tid] = t;
    __syncthreads();
    for (int w = FMDBZP_NTHR / 2; w > 0; w >>= 1) {
        if (tid < w) ss[tid] += ss[tid + w];
        __syncthreads();
    }
    if (tid == 0) {
        int c = win0 + o;
        if (c >= spc) c -= spc;
        colsum[(size_t)p * spc_eff + (size_t)q * spc + c] = ss[0];
    }
}

// Merge of chunk partials per row, carrying the best cell's neighbours.
// grid (ceil(ndop / NTHR), batch).
__global__ void __launch_bounds__(FMDBZP_NTHR)
k_merge_rows_nbr(const double* __restrict__ psum, const float* __restrict__ pbest_v,
                 const uint64_t* __restrict__ pbest_k, const float4* __restrict__ pnbr, int nparts, int ndop,
                 double* __restrict__ rowsum, float* __restrict__ rowbest_v, uint64_t* __restrict__ rowbest_k,
                 float4* __restrict__ rownbr)
{
    const int row = blockIdx.x * FMDBZP_NTHR + threadIdx.x, p = blockIdx.y;
    if (row >= ndop) return;
    double s = 0.0;
    float bv = -INFINITY;
    uint64_t bk = ~0ull;
    float4 nb4 = make_float4(0.f, 0.f, 0.f, 0.f);
    for (int c = 0; c < nparts; c++) {
        const size_t o = ((size_t)p * nparts + c) * ndop + row;
        s += psum[o];
        if (better(pbest_v[o], pbest_k[o], bv, bk)) { bv = pbest_v[o]; bk = pbest_k[o]; nb4 = pnbr[o]; }
    }
    rowsum[(size_t)p * ndop + row] = s;
    rowbest_v[(size_t)p * ndop + row] = bv;
    rowbest_k[(size_t)p * ndop + row] = bk;
    rownbr[(size_t)p * ndop + row] = nb4;
}

// Peak, noise and neighbours of a search accumulated in code-column chunks:
// k_finalize without reading the accumulator. The neighbours come with each
// row's best cell; GlobalMean excludes columns [col - spchip, col + spchip]
// (clipped) through the per-column sums. grid (batch).
__global__ void __launch_bounds__(FMDBZP_NTHR)
k_finalize_chunked(const double* __restrict__ rowsum, const float* __restrict__ rowbest_v,
                   const uint64_t* __restrict__ rowbest_k, const float4* __restrict__ rownbr,
                   const double* __restrict__ colsum, int ndop, int spc, int spc_eff, int R, int streamed_rot,
                   int noise_est, int spchip, fmdbzp_prn_stats* __restrict__ stats)
{
    __shared__ double ssum[FMDBZP_NTHR];
    __shared__ float sv[FMDBZP_NTHR];
    __shared__ uint64_t sk[FMDBZP_NTHR];
    __shared__ int srow[FMDBZP_NTHR];
    const int p = blockIdx.x, tid = threadIdx.x;
    float bv = -INFINITY;
    uint64_t bk = ~0ull;
    int br = 0;
    double tot = 0.0;
    for (int r = tid; r < ndop; r += FMDBZP_NTHR) {
        const float v = rowbest_v[(size_t)p * ndop + r];
        const uint64_t k = rowbest_k[(size_t)p * ndop + r];
        if (better(v, k, bv, bk)) { bv = v; bk = k; br = r; }
        tot += rowsum[(size_t)p * ndop + r];
    }
    sv[tid] = bv;
    sk[tid] = bk;
    srow[tid] = br;
    ssum[tid] = tot;
    __syncthreads();
    for (int w = FMDBZP_NTHR / 2; w > 0; w >>= 1) {
        if (tid < w) {
            ssum[tid] += ssum[tid + w];
            if (better(sv[tid + w], sk[tid + w], sv[tid], sk[tid])) {
                sv[tid] = sv[tid + w];
                sk[tid] = sk[tid + w];
                srow[tid] = srow[tid + w];
            }
        }
        __syncthreads();
    }
    const double total = ssum[0];
    const float peak = sv[0];
    const uint64_t key = sk[0];
    int row, col;
    if (streamed_rot) {
        row = (int)(key % (uint64_t)ndop);
        const uint64_t rest = key / (uint64_t)ndop;
        const int slice = (int)(rest % (uint64_t)R);
        const int cp = (int)(rest / (uint64_t)R);
        col = slice * spc + cp;
    } else {
        row = (int)(key % (uint64_t)ndop);
        col = (int)(key / (uint64_t)ndop);
    }
    const bool none = key == ~0ull || row < 0 || row >= ndop || col < 0 || col >= spc_eff;
    if (none) {
        row = 0;
        col = 0;
    }
    int lo = col - spchip;
    if (lo < 0) lo = 0;
    int hi = col + spchip;
    if (hi > spc_eff - 1) hi = spc_eff - 1;
    const int nex = hi - lo + 1;
    double ex = 0.0;
    if (noise_est == FMDBZP_NOISE_GLOBAL_MEAN)
        for (int c = lo + tid; c <= hi; c += FMDBZP_NTHR) ex += colsum[(size_t)p * spc_eff + c];
    __syncthreads();
    ssum[tid] = ex;
    __syncthreads();
    for (int w = FMDBZP_NTHR / 2; w > 0; w >>= 1) {
        if (tid < w) ssum[tid] += ssum[tid + w];
        __syncthreads();
    }
    if (tid == 0) {
        fmdbzp_prn_stats st;
        st.peak_power = peak;
        st.peak_row = row;
        st.peak_col = col;
        if (noise_est == FMDBZP_NOISE_GLOBAL_MEAN) {
            const double s = total - ssum[0];
            const int64_t cnt = (int64_t)(spc_eff - nex) * ndop;
            st.noise_sum = s;
            st.noise_cells = cnt;
            st.noise_power = (float)s / (float)cnt;
        } else {
            const int opp = (row + ndop / 2) % ndop;
            const double s = rowsum[(size_t)p * ndop + opp];
            st.noise_sum = s;
            st.noise_cells = spc_eff;
            st.noise_power = (float)s / (float)spc_eff;
        }
        const float4 nb4 = none ? make_float4(0.f, 0.f, 0.f, 0.f) : rownbr[(size_t)p * ndop + row];
        st.code_left = nb4.x;
        st.code_right = nb4.y;
        st.dop_left = nb4.z;
        st.dop_right = nb4.w;
        stats[p] = st;
    }
}

// Surface export from a column-major accumulator (column pitch ldc): a
// strided copy into the Julia column-major (ndop, spc_eff) layout.
// grid (spc_eff, ceil(ndop / NTHR))
__global__ void __launch_bounds__(FMDBZP_NTHR)
k_export_cm(const float* __restrict__ acc, float* __restrict__ out, int ndop, int ldc)
{
    const int col = blockIdx.x, row = blockIdx.y * FMDBZP_NTHR + threadIdx.x;
    if (row < ndop) out[(size_t)col * ndop + row] = acc[(size_t)col * ldc + row];
}

// Secondary-code phase of a detected PRN (`_estimate_secondary_code_phase`,
// src/acquire.jl:503-538), in the reference's order of operations: period k is
// despread sequentially, acc += (x * carr) * code with ComplexF32 products (no
// fused multiply-add) and carr *= dphi, the phasor reset per period from an
// FP64 sincos; the L rotations of the secondary code are then summed in order
// and the first largest |s|^2 is kept. grid (requests), L <= 64.
//
// Two chains are serial by that definition: the phasor of a period (two
// dependent operations per sample) and its sum (one add). Everything else is
// not, so the workgroup is a pipeline over chunks of 64 samples, all periods at
// once, one barrier per chunk: wave 0 writes the phasors of chunk i to LDS
// (lane = period), waves 2-7 form the despread products of chunk i - 1 and
// load the samples of chunk i (lane = sample, wave 2 + g has the periods g,
// g + 6, ...), wave 1 sums chunk i - 2 (lane = period). The loop runs two chunks
// per turn with the samples in two register sets: moving them from one to the
// other waited for the loads of the chunk just begun. The LDS pitch LP, odd and
// above the largest L of the launch, is a constant, so that the chains' LDS
// accesses carry their offsets; the four buffers take 35 to 133 KB. Bound by the
// phasor chain (20 ns a sample on one wave): 10 periods of 30690 samples take
// 684 us, 25 of 100000 2.06 ms (842 us and 2.37 ms with the samples moved and a
// pitch of the request's L; chunks of 4096 products took 762 us and 3.77 ms).
struct SecReqDev {
    const int8_t* code;  // spc samples at the estimated code phase
    const int8_t* sec;   // L secondary chips
    double phase_step;   // -2 pi (IF + Doppler) / fs
    int L;
    int pad;
};
#define FMDBZP_SEC_NTHR 512
#define FMDBZP_SEC_C 64
__host__ __device__ constexpr size_t sec_lds(int LP) { return (size_t)4 * FMDBZP_SEC_C * LP * sizeof(float2); }
// LP: 17, 33 or 65, L < LP
template <int ELT, int LP>
__global__ void __launch_bounds__(FMDBZP_SEC_NTHR)
k_secondary_phase(const void* __restrict__ sig, int spc, const SecReqDev* __restrict__ reqs,
                  int32_t* __restrict__ out)
{
#pragma clang fp contract(off)
    constexpr int C = FMDBZP_SEC_C, G = FMDBZP_SEC_NTHR / 64 - 2, NI = (LP - 1 + G - 1) / G;
    const SecReqDev R = reqs[blockIdx.x];
    extern __shared__ float2 lds[];
    __shared__ float zr[64], zi[64], mags[64];
    const int tid = threadIdx.x, k = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int L = R.L;
    float2* ph = lds;              // [2][C][LP] phasors
    float2* qq = lds + 2 * C * LP; // [2][C][LP] despread products
    const int nch = (spc + C - 1) / C;
    // wave 0: phasor of period k
    float cr = 1.0f, ci = 0.0f, dre = 1.0f, dim = 0.0f;
    if (wave == 0 && k < L) {
        const double a = R.phase_step * (double)((int64_t)k * spc);
        cr = (float)cos(a);
        ci = (float)sin(a);
        dre = (float)cos(R.phase_step);
        dim = (float)sin(R.phase_step);
    }
    float ar = 0.0f, ai = 0.0f;  // wave 1: sum of period k
    // product waves: samples of periods g + G u and the code, one set per chunk parity
    float2 x0[NI], x1[NI];
    int8_t c0 = 0, c1 = 0;
    auto step = [&](int i, float2(&xn)[NI], int8_t& cn, const float2(&xs)[NI], const int8_t& cs) {
        if (wave == 0) {
            if (i < nch && k < L) {
                float2* p = ph + (i & 1) * C * LP + k;
                auto next = [&](int n) {
                    p[n * LP] = make_float2(cr, ci);
                    const float ncr = cr * dre - ci * dim, nci = cr * dim + ci * dre;
                    cr = ncr;
                    ci = nci;
                };
                const int m = min(C, spc - i * C);
                if (m == C) {
#pragma unroll 16
                    for (int n = 0; n < C; n++) next(n);
                } else
                    for (int n = 0; n < m; n++) next(n);
            }
        } else if (wave == 1) {
            if (i >= 2 && k < L) {
                const float2* q = qq + (i & 1) * C * LP + k;
                const int m = min(C, spc - (i - 2) * C);
                if (m == C) {
#pragma unroll 16
                    for (int n = 0; n < C; n++) {
                        const float2 v = q[n * LP];
                        ar += v.x;
                        ai += v.y;
                    }
                } else
                    for (int n = 0; n < m; n++) {
                        const float2 v = q[n * LP];
                        ar += v.x;
                        ai += v.y;
                    }
            }
        } else {
            const int g = wave - 2;
            if (i < nch) {
                const int n = min(i * C + k, spc - 1);
                cn = R.code[n];
#pragma unroll
                for (int u = 0; u < NI; u++)
                    if (g + G * u < L) xn[u] = load_sample(sig, ELT, (int64_t)(g + G * u) * spc + n);
            }
            if (i >= 1 && i <= nch) {
                const int at = ((i - 1) & 1) * C * LP + k * LP + g;
                const float c = (float)cs;
#pragma unroll
                for (int u = 0; u < NI; u++)
                    if (g + G * u < L) {
                        const float2 x = xs[u], w = ph[at + G * u];
                        const float pr = x.x * w.x - x.y * w.y, pim = x.x * w.y + x.y * w.x;
                        qq[at + G * u] = make_float2(pr * c - pim * 0.0f, pr * 0.0f + pim * c);
                    }
            }
        }
        __syncthreads();
    };
#pragma unroll
    for (int u = 0; u < NI; u++) x0[u] = x1[u] = make_float2(0.f, 0.f);
    for (int i = 0; i < nch + 2; i += 2) {
        step(i, x0, c0, x1, c1);
        step(i + 1, x1, c1, x0, c0);  // past the last chunk: nothing but the barrier
    }
    if (wave == 1 && k < L) {
        zr[k] = ar;
        zi[k] = ai;
    }
    __syncthreads();
    if (tid < L) {  // rotation r = tid
        float sr = 0.0f, si = 0.0f;
        for (int q = 0; q < L; q++) {
            int j = q + tid;
            if (j >= L) j -= L;
            const float sv = (float)R.sec[j];
            sr += sv * zr[q];
            si += sv * zi[q];
        }
        mags[tid] = sr * sr + si * si;
    }
    __syncthreads();
    if (tid == 0) {
        int best_r = 0;
        float best = -1.0f;
        for (int r = 0; r < L; r++)
            if (mags[r] > best) {
                best = mags[r];
                best_r = r;
            }
        out[blockIdx.x] = best_r;
    }
}

// Chip-ordered surface export (fmdbzp_plan_set_surface_layout): grid (nbins,
// ceil(ndop / NTHR)). Bin b holds, per sorted Doppler row, the maximum over
// the code columns order[b spc / nbins .. (b + 1) spc / nbins) (ascending code
// phase, src/plot.jl:35-57) and over the R rotation slices of each;
// out is column-major (ndop, nbins).
__global__ void __launch_bounds__(FMDBZP_NTHR)
k_export_chip(const float* __restrict__ acc, float* __restrict__ out, const int32_t* __restrict__ order, int ndop,
              int spc, int R, int nbins, int ldr, int ldc)
{
    const int b = blockIdx.x, row = blockIdx.y * FMDBZP_NTHR + threadIdx.x;
    if (row >= ndop) return;
    const int i0 = (int)((int64_t)b * spc / nbins), i1 = (int)((int64_t)(b + 1) * spc / nbins);
    const float* a = acc + (size_t)row * ldr;
    float m = -INFINITY;
    for (int i = i0; i < i1; i++) {
        const int c = order[i];
        for (int sl = 0; sl < R; sl++) m = fmaxf(m, a[((size_t)sl * spc + c) * ldc]);
    }
    out[(size_t)b * ndop + row] = m;
}

// Surface export for store_power_bins: acc[row][col] (row pitch ap) -> Julia column-major
// (ndop, spc_eff), i.e. out[col * ndop + row]. 32x32 LDS-tiled transpose.
// grid (ceil(spc_eff/32), ceil(ndop/32)), block (32, 8)
__global__ void k_export(const float* __restrict__ acc, float* __restrict__ out, int ndop, int spc_eff, int ap)
{
    __shared__ float t[32][33];
    const int c0 = blockIdx.x * 32, r0 = blockIdx.y * 32;
    for (int i = threadIdx.y; i < 32; i += 8) {
        const int r = r0 + i, c = c0 + threadIdx.x;
        if (r < ndop && c < spc_eff) t[i][threadIdx.x] = acc[(size_t)r * ap + c];
    }
    __syncthreads();
    for (int i = threadIdx.y; i < 32; i += 8) {
        const int c = c0 + i, r = r0 + threadIdx.x;
        if (r < ndop && c < spc_eff) out[(size_t)c * ndop + r] = t[threadIdx.x][i];
    }
}
