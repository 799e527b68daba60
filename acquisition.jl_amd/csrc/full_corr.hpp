// full_corr.hpp — full-period correlation search (simple path) for gfx950.
//
// The simple path of the search (src/acquire.jl:335-385 and
// src/noncoherent_integration.jl:482-592 on the tile of
// src/coherent_integration.jl:136-171) is, for raw Doppler bin w and column
// (block r, lag), with k = p nb + j (period p, block j) and N = ndop = P nb,
//   X[w][r][lag] = sum_p sum_j W_N^(w k) sum_i x[k bs + lag + i] c[((j + r) mod nb) bs + i].
// With s = w mod P the sum over p does not depend on the PRN or on j:
//   z_s[n] = sum_p W_P^(s p) x[p spc + n],  z_s[n + spc] = W_P^(-s) z_s[n],
// and with m = ((j + r) mod nb) bs + i the rest is one correlation over the code
// period, at delay tau = lag - r bs (mod spc):
//   X = W_N^(-w r) sum_m c[m] W_N^(w floor(m / bs)) z_s[m + tau].
// The factors of modulus one that depend on the output cell drop out of |X|^2,
// so with the periodic z'_s[n] = z_s[n] e^(-2 pi i s n / (P spc)) and the
// ramped code a_w[m] = c[m] W_N^(w floor(m / bs)) e^(2 pi i s m / (P spc)) a
// Doppler row is ONE circular correlation of spc points,
//   |X[w][tau]|^2 = |IDFT(Z'_s conj(DFT(conj a_w)))[tau]|^2,
// instead of nb zero-padded ones of 2 bs points and a column transform: about
// half the arithmetic, and no coherent tile in memory. The code spectra are
// plan data (8 ndop spc bytes per PRN).
//
// A transform lives in one LDS buffer (spc <= 20480 - padding). Forward:
// decimation in frequency, natural order in, digit-reversed out; inverse:
// decimation in time, digit-reversed in, natural out; the product is formed in
// the permuted order, so nothing is ever reordered. Every stage reads and
// writes the same LDS slots per butterfly: one barrier per stage, and the
// slots of a butterfly are base + r * pitch (one add each).
#pragma once
#include "kernels.hpp"
#include <type_traits>

#define FC_MAX_STAGES 6

// Stage t combines radix[t] sub-transforms of ns[t] = radix[0] ... radix[t-1]
// points. pad_shift: one LDS pad slot every 2^pad_shift elements (n a power
// of two, radix[0] = 2^pad_shift); 31: none, radix[0] is odd, which spreads
// the strides over the banks. twoff: the stage's twiddles [r - 1][k],
// exp(-2 pi i r k / (ns radix)), in the plan's table.
struct FullPlanDev {
    int n, nst, pad_shift;
    int radix[FC_MAX_STAGES], ns[FC_MAX_STAGES], twoff[FC_MAX_STAGES];
    float inv_ns[FC_MAX_STAGES];
};

// ---------------------------------------------------------------------------
// In-register DFTs beyond fft_lds.hpp: primes by their conjugate symmetry
// (real and imaginary parts share cos and sin products), coprime products by
// Good-Thomas (no internal twiddles), 9 and 25 as square Cooley-Tukey.
// ---------------------------------------------------------------------------
template <int R>
struct PrimeTab;
template <> struct PrimeTab<7> {
    static constexpr float c[7] = {1.0f, 0.6234898018587336f, -0.22252093395631434f, -0.900968867902419f,
        -0.9009688679024191f, -0.2225209339563146f, 0.6234898018587334f};
    static constexpr float s[7] = {0.0f, 0.7818314824680298f, 0.9749279121818236f, 0.43388373911755823f,
        -0.433883739117558f, -0.9749279121818236f, -0.7818314824680299f};
};
template <> struct PrimeTab<11> {
    static constexpr float c[11] = {1.0f, 0.8412535328311812f, 0.41541501300188644f, -0.142314838273285f,
        -0.654860733945285f, -0.9594929736144974f, -0.9594929736144975f, -0.6548607339452852f, -0.14231483827328523f,
        0.41541501300188605f, 0.8412535328311812f};
    static constexpr float s[11] = {0.0f, 0.5406408174555976f, 0.9096319953545183f, 0.9898214418809328f,
        0.7557495743542583f, 0.28173255684142967f, -0.2817325568414294f, -0.7557495743542582f, -0.9898214418809327f,
        -0.9096319953545186f, -0.5406408174555974f};
};
template <> struct PrimeTab<13> {
    static constexpr float c[13] = {1.0f, 0.8854560256532099f, 0.5680647467311559f, 0.120536680255323f,
        -0.35460488704253545f, -0.7485107481711012f, -0.970941817426052f, -0.9709418174260521f, -0.7485107481711013f,
        -0.3546048870425359f, 0.1205366802553232f, 0.5680647467311548f, 0.88545602565321f};
    static constexpr float s[13] = {0.0f, 0.4647231720437685f, 0.8229838658936564f, 0.992708874098054f,
        0.9350162426854148f, 0.6631226582407952f, 0.23931566428755768f, -0.23931566428755743f, -0.663122658240795f,
        -0.9350162426854147f, -0.992708874098054f, -0.822983865893657f, -0.4647231720437684f};
};
template <> struct PrimeTab<31> {
    static constexpr float c[31] = {1.0f, 0.9795299412524945f, 0.9189578116202306f, 0.8207634412072763f,
        0.6889669190756866f, 0.5289640103269624f, 0.3473052528448203f, 0.1514277775045767f, -0.05064916883871264f,
        -0.2506525322587204f, -0.4403941515576344f, -0.6121059825476626f, -0.7587581226927909f, -0.8743466161445821f,
        -0.9541392564000488f, -0.994869323391895f, -0.9948693233918952f, -0.9541392564000488f, -0.8743466161445822f,
        -0.7587581226927911f, -0.6121059825476627f, -0.44039415155763423f, -0.2506525322587213f,
        -0.05064916883871355f, 0.15142777750457667f, 0.3473052528448203f, 0.5289640103269624f, 0.6889669190756865f,
        0.8207634412072763f, 0.9189578116202306f, 0.9795299412524943f};
    static constexpr float s[31] = {0.0f, 0.20129852008866006f, 0.39435585511331855f, 0.5712682150947923f,
        0.7247927872291199f, 0.8486442574947509f, 0.9377521321470804f, 0.9884683243281114f, 0.9987165071710528f,
        0.9680771188662043f, 0.8978045395707416f, 0.7907757369376989f, 0.6513724827222223f, 0.48530196253108104f,
        0.29936312297335804f, 0.10116832198743272f, -0.10116832198743204f, -0.2993631229733582f, -0.4853019625310808f,
        -0.651372482722222f, -0.7907757369376986f, -0.8978045395707417f, -0.9680771188662041f, -0.9987165071710528f,
        -0.9884683243281114f, -0.9377521321470804f, -0.848644257494751f, -0.72479278722912f, -0.5712682150947924f,
        -0.3943558551133187f, -0.20129852008866114f};
};

template <int R, bool INV, class Put>
__device__ __forceinline__ void dft_prime(const float2* v, Put&& put)
{
    constexpr int H = (R - 1) / 2;
    float2 e[H], o[H];
    float2 sum = v[0];
#pragma unroll
    for (int i = 0; i < H; i++) {
        e[i] = caddf(v[i + 1], v[R - 1 - i]);
        o[i] = csubf(v[i + 1], v[R - 1 - i]);
        sum = caddf(sum, e[i]);
    }
    const float2 x0 = v[0];
    put(std::integral_constant<int, 0>{}, sum);
    [&]<int... K>(std::integer_sequence<int, K...>) {
        (([&] {
             constexpr int k = K + 1;
             float2 a = x0, b = make_float2(0.f, 0.f);
#pragma unroll
             for (int i = 0; i < H; i++) {
                 const float c = PrimeTab<R>::c[((i + 1) * k) % R], s = PrimeTab<R>::s[((i + 1) * k) % R];
                 a.x = fmaf(e[i].x, c, a.x);
                 a.y = fmaf(e[i].y, c, a.y);
                 b.x = fmaf(o[i].x, s, b.x);
                 b.y = fmaf(o[i].y, s, b.y);
             }
             const float2 mb = mul_mi<INV>(b);  // -i b forward, +i b inverse
             put(std::integral_constant<int, k>{}, caddf(a, mb));
             put(std::integral_constant<int, R - k>{}, csubf(a, mb));
         }()),
         ...);
    }(std::make_integer_sequence<int, H>{});
}

template <int R, bool INV>
__device__ __forceinline__ void dft_reg(float2* v);

constexpr int inv_mod(int a, int m)
{
    for (int x = 1; x < m; x++)
        if (a * x % m == 1) return x;
    return 1;
}

template <int A, int B, bool INV>
__device__ __forceinline__ void dft_pfa(float2* v)
{
    constexpr int R = A * B;
    float2 t[A][B];
#pragma unroll
    for (int n2 = 0; n2 < B; n2++) {
        float2 u[A];
#pragma unroll
        for (int n1 = 0; n1 < A; n1++) u[n1] = v[(B * n1 + A * n2) % R];
        dft_reg<A, INV>(u);
#pragma unroll
        for (int k1 = 0; k1 < A; k1++) t[k1][n2] = u[k1];
    }
#pragma unroll
    for (int k1 = 0; k1 < A; k1++) {
        dft_reg<B, INV>(t[k1]);
        // long products: one sub-transform at a time, or their temporaries are all live at once
        if constexpr (R > 24) __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int k2 = 0; k2 < B; k2++) v[(k1 * B * inv_mod(B % A, A) + k2 * A * inv_mod(A % B, B)) % R] = t[k1][k2];
    }
}

// 9 = 3 x 3 and 25 = 5 x 5: v[a + Q b], DFTs over b, twiddles W^(a k), DFTs over a
template <int Q, bool INV>
__device__ __forceinline__ void dft_square(float2* v)
{
    constexpr int R = Q * Q;
    float2 t[Q][Q];
#pragma unroll
    for (int a = 0; a < Q; a++) {
#pragma unroll
        for (int b = 0; b < Q; b++) t[a][b] = v[a + Q * b];
        bfly<Q, INV>(t[a]);
#pragma unroll
        for (int k = 1; k < Q; k++)
            if (a) {
                // W_R^(a k): exact FP32 constants of the forward transform
                constexpr float c9[5] = {1.f, 0.76604444311897804f, 0.17364817766693035f, -0.5f, -0.93969262078590838f};
                constexpr float s9[5] = {0.f, 0.64278760968653933f, 0.98480775301220806f, 0.86602540378443865f,
                                         0.34202014332566873f};
                if constexpr (Q == 3) t[a][k] = cmul_const<INV>(t[a][k], c9[a * k], -s9[a * k]);
                else t[a][k] = cmul_const<INV>(t[a][k], kW25[a * k].x, kW25[a * k].y);
            }
    }
#pragma unroll
    for (int k = 0; k < Q; k++) {
        float2 u[Q];
#pragma unroll
        for (int a = 0; a < Q; a++) u[a] = t[a][k];
        bfly<Q, INV>(u);
#pragma unroll
        for (int q = 0; q < Q; q++) v[k + Q * q] = u[q];
    }
    static_assert(R == 9 || R == 25, "square radices");
}

// 32 = 2 x 16: even and odd samples, twiddles W_32^k on the odd half
template <bool INV>
__device__ __forceinline__ void dft_32(float2* v)
{
    constexpr float c32[16] = {1.f, 0.98078528040323043f, 0.92387953251128674f, 0.83146961230254524f,
                               0.70710678118654757f, 0.55557023301960229f, 0.38268343236508984f, 0.19509032201612833f,
                               0.f, -0.19509032201612819f, -0.38268343236508973f, -0.55557023301960196f,
                               -0.70710678118654746f, -0.83146961230254535f, -0.92387953251128674f, -0.98078528040323043f};
    constexpr float s32[16] = {0.f, 0.19509032201612825f, 0.38268343236508978f, 0.55557023301960218f,
                               0.70710678118654746f, 0.83146961230254524f, 0.92387953251128674f, 0.98078528040323043f,
                               1.f, 0.98078528040323043f, 0.92387953251128674f, 0.83146961230254546f,
                               0.70710678118654757f, 0.55557023301960218f, 0.38268343236508989f, 0.19509032201612861f};
    float2 a[16], b[16];
#pragma unroll
    for (int i = 0; i < 16; i++) {
        a[i] = v[2 * i];
        b[i] = v[2 * i + 1];
    }
    dft_reg<16, INV>(a);
    dft_reg<16, INV>(b);
#pragma unroll
    for (int k = 0; k < 16; k++) {
        const float2 u = k ? cmul_const<INV>(b[k], c32[k], -s32[k]) : b[k];
        v[k] = make_float2(a[k].x + u.x, a[k].y + u.y);
        v[k + 16] = make_float2(a[k].x - u.x, a[k].y - u.y);
    }
}

template <int R, bool INV>
__device__ __forceinline__ void dft_reg(float2* v)
{
    if constexpr (R == 6) dft_pfa<2, 3, INV>(v);
    else if constexpr (R == 12) dft_pfa<3, 4, INV>(v);
    else if constexpr (R == 15) dft_pfa<3, 5, INV>(v);
    else if constexpr (R == 20) dft_pfa<4, 5, INV>(v);
    else if constexpr (R == 22) dft_pfa<2, 11, INV>(v);
    else if constexpr (R == 24) dft_pfa<3, 8, INV>(v);
    else if constexpr (R == 33) dft_pfa<3, 11, INV>(v);
    else if constexpr (R == 18) dft_pfa<2, 9, INV>(v);
    else if constexpr (R == 21) dft_pfa<3, 7, INV>(v);
    else if constexpr (R == 30) dft_pfa<2, 15, INV>(v);
    else if constexpr (R == 32) dft_32<INV>(v);
    else if constexpr (R == 9) dft_square<3, INV>(v);
    else if constexpr (R == 25) dft_square<5, INV>(v);
    else if constexpr (R == 7 || R == 11 || R == 13 || R == 31) {
        float2 t[R];
        dft_prime<R, INV>(v, [&](auto k, float2 x) { t[k] = x; });
#pragma unroll
        for (int r = 0; r < R; r++) v[r] = t[r];
    } else bfly<R, INV>(v);
}

// DFT of v with each output handed to put(index, value) as it is formed
template <int R, bool INV, class Put>
__device__ __forceinline__ void dft_out(float2* v, Put&& put)
{
    if constexpr (R == 31) {
        dft_prime<R, INV>(v, put);
    } else {
        dft_reg<R, INV>(v);
        [&]<int... K>(std::integer_sequence<int, K...>) {
            (put(std::integral_constant<int, K>{}, v[K]), ...);
        }(std::make_integer_sequence<int, R>{});
    }
}

// op(std::integral_constant<int, R>) for a runtime radix (uniform branch)
#define FC_RADIX_SWITCH(R, OP)                                        \
    switch (R) {                                                      \
    case 2: OP(std::integral_constant<int, 2>{}); break;              \
    case 3: OP(std::integral_constant<int, 3>{}); break;              \
    case 4: OP(std::integral_constant<int, 4>{}); break;              \
    case 5: OP(std::integral_constant<int, 5>{}); break;              \
    case 6: OP(std::integral_constant<int, 6>{}); break;              \
    case 7: OP(std::integral_constant<int, 7>{}); break;              \
    case 8: OP(std::integral_constant<int, 8>{}); break;              \
    case 9: OP(std::integral_constant<int, 9>{}); break;              \
    case 10: OP(std::integral_constant<int, 10>{}); break;            \
    case 11: OP(std::integral_constant<int, 11>{}); break;            \
    case 12: OP(std::integral_constant<int, 12>{}); break;            \
    case 13: OP(std::integral_constant<int, 13>{}); break;            \
    case 15: OP(std::integral_constant<int, 15>{}); break;            \
    default: OP(std::integral_constant<int, 16>{}); break;            \
    }
// With one noncoherent step a middle stage also has 20 and 22 and the first
// one 25. With several, the cells kept between the steps leave no room for
// them at four waves per SIMD (128 registers): 20 and 22 spilled 190.
#define FC_RADIX_SWITCH_MID(R, OP)                                    \
    switch (R) {                                                      \
    case 20: OP(std::integral_constant<int, 20>{}); break;            \
    case 22: OP(std::integral_constant<int, 22>{}); break;            \
    default: FC_RADIX_SWITCH(R, OP)                                   \
    }
#define FC_RADIX_SWITCH_FIRST(R, OP)                                  \
    switch (R) {                                                      \
    case 25: OP(std::integral_constant<int, 25>{}); break;            \
    default: FC_RADIX_SWITCH(R, OP)                                   \
    }

// element i of the LDS buffer
__device__ __forceinline__ int fc_addr(int i, int pad_shift) { return i + (i >> pad_shift); }
inline int fc_lds_span(const FullPlanDev& f) { return f.n + (f.n >> f.pad_shift) + 1; }

// p[i] with a 32-bit byte offset from a uniform base
__device__ __forceinline__ float2 fc_ld(const float2* __restrict__ p, int i)
{
    return *(const float2*)((const char*)p + (uint32_t)i * (uint32_t)sizeof(float2));
}

// fdivmod without branches
__device__ __forceinline__ int fc_divmod(int x, int d, float inv_d, int* r)
{
    int q = (int)((float)x * inv_d);
    int m = x - q * d;
    const int up = m >= d ? 1 : 0, down = m < 0 ? 1 : 0;
    q += up - down;
    m += down ? d : 0;
    m -= up ? d : 0;
    *r = m;
    return q;
}

// R elements a pitch (in elements) apart, from element i on; all loads are
// issued before anything after fc_issued() runs: left alone, the compiler
// waits for each pair of loads where it first uses it.
template <int R>
__device__ __forceinline__ void fc_ld_run(float2 (&v)[R], const float2* __restrict__ p, int i, int pitch)
{
    uint32_t off = (uint32_t)i * (uint32_t)sizeof(float2);
#pragma unroll
    for (int r = 0; r < R; r++) {
        v[r] = *(const float2*)((const char*)p + off);
        off += (uint32_t)pitch * (uint32_t)sizeof(float2);
    }
}
__device__ __forceinline__ void fc_issued() { __builtin_amdgcn_sched_barrier(0); }
// the same value, unknown to the compiler: index arithmetic on it stays where
// it is used instead of being hoisted out of the step loop into registers
__device__ __forceinline__ int fc_opaque(int x)
{
    asm volatile("" : "+v"(x));
    return x;
}

// Stage t >= 1, one butterfly per call of body(a, pn, k): its slots are
// lds[a + r pn], its position within the sub-transform k.
template <int R, int NTHR, class Body>
__device__ __forceinline__ void fc_butterflies(const FullPlanDev& f, int t, int tid, Body&& body)
{
    const int ns = f.ns[t], m = f.n / R;
    const int pn = ns + (ns >> f.pad_shift), pb = R * pn;
    for (int j = tid; j < m; j += NTHR) {
        int k;
        const int b = fc_divmod(j, ns, f.inv_ns[t], &k);
        body(b * pb + fc_addr(k, f.pad_shift), pn, k);
    }
}

// Forward transform: in(i) -> out(i) in the stage-0 order r * (n / radix[0]) + j.
template <int NTHR, class In, class Out>
__device__ __forceinline__ void fc_forward(float2* lds, const FullPlanDev& f, const float2* __restrict__ tw, int tid,
                                           const In& in, const Out& out)
{
    for (int i = tid; i < f.n; i += NTHR) lds[fc_addr(i, f.pad_shift)] = in(i);
    __syncthreads();
    for (int t = f.nst - 1; t >= 1; t--) {
        const float2* twt = tw + f.twoff[t];
        const int ns = f.ns[t];
        auto op = [&](auto rc) {
            constexpr int R = decltype(rc)::value;
            fc_butterflies<R, NTHR>(f, t, tid, [&](int a, int pn, int k) {
                float2 v[R], tv[R - 1];
                fc_ld_run(tv, twt, k, ns);
#pragma unroll
                for (int r = 0; r < R; r++) v[r] = lds[a + r * pn];
                fc_issued();
                dft_reg<R, false>(v);
                lds[a] = v[0];
#pragma unroll
                for (int r = 1; r < R; r++) lds[a + r * pn] = cmulf(v[r], tv[r - 1]);
            });
        };
        FC_RADIX_SWITCH_MID(f.radix[t], op)
        __syncthreads();
    }
    const int m0 = f.n / f.radix[0], p1 = f.radix[0] + (f.pad_shift < 31 ? 1 : 0);
    auto op = [&](auto rc) {
        constexpr int R = decltype(rc)::value;
        for (int j = tid; j < m0; j += NTHR) {
            float2 v[R];
#pragma unroll
            for (int r = 0; r < R; r++) v[r] = lds[j * p1 + r];
            dft_out<R, false>(v, [&](auto r, float2 x) { out(r * m0 + j, x); });
        }
    };
    FC_RADIX_SWITCH_FIRST(f.radix[0], op)
}

// ---------------------------------------------------------------------------
// Tables (plan time), FP64 angles on the device: on the host the sines of a
// 20000-point plan took 0.4 ms, as long as the rest of its creation.
// ---------------------------------------------------------------------------
inline int fc_tw_count(const FullPlanDev& f)
{
    const int t = f.nst - 1;
    return f.twoff[t] + (f.radix[t] - 1) * f.ns[t];
}
// twiddles of the stages, in their order. grid (ceil(fc_tw_count / 256))
__global__ void __launch_bounds__(256)
k_fc_twiddles(FullPlanDev f, float2* __restrict__ tw, int count)
{
    const int e = blockIdx.x * 256 + threadIdx.x;
    if (e >= count) return;
    int t = f.nst - 1;
    while (t > 1 && e < f.twoff[t]) t--;
    const int ns = f.ns[t], r = (e - f.twoff[t]) / ns + 1, k = (e - f.twoff[t]) % ns;
    double sn, cs;
    sincospi(-2.0 * (double)((int64_t)r * k) / ((double)ns * f.radix[t]), &sn, &cs);
    tw[e] = make_float2((float)cs, (float)sn);
}
// column of delay tau: block (nb - tau / bs) mod nb, lag tau mod bs
__device__ __forceinline__ uint16_t full_column(int tau, int nb, int bs)
{
    const int r = tau / bs;
    return (uint16_t)((r ? nb - r : 0) * bs + tau % bs);
}
// grid (ceil(n / 256))
__global__ void __launch_bounds__(256)
k_full_map(uint16_t* __restrict__ map, int n, int nb, int bs)
{
    const int tau = blockIdx.x * 256 + threadIdx.x;
    if (tau < n) map[tau] = full_column(tau, nb, bs);
}

// ---------------------------------------------------------------------------
// Code spectra (plan time): conj(DFT(conj a_w)) / spc. grid (ndop, nprn)
// ---------------------------------------------------------------------------
#define FC_FWD_NTHR 512
// conj a_w[m]: exp(2 pi i (w bs floor(m / bs) - s m) / (ncoh spc)) times the
// code sample, the angle an exact integer over ncoh spc. (The sincospi is not
// what bounds these kernels: with the angle's two factors from tables they took
// 50.9 instead of 56.9 us at 8 x 80 rows of 10000 points and 543 instead of 538 at
// 32 x 160 of 16368.)
__device__ __forceinline__ float2 full_code_in(const int8_t* c, int m, int w, int s, int bs, double two_over_d)
{
    const double t = (double)((int64_t)w * ((m / bs) * bs) - (int64_t)s * m);
    double sn, cs;
    sincospi(t * two_over_d, &sn, &cs);
    const float v = (float)c[m];
    return make_float2(v * (float)cs, v * (float)sn);
}

__global__ void __launch_bounds__(FC_FWD_NTHR)
k_full_code(const int8_t* __restrict__ codes, float2* __restrict__ spec, FullPlanDev f, const float2* __restrict__ tw,
            int bs, int ncoh, float scale)
{
    extern __shared__ float2 lds[];
    const int w = blockIdx.x, prn = blockIdx.y, n = f.n, s = w % ncoh;
    const int8_t* c = codes + (size_t)prn * n;
    const double two_over_d = 2.0 / ((double)ncoh * n);
    float2* out = spec + ((size_t)prn * gridDim.x + w) * n;
    fc_forward<FC_FWD_NTHR>(
        lds, f, tw, threadIdx.x,
        [&](int m) { return full_code_in(c, m, w, s, bs, two_over_d); },
        [&](int i, float2 x) { out[i] = make_float2(x.x * scale, -x.y * scale); });
}

// ---------------------------------------------------------------------------
// Periods folded: z'_s[n], s < ncoh, per step (ncoh > 1). A thread owns one n
// and SB values of s, so the samples of its column are read and downconverted
// once per SB outputs. grid (ceil(spc / 256), ceil(ncoh / SB), nnc)
// ---------------------------------------------------------------------------
#define FC_FOLD_SB 10
__global__ void __launch_bounds__(256)
k_full_fold(const void* __restrict__ sig, int eltype, float2* __restrict__ z, int spc, int ncoh, int do_if,
            float phase_step, double phase_step64)
{
    extern __shared__ float2 wp[];  // W_ncoh^i
    const int n = blockIdx.x * 256 + threadIdx.x, s0 = blockIdx.y * FC_FOLD_SB, step = blockIdx.z;
    for (int i = threadIdx.x; i < ncoh; i += 256) {
        double sn, cs;
        sincospi(-2.0 * i / ncoh, &sn, &cs);
        wp[i] = make_float2((float)cs, (float)sn);
    }
    __syncthreads();
    if (n >= spc) return;
    const int64_t seglen = (int64_t)ncoh * spc, seg0 = step * seglen;
    const DownconvIn in{sig, eltype, seg0, seglen, 0, (int)seglen, do_if, __fmul_rn((float)seg0, phase_step), phase_step,
                        phase_step64};
    float2 a[FC_FOLD_SB];
    int at[FC_FOLD_SB];  // s p mod ncoh
#pragma unroll
    for (int i = 0; i < FC_FOLD_SB; i++) {
        a[i] = make_float2(0.f, 0.f);
        at[i] = 0;
    }
    for (int p = 0; p < ncoh; p++) {
        const float2 x = in(0, p * spc + n);
#pragma unroll
        for (int i = 0; i < FC_FOLD_SB; i++) {
            const float2 w = wp[at[i]];
            a[i].x = fmaf(x.x, w.x, fmaf(-x.y, w.y, a[i].x));
            a[i].y = fmaf(x.x, w.y, fmaf(x.y, w.x, a[i].y));
            const int s = s0 + i < ncoh ? s0 + i : 0;
            at[i] += s;
            if (at[i] >= ncoh) at[i] -= ncoh;
        }
    }
    const double two_over_d = 2.0 / ((double)ncoh * spc);
#pragma unroll
    for (int i = 0; i < FC_FOLD_SB; i++) {
        const int s = s0 + i;
        if (s < ncoh) {
            double sn, cs;
            sincospi(-(double)((int64_t)s * n) * two_over_d, &sn, &cs);
            z[((size_t)step * ncoh + s) * spc + n] = cmulf(a[i], make_float2((float)cs, (float)sn));
        }
    }
}

// Signal spectra, in place on z (ncoh > 1) or straight from the samples
// (ncoh == 1). grid (ncoh, nnc)
template <int NTHR>
__global__ void __launch_bounds__(NTHR)
k_full_signal(const void* __restrict__ sig, int eltype, float2* z, FullPlanDev f, const float2* __restrict__ tw,
              int do_if, float phase_step, double phase_step64)
{
    extern __shared__ float2 lds[];
    const int n = f.n;
    const int64_t seg0 = (int64_t)blockIdx.y * n;
    float2* zz = z + ((size_t)blockIdx.y * gridDim.x + blockIdx.x) * n;
    const DownconvIn in{sig, eltype, seg0, n, 0, n, do_if, __fmul_rn((float)seg0, phase_step), phase_step, phase_step64};
    const bool folded = gridDim.x > 1;
    fc_forward<NTHR>(
        lds, f, tw, threadIdx.x, [&](int i) { return folded ? zz[i] : in(0, i); },
        [&](int i, float2 x) { zz[i] = x; });
}

// ---------------------------------------------------------------------------
// The search: one workgroup per (Doppler row, PRN), all noncoherent steps.
// Per step: product of the signal and code spectra in the first stage, the
// inverse transform in LDS, and the powers through LDS, over the consumed
// transform, to the threads that own their drifted columns. A row's cells stay
// in registers between the steps and are written once; the row's FP64 sum and
// best cell come from the same registers.
// ---------------------------------------------------------------------------
// The product of two spectra and all but the last stage of its inverse
// transform, ending with a barrier. WIDE: the radices of FC_RADIX_SWITCH_FIRST
// and FC_RADIX_SWITCH_MID.
template <int NTHR, bool WIDE>
__device__ __forceinline__ void fc_inverse_head(float2* lds, const FullPlanDev& f, const float2* __restrict__ tw, int tid,
                                                const float2* __restrict__ Z, const float2* __restrict__ G)
{
    {
        const int m0 = f.n / f.radix[0], p1 = f.radix[0] + (f.pad_shift < 31 ? 1 : 0);
        auto op = [&](auto rc) {
            constexpr int R = decltype(rc)::value;
            for (int j = fc_opaque(tid); j < m0; j += NTHR) {
                float2 v[R], gv[R];
                fc_ld_run(gv, G, j, m0);
                fc_ld_run(v, Z, j, m0);
                fc_issued();
#pragma unroll
                for (int r = 0; r < R; r++) v[r] = cmulf(v[r], gv[r]);
                float2* dst = lds + j * p1;
                dft_reg<R, true>(v);
#pragma unroll
                for (int r = 0; r < R; r++) dst[r] = v[r];
            }
        };
        if constexpr (WIDE) {
            FC_RADIX_SWITCH_FIRST(f.radix[0], op)
        } else {
            FC_RADIX_SWITCH(f.radix[0], op)
        }
    }
    __syncthreads();
    for (int t = 1; t + 1 < f.nst; t++) {
        const float2* twt = tw + f.twoff[t];
        const int ns = f.ns[t];
        auto op = [&](auto rc) {
            constexpr int R = decltype(rc)::value;
            fc_butterflies<R, NTHR>(f, t, fc_opaque(tid), [&](int a, int pn, int k) {
                float2 v[R], tv[R - 1];
                fc_ld_run(tv, twt, k, ns);
#pragma unroll
                for (int r = 0; r < R; r++) v[r] = lds[a + r * pn];
                fc_issued();
#pragma unroll
                for (int r = 1; r < R; r++) v[r] = cmulf(v[r], make_float2(tv[r - 1].x, -tv[r - 1].y));
                dft_reg<R, true>(v);
#pragma unroll
                for (int r = 0; r < R; r++) lds[a + r * pn] = v[r];
            });
        };
        if constexpr (WIDE) {
            FC_RADIX_SWITCH_MID(f.radix[t], op)
        } else {
            FC_RADIX_SWITCH(f.radix[t], op)
        }
        __syncthreads();
    }
}

// Row sum and best cell over the workgroup's threads (the lowest column on
// ties: the visit order within a row). The LDS buffer is free.
template <int NTHR>
__device__ __forceinline__ void full_row_reduce(float2* lds, double sum, float bv, int bc, double* rowsum,
                                                float* rowbest_v, uint64_t* rowbest_k, size_t base, int row, int ndop)
{
    const int tid = threadIdx.x;
    double* ssum = (double*)lds;
    float* sv = (float*)(ssum + NTHR / 64);
    int* sc = (int*)(sv + NTHR / 64);
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) {
        sum += __shfl_xor(sum, o);
        const float ov = __shfl_xor(bv, o);
        const int oc = __shfl_xor(bc, o);
        if (ov > bv || (ov == bv && oc < bc)) {
            bv = ov;
            bc = oc;
        }
    }
    if ((tid & 63) == 0) {
        ssum[tid >> 6] = sum;
        sv[tid >> 6] = bv;
        sc[tid >> 6] = bc;
    }
    __syncthreads();
    if (tid == 0) {
        for (int i = 1; i < NTHR / 64; i++) {
            sum += ssum[i];
            if (sv[i] > bv || (sv[i] == bv && sc[i] < bc)) {
                bv = sv[i];
                bc = sc[i];
            }
        }
        rowsum[base + row] = sum;
        rowbest_v[base + row] = bv;
        rowbest_k[base + row] = bc == 0x7fffffff ? ~0ull : (uint64_t)bc * ndop + row;
    }
}

// The powers of a step lie in LDS by drifted column; a thread's cells are
// columns tid + NTHR i, in registers between the steps. Beyond n: other LDS
// contents of the buffer (host: at least n rounded up to 4 NTHR floats).
#define FC_CELLS 20
template <int NTHR, int NC>
__device__ __forceinline__ void fc_accumulate(float (&acc)[NC], const float* pws, int n, bool first)
{
    static_assert(NC % 4 == 0, "cells in groups of four");
    const float* own = pws + fc_opaque(threadIdx.x);
#pragma unroll
    for (int i0 = 0; i0 < NC; i0 += 4) {
        if (NTHR * i0 < n) {
            float pw[4];
#pragma unroll
            for (int i = 0; i < 4; i++) pw[i] = own[NTHR * (i0 + i)];
#pragma unroll
            for (int i = 0; i < 4; i++) acc[i0 + i] = first ? pw[i] : acc[i0 + i] + pw[i];
        }
    }
}
template <int NTHR, int NC>
__device__ __forceinline__ void fc_store_cells(const float (&acc)[NC], float* accp, int n, double& sum, float& bv,
                                               int& bc)
{
#pragma unroll
    for (int i = 0; i < NC; i++) {
        const int dc = (int)threadIdx.x + NTHR * i;
        if (dc < n) {
            accp[dc] = acc[i];
            sum += (double)acc[i];
            if (acc[i] > bv) {  // columns ascend with i: the lowest on ties
                bv = acc[i];
                bc = dc;
            }
        }
    }
}

struct FullArgs {
    FullPlanDev f;
    const float2* tw;
    const float2* spec;      // [nnc][ncoh][n]
    const float2* code;      // [nprn][ndop][n]
    const uint16_t* colmap;  // [n] column of delay tau
    const int32_t* shifts;   // [nnc][ndop] drift of the sorted rows
    const int32_t* req;
    float* acc;              // [cnt][ndop][ap]
    double* rowsum;
    float* rowbest_v;
    uint64_t* rowbest_k;
    int ncoh, ndop, nnc, cnt, ap;
};

// MULTI: several noncoherent steps.
template <int NTHR, bool MULTI>
__global__ void __launch_bounds__(NTHR)
__attribute__((amdgpu_waves_per_eu(4))) k_full_corr(FullArgs A)
{
    extern __shared__ float2 lds[];
    const FullPlanDev& f = A.f;
    const int tid = threadIdx.x, n = f.n;
    // PRNs fastest, then the rows of one s: an XCD's workgroups share the
    // spectra of a few s in its L2
    const int lbk = xcd_logical_block();
    const int p = __builtin_amdgcn_readfirstlane(lbk % A.cnt);
    const int wi = __builtin_amdgcn_readfirstlane(lbk / A.cnt);
    const int nb = A.ndop / A.ncoh, s = wi / nb, w = s + A.ncoh * (wi - s * nb);
    int row = w + A.ndop / 2;
    if (row >= A.ndop) row -= A.ndop;
    const float2* G = A.code + ((size_t)A.req[p] * A.ndop + w) * n;
    float* accp = A.acc + ((size_t)p * A.ndop + row) * A.ap;
    double sum = 0.0;
    float bv = -INFINITY;
    int bc = 0x7fffffff;
    float acc[MULTI ? FC_CELLS : 1];
#pragma unroll
    for (int i = 0; i < (MULTI ? FC_CELLS : 1); i++) acc[i] = 0.f;
    for (int step = 0; step < A.nnc; step++) {
        const float2* Z = A.spec + ((size_t)step * A.ncoh + s) * n;
        fc_inverse_head<NTHR, !MULTI>(lds, f, A.tw, tid, Z, G);
        const uint32_t shift = (uint32_t)A.shifts[(size_t)step * A.ndop + row];
        {
            const int t = f.nst - 1, ns = f.ns[t];
            const float2* twt = A.tw + f.twoff[t];
            const int pn = ns + (ns >> f.pad_shift);
            auto op = [&](auto rc) {
                constexpr int R = decltype(rc)::value;
                constexpr int Q = FC_CELLS / R;  // butterflies per thread (host: ns <= Q NTHR)
                float pw[Q][R];
                const int k0 = fc_opaque(tid);
#pragma unroll
                for (int q = 0; q < Q; q++) {
                    const int k = k0 + NTHR * q;
                    if (k < ns) {
                        float2 v[R], tv[R - 1];
                        fc_ld_run(tv, twt, k, ns);
                        const float2* src = lds + fc_addr(k, f.pad_shift);
#pragma unroll
                        for (int r = 0; r < R; r++) v[r] = src[r * pn];
                        fc_issued();
#pragma unroll
                        for (int r = 1; r < R; r++) v[r] = cmulf(v[r], make_float2(tv[r - 1].x, -tv[r - 1].y));
                        dft_reg<R, true>(v);
#pragma unroll
                        for (int r = 0; r < R; r++) pw[q][r] = abs2_exact(v[r]);
                    }
                }
                fc_issued();
                uint32_t dc[Q][R];
#pragma unroll
                for (int q = 0; q < Q; q++) {
                    uint32_t off = (uint32_t)min(k0 + NTHR * q, ns - 1) * 2u;
#pragma unroll
                    for (int r = 0; r < R; r++) {
                        dc[q][r] = *(const uint16_t*)((const char*)A.colmap + off);
                        off += (uint32_t)ns * 2u;
                    }
                }
                fc_issued();
                if constexpr (MULTI) __syncthreads();  // every butterfly of the last stage is read
#pragma unroll
                for (int q = 0; q < Q; q++) {
#pragma unroll
                    for (int r = 0; r < R; r++) {
                        const uint32_t c = dc[q][r] + shift;
                        dc[q][r] = min(c, c - (uint32_t)n);  // c mod n for c < 2 n
                    }
                    if (k0 + NTHR * q < ns) {
#pragma unroll
                        for (int r = 0; r < R; r++) {
                            if constexpr (MULTI) {
                                *(float*)((char*)lds + dc[q][r] * 4u) = pw[q][r];
                            } else {  // one step: the cells go straight out
                                *(float*)((char*)accp + dc[q][r] * 4u) = pw[q][r];
                                sum += (double)pw[q][r];
                                if (pw[q][r] > bv || (pw[q][r] == bv && (int)dc[q][r] < bc)) {
                                    bv = pw[q][r];
                                    bc = (int)dc[q][r];
                                }
                            }
                        }
                    }
                }
            };
            FC_RADIX_SWITCH(f.radix[t], op)
        }
        if constexpr (MULTI) {
            __syncthreads();
            fc_accumulate<NTHR, FC_CELLS>(acc, (const float*)lds, n, step == 0);
        }
        __syncthreads();
    }
    if constexpr (MULTI) fc_store_cells<NTHR, FC_CELLS>(acc, accp, n, sum, bv, bc);
    full_row_reduce<NTHR>(lds, sum, bv, bc, A.rowsum, A.rowbest_v, A.rowbest_k, (size_t)p * A.ndop, row, A.ndop);
}

// ---------------------------------------------------------------------------
// The tile's block correlation (k_corr_tile: row k of column block r is signal
// double block k times code sub-block (k mod nb + r) mod nb, lags < bs) on the
// same in-place transforms, for the sizes that k_corr_tile runs with one
// transform per pass and runtime radices: more than 2048 points, or a radix
// above 5 in a middle stage, where it computes each output of a prime radix by
// its own sum. F 5600 (L5-like 30.69 MHz, 110 rows, 11 blocks, 6 PRNs) took
// 1.89 ms per launch there. grid (ndop, batch, split)
// ---------------------------------------------------------------------------
template <int NTHR, class TileT>
__global__ void __launch_bounds__(NTHR)
__attribute__((amdgpu_waves_per_eu(4)))
k_corr_fc(const float2* __restrict__ sigfft_step, const float2* __restrict__ prnconj, const int32_t* __restrict__ req,
          TileT* __restrict__ tile, FullPlanDev f, const float2* __restrict__ tw, int nb, int bs, int tp, int ndop,
          float hscale, int rb0, int nrb)
{
    extern __shared__ float2 lds[];
    const int tid = threadIdx.x;
    const int lbk = xcd_logical_block();
    const int k = __builtin_amdgcn_readfirstlane(lbk % gridDim.x);
    const int rest = __builtin_amdgcn_readfirstlane(lbk / gridDim.x);
    const int p = rest % gridDim.y, sp = rest / gridDim.y;
    const int chunk = (nrb + gridDim.z - 1) / gridDim.z;
    const int r_end = min(nrb, (sp + 1) * chunk);
    const float2* S = sigfft_step + (size_t)k * f.n;
    const float2* Pp = prnconj + (size_t)req[p] * nb * f.n;
    for (int rr = sp * chunk; rr < r_end; rr++) {
        const int b = (k % nb + rb0 + rr) % nb;
        fc_inverse_head<NTHR, true>(lds, f, tw, tid, S, Pp + (size_t)b * f.n);
        const LagOut<TileT, false> out{tile + (((size_t)p * nrb + rr) * ndop + k) * tp, 0, bs, 1.0f, 1, hscale};
        const int t = f.nst - 1, ns = f.ns[t];
        const float2* twt = tw + f.twoff[t];
        const int pn = ns + (ns >> f.pad_shift);
        auto op = [&](auto rc) {
            constexpr int R = decltype(rc)::value;
            for (int j = fc_opaque(tid); j < ns; j += NTHR) {
                float2 v[R], tv[R - 1];
                fc_ld_run(tv, twt, j, ns);
                const float2* src = lds + fc_addr(j, f.pad_shift);
#pragma unroll
                for (int r = 0; r < R; r++) v[r] = src[r * pn];
                fc_issued();
#pragma unroll
                for (int r = 1; r < R; r++) v[r] = cmulf(v[r], make_float2(tv[r - 1].x, -tv[r - 1].y));
                dft_reg<R, true>(v);
                // lags below bs <= F / 2: outputs r <= R / 2
#pragma unroll
                for (int r = 0; r <= R / 2; r++) out(0, j + r * ns, v[r]);
            }
        };
        FC_RADIX_SWITCH(f.radix[t], op)
        __syncthreads();
    }
}

// Spectra for k_corr_fc: signal double blocks (grid (ndop, nnc)) and conj code
// sub-blocks times 1 / F (grid (nb, nprn)).
template <int NTHR>
__global__ void __launch_bounds__(NTHR)
k_fc_signal(const void* __restrict__ sig, int eltype, float2* __restrict__ sigfft, FullPlanDev f,
            const float2* __restrict__ tw, int bs, int64_t seglen, int ndop, int do_if, float phase_step,
            double phase_step64)
{
    extern __shared__ float2 lds[];
    const int64_t seg0 = (int64_t)blockIdx.y * seglen;
    const DownconvIn in{sig, eltype, seg0, seglen, (int64_t)blockIdx.x * bs, 2 * bs, do_if,
                        __fmul_rn((float)seg0, phase_step), phase_step, phase_step64};
    float2* out = sigfft + ((size_t)blockIdx.y * ndop + blockIdx.x) * f.n;
    fc_forward<NTHR>(
        lds, f, tw, threadIdx.x, [&](int i) { return in(0, i); }, [&](int i, float2 x) { out[i] = x; });
}
template <int NTHR>
__global__ void __launch_bounds__(NTHR)
k_fc_code(const int8_t* __restrict__ codes, float2* __restrict__ prnconj, FullPlanDev f, const float2* __restrict__ tw,
          int spc, int nb, int bs, float scale)
{
    extern __shared__ float2 lds[];
    const CodeIn in{codes + (size_t)blockIdx.y * spc + (size_t)blockIdx.x * bs, bs};
    float2* out = prnconj + ((size_t)blockIdx.y * nb + blockIdx.x) * f.n;
    fc_forward<NTHR>(
        lds, f, tw, threadIdx.x, [&](int i) { return in(0, i); },
        [&](int i, float2 x) { out[i] = make_float2(x.x * scale, -x.y * scale); });
}

// ---------------------------------------------------------------------------
// Column stage of the simple path (k_column_simple) with few Doppler rows: a
// thread owns a code column, reads its N tile values (consecutive lanes,
// consecutive lags), transforms them in registers and adds the powers to its
// N cells. No LDS and one round trip to memory: bound by the tile and the
// accumulator's read-modify-write, 8 N + 8 N bytes per column. k_column_simple
// gathers blocks of columns into LDS for transforms of any length: 46 us per
// step at N 15, 30690 columns, 12 PRNs (88 MB), this 15.7 us (5.6 TB/s).
// grid (ceil(bs / 256), nb, batch)
// ---------------------------------------------------------------------------
#define COLREG_NTHR 256
template <int N>
__global__ void __launch_bounds__(COLREG_NTHR)
k_column_reg(ColumnArgs A)
{
    const int lbk = xcd_logical_block();
    const int lb = __builtin_amdgcn_readfirstlane(lbk % gridDim.x);
    const int r = __builtin_amdgcn_readfirstlane((lbk / gridDim.x) % gridDim.y);
    const int p = __builtin_amdgcn_readfirstlane(lbk / (gridDim.x * gridDim.y));
    const int lag = lb * COLREG_NTHR + threadIdx.x;
    if (lag >= A.bs) return;
    const char* T = (const char*)(A.tile + ((size_t)p * A.nb + r) * N * A.tp);
    char* acc = (char*)(A.acc + (size_t)p * A.acc_ps);
    const int pc = r * A.bs + lag;
    float2 v[N];
    float prev[N];
    uint32_t off[N];
#pragma unroll
    for (int n = 0; n < N; n++) v[n] = *(const float2*)(T + (uint32_t)(n * A.tp + lag) * (uint32_t)sizeof(float2));
    // raw bin k -> row (k + N / 2) mod N (src/plan.jl:528), drifted column
#pragma unroll
    for (int k = 0; k < N; k++) {
        const int row = (k + N / 2) % N;
        int dc = pc + A.shifts[row];
        if (dc >= A.spc) dc -= A.spc;
        off[k] = (uint32_t)(row * A.ap + dc) * (uint32_t)sizeof(float);
        prev[k] = 0.f;
    }
    if (!A.first_step) {
#pragma unroll
        for (int k = 0; k < N; k++) prev[k] = *(const float*)(acc + off[k]);
    }
    fc_issued();
    dft_reg<N, false>(v);
#pragma unroll
    for (int k = 0; k < N; k++) *(float*)(acc + off[k]) = prev[k] + abs2_exact(v[k]);
}
// OP(N) for the compiled row counts
#define COLREG_ALL(OP)                                                                                           \
    OP(4) OP(5) OP(6) OP(7) OP(8) OP(9) OP(10) OP(11) OP(12) OP(13) OP(15) OP(16) OP(18) OP(20) OP(21) OP(22) \
    OP(24) OP(25) OP(30) OP(32)

// ---------------------------------------------------------------------------
// Direct rotation search (k_column_rotation with one pattern per rotation
// slice) of few Doppler rows, ndop = P nb with P coherent periods: rows
// n = p nb + m, raw bins w = s + P k,
//   X_q[s + P k] = sum_m W_nb^(k m) W_N^(s m) sum_p sigma_q[p] W_P^(s p) x[p nb + m].
// A workgroup owns C lags; thread (lag, m) holds its P samples (the column
// rotated by its alignment) for all rotations, thread (lag, s) the nb
// accumulator cells of its bins. Per rotation: signs, a P-point DFT and the
// twiddles in registers, one LDS transpose, an nb-point DFT in registers, and
// the cells' read-modify-write, whose reads go out ahead of the transforms.
// Lanes run along lags throughout: LDS and the row-major accumulator are
// accessed in runs of C. k_column_rotation restarts from LDS per rotation with
// runtime radices (11 as a direct sum): 4.72 ms per step at ndop 110, R 10,
// 30690 columns, 6 PRNs. grid (ceil(bs / C), nb, batch)
// ---------------------------------------------------------------------------
#define ROTSPLIT_NTHR 512
// dynamic LDS pitch of a bin class (float2): two classes of half a wave fall on
// distinct banks
__host__ __device__ constexpr int rotsplit_pitch(int nb, int C) { return nb * C + (nb % 2 == 0 ? 16 : 0); }
template <int P, int NB>
__global__ void __launch_bounds__(ROTSPLIT_NTHR)
k_column_rotsplit(ColumnArgs A, int C)
{
    extern __shared__ float2 lds[];
    __shared__ uint32_t smask[64];
    constexpr int N = P * NB, HALF = N / 2;
    const int tid = threadIdx.x;
    const int lbk = xcd_logical_block();
    const int lb = __builtin_amdgcn_readfirstlane(lbk % gridDim.x);
    const int r = __builtin_amdgcn_readfirstlane((lbk / gridDim.x) % gridDim.y);
    const int p = __builtin_amdgcn_readfirstlane(lbk / (gridDim.x * gridDim.y));
    const int lag0 = lb * C, ncol = min(C, A.bs - lag0);
    const int c = tid & (C - 1), m = tid / C;  // m: lag within the period, and the bin class s
    const int pitch = rotsplit_pitch(NB, C);
    const bool act1 = m < NB && c < ncol, act2 = m < P && c < ncol;
    const int pc = r * A.bs + lag0 + min(c, ncol - 1);
    if (tid < A.R) {
        const float* pat = A.patterns + ((size_t)A.pset[A.req[p]] * A.Q + tid) * A.ncoh;
        uint32_t msk = 0;
        for (int i = 0; i < P; i++)
            if (pat[i] < 0.f) msk |= 1u << i;
        smask[tid] = msk;
    }
    // samples and twiddles W_N^(s m) of thread (c, m)
    float2 x[P], tw[P];
    {
        const int lag = lag0 + min(c, ncol - 1);
        const int wrap = ((NB - pc / A.bs) % NB) * A.bs + (pc % A.bs);  // src/noncoherent_integration.jl:212-215
        const int eff = ((wrap + (A.bs >> 1)) / A.bs) % NB;
        const float2* T = A.tile + (((size_t)p * NB + r) * N) * A.tp + lag;
        const int mm = min(m, NB - 1);
#pragma unroll
        for (int q = 0; q < P; q++) {
            int src = q * NB + mm + eff;
            if (src >= N) src -= N;
            x[q] = T[(size_t)src * A.tp];
        }
#pragma unroll
        for (int q = 0; q < P; q++) tw[q] = A.twD[q * mm];
    }
    // cells of thread (c, s): raw bin s + P k -> row (w + N / 2) mod N, drifted column
    uint32_t off[NB];
    {
        const int s = min(m, P - 1);
#pragma unroll
        for (int k = 0; k < NB; k++) {
            int row = s + P * k + HALF;
            if (row >= N) row -= N;
            int dc = pc + A.shifts[row];
            if (dc >= A.spc) dc -= A.spc;
            off[k] = (uint32_t)(row * A.ap + dc) * (uint32_t)sizeof(float);
        }
    }
    float* accp = A.acc + (size_t)p * A.acc_ps;
    const bool first = A.first_step != 0;
    __syncthreads();  // masks
    for (int q = 0; q < A.R; q++) {
        char* base = (char*)(accp + (size_t)q * A.spc);
        float prev[NB];
        if (!first && act2) {
#pragma unroll
            for (int k = 0; k < NB; k++) prev[k] = *(const float*)(base + off[k]);
        }
        const uint32_t mq = smask[q];
        if (act1) {
            float2 u[P];
#pragma unroll
            for (int i = 0; i < P; i++) {
                const uint32_t sg = ((mq >> i) & 1u) << 31;
                u[i] = make_float2(__uint_as_float(__float_as_uint(x[i].x) ^ sg),
                                   __uint_as_float(__float_as_uint(x[i].y) ^ sg));
            }
            dft_reg<P, false>(u);
            float2* dst = lds + m * C + c;
            dst[0] = u[0];
#pragma unroll
            for (int s = 1; s < P; s++) dst[s * pitch] = cmulf(u[s], tw[s]);
        }
        __syncthreads();
        float2 v[NB];
        if (act2) {
            const float2* src = lds + m * pitch + c;
#pragma unroll
            for (int i = 0; i < NB; i++) v[i] = src[i * C];
        }
        __syncthreads();  // the transpose is consumed
        if (act2) {
            dft_reg<NB, false>(v);
#pragma unroll
            for (int k = 0; k < NB; k++) {
                // muladd(re, re, im * im), the reference's rotation power
                const float pw = fmaf(v[k].x, v[k].x, __fmul_rn(v[k].y, v[k].y));
                *(float*)(base + off[k]) = first ? pw : prev[k] + pw;
            }
        }
    }
}
// OP(P, NB) for the compiled periods and row lengths
#define ROTSPLIT_NB(P, OP)                                                                                     \
    OP(P, 4) OP(P, 5) OP(P, 6) OP(P, 7) OP(P, 8) OP(P, 9) OP(P, 10) OP(P, 11) OP(P, 12) OP(P, 13) OP(P, 15) \
    OP(P, 16) OP(P, 20) OP(P, 22)
#define ROTSPLIT_ALL(OP) ROTSPLIT_NB(10, OP) ROTSPLIT_NB(20, OP)

// ---------------------------------------------------------------------------
// Direct rotation search of 25 coherent periods, ndop = 25 NB (the E1-like
// searches): rows n = p NB + m, raw bins w = s + 25 k, as k_column_rotbig,
//   X_q[s + 25 k] = sum_m W_NB^(k m) W_N^(s m) sum_p sigma_q[p] W_25^(s p) x[p NB + m].
// A workgroup owns C code columns. Thread (column, m) keeps the 25 samples
// of its lag in registers for all rotations; per rotation it applies the
// signs (flips of the float sign bit), a 5 x 5 DFT over p and the twiddles,
// and writes the 25 classes s to LDS. The NB-point transforms of the 25 C
// rows follow as RA x RB in place, and the last stage adds the powers to the
// cells straight from its registers: butterfly (s, i) of a column has rows
// s + 25 i + 25 RA k2, so consecutive threads hold consecutive rows of the
// column-major accumulator. Offsets of the cells stay in registers, and their
// previous values are read ahead of the rotation's first stage.
// CHUNK: cells outside a code-column window are dropped and the tile holds
// blocks rb0 .. rb0 + nrb (launch_rotbig); else the whole code period.
// grid (ceil(bs / C), column blocks, batch)
// Bound by vector instructions. At NB 80: 2130 per column and rotation against
// 2600 of k_column_rot2000, 8.5 ms at 100000 columns and R 25 if
// nothing waited, next to 41.9 GB of cells (8.5 ms at a copy's rate). Three
// columns make four waves, one per SIMD, and two workgroups per CU leave the
// 231 registers for all 30 offsets and values: four columns in five waves, two
// and a half per SIMD with one butterfly's cells ahead, took 14.4 ms
// and k_column_rot2000 15.1 ms; this takes 10.5 ms per PRN-step. The other row
// lengths take C and RA x RB that keep 200 to 250 of 256 threads (500 of 512)
// busy in the 25-point stage with at most 30 cells each; against
// k_column_rotbig with compile-time rows, per PRN-step at 25 MHz: 8.9 -> 6.3 ms
// at NB 50, 17.6 -> 12.9 at 100, 55.6 -> 32.3 at 250, 132 -> 72 at 500 (windows
// of a PRN added up, one step).
template <int NB>
struct Rot25;
template <> struct Rot25<50> { static constexpr int RA = 10, RB = 5, C = 5, NT = 256; };
template <> struct Rot25<80> { static constexpr int RA = 8, RB = 10, C = 3, NT = 256; };
template <> struct Rot25<100> { static constexpr int RA = 10, RB = 10, C = 2, NT = 256; };
template <> struct Rot25<250> { static constexpr int RA = 10, RB = 25, C = 1, NT = 256; };
template <> struct Rot25<500> { static constexpr int RA = 20, RB = 25, C = 1, NT = 512; };
// pitches of a row and of a column: odd, and about 32 / C mod 32, so that lanes
// along rows and along columns spread over the banks
template <int NB>
constexpr int rot25_row() { return NB | 1; }
template <int NB>
constexpr int rot25_col()
{
    constexpr int C = Rot25<NB>::C, n = 25 * rot25_row<NB>();
    return n + (((32 + C - 1) / C - n) % 32 + 32) % 32;
}
template <int NB>
constexpr size_t rot25_lds() { return (size_t)(Rot25<NB>::C * rot25_col<NB>() + NB) * sizeof(float2); }

template <int NB, bool CHUNK>
__global__ void __launch_bounds__(Rot25<NB>::NT)
__attribute__((amdgpu_waves_per_eu(2, 2)))
k_column_rot25(ColumnArgs A)
{
    constexpr int P = 25, N = P * NB, RA = Rot25<NB>::RA, RB = Rot25<NB>::RB, C = Rot25<NB>::C, NT = Rot25<NB>::NT;
    constexpr int RP = rot25_row<NB>(), CP = rot25_col<NB>();
    constexpr int ITA = (C * P * RB + NT - 1) / NT, ITB = (C * P * RA + NT - 1) / NT;
    static_assert(C * NB <= NT && RA * RB == NB && N % 2 == 0 && C * CP < 65536 && NT >= 64, "work split");
    extern __shared__ float2 lds[];
    float2* stw = lds + C * CP;                // W_NB^(i j) at [j][i], i < RA, j < RB
    __shared__ uint32_t smask[64];
    const int tid = threadIdx.x;
    const int lbk = xcd_logical_block();
    const int lb = __builtin_amdgcn_readfirstlane(lbk % gridDim.x);
    const int rr = __builtin_amdgcn_readfirstlane((lbk / gridDim.x) % gridDim.y);  // tile block
    const int p = __builtin_amdgcn_readfirstlane(lbk / (gridDim.x * gridDim.y));
    const int nrb = CHUNK ? A.nrb : NB;
    int r = CHUNK ? A.rb0 + rr : rr;
    if (CHUNK && r >= NB) r -= NB;
    const int lag0 = lb * C, ncol = min(C, A.bs - lag0);
    for (int j = tid; j < NB; j += NT) stw[j] = A.twD[P * (j % RA) * (j / RA)];
    if (tid < A.R) {
        const float* pat = A.patterns + ((size_t)A.pset[A.req[p]] * A.Q + tid) * A.ncoh;
        uint32_t msk = 0;
        for (int q = 0; q < P; q++)
            if (pat[q] < 0.f) msk |= 1u << q;
        smask[tid] = msk;
    }
    // lag m of column c: 25 samples of the column rotated by its alignment
    // (src/noncoherent_integration.jl:212-215), factors of W_N^(s m), s = s1 + 5 s2
    const int c1 = tid % C, m = min(tid / C, NB - 1);
    float2 x[P], tw1[5], tw5[5];
    {
        const int lag = lag0 + min(c1, ncol - 1), pc = r * A.bs + lag;
        const int wrap = ((NB - pc / A.bs) % NB) * A.bs + (pc % A.bs);
        const int eff = ((wrap + (A.bs >> 1)) / A.bs) % NB;
        const float2* T = A.tile + (((size_t)p * nrb + rr) * N) * A.tp + lag;
#pragma unroll
        for (int q = 0; q < P; q++) {
            int src = q * NB + m + eff;
            if (src >= N) src -= N;
            // neighbouring workgroups (the next lags) read the same tile lines: plain, cached loads
            x[q] = T[(size_t)src * A.tp];
        }
#pragma unroll
        for (int i = 1; i < 5; i++) {
            tw1[i] = A.twD[i * m];
            tw5[i] = A.twD[5 * i * m];
        }
    }
    float* accp = A.acc + (size_t)p * A.acc_ps;
    const size_t slice = (size_t)(CHUNK ? A.slice_cols : A.spc) * A.acc_ldc * 4;  // bytes of a rotation slice (below 2^32)
    const bool first = A.first_step != 0;
    const bool whole = !CHUNK || A.winlen >= A.spc;  // no cell falls outside the window
    // The stages' butterflies (their index arithmetic is full of slow
    // multiplications). Radix RA: LDS index | j << 16, all ones past the end.
    // Radix RB: LDS index and the byte offsets of the cells in a slice; it takes
    // the threads in reverse, so that the remainders of the two stages fall to
    // different waves.
    uint32_t pa[ITA], pb[ITB], off[ITB][RB];
#pragma unroll
    for (int it = 0; it < ITA; it++) {
        const uint32_t idx = tid + it * NT, c = idx / (P * RB), b = idx % (P * RB), j = b / P, s = b % P;
        pa[it] = idx < C * P * RB ? (c * CP + s * RP + j) | j << 16 : 0xffffffffu;
    }
#pragma unroll
    for (int it = 0; it < ITB; it++) {
        const uint32_t idx = NT - 1 - tid + it * NT, c = idx / (P * RA), b = idx % (P * RA), i = b / P, s = b % P;
        const bool act = idx < C * P * RA && c < (uint32_t)ncol;
        pb[it] = act ? c * CP + s * RP + RB * i : 0xffffffffu;
#pragma unroll
        for (int k2 = 0; k2 < RB; k2++) {
            // raw bin b + 25 RA k2, its sorted row (N / 2 further), column + its drift (mod spc)
            int row = (int)b + P * RA * k2 + N / 2;
            if (row >= N) row -= N;
            int dc = r * A.bs + lag0 + (act ? (int)c : 0) + A.shifts[row];
            if (dc >= A.spc) dc -= A.spc;
            if (CHUNK) {
                dc -= A.win0;
                if (dc < 0) dc += A.spc;
            }
            off[it][k2] = ((uint32_t)row + (uint32_t)dc * (uint32_t)A.acc_ldc) * 4u;
            if (CHUNK && dc >= A.winlen) off[it][k2] = ~0u;
        }
    }
    __syncthreads();  // tables and masks
#pragma unroll 1
    for (int q = 0; q < A.R; q++) {
        // opaque copies: what follows from them is not hoisted into registers
        uint32_t ia[ITA], ib[ITB];
#pragma unroll
        for (int it = 0; it < ITA; it++) {
            ia[it] = pa[it];
            asm volatile("" : "+v"(ia[it]));
        }
#pragma unroll
        for (int it = 0; it < ITB; it++) {
            ib[it] = pb[it];
            asm volatile("" : "+v"(ib[it]));
        }
        const uint32_t mq = __builtin_amdgcn_readfirstlane(smask[q]);
        char* base = (char*)accp + (size_t)q * slice;
        // opaque copies of the offsets: loads and stores take the form of a
        // scalar base and a 32-bit offset
        uint32_t po[ITB][RB];
#pragma unroll
        for (int it = 0; it < ITB; it++)
#pragma unroll
            for (int k2 = 0; k2 < RB; k2++) {
                po[it][k2] = off[it][k2];
                asm volatile("" : "+v"(po[it][k2]));
            }
        // previous values of the cells
        float prev[ITB][RB];
#pragma unroll
        for (int it = 0; it < ITB; it++)
#pragma unroll
            for (int k2 = 0; k2 < RB; k2++) prev[it][k2] = 0.f;
        if (!first) {
#pragma unroll
            for (int it = 0; it < ITB; it++)
#pragma unroll
                for (int k2 = 0; k2 < RB; k2++) {
                    // outside the window: the slice's first cell instead, no branch
                    const uint32_t o = CHUNK && po[it][k2] == ~0u ? 0u : po[it][k2];
                    prev[it][k2] = *(const float*)(base + o);
                }
            __builtin_amdgcn_sched_barrier(0);
        }
        {
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
            float2* dst = lds + c1 * CP + m;
            if (tid < C * NB) {
#pragma unroll
                for (int s1 = 0; s1 < 5; s1++) {
                    float2 w5[5];
#pragma unroll
                    for (int p2 = 0; p2 < 5; p2++) w5[p2] = s1 ? cmulf(u[p2][s1], tw1[s1]) : u[p2][s1];
                    bfly5<false>(w5);
#pragma unroll
                    for (int s2 = 0; s2 < 5; s2++) dst[(s1 + 5 * s2) * RP] = s2 ? cmulf(w5[s2], tw5[s2]) : w5[s2];
                }
            }
        }
        __syncthreads();
        // radix RA over m = j + RB i: output i at slot RB i + j, times W_NB^(i j)
#pragma unroll
        for (int it = 0; it < ITA; it++) {
            if (ia[it] != 0xffffffffu) {
                float2* a = lds + (ia[it] & 0xffffu);
                const float2* w = stw + RA * (ia[it] >> 16);
                float2 v[RA], tw[RA];
#pragma unroll
                for (int i = 0; i < RA; i++) v[i] = a[RB * i];
#pragma unroll
                for (int i = 1; i < RA; i++) tw[i] = w[i];
                __builtin_amdgcn_sched_barrier(0);
                dft_reg<RA, false>(v);
                a[0] = v[0];
#pragma unroll
                for (int i = 1; i < RA; i++) a[RB * i] = cmulf(v[i], tw[i]);
            }
        }
        __syncthreads();
        // radix RB over j of (s, i): raw bins s + 25 (i + RA k2)
#pragma unroll
        for (int it = 0; it < ITB; it++) {
            const bool act = ib[it] != 0xffffffffu;
            float2 v[RB];
            const float2* a = lds + (act ? ib[it] : 0u);
#pragma unroll
            for (int j = 0; j < RB; j++) v[j] = a[j];
            __builtin_amdgcn_sched_barrier(0);
            dft_reg<RB, false>(v);
            if (act) {
#pragma unroll
                for (int k2 = 0; k2 < RB; k2++) {
                    // muladd(re, re, im * im), the reference's rotation power
                    const float pw = fmaf(v[k2].x, v[k2].x, __fmul_rn(v[k2].y, v[k2].y));
                    if (whole || po[it][k2] != ~0u) *(float*)(base + po[it][k2]) = prev[it][k2] + pw;
                }
            }
        }
        __syncthreads();  // the rows are consumed
    }
}

// ---------------------------------------------------------------------------
// Data-bit search (k_column_sign) of two 20-period bits, ndop = 40 nb: for
// every edge offset and sign combination the window's two bits are added onto
// each other, x_e[i] +- x_e[i + 20] at period i < 20, and transformed with
// 20 periods of zeros behind them; a cell is the largest power of the set.
//   X[w] = sum_m W_nb^(k m) W_N^(w' m) DFT20_s(W_40^(o i) y[i nb + m]),
// w' = 2 s + o, w = w' + 40 k: the zeros cost nothing, both parities o are
// 20-point transforms of the same y. A workgroup owns C = 16 lags; thread
// (lag, m) adds the bits and transforms over the periods in registers, thread
// (lag, s) takes the nb-point rows after one LDS transpose and keeps the
// maxima of its 2 nb cells in registers, lanes along lags throughout. The tile
// is read again for each edge and combination, from L2 mostly: 80 registers of
// samples, or as much LDS, would leave one workgroup per CU.
// k_column_sign runs the padded transforms with runtime radices in LDS, and
// its maxima too: 781 us at ndop 640, 4000 columns, 8 PRNs, two edges and two
// combinations; this takes 210 us. grid (ceil(bs / 16), nb, batch)
// ---------------------------------------------------------------------------
#define BITSPLIT_C 16
#define BITSPLIT_NTHR 384
// W_40^i = exp(-2 pi i / 40)
__constant__ float2 kW40[20] = {
    {1.0f, 0.0f}, {0.98768834059513777f, -0.15643446504023087f},
    {0.95105651629515353f, -0.3090169943749474f}, {0.8910065241883679f, -0.45399049973954675f},
    {0.80901699437494745f, -0.58778525229247314f}, {0.70710678118654757f, -0.70710678118654746f},
    {0.58778525229247314f, -0.80901699437494745f}, {0.4539904997395468f, -0.89100652418836779f},
    {0.30901699437494745f, -0.95105651629515353f}, {0.15643446504023092f, -0.98768834059513777f},
    {0.0f, -1.0f}, {-0.15643446504023059f, -0.98768834059513777f},
    {-0.30901699437494734f, -0.95105651629515364f}, {-0.45399049973954669f, -0.8910065241883679f},
    {-0.58778525229247303f, -0.80901699437494745f}, {-0.70710678118654746f, -0.70710678118654757f},
    {-0.80901699437494734f, -0.58778525229247325f}, {-0.89100652418836779f, -0.45399049973954686f},
    {-0.95105651629515353f, -0.30901699437494751f}, {-0.98768834059513766f, -0.15643446504023098f}};
constexpr size_t bitsplit_lds(int nb)
{
    return ((size_t)20 * rotsplit_pitch(nb, BITSPLIT_C) + (size_t)40 * nb) * sizeof(float2);
}
template <int NB>
__global__ void __launch_bounds__(BITSPLIT_NTHR)
__attribute__((amdgpu_waves_per_eu(3)))
k_column_bitsplit(ColumnArgs A)
{
    extern __shared__ float2 lds[];
    constexpr int PB = 20, P = 2 * PB, N = P * NB, C = BITSPLIT_C, pitch = rotsplit_pitch(NB, C);
    float2* stw = lds + PB * pitch;  // W_N^(s m) at [s][m]
    const int tid = threadIdx.x;
    const int lbk = xcd_logical_block();
    const int lb = __builtin_amdgcn_readfirstlane(lbk % gridDim.x);
    const int r = __builtin_amdgcn_readfirstlane((lbk / gridDim.x) % gridDim.y);
    const int p = __builtin_amdgcn_readfirstlane(lbk / (gridDim.x * gridDim.y));
    const int lag0 = lb * C, ncol = min(C, A.bs - lag0);
    const int c = tid % C, m = tid / C;  // m: lag within the period, and the bin class s
    const bool act1 = m < NB && c < ncol, act2 = m < PB && c < ncol;
    for (int i = tid; i < N; i += blockDim.x) stw[i] = A.twD[(i / NB) * (i % NB)];
    const float* pat = A.patterns + (size_t)A.pset[A.req[p]] * A.ncoh * A.Q;
    const float2* T = A.tile + (((size_t)p * NB + r) * N) * A.tp + lag0;
    const uint32_t voff = (uint32_t)(min(m, NB - 1) * A.tp + min(c, ncol - 1)) * (uint32_t)sizeof(float2);
    const int es = __builtin_amdgcn_readfirstlane(PB / A.E);
    const uint32_t bit = (uint32_t)(PB * NB * A.tp) * (uint32_t)sizeof(float2);
    const uint32_t period = bit / PB;  // bytes of a period's rows; the 40 below 2^31
    float* accp = A.acc + (size_t)p * A.acc_ps;
    const int pc = r * A.bs + lag0 + min(c, ncol - 1);
    __syncthreads();  // twiddles
    // both parities per read of the tile where their maxima fit the registers
    // with the transforms, else one after the other
    constexpr int NO = NB <= 16 ? 2 : 1;
#pragma unroll
    for (int o0 = 0; o0 < 2; o0 += NO) {
        float mx[NO][NB];
#pragma unroll
        for (int k = 0; k < NB; k++) mx[0][k] = mx[NO - 1][k] = 0.f;
#pragma unroll 1
        for (int e = 0; e < A.E; e++) {
#pragma unroll 1
            for (int d = 0; d < A.Q; d++) {
                // the power does not see a common sign: the second bit relative to the first
                const uint32_t sg = __builtin_amdgcn_readfirstlane(
                    (__float_as_uint(pat[(size_t)d * P]) ^ __float_as_uint(pat[(size_t)d * P + PB])) & 0x80000000u);
                float2 y[PB];
                {
                    float2 b1[PB];
                    uint32_t vo = voff, q0 = e * es * period;
                    asm volatile("" : "+v"(vo), "+s"(q0));  // opaque: no addresses kept across combinations
#pragma unroll
                    for (int i = 0; i < PB; i++) {
                        const uint32_t q1 = q0 >= bit ? q0 - bit : q0 + bit;
                        y[i] = *(const float2*)((const char*)T + (q0 + vo));
                        b1[i] = *(const float2*)((const char*)T + (q1 + vo));
                        q0 += period;
                    }
                    fc_issued();
#pragma unroll
                    for (int i = 0; i < PB; i++) {
                        y[i].x += __uint_as_float(__float_as_uint(b1[i].x) ^ sg);
                        y[i].y += __uint_as_float(__float_as_uint(b1[i].y) ^ sg);
                    }
                }
#pragma unroll
                for (int o1 = 0; o1 < NO; o1++) {
                    const int o = o0 + o1;
                    if (act1) {
                        float2 u[PB];
#pragma unroll
                        for (int i = 0; i < PB; i++) u[i] = o && i ? cmulf(y[i], kW40[i]) : y[i];
                        dft_reg<PB, false>(u);
                        float2* dst = lds + m * C + c;
                        const float2* w = stw + o * NB + m;
#pragma unroll
                        for (int s = 0; s < PB; s++) dst[s * pitch] = s + o ? cmulf(u[s], w[2 * s * NB]) : u[s];
                    }
                    __syncthreads();
                    __builtin_amdgcn_sched_barrier(0);
                    float2 v[NB];
                    if (act2) {
                        const float2* src = lds + m * pitch + c;
#pragma unroll
                        for (int i = 0; i < NB; i++) v[i] = src[i * C];
                    }
                    __syncthreads();  // the transpose is consumed
                    __builtin_amdgcn_sched_barrier(0);
                    if (act2) {
                        dft_reg<NB, false>(v);
#pragma unroll
                        for (int k = 0; k < NB; k++) {
                            const float pw = abs2_exact(v[k]);
                            mx[o1][k] = pw > mx[o1][k] ? pw : mx[o1][k];
                        }
                    }
                }
            }
        }
        if (act2) {
            // raw bin w = 2 s + o + 40 k -> row (w + N / 2) mod N, drifted column
#pragma unroll
            for (int o1 = 0; o1 < NO; o1++) {
                uint32_t off[NB];
#pragma unroll
                for (int k = 0; k < NB; k++) {
                    int row = 2 * m + o0 + o1 + P * k + N / 2;
                    if (row >= N) row -= N;
                    int dc = pc + A.shifts[row];
                    if (dc >= A.spc) dc -= A.spc;
                    off[k] = (uint32_t)(row * A.ap + dc) * (uint32_t)sizeof(float);
                }
                if (!A.first_step) {
                    float prev[NB];
#pragma unroll
                    for (int k = 0; k < NB; k++) prev[k] = *(const float*)((const char*)accp + off[k]);
#pragma unroll
                    for (int k = 0; k < NB; k++) mx[o1][k] = prev[k] + mx[o1][k];
                }
#pragma unroll
                for (int k = 0; k < NB; k++) *(float*)((char*)accp + off[k]) = mx[o1][k];
            }
        }
    }
}
// OP(NB) for the compiled row lengths
#define BITSPLIT_ALL(OP) OP(10) OP(11) OP(12) OP(15) OP(16) OP(20) OP(22)

// ---------------------------------------------------------------------------
// Code periods of 31 RB RC samples with 31, RB and RC pairwise coprime, RB and
// RC radices of the switches below, at most 16384 samples: of the multiples of
// the 1.023 MHz chip rate (1023 = 3 11 31) the 2, 3, 4, 5, 6, 8, 10 and 16 fold. The
// others (7, 9, 11 to 15, 17 to 20) have no such axes or do not fit, and a
// factor 31 no radix in k_full_corr: they run on the tile. By
// Good-Thomas the transform is three independent DFTs along the axes of a
// 31 x RB x RC array, with no twiddles: f = sum_i f_i N / q_i, n and tau by
// their residues. The 31-point DFTs, the largest part of the arithmetic on
// the vector unit (34 operations per point), run on the matrix cores in FP32:
// with E_n = x_n + x_(31-n), O_n = x_n - x_(31-n) (E_0 = x_0, O_0 = 0) a DFT is
// one real 16 x 16 cosine product on E and one sine product on O, so 16
// columns take 16 v_mfma_f32_16x16x4_f32 (re and im of both), whose lane
// layout the spectra's loads and the LDS stores follow directly.
// ---------------------------------------------------------------------------
// cos and sin of 2 pi k / 31
__constant__ float k31cos[31] = {1.0f, 0.97952994125249448f, 0.9189578116202306f, 0.82076344120727629f,
    0.68896691907568663f, 0.52896401032696239f, 0.34730525284482028f, 0.1514277775045767f, -0.050649168838712642f,
    -0.25065253225872042f, -0.44039415155763439f, -0.61210598254766257f, -0.75875812269279086f, -0.87434661614458209f,
    -0.95413925640004882f, -0.99486932339189504f, -0.99486932339189516f, -0.95413925640004882f, -0.8743466161445822f,
    -0.75875812269279108f, -0.61210598254766269f, -0.44039415155763423f, -0.25065253225872131f,
    -0.050649168838713551f, 0.15142777750457667f, 0.34730525284482028f, 0.52896401032696239f, 0.68896691907568652f,
    0.82076344120727629f, 0.9189578116202306f, 0.97952994125249426f};
__constant__ float k31sin[31] = {0.0f, 0.20129852008866006f, 0.39435585511331855f, 0.57126821509479231f,
    0.72479278722911988f, 0.84864425749475092f, 0.93775213214708042f, 0.98846832432811138f, 0.99871650717105276f,
    0.96807711886620429f, 0.89780453957074158f, 0.79077573693769887f, 0.65137248272222226f, 0.48530196253108104f,
    0.29936312297335804f, 0.10116832198743272f, -0.10116832198743204f, -0.29936312297335821f, -0.48530196253108082f,
    -0.65137248272222203f, -0.79077573693769865f, -0.89780453957074169f, -0.96807711886620407f, -0.99871650717105276f,
    -0.98846832432811138f, -0.93775213214708042f, -0.84864425749475103f, -0.72479278722911999f, -0.57126821509479242f,
    -0.39435585511331872f, -0.20129852008866114f};

struct Full31Dev {
    int n, m0, rb, rc;  // m0 = rb rc; column j = b rc + c
    int pc, pk;         // LDS: element (k, b, c) at k pk + b pc + c
    float inv_rb, inv_rc;
};
inline int fc31_lds_span(const Full31Dev& f) { return 32 * f.pk; }  // row 31: spare (k_full31_corr)

#define FC31_SWITCH_B(R, OP)                                \
    switch (R) {                                            \
    case 2: OP(std::integral_constant<int, 2>{}); break;    \
    case 4: OP(std::integral_constant<int, 4>{}); break;    \
    case 5: OP(std::integral_constant<int, 5>{}); break;    \
    case 6: OP(std::integral_constant<int, 6>{}); break;    \
    case 8: OP(std::integral_constant<int, 8>{}); break;    \
    case 9: OP(std::integral_constant<int, 9>{}); break;    \
    case 10: OP(std::integral_constant<int, 10>{}); break;  \
    case 16: OP(std::integral_constant<int, 16>{}); break;  \
    case 20: OP(std::integral_constant<int, 20>{}); break;  \
    case 22: OP(std::integral_constant<int, 22>{}); break;  \
    default: OP(std::integral_constant<int, 24>{}); break;  \
    }
#define FC31_SWITCH_C(R, OP)                                \
    switch (R) {                                            \
    case 3: OP(std::integral_constant<int, 3>{}); break;    \
    case 5: OP(std::integral_constant<int, 5>{}); break;    \
    case 9: OP(std::integral_constant<int, 9>{}); break;    \
    case 11: OP(std::integral_constant<int, 11>{}); break;  \
    case 15: OP(std::integral_constant<int, 15>{}); break;  \
    case 22: OP(std::integral_constant<int, 22>{}); break;  \
    case 25: OP(std::integral_constant<int, 25>{}); break;  \
    default: OP(std::integral_constant<int, 33>{}); break;  \
    }
inline bool fc31_b_ok(int r)
{
    for (int x : {2, 4, 5, 6, 8, 9, 10, 16, 20, 22, 24})
        if (r == x) return true;
    return false;
}
inline bool fc31_c_ok(int r)
{
    for (int x : {3, 5, 9, 11, 15, 22, 25, 33})
        if (r == x) return true;
    return false;
}

// DFTs along b, in place: butterfly (k, c)
template <bool INV, int NTHR>
__device__ __forceinline__ void fc31_axis_b(float2* lds, const Full31Dev& f, int tid)
{
    const int m = 31 * f.rc, pc = f.pc;
    auto op = [&](auto rcst) {
        constexpr int R = decltype(rcst)::value;
        for (int j = tid; j < m; j += NTHR) {
            int c;
            const int k = fc_divmod(j, f.rc, f.inv_rc, &c);
            float2* a = lds + k * f.pk + c;
            float2 v[R];
#pragma unroll
            for (int r = 0; r < R; r++) v[r] = a[r * pc];
            dft_reg<R, INV>(v);
#pragma unroll
            for (int r = 0; r < R; r++) a[r * pc] = v[r];
        }
    };
    FC31_SWITCH_B(f.rb, op)
}

// Forward transform of in(n) -> out(k m0 + j)
template <int NTHR, class In, class Out>
__device__ __forceinline__ void fc31_forward(float2* lds, const Full31Dev& f, int tid, const In& in, const Out& out)
{
    const float inv31 = 1.0f / 31.0f;
    for (int i = tid; i < f.n; i += NTHR) {
        int k, b, c;
        (void)fc_divmod(i, 31, inv31, &k);
        (void)fc_divmod(i, f.rb, f.inv_rb, &b);
        (void)fc_divmod(i, f.rc, f.inv_rc, &c);
        lds[k * f.pk + b * f.pc + c] = in(i);
    }
    __syncthreads();
    {
        const int m = 31 * f.rb;
        auto op = [&](auto rcst) {
            constexpr int R = decltype(rcst)::value;
            for (int j = tid; j < m; j += NTHR) {
                int b;
                const int k = fc_divmod(j, f.rb, f.inv_rb, &b);
                float2* a = lds + k * f.pk + b * f.pc;
                float2 v[R];
#pragma unroll
                for (int r = 0; r < R; r++) v[r] = a[r];
                dft_reg<R, false>(v);
#pragma unroll
                for (int r = 0; r < R; r++) a[r] = v[r];
            }
        };
        FC31_SWITCH_C(f.rc, op)
    }
    __syncthreads();
    fc31_axis_b<false, NTHR>(lds, f, tid);
    __syncthreads();
    for (int j = tid; j < f.m0; j += NTHR) {
        int c;
        const int b = fc_divmod(j, f.rc, f.inv_rc, &c);
        const float2* a = lds + b * f.pc + c;
        float2 v[31];
#pragma unroll
        for (int r = 0; r < 31; r++) v[r] = a[r * f.pk];
        dft_prime<31, false>(v, [&](auto r, float2 x) { out(r * f.m0 + j, x); });
    }
}

__global__ void __launch_bounds__(FC_FWD_NTHR)
k_full31_code(const int8_t* __restrict__ codes, float2* __restrict__ spec, Full31Dev f, int bs, int ncoh, float scale)
{
    extern __shared__ float2 lds[];
    const int w = blockIdx.x, prn = blockIdx.y, n = f.n, s = w % ncoh;
    const int8_t* c = codes + (size_t)prn * n;
    const double two_over_d = 2.0 / ((double)ncoh * n);
    float2* out = spec + ((size_t)prn * gridDim.x + w) * n;
    fc31_forward<FC_FWD_NTHR>(
        lds, f, threadIdx.x, [&](int m) { return full_code_in(c, m, w, s, bs, two_over_d); },
        [&](int i, float2 x) { out[i] = make_float2(x.x * scale, -x.y * scale); });
}
// columns of k_full31_corr's last stage: [(rc + 1) / 2][31 rb] pairs of outputs
// c = 2 i, 2 i + 1 of (k, b); the partner of an odd rc's last output is 0.
// grid (ceil(n / 256))
__global__ void __launch_bounds__(256)
k_full31_map(uint16_t* __restrict__ map, Full31Dev f, int nb, int bs)
{
    const int tau = blockIdx.x * 256 + threadIdx.x;
    if (tau >= f.n) return;
    const int c = tau % f.rc;
    uint16_t* at = map + ((size_t)(c / 2) * 31 * f.rb + (tau % 31) * f.rb + tau % f.rb) * 2;
    at[c & 1] = full_column(tau, nb, bs);
    if (c == f.rc - 1 && !(c & 1)) at[1] = 0;
}

template <int NTHR>
__global__ void __launch_bounds__(NTHR)
k_full31_signal(const void* __restrict__ sig, int eltype, float2* z, Full31Dev f, int do_if, float phase_step,
                double phase_step64)
{
    extern __shared__ float2 lds[];
    const int n = f.n;
    const int64_t seg0 = (int64_t)blockIdx.y * n;
    float2* zz = z + ((size_t)blockIdx.y * gridDim.x + blockIdx.x) * n;
    const DownconvIn in{sig, eltype, seg0, n, 0, n, do_if, __fmul_rn((float)seg0, phase_step), phase_step, phase_step64};
    const bool folded = gridDim.x > 1;
    fc31_forward<NTHR>(
        lds, f, threadIdx.x, [&](int i) { return folded ? zz[i] : in(0, i); },
        [&](int i, float2 x) { zz[i] = x; });
}

// The search, one workgroup per (Doppler row, PRN) as k_full_corr. Cells of a
// thread are columns tid + NTHR i (i < NACC, host: n <= NACC NTHR); the powers of a
// step go through LDS, over the consumed transform, to the threads that own
// their drifted columns, and stay there in registers between steps.
struct Full31Args {
    Full31Dev f;
    const float2* spec;      // [nnc][ncoh][n]
    const float2* code;      // [nprn][ndop][n]
    const uint32_t* colmap;  // [(rc + 1) / 2][31 rb] columns of outputs c = 2 i, 2 i + 1 of (k, b)
    const int32_t* shifts;
    const int32_t* req;
    float* acc;
    double* rowsum;
    float* rowbest_v;
    uint64_t* rowbest_k;
    int ncoh, ndop, nnc, cnt, ap;
};

template <int NTHR>
__global__ void __launch_bounds__(NTHR)
__attribute__((amdgpu_waves_per_eu(2))) k_full31_corr(Full31Args A)
{
    constexpr int NACC = NTHR == 256 ? 24 : 32;
    extern __shared__ float2 lds[];
    typedef float v4f __attribute__((ext_vector_type(4)));
    const Full31Dev& f = A.f;
    const int tid = threadIdx.x, n = f.n, m0 = f.m0;
    const int lbk = xcd_logical_block();
    const int p = __builtin_amdgcn_readfirstlane(lbk % A.cnt);
    const int wi = __builtin_amdgcn_readfirstlane(lbk / A.cnt);
    const int nb = A.ndop / A.ncoh, s = wi / nb, w = s + A.ncoh * (wi - s * nb);
    int row = w + A.ndop / 2;
    if (row >= A.ndop) row -= A.ndop;
    const float2* G = A.code + ((size_t)A.req[p] * A.ndop + w) * n;
    // matrix operands of the 31-point DFT: row l & 15, K index 4 t + (l >> 4)
    const int lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6), l16 = lane & 15, g = lane >> 4;
    float ca[4], sa[4];
#pragma unroll
    for (int t = 0; t < 4; t++) {
        const int e = (l16 * (4 * t + g)) % 31;
        ca[t] = k31cos[e];
        sa[t] = k31sin[e];
    }
    // columns of this thread's last-stage outputs, two to a word
    uint32_t cm[17];
    {
        const int m = 31 * f.rb;
#pragma unroll
        for (int i = 0; i < 17; i++)
            cm[i] = 2 * i < f.rc ? A.colmap[(size_t)i * m + min(tid, m - 1)] : 0u;
    }
    float acc[NACC];
#pragma unroll
    for (int i = 0; i < NACC; i++) acc[i] = 0.f;
    // A wave's groups of 32 columns of the spectra: rows r = 4 t + g and their
    // partners 31 - r (row 0 has none), columns 2 l16 and 2 l16 + 1 per lane as
    // one 16-byte load; the even and the odd columns are one 16-column tile
    // each. The code spectra come from beyond L2 (about 2400 cycles): a group's
    // loads go out when the previous one's registers are consumed, the first
    // one's before the previous step's accumulation. Loaded where used, this
    // stage took 37000 cycles per transform at 16368 points. A group's lanes
    // beyond m0 read the next row's values (host: 32 elements behind the
    // arrays) and are dropped.
    typedef float f4u __attribute__((ext_vector_type(4), aligned(8)));
    struct Group {
        f4u zx[4], zy[4], gx[4], gy[4];
    };
    constexpr int GSTEP = NTHR / 2;  // columns of the workgroup's waves
    uint32_t vx[4], vy[4];
#pragma unroll
    for (int t = 0; t < 4; t++) {
        const int r = 4 * t + g;
        vx[t] = (uint32_t)(r * m0 + 2 * l16) * (uint32_t)sizeof(float2);
        vy[t] = (uint32_t)((r ? 31 - r : 0) * m0 + 2 * l16) * (uint32_t)sizeof(float2);
    }
    Group ga;
    auto load_group = [&](Group& o, const float2* Zs, int j0) {
        const char* zb = (const char*)(Zs + j0);
        const char* cb = (const char*)(G + j0);
#pragma unroll
        for (int t = 0; t < 4; t++) {
            o.gx[t] = *(const f4u*)(cb + vx[t]);
            o.gy[t] = *(const f4u*)(cb + vy[t]);
            o.zx[t] = *(const f4u*)(zb + vx[t]);
            o.zy[t] = *(const f4u*)(zb + vy[t]);
        }
    };
    const int w0 = wave * 32;
    auto load_first = [&](const float2* Zs) {
#pragma unroll
        for (int t = 0; t < 4; t++) {
            vx[t] = fc_opaque(vx[t]);  // or the addresses of the code spectra stay in registers
            vy[t] = fc_opaque(vy[t]);
        }
        load_group(ga, Zs, w0 < m0 ? w0 : 0);  // a wave with no group: any columns
    };
    load_first(A.spec + (size_t)s * n);
    for (int step = 0; step < A.nnc; step++) {
        const float2* Z = A.spec + ((size_t)step * A.ncoh + s) * n;
        // E and O of half h of a group (matrix operands), the products, and the
        // outputs. The two waves of a SIMD run this stage in step, so a wave has
        // to fill its own matrix cycles: a half's products are interleaved with
        // the previous half's outputs. In sequence, matrix and vector time added
        // up (10000 cycles; 5300 without the products).
        struct Half {
            float2 e[4], o[4];
            v4f er, ei, orr, oi;
        };
        auto operands = [&](const Group& in, int h, Half& u) {
#pragma unroll
            for (int t = 0; t < 4; t++) {
                const float2 x = cmulf(make_float2(in.zx[t][2 * h], in.zx[t][2 * h + 1]),
                                       make_float2(in.gx[t][2 * h], in.gx[t][2 * h + 1]));
                float2 y = cmulf(make_float2(in.zy[t][2 * h], in.zy[t][2 * h + 1]),
                                 make_float2(in.gy[t][2 * h], in.gy[t][2 * h + 1]));
                if (t == 0) y = make_float2(g ? y.x : 0.f, g ? y.y : 0.f);
                u.e[t] = caddf(x, y);
                u.o[t] = csubf(x, y);
                if (t == 0) u.o[t] = make_float2(g ? u.o[t].x : 0.f, g ? u.o[t].y : 0.f);
            }
        };
        auto products = [&](Half& u) {
            u.er = u.ei = u.orr = u.oi = v4f{};
#pragma unroll
            for (int t = 0; t < 4; t++) {
                u.er = __builtin_amdgcn_mfma_f32_16x16x4f32(ca[t], u.e[t].x, u.er, 0, 0, 0);
                u.ei = __builtin_amdgcn_mfma_f32_16x16x4f32(ca[t], u.e[t].y, u.ei, 0, 0, 0);
                u.orr = __builtin_amdgcn_mfma_f32_16x16x4f32(sa[t], u.o[t].x, u.orr, 0, 0, 0);
                u.oi = __builtin_amdgcn_mfma_f32_16x16x4f32(sa[t], u.o[t].y, u.oi, 0, 0, 0);
            }
        };
        // a b (Y_k) and its mirror (Y_(31-k)), k = 4 g + r; columns beyond m0 go to
        // the pitch's spare slots, Y_31 of k = 0 to the spare row 31: no branches
        auto outputs = [&](const Half& u, int jj) {
            int c;
            const int b = fc_divmod(jj, f.rc, f.inv_rc, &c);
            const int col = jj < m0 ? b * f.pc + c : f.pk - 1;
            float2* up = lds + col + 4 * g * f.pk;
            float2* dn = lds + col + (31 - 4 * g) * f.pk;
#pragma unroll
            for (int r = 0; r < 4; r++) {  // inverse: a + i b and a - i b
                up[r * f.pk] = make_float2(u.er[r] - u.oi[r], u.ei[r] + u.orr[r]);
                dn[-r * f.pk] = make_float2(u.er[r] + u.oi[r], u.ei[r] - u.orr[r]);
            }
        };
        auto interleave = [&] {  // one matrix product, seven vector instructions, one LDS store
#pragma unroll
            for (int i = 0; i < 16; i++) {
                __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
                __builtin_amdgcn_sched_group_barrier(0x002, 7, 0);
                __builtin_amdgcn_sched_group_barrier(0x200, 1, 0);
            }
            fc_issued();
        };
        {
            Half u0, u1, last;
            last.er = last.ei = last.orr = last.oi = v4f{};
            int jl = m0;  // no outputs yet: the spare slots
#pragma unroll 1
            for (int j0 = w0; j0 < m0; j0 += GSTEP) {
                const int jj = j0 + 2 * fc_opaque(l16);
                operands(ga, 0, u0);
                operands(ga, 1, u1);
                fc_issued();
                load_group(ga, Z, j0 + GSTEP < m0 ? j0 + GSTEP : 0);
                products(u0);
                outputs(last, jl);
                interleave();
                products(u1);
                outputs(u0, jj);
                interleave();
                last.er = u1.er;
                last.ei = u1.ei;
                last.orr = u1.orr;
                last.oi = u1.oi;
                jl = jj + 1;
            }
            outputs(last, jl);
        }
        __syncthreads();
        fc31_axis_b<true, NTHR>(lds, f, fc_opaque(tid));
        __syncthreads();
        // DFTs along c; one butterfly (k, b) per thread (31 rb <= NTHR)
        const uint32_t shift = (uint32_t)A.shifts[(size_t)step * A.ndop + row];
        float* pws = (float*)lds;
        {
            const int m = 31 * f.rb, q = fc_opaque(tid);
            auto op = [&](auto rcst) {
                constexpr int R = decltype(rcst)::value;
                float2 v[R];
                if (q < m) {
                    int b;
                    const int k = fc_divmod(q, f.rb, f.inv_rb, &b);
                    const float2* a = lds + k * f.pk + b * f.pc;
#pragma unroll
                    for (int r = 0; r < R; r++) v[r] = a[r];
                }
                __syncthreads();
                if (q < m) {
                    dft_reg<R, true>(v);
#pragma unroll
                    for (int r = 0; r < R; r++) {
                        const uint32_t c = ((cm[r >> 1] >> (16 * (r & 1))) & 0xffffu) + shift;
                        pws[min(c, c - (uint32_t)n)] = abs2_exact(v[r]);  // drifted column mod n
                    }
                }
            };
            FC31_SWITCH_C(f.rc, op)
        }
        __syncthreads();
        // the next step's first tiles, behind the accumulation
        load_first(step + 1 < A.nnc ? Z + (size_t)A.ncoh * n : Z);
        fc_accumulate<NTHR, NACC>(acc, pws, n, step == 0);
        __syncthreads();
    }
    double sum = 0.0;
    float bv = -INFINITY;
    int bc = 0x7fffffff;
    fc_store_cells<NTHR, NACC>(acc, A.acc + ((size_t)p * A.ndop + row) * A.ap, n, sum, bv, bc);
    full_row_reduce<NTHR>(lds, sum, bv, bc, A.rowsum, A.rowbest_v, A.rowbest_k, (size_t)p * A.ndop, row, A.ndop);
}
