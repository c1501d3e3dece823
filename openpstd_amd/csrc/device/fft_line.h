// Register/LDS Stockham FFT building blocks for the line-derivative kernels (gfx950).
//
// A "line pair" is two real lines packed as one complex sequence
// z = x1 + i*x2 of length F (F a power of two, 128..8192).  T threads work on one
// pair; thread t holds the V = F/T elements t + m*T (m = 0..V-1) in registers
// ("natural layout") at the start and end of the transform.  A Stockham radix-R
// pass (R in {2, 4, 8}; the first and the last are radix 8) does V/R butterflies
// per thread and exchanges through LDS; the last one leaves natural layout
// without touching LDS.  Only the forward transform exists: the inverse is the
// conjugate of the forward transform of the conjugate (the same roundings), so
// one piece of code runs twice (it is straight-line and long).
//
// V = 16 from F = 1024 on, in launches of many wavefronts: a 1024-point pair fits one
// wavefront (no workgroup barrier in its tile), the butterflies of a thread share
// their twiddles in the passes of span <= T, and address, halo and update work is
// shared by twice the values.  V = 8 up to 512 points, and for 1024 and 2048 points in
// launches of few wavefronts (the caller's choice): these are bound by one
// wavefront's instruction stream, which is half as long.  V changes no result: which
// values a butterfly combines depends on F alone.  One LDS buffer per pair
// (17/16 F complex values): 16 wavefronts fit a CU.
#pragma once

#include <hip/hip_runtime.h>

namespace pstdamd {
namespace dev {

__device__ __forceinline__ float2 cadd(float2 a, float2 b) { return make_float2(a.x + b.x, a.y + b.y); }
__device__ __forceinline__ float2 csub(float2 a, float2 b) { return make_float2(a.x - b.x, a.y - b.y); }
// Explicit FMAs (the device code is built without implicit contraction, so
// the rounding is the same in every instantiation).
__device__ __forceinline__ float2 cmul(float2 a, float2 b) {
    return make_float2(__builtin_fmaf(a.x, b.x, -(a.y * b.y)), __builtin_fmaf(a.x, b.y, a.y * b.x));
}
// multiply by -i, by exp(-i pi/4)
__device__ __forceinline__ float2 mul_i(float2 a) { return make_float2(a.y, -a.x); }
__device__ __forceinline__ float2 mul_8(float2 a) {
    const float c = 0.70710678118654752440f;
    return make_float2(c * (a.x + a.y), c * (a.y - a.x));
}

__device__ __forceinline__ void dft2(float2 &a0, float2 &a1) {
    float2 t = a0;
    a0 = cadd(t, a1);
    a1 = csub(t, a1);
}

__device__ __forceinline__ void dft4(float2 &a0, float2 &a1, float2 &a2, float2 &a3) {
    float2 t0 = cadd(a0, a2), t1 = csub(a0, a2), t2 = cadd(a1, a3), t3 = mul_i(csub(a1, a3));
    a0 = cadd(t0, t2);
    a2 = csub(t0, t2);
    a1 = cadd(t1, t3);
    a3 = csub(t1, t3);
}

__device__ __forceinline__ void dft8(float2 *a) {
    // even/odd split: E = DFT4(a0,a2,a4,a6), O = DFT4(a1,a3,a5,a7)
    dft4(a[0], a[2], a[4], a[6]);
    dft4(a[1], a[3], a[5], a[7]);
    const float2 w1 = mul_8(a[3]), w2 = mul_i(a[5]), w3 = mul_i(mul_8(a[7]));
    const float2 e0 = a[0], e1 = a[2], e2 = a[4], e3 = a[6], o0 = a[1];
    a[0] = cadd(e0, o0);
    a[4] = csub(e0, o0);
    a[1] = cadd(e1, w1);
    a[5] = csub(e1, w1);
    a[2] = cadd(e2, w2);
    a[6] = csub(e2, w2);
    a[3] = cadd(e3, w3);
    a[7] = csub(e3, w3);
}

template <int R>
__device__ __forceinline__ void dft(float2 *a) {
    if constexpr (R == 2) dft2(a[0], a[1]);
    else if constexpr (R == 4) dft4(a[0], a[1], a[2], a[3]);
    else dft8(a);
}

// Values per thread (1024 and 2048 points: or 8, fft_run's V); pass schedule: radix of
// pass p for length F <= 4096.  An
// 8192-point pair is two 4096-point sequences (split_first), each with 8 values
// per thread: T = 512, 16 values in all.
__host__ __device__ constexpr int fft_values(int F) { return F <= 512 ? 8 : 16; }
__host__ __device__ constexpr int fft_npasses(int F) { return F <= 512 ? 3 : 4; }
__host__ __device__ constexpr int fft_radix(int F, int p) {
    return (p == 0 || p == fft_npasses(F) - 1) ? 8
           : F == 128  ? 2
           : F == 256  ? 4
           : F == 512  ? 8
           : F == 1024 ? 4
           : F == 2048 ? (p == 1 ? 8 : 4)
                       : 8;
}
__host__ __device__ constexpr int fft_span(int F, int p) {  // product of radices before pass p
    return p == 0 ? 1 : fft_span(F, p - 1) * fft_radix(F, p - 1);
}
// The twiddle table of length F <= 4096: for every pass p >= 1 the factors
// exp(-2 pi i r k / (span * radix)) as [r / 2][k = 0 .. span-1][r % 2] (r = 0: 1,
// unused).  A wavefront's lanes (consecutive k) read two factors each with one
// 16-byte load, 64 bytes a cycle from the L1; an 8-byte load moves 32 and the
// table reads then cost more L1 cycles than the lines do (16 sources of 512 x 1024
// twice: 414 us per stage with 8-byte loads, 369 with 16-byte ones).
// Length 8192: the table of 4096, then exp(-2 pi i n / 8192), n = t + 512 m < 4096,
// as [m / 2][t][m % 2].
__host__ __device__ constexpr int fft_tw_base(int F, int p) {
    return p <= 1 ? 0 : fft_tw_base(F, p - 1) + fft_radix(F, p - 1) * fft_span(F, p - 1);
}
__host__ __device__ constexpr int fft_tw_size(int F) { return fft_tw_base(F, fft_npasses(F)); }

// LDS slot of element idx of a pair: one pad slot per 16 elements.  The first
// pass writes elements 8 t + r: without the pad every lane of a wavefront
// would be on the same banks.
__host__ __device__ constexpr int lds_slot(int idx) { return idx + (idx >> 4); }
// Distance of the pairs' buffers: four slots more, so that the same element of
// four neighbouring pairs lies on different banks.
__host__ __device__ constexpr int lds_pitch(int F) { return lds_slot(F) + 4; }

// A table of complex values in memory: lane offset and uniform offset in bytes.
struct Table {
    __amdgpu_buffer_rsrc_t r;
    // two consecutive values
    __device__ __forceinline__ void pair(float2 &a, float2 &b, int lane, int uniform) const {
        const float4 x = __builtin_bit_cast(float4, __builtin_amdgcn_raw_buffer_load_b128(r, lane, uniform, 0));
        a = make_float2(x.x, x.y);
        b = make_float2(x.z, x.w);
    }
};

// Twiddles of one pass for thread t: one set of R factors for all of its V/R
// butterflies where the span divides T (j mod span = t mod span), otherwise one
// each (span = T V/R, the last pass).
constexpr int kTwPass = 16;
template <int F, int T, int PASS>
__device__ __forceinline__ void fft_pass_twiddles(float2 (&w)[kTwPass], int t, const Table &tab, int tw) {
    if constexpr (PASS >= 1 && PASS < fft_npasses(F)) {
        constexpr int R = fft_radix(F, PASS), NS = fft_span(F, PASS), sets = NS <= T ? 1 : NS / T;
        constexpr int base = fft_tw_base(F, PASS);
        static_assert(sets * R <= kTwPass, "twiddle registers");
        const int k = t & ((NS <= T ? NS : T) - 1);
#pragma unroll
        for (int s = 0; s < sets; ++s)
#pragma unroll
            for (int r = 0; r < R; r += 2)
                tab.pair(w[s * R + r], w[s * R + r + 1], k * 16, tw + (base + r * NS + 2 * s * T) * 8);
    }
}

// One Stockham pass on natural-layout registers.  Non-last passes write their
// outputs to `lds` (the sequence's buffer); the last one leaves them in v.
template <int F, int T, int PASS>
__device__ __forceinline__ void fft_pass(float2 *v, int t, float2 *lds, const float2 (&w)[kTwPass]) {
    constexpr int V = F / T, R = fft_radix(F, PASS), NS = fft_span(F, PASS), NB = V / R;
#pragma unroll
    for (int s = 0; s < NB; ++s) {
        float2 a[R];
#pragma unroll
        for (int r = 0; r < R; ++r) a[r] = v[s + r * NB];
        if constexpr (PASS > 0) {
#pragma unroll
            for (int r = 1; r < R; ++r) a[r] = cmul(a[r], w[(NS <= T ? 0 : s * R) + r]);
        }
        dft<R>(a);
        if constexpr (PASS == fft_npasses(F) - 1) {
#pragma unroll
            for (int r = 0; r < R; ++r) v[s + r * NB] = a[r];
        } else {
            const int j = t + s * T, k = j & (NS - 1), base = (j - k) * R + k;
            const int at = lds_slot(base);
            // slot(base + r NS) - slot(base): NS = 1 and base a multiple of 8 (no pad lies
            // between), NS = 8 and base = k < 8 mod 16, or NS a multiple of 16
#pragma unroll
            for (int r = 0; r < R; ++r) lds[at + r * NS + ((r * NS) >> 4)] = a[r];
        }
    }
}

// Exchange point.  Pairs of up to 64 threads lie inside one wavefront and own
// their LDS slots; the LDS executes one wavefront's accesses in issue order, so a
// compiler fence is enough.  Longer ones synchronise the workgroup.
template <int T>
__device__ __forceinline__ void pass_sync() {
    if constexpr (T <= 64) __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
    else __syncthreads();
}

// Full forward transform, natural layout in and out, of SETS sequences of F points
// (v: V values of each; LDS buffers lds_slot(F) apart).  The twiddles of each pass
// are loaded one pass ahead: in flight while the pass before computes and
// exchanges.  Every thread of the block calls it (T > 64 synchronises).
template <int F, int T, int SETS, int PASS>
__device__ __forceinline__ void fft_passes(float2 *v, int t, float2 *lds, const Table &tab, int tw,
                                           const float2 (&wcur)[kTwPass]) {
    constexpr int V = F / T, NP = fft_npasses(F);
    float2 wnext[kTwPass];
    if constexpr (PASS + 1 < NP) fft_pass_twiddles<F, T, PASS + 1>(wnext, t, tab, tw);
    if constexpr (PASS + 1 < NP) pass_sync<T>();  // what the slots held before has been read
#pragma unroll
    for (int q = 0; q < SETS; ++q) fft_pass<F, T, PASS>(v + q * V, t, lds + q * lds_slot(F), wcur);
    if constexpr (PASS + 1 < NP) {
        pass_sync<T>();
        const int at = lds_slot(t);
        // slot(t + m T): T is a multiple of 16
#pragma unroll
        for (int q = 0; q < SETS; ++q)
#pragma unroll
            for (int m = 0; m < V; ++m) v[q * V + m] = lds[q * lds_slot(F) + at + m * T + ((m * T) >> 4)];
        fft_passes<F, T, SETS, PASS + 1>(v, t, lds, tab, tw, wnext);
    }
}

template <int F, int V>
__device__ __forceinline__ void fft_run(float2 *v, int t, float2 *lds, const Table &tab, int tw) {
    const float2 w0[kTwPass] = {};
    if constexpr (F == 8192) fft_passes<4096, 512, 2, 0>(v, t, lds, tab, tw, w0);
    else fft_passes<F, F / V, 1, 0>(v, t, lds, tab, tw, w0);
}

// 8192 points as two sequences of 4096: with W = exp(-2 pi i / 8192), the even bins
// are the transform of z[n] + z[n + 4096], the odd ones that of (z[n] - z[n + 4096])
// W^n; n = t + 512 m, values m and m + 8 of the thread.  The inverse recombines
// y[n], y[n + 4096] = e[n] +- W^-n o[n] in the same threads (on conjugates: W^n).
__device__ __forceinline__ void split_first(float2 (&v)[16], int t, const Table &tab, int tw) {
#pragma unroll
    for (int m = 0; m < 8; m += 2) {
        float2 w[2];
        tab.pair(w[0], w[1], t * 16, tw + (fft_tw_size(4096) + m * 512) * 8);
#pragma unroll
        for (int q = 0; q < 2; ++q) {
            const float2 x = v[m + q], y = v[m + q + 8];
            v[m + q] = cadd(x, y);
            v[m + q + 8] = cmul(csub(x, y), w[q]);
        }
    }
}
__device__ __forceinline__ void split_last(float2 (&v)[16], int t, const Table &tab, int tw) {
#pragma unroll
    for (int m = 0; m < 8; m += 2) {
        float2 w[2];
        tab.pair(w[0], w[1], t * 16, tw + (fft_tw_size(4096) + m * 512) * 8);
#pragma unroll
        for (int q = 0; q < 2; ++q) {
            const float2 e = v[m + q], o = cmul(v[m + q + 8], w[q]);
            v[m + q] = cadd(e, o);
            v[m + q + 8] = csub(e, o);
        }
    }
}

}  // namespace dev
}  // namespace pstdamd
