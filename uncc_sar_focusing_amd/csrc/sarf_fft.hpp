// sarf_fft.hpp -- register/LDS building blocks of the power-of-two FFTs
// (range compression, PGA row transforms): radix-2 DIF networks on up to 16
// registers with exact trivial rotations, and a self-sorting Stockham
// transform of length N = 2^LOG2N by N/16 lanes (16 values per lane, radix-16
// passes through a padded LDS row).
#pragma once

#include "sarf_cis.hpp"
#include "sarf_internal.hpp"

namespace sarf {
namespace fft {

// cos(2 pi m / 16) for m = 0..15; sin(x) is cos(x - pi/2).
template <int M>
struct Tw16 {
    static constexpr double c() {
        constexpr double t[16] = {1.0, 0.92387953251128674, 0.70710678118654752,
                                  0.38268343236508978, 0.0, -0.38268343236508978,
                                  -0.70710678118654752, -0.92387953251128674, -1.0,
                                  -0.92387953251128674, -0.70710678118654752,
                                  -0.38268343236508978, 0.0, 0.38268343236508978,
                                  0.70710678118654752, 0.92387953251128674};
        return t[M & 15];
    }
    static constexpr double s() { return Tw16<(M + 12) & 15>::c(); }  // sin x = cos(x - pi/2)
};

__device__ __forceinline__ float2 complex_of(float x, float y) { return make_float2(x, y); }
__device__ __forceinline__ double2 complex_of(double x, double y) { return make_double2(x, y); }

// d * e^{SIGN j 2 pi M / 16}, with the trivial rotations done exactly
// (T2 = float2 or double2).
template <int SIGN, int M, typename T2>
__device__ __forceinline__ T2 rot16(T2 d) {
    constexpr int m = M & 15;
    if constexpr (m == 0) {
        return d;
    } else if constexpr (m == 8) {
        return complex_of(-d.x, -d.y);
    } else if constexpr (m == 4) {  // e^{SIGN j pi/2} = SIGN j
        return SIGN > 0 ? complex_of(-d.y, d.x) : complex_of(d.y, -d.x);
    } else if constexpr (m == 12) {
        return SIGN > 0 ? complex_of(d.y, -d.x) : complex_of(-d.y, d.x);
    } else {
        using Re = decltype(T2{}.x);
        constexpr Re c = (Re)Tw16<m>::c();
        constexpr Re s = (Re)(SIGN * Tw16<m>::s());
        return complex_of(d.x * c - d.y * s, d.x * s + d.y * c);
    }
}

// Radix-2 decimation-in-frequency network on R registers (R = 2,4,8,16),
// natural-order input, bit-reversed output.
template <int SIGN, int L, int S, int K>
struct DifBfly {
    template <typename T2>
    static __device__ __forceinline__ void run(T2 *v) {
        if constexpr (K < L / 2) {
            T2 a = v[S + K], b = v[S + K + L / 2];
            v[S + K] = cadd(a, b);
            v[S + K + L / 2] = rot16<SIGN, (K * 16 / L)>(csub(a, b));
            DifBfly<SIGN, L, S, K + 1>::run(v);
        }
    }
};
template <int SIGN, int R, int L, int S>
struct DifStage {
    template <typename T2>
    static __device__ __forceinline__ void run(T2 *v) {
        if constexpr (S < R) {
            DifBfly<SIGN, L, S, 0>::run(v);
            DifStage<SIGN, R, L, S + L>::run(v);
        }
    }
};
template <int SIGN, int R, int L>
struct DifAll {
    template <typename T2>
    static __device__ __forceinline__ void run(T2 *v) {
        if constexpr (L >= 2) {
            DifStage<SIGN, R, L, 0>::run(v);
            DifAll<SIGN, R, L / 2>::run(v);
        }
    }
};
template <int R>
__host__ __device__ constexpr int bitrev(int x) {
    int r = 0;
    for (int b = 1; b < R; b <<= 1) {
        r = (r << 1) | (x & 1);
        x >>= 1;
    }
    return r;
}

// In-place R-point DFT (sign SIGN) of v[0..R-1], result in natural order.
template <int SIGN, int R, typename T2>
__device__ __forceinline__ void dft(T2 *v) {
    DifAll<SIGN, R, R>::run(v);
    T2 t[R];
#pragma unroll
    for (int i = 0; i < R; i++) t[i] = v[bitrev<R>(i)];
#pragma unroll
    for (int i = 0; i < R; i++) v[i] = t[i];
}

// cos(2 pi m / 16) less its value rounded to FP64, for m = 1, 2, 3.
template <int M>
constexpr double cos16_rest() {
    constexpr int m = M & 15, f = m > 8 ? 16 - m : m, q = f > 4 ? 8 - f : f;
    constexpr double t[5] = {0.0, 1.764504708433667706e-17, -4.833646656726456726e-17,
                             -1.00507726964615876e-17, 0.0};
    return f > 4 ? -t[q] : t[q];
}

__device__ __forceinline__ float madd(float a, float b, float c) { return fmaf(a, b, c); }
__device__ __forceinline__ double madd(double a, double b, double c) { return fma(a, b, c); }

// rot16<+1, M> with cosine and sine in two parts.  Rounded to FP32, the three
// constants are all too small, by 1.2e-8 to 2.8e-8, so that every 16-point step
// shrinks its results: a transform of 2^16, which has four of them, by 5e-8.
template <int M, typename T2>
__device__ __forceinline__ T2 rot16_split(T2 d) {
    constexpr int m = M & 15;
    if constexpr (m % 4 == 0) {
        return rot16<+1, m>(d);
    } else {
        using Re = decltype(T2{}.x);
        constexpr double C = Tw16<m>::c(), S = Tw16<m>::s();
        constexpr Re c = (Re)C, s = (Re)S;
        constexpr Re cl = (Re)((C - (double)c) + cos16_rest<m>());
        constexpr Re sl = (Re)((S - (double)s) + cos16_rest<m + 12>());
        return complex_of(madd(d.x, c, madd(-d.y, s, madd(d.x, cl, -d.y * sl))),
                          madd(d.x, s, madd(d.y, c, madd(d.x, sl, d.y * cl))));
    }
}

template <typename T2>
__device__ __forceinline__ void idft4(T2 &v0, T2 &v1, T2 &v2, T2 &v3) {
    const T2 a = cadd(v0, v2), b = csub(v0, v2), c = cadd(v1, v3), d = rot16<+1, 4>(csub(v1, v3));
    v0 = cadd(a, c);
    v1 = cadd(b, d);
    v2 = csub(a, c);
    v3 = csub(b, d);
}

// In-place R-point inverse DFT, natural order in and out, with the fewest
// roundings: radix 4 (one rotation per 16 points where radix 2 has two) and
// rot16_split.  Transforms of 2^16 samples in FP32: rel-L2 1.23e-7 of this and
// cis_rev, 1.39e-7 of dft<+1, R>, 1.28e-7 of radix-4 passes with table twiddles.
template <int R, typename T2>
__device__ __forceinline__ void idft_split(T2 *v) {
    static_assert(R == 2 || R == 4 || R == 8 || R == 16, "radix");
    if constexpr (R == 2) {
        const T2 a = v[0], b = v[1];
        v[0] = cadd(a, b);
        v[1] = csub(a, b);
    } else if constexpr (R == 4) {
        idft4(v[0], v[1], v[2], v[3]);
    } else if constexpr (R == 8) {
        T2 o[4];
#pragma unroll
        for (int i = 0; i < 4; i++) {
            o[i] = csub(v[i], v[i + 4]);
            v[i] = cadd(v[i], v[i + 4]);
        }
        o[1] = rot16_split<2>(o[1]);
        o[2] = rot16_split<4>(o[2]);
        o[3] = rot16_split<6>(o[3]);
        idft4(v[0], v[1], v[2], v[3]);
        idft4(o[0], o[1], o[2], o[3]);
        v[6] = v[3];
        v[4] = v[2];
        v[2] = v[1];
#pragma unroll
        for (int i = 0; i < 4; i++) v[2 * i + 1] = o[i];
    } else {
#pragma unroll
        for (int i = 0; i < 4; i++) idft4(v[i], v[i + 4], v[i + 8], v[i + 12]);
        v[5] = rot16_split<1>(v[5]);
        v[9] = rot16_split<2>(v[9]);
        v[13] = rot16_split<3>(v[13]);
        v[6] = rot16_split<2>(v[6]);
        v[10] = rot16_split<4>(v[10]);
        v[14] = rot16_split<6>(v[14]);
        v[7] = rot16_split<3>(v[7]);
        v[11] = rot16_split<6>(v[11]);
        v[15] = rot16_split<9>(v[15]);
#pragma unroll
        for (int i = 0; i < 4; i++) idft4(v[4 * i], v[4 * i + 1], v[4 * i + 2], v[4 * i + 3]);
        T2 t[16];
#pragma unroll
        for (int i = 0; i < 16; i++) t[i] = v[4 * (i & 3) + (i >> 2)];
#pragma unroll
        for (int i = 0; i < 16; i++) v[i] = t[i];
    }
}

__device__ __forceinline__ int lpad(int i) { return i + (i >> 4); }

// e^{j 2 pi r rev} for r = 1..15 from the sine/cosine unit, which takes
// revolutions (rev = k / (Ns 16) is exact, so each twiddle is one rounding
// of the unit, about 1e-7).
__device__ __forceinline__ void powers16_rev(float rev, float2 *p) {
#pragma unroll
    for (int r = 1; r < 16; r++) {
        const float a = rev * (float)r;
        p[r] = make_float2(__builtin_amdgcn_cosf(a), __builtin_amdgcn_sinf(a));
    }
}

// w^r for r = 0..15 from w (r = 0 unused); error <= ~4 roundings.
__device__ __forceinline__ void powers16(float2 w, float2 *p) {
    p[1] = w;
    p[2] = cmul(w, w);
    p[3] = cmul(p[2], w);
    p[4] = cmul(p[2], p[2]);
    p[5] = cmul(p[4], w);
    p[6] = cmul(p[4], p[2]);
    p[7] = cmul(p[4], p[3]);
    p[8] = cmul(p[4], p[4]);
#pragma unroll
    for (int r = 9; r < 16; r++) p[r] = cmul(p[8], p[r - 8]);
}

// Pass twiddles of a length-2^LOG2N transform for k = j mod Ns.  Up to 2^13
// from the sine/cosine unit: measured on MI355X, a batch of range
// compressions at 2^11-2^13 points ran 7 % faster and single ones as fast,
// with rel-L2 against FP64 of 1.5-2.2e-7 instead of 2.9-3.6e-7.  At 2^14 and
// above from the table entry w = tw[k N / (Ns 16)] and its products
// (powers16), which measured faster there (2^14: 0.191 against 0.196 ms for
// 4096 x 2048 -> 16384).
template <int LOG2N>
__device__ __forceinline__ void pass_twiddles(const float2 *__restrict__ tw, int k, int Ns,
                                              float2 *p) {
    constexpr int N = 1 << LOG2N;
    if constexpr (LOG2N <= 13) {
        powers16_rev((float)k / (float)(Ns * 16), p);
    } else {
        powers16(tw[k * (N / (Ns * 16))], p);
    }
}


// Lanes and workgroup size of a transform of length 2^log2n: N/16 lanes per
// row, rows packed so a workgroup has at least 256 lanes.
constexpr int lanes(int log2n) { return (1 << log2n) / 16; }
constexpr int rows_per_group(int log2n) { return lanes(log2n) >= 256 ? 1 : 256 / lanes(log2n); }
constexpr int group_threads(int log2n) { return lanes(log2n) * rows_per_group(log2n); }
constexpr int padded(int log2n) { return (1 << log2n) + (1 << log2n) / 16; }

// First-pass radix and butterflies per lane of a length-2^LOG2N transform.
template <int LOG2N>
struct Shape {
    static constexpr int N = 1 << LOG2N;
    static constexpr int T = N / 16;
    static constexpr int B = LOG2N % 4;
    static constexpr int R0 = B == 0 ? 16 : (1 << B);
    static constexpr int NB0 = 16 / R0;
    static constexpr int NPASS16 = (LOG2N - (B == 0 ? 4 : B)) / 4;
    static_assert(LOG2N >= 5, "at least one radix-16 pass after the first");
};

// Unnormalised inverse transform (e^{+j 2 pi k m / N}) of one row by its T
// lanes (lane j < T), through the row's padded LDS buffer L (padded(LOG2N)
// float2).  tw[t] = e^{+j 2 pi t / N}.
//   in:  v[b*R0 + r] = x[j + b*T + r*(N/R0)]  (b < NB0, r < R0)
//   out: v[r]        = X[j + r*T]             (r < 16)
// Starts with a barrier, so the caller may have just read L; every thread
// of the workgroup must call it.  The forward transform is conj(ifft(conj)).
// With active = false a thread only takes part in the barriers (for a
// workgroup wider than the row's T lanes); its v is left unchanged.  SPLIT: by
// idft_split.
template <int LOG2N, bool SPLIT = false>
__device__ __forceinline__ void ifft_regs(float2 (&v)[16], float2 *L, int j,
                                          const float2 *__restrict__ tw, bool active = true) {
    using S = Shape<LOG2N>;
    constexpr int N = S::N, T = S::T, R0 = S::R0, NB0 = S::NB0;
    __syncthreads();
    if (active) {
#pragma unroll
        for (int b = 0; b < NB0; b++) {
            const int jb = j + b * T;
            if constexpr (SPLIT) idft_split<R0>(v + b * R0);
            else dft<+1, R0>(v + b * R0);
#pragma unroll
            for (int r = 0; r < R0; r++) L[lpad(jb * R0 + r)] = v[b * R0 + r];
        }
    }
    __syncthreads();
    int Ns = R0;
#pragma unroll
    for (int pass = 0; pass < S::NPASS16; pass++) {
        const bool last = (pass == S::NPASS16 - 1);
        const int k = j & (Ns - 1);
        if (active) {
#pragma unroll
            for (int r = 0; r < 16; r++) v[r] = L[lpad(j + r * (N / 16))];
            if (k != 0) {
                float2 p[16];
                pass_twiddles<LOG2N>(tw, k, Ns, p);
#pragma unroll
                for (int r = 1; r < 16; r++) v[r] = cmul(v[r], p[r]);
            }
            if constexpr (SPLIT) idft_split<16>(v);
            else dft<+1, 16>(v);
        }
        if (!last) {
            __syncthreads();  // every lane has read before anyone overwrites
            if (active) {
                const int base = (j - k) * 16 + k;
#pragma unroll
                for (int r = 0; r < 16; r++) L[lpad(base + r * Ns)] = v[r];
            }
            __syncthreads();
        }
        Ns *= 16;
    }
}

// Natural-order output of ifft_regs (u[r] = X[j + r*T]) rearranged into the
// pass-0 input order of the next transform of the same length.
template <int LOG2N>
__device__ __forceinline__ void to_input_order(const float2 (&u)[16], float2 (&v)[16]) {
    using S = Shape<LOG2N>;
#pragma unroll
    for (int b = 0; b < S::NB0; b++)
#pragma unroll
        for (int r = 0; r < S::R0; r++) v[b * S::R0 + r] = u[b + r * S::NB0];
}

}  // namespace fft
}  // namespace sarf
