// sarf_mf.hip -- matched-filter image formation.
//
// Semantics of run_mf / computeDifferentialRangeAndPhaseCorrectionsMF
// (src/cpuBackProjection/cpuBackProjection.hpp:165-228) and mfBasic.m:66-89:
//   img[x*Ny + y] += sum_n sum_k ph[n][k] exp(j 4 pi f_{n,k} dR_n / c),
//   f_{n,k} = f0_n + k df_n, dR_n = |a_n - p| - R0_n, target z = 0,
// for every pixel and pulse (no swath gate, no interpolation).
//
// gfx950 formulation.  Summing the K samples at every pixel costs 4 K FMA per
// pixel and pulse (a Horner recurrence measured 1400 us at 256^2 pixels,
// 512 pulses of 424 samples, bound by FP32 issue).  But with u = 2 df dR / c
// the sum over k is a trigonometric polynomial of u with period 1, the same
// for every pixel of a pulse, so it is tabulated once per pulse and
// interpolated:
//   * N >= 4 K bins (a power of two) per period, u = (b + f) / N, |f| <= 1/2;
//     with Kc = K / 2 and s = 2 f,
//       sum_k ph_k e^{j 2 pi k u}
//         = e^{j 2 pi Kc f / N} sum_k ph_k e^{j x_k s} e^{j 2 pi k b / N},
//       x_k = pi (k - Kc) / N,  |x_k| <= pi / 8;
//   * cos(x s) = sum over even m, sin(x s) = sum over odd m, of g_m(x) s^m (the
//     Chebyshev interpolants in s on [-1, 1]): degree 5 (6 terms) leaves at
//     most 1.8e-7 of e^{j x s} (rms 3.4e-8), so the bin's polynomial has the 6
//     coefficients (times j for odd m)
//       Y_m[b] = sum_k ph_k g_m(x_k) e^{j 2 pi k b / N}:
//     6 transforms of length N per pulse (mf_table).  Above 4096 samples N
//     stays 16384 (the longest transform held in LDS), |x| <= pi / 4 there and
//     the degree is 7 (at most 6.4e-8).
// mf_interp then spends about 40 instructions per pixel and pulse: the range
// dR = |a_n - p| - R0, the revolutions th0 = frac(2 f0 dR / c) and the bin
// position in FP64, the polynomial and the rotation in FP32, the bins of a
// tile staged through LDS.  Same sizes: 80 us (transforms 20, interpolation 62
// at 0.54 T pixel-pulses/s, bound by FP64 and FP32 issue; sum of the partial
// images 4, traced), and rel-L2 against FP64 2.1e-7 where the recurrence had
// 2.0e-6 (its rounding of e^{j 2 pi u} to FP32 grows with k).
#include <algorithm>
#include <cmath>

#include "sarf_fft.hpp"

namespace sarf {
namespace {

constexpr int kMfThreads = 256;
constexpr int kMfPX = 4;       // pixels per lane
constexpr int kMfTX = 8 * kMfPX, kMfTY = 32;
constexpr int kMfChunk = 32;   // pulses staged per chunk
constexpr int kMfLds = 36864;  // LDS of the staged bins: four workgroups per CU
constexpr int kMfMaxK = 8192;
// Key offset of the weight tables in sarf_ctx::rc_blue.
constexpr long kMfTableKey = 1L << 41;
// Device memory of the coefficient table: pulses are processed in slabs that
// fit (all 512 pulses of the 256^2 configuration take 50 MB).
constexpr size_t kMfSlabBytes = size_t(128) << 20;

struct MfArgs {
    int Nx, Ny, Kc, N, Np;  // Np pulses in this slab
    int tiles_x, tiles_y, splits;
    int accumulate;
    long split_stride;
    double left, bottom, dx, dy;
};

// What every tile needs of a pulse, in device memory so that the wave-uniform
// reads are scalar loads: antenna x, y, z^2, R0, 2 f0 / c, 2 df N / c (bins per
// metre).
struct MfPulse {
    double ax, ay, az2, r0, rev, bins;
};

// Coefficient table of one slab: plane q of pulse n, tab[(n * NPL + q) * N + b]
// = (Y_2q[b], Y_2q+1[b]).  One row of N/16 lanes per (pulse, plane) runs both
// transforms (sarf_fft.hpp), so a bin's pair leaves as one 16-byte store.
// Bound by FP32 issue, as range compression is.
template <int LOG2N, int NPL>
__global__ __launch_bounds__(fft::group_threads(LOG2N)) void mf_table(
    const float2 *__restrict__ ph, int K, int rows, const float *__restrict__ wts,
    const float2 *__restrict__ tw, const double *__restrict__ ant, const double *__restrict__ r0,
    const double *__restrict__ f0, const double *__restrict__ df, float4 *__restrict__ tab,
    MfPulse *__restrict__ pulses) {
    using S = fft::Shape<LOG2N>;
    constexpr int N = S::N, T = S::T, P = fft::rows_per_group(LOG2N);
    __shared__ float2 lds[P * fft::padded(LOG2N)];
    const int lp = threadIdx.x / T;
    const int row = blockIdx.x * P + lp;
    const bool active = row < rows;
    const int n = active ? row / NPL : 0, q = active ? row - n * NPL : 0;
    if (active && q == 0 && threadIdx.x % T == 0) {
        const double az = ant[3 * n + 2];
        pulses[n] = MfPulse{ant[3 * n], ant[3 * n + 1], az * az, r0[n], 2.0 * f0[n] / kClight,
                            2.0 * df[n] / kClight * N};
    }
    const float2 *x = ph + (size_t)n * K;
    const float *g0 = wts + (size_t)(2 * q) * K, *g1 = g0 + K;
    float2 *Lr = lds + lp * fft::padded(LOG2N);
    float2 y[2][16];
#pragma unroll
    for (int m = 0; m < 2; m++) {
        // opaque copy of the lane index: keeps the addresses of both
        // transforms from being held in registers at once
        int j = threadIdx.x % T;
        __asm__ volatile("" : "+v"(j));
#pragma unroll
        for (int b = 0; b < S::NB0; b++)
#pragma unroll
            for (int r = 0; r < S::R0; r++) {
                const int k = j + b * T + r * (N / S::R0);
                float2 v = make_float2(0.f, 0.f);
                if (k < K && active) {
                    const float2 s = x[k];
                    const float g = (m ? g1 : g0)[k];
                    v = m ? make_float2(-s.y * g, s.x * g) : make_float2(s.x * g, s.y * g);
                }
                y[m][b * S::R0 + r] = v;
            }
        fft::ifft_regs<LOG2N>(y[m], Lr, j, tw);
    }
    if (!active) return;
    float4 *o = tab + (size_t)row * N + threadIdx.x % T;
#pragma unroll
    for (int r = 0; r < 16; r++)
        o[r * T] = make_float4(y[0][r].x, y[0][r].y, y[1][r].x, y[1][r].y);
}

// Square root to about an ulp of FP64, a third of the instructions of sqrt():
// y = rsq(v) in FP32, e = 1 - v y^2 (below 1e-6), v y (1 + e/2 + 3 e^2/8).
__device__ __forceinline__ double mf_sqrt(double v) {
    const double y = (double)__builtin_amdgcn_rsqf(fmaxf((float)v, 1e-30f));
    const double g = v * y;
    const double e = fma(-g, y, 1.0);
    return fma(g * e, fma(e, 0.375, 0.5), g);
}

// Staged state of a chunk: bins of up to kMfChunk pulses, planes apart.
template <int NPL>
struct MfStage {
    static constexpr int kCap = kMfLds / (16 * NPL);  // bins
    float4 win[NPL][kCap];
    int4 pI[kMfChunk];    // LDS offset, bins, first bin mod N, staged
    double pS[kMfChunk];  // first bin
    int nc, tot;
};

// A workgroup (4 wave64) owns a 32 x 32 pixel tile, each wave 8 rows; a lane's 4
// pixels are 8 columns apart, and 16 lanes in a row cover 4 x 4 pixels: of any
// line of sight they read a few bins only (lanes along y, two bins apart at
// 0.1 m, had two-way bank conflicts).  Per chunk one lane per pulse bounds the bins its tile needs; the
// pulses whose bins fit are staged together.  A pulse that needs more bins
// than fit at all (pixels far apart) is read from the table directly, at any
// spacing.  At 256^2 pixels and 512 pulses the tile needs about 75 bins and 10
// pulses go together.
template <int NPL>
__global__ __launch_bounds__(kMfThreads) __attribute__((amdgpu_waves_per_eu(4))) void mf_interp(
    MfArgs a, const float4 *__restrict__ tab, const MfPulse *__restrict__ pulses,
    float2 *__restrict__ img) {
    using St = MfStage<NPL>;
    __shared__ St L;
    const int ntiles = a.tiles_x * a.tiles_y;
    const int split = blockIdx.x / ntiles;
    const int t = blockIdx.x - split * ntiles;
    const int tx = t % a.tiles_x, ty = t / a.tiles_x;
    const int per = (a.Np + a.splits - 1) / a.splits;
    const int nbeg = min(a.Np, split * per), nend = min(a.Np, nbeg + per);
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int xb = tx * kMfTX, yb = ty * kMfTY, N = a.N;
    const int x0 = xb + ((lane >> 2) & 3) + 4 * (lane >> 5);
    const int y = yb + 8 * wave + (lane & 3) + 4 * ((lane >> 4) & 1);
    const double py = a.bottom + y * a.dy;
    double px[kMfPX];
#pragma unroll
    for (int j = 0; j < kMfPX; j++) px[j] = a.left + (x0 + 8 * j) * a.dx;
    // tile centre and half extents
    const double hx = 0.5 * (kMfTX - 1) * a.dx, hy = 0.5 * (kMfTY - 1) * a.dy;
    const double pcx = a.left + xb * a.dx + hx, pcy = a.bottom + yb * a.dy + hy;
    const double q2 = hx * hx + hy * hy;
    const float kcn = (float)((double)a.Kc / N);
    float2 acc[kMfPX];
#pragma unroll
    for (int j = 0; j < kMfPX; j++) acc[j] = make_float2(0.f, 0.f);

    for (int n0 = nbeg; n0 < nend;) {
        const int cmax = min(kMfChunk, nend - n0);
        __syncthreads();  // previous users of L are done
        if (tid < 64) {
            int W = 0, wl = 0, start = 0, staged = 0;
            if (tid < cmax) {
                const MfPulse p = pulses[n0 + tid];
                const double ux = p.ax - pcx, uy = p.ay - pcy, bins = p.bins;
                const double Rc = sqrt(ux * ux + uy * uy + p.az2);
                // |dR - dR_c| over the tile: with s = uh . q and |q|^2 <= q2,
                // Rc - s <= R <= Rc - s + |q|^2 / (2 (Rc - s)), and never more
                // than |q|
                const double s = (fabs(ux) * hx + fabs(uy) * hy) / Rc;
                double ext = sqrt(q2);
                if (Rc > s) ext = fmin(ext, s + 0.5 * q2 / (Rc - s));
                const double pc = bins * (Rc - p.r0), span = fabs(bins) * ext;
                double st = 0.0;
                // false as well for a position that is no number
                if (span < 1e8 && fabs(pc) < 1e15) {
                    st = floor(pc - span) - 1.0;
                    W = (int)(ceil(pc + span) - st) + 2;
                    staged = W <= St::kCap;
                    wl = staged ? W : 0;
                    start = (int)((long)st & (N - 1));
                }
                L.pS[tid] = st;
            }
            // windows back to back: offsets are the exclusive prefix sum of
            // wl, the pulses that fit a prefix of the chunk
            int incl = wl;
#pragma unroll
            for (int d = 1; d < kMfChunk; d <<= 1) {
                const int v = __shfl_up(incl, d, 64);
                if (tid >= d) incl += v;
            }
            const int nc = __popcll(__ballot(tid < cmax && incl <= St::kCap));
            if (tid < cmax) L.pI[tid] = make_int4(incl - wl, wl, start, staged);
            if (tid == nc - 1) {
                L.nc = nc;
                L.tot = incl;
            }
        }
        __syncthreads();
        const int nc = L.nc, tot = L.tot;
        for (int f = tid; f < tot; f += kMfThreads) {
            int c = 0;
#pragma unroll
            for (int step = kMfChunk / 2; step >= 1; step >>= 1)
                if (c + step < nc && L.pI[c + step].x <= f) c += step;
            const int4 I = L.pI[c];
            const float4 *src = tab + (size_t)(n0 + c) * NPL * N + ((I.z + (f - I.x)) & (N - 1));
            float4 v[NPL];
#pragma unroll
            for (int q = 0; q < NPL; q++) v[q] = src[(size_t)q * N];
#pragma unroll
            for (int q = 0; q < NPL; q++) L.win[q][f] = v[q];
        }
        __syncthreads();
        for (int c = 0; c < nc; c++) {
            const MfPulse p = pulses[n0 + c];
            const int4 I = L.pI[c];
            const double st = L.pS[c] - 0.5;
            const double ddy = p.ay - py;
            const double yz = fma(ddy, ddy, p.az2);
            const int off = __builtin_amdgcn_readfirstlane(I.x), top = I.y - 1;
            const float4 *src = tab + (size_t)(n0 + c) * NPL * N;
            auto pixels = [&](auto coefs) {
#pragma unroll
                for (int j = 0; j < kMfPX; j++) {
                    const double ddx = p.ax - px[j];
                    const double dR = mf_sqrt(fma(ddx, ddx, yz)) - p.r0;
                    const float th = (float)__builtin_amdgcn_fract(p.rev * dR);
                    // from half a bin below the first: floor is the bin
                    const double pos = fma(p.bins, dR, -st);
                    const float f = (float)__builtin_amdgcn_fract(pos) - 0.5f, s = f + f;
                    float4 cf[NPL];
                    coefs(pos, cf);
                    float hr = cf[NPL - 1].z, hi = cf[NPL - 1].w;
#pragma unroll
                    for (int q = NPL - 1; q >= 0; q--) {
                        if (q < NPL - 1) {
                            hr = fmaf(hr, s, cf[q].z);
                            hi = fmaf(hi, s, cf[q].w);
                        }
                        hr = fmaf(hr, s, cf[q].x);
                        hi = fmaf(hi, s, cf[q].y);
                    }
                    const float ph = fmaf(f, kcn, th);  // revolutions
                    const float sn = __builtin_amdgcn_sinf(ph), cs = __builtin_amdgcn_cosf(ph);
                    acc[j].x = fmaf(hr, cs, fmaf(-hi, sn, acc[j].x));
                    acc[j].y = fmaf(hr, sn, fmaf(hi, cs, acc[j].y));
                }
            };
            if (__builtin_amdgcn_readfirstlane(I.w)) {
                pixels([&](double pos, float4 *cf) {
                    const int w = off + max(0, min((int)pos, top));
#pragma unroll
                    for (int q = 0; q < NPL; q++) cf[q] = L.win[q][w];
                });
            } else {
                pixels([&](double pos, float4 *cf) {
                    const int b = (int)((long)I.z + (long)floor(pos)) & (N - 1);
#pragma unroll
                    for (int q = 0; q < NPL; q++) cf[q] = src[(size_t)q * N + b];
                });
            }
        }
        n0 += nc;
    }
    if (y >= a.Ny) return;
    float2 *o = img + (size_t)split * a.split_stride;
#pragma unroll
    for (int q = 0; q < kMfPX; q++) {
        const int x = x0 + 8 * q;
        if (x >= a.Nx) continue;
        const size_t idx = (size_t)x * a.Ny + y;
        o[idx] = a.accumulate ? cadd(o[idx], acc[q]) : acc[q];
    }
}

// Weights g_m(x_k), m < nc, k < K (the sign of j^m folded in, m even: (-1)^(m/2),
// m odd: (-1)^((m-1)/2)), kept in the context per (K, N): Chebyshev
// interpolation of cos(x s) (m even) and sin(x s) (m odd) on [-1, 1], converted
// to powers of s, in FP64.
int mf_weights(sarf_ctx *ctx, int K, int N, int nc, const float **out) {
    std::lock_guard<std::mutex> lk(ctx->mu);
    auto it = ctx->rc_blue.find(kMfTableKey + K);
    if (it == ctx->rc_blue.end()) {
        constexpr int kNodes = 32, kMax = 8;
        double T[kMax][kNodes], pow_of[kMax][kMax] = {};  // T_m at the nodes; its powers
        for (int i = 0; i < kNodes; i++) {
            const double s = std::cos(kPi * (i + 0.5) / kNodes);
            T[0][i] = 1.0;
            T[1][i] = s;
            for (int m = 2; m < nc; m++) T[m][i] = 2.0 * s * T[m - 1][i] - T[m - 2][i];
        }
        pow_of[0][0] = pow_of[1][1] = 1.0;
        for (int m = 2; m < nc; m++)
            for (int p = 0; p <= m; p++)
                pow_of[m][p] = (p > 0 ? 2.0 * pow_of[m - 1][p - 1] : 0.0) - pow_of[m - 2][p];
        std::vector<float> h((size_t)nc * K);
        for (int k = 0; k < K; k++) {
            const double x = kPi * (double)(k - K / 2) / (double)N;
            double c[kMax] = {}, g[kMax] = {};
            for (int i = 0; i < kNodes; i++) {
                const double co = std::cos(x * T[1][i]), si = std::sin(x * T[1][i]);
                for (int m = 0; m < nc; m++)
                    c[m] += (m ? 2.0 : 1.0) / kNodes * T[m][i] * ((m & 1) ? si : co);
            }
            for (int m = 0; m < nc; m++)
                for (int p = 0; p <= m; p++) g[p] += c[m] * pow_of[m][p];
            for (int m = 0; m < nc; m++) h[(size_t)m * K + k] = (float)g[m];
        }
        void *dv = nullptr;
        hipError_t e = hipMalloc(&dv, sizeof(float) * h.size());
        if (e != hipSuccess)
            return fail(SARF_ERR_NOMEM, "sarf_matched_filter: weights: %s", hipGetErrorString(e));
        e = hipMemcpy(dv, h.data(), sizeof(float) * h.size(), hipMemcpyHostToDevice);
        if (e != hipSuccess) {
            (void)hipFree(dv);
            return fail(SARF_ERR_HIP, "sarf_matched_filter: weights: %s", hipGetErrorString(e));
        }
        it = ctx->rc_blue.emplace(kMfTableKey + K, dv).first;
    }
    *out = (const float *)it->second;
    return SARF_OK;
}

template <int LOG2N, int NPL>
void launch_table_t(const float2 *ph, int K, int Np, const float *wts, const float2 *tw,
                    const double *const (&geo)[4], float4 *tab, MfPulse *pulses, hipStream_t s) {
    constexpr int P = fft::rows_per_group(LOG2N);
    const int rows = Np * NPL;
    hipLaunchKernelGGL((mf_table<LOG2N, NPL>), dim3((rows + P - 1) / P),
                       dim3(fft::group_threads(LOG2N)), 0, s, ph, K, rows, wts, tw, geo[0],
                       geo[1], geo[2], geo[3], tab, pulses);
}

}  // namespace
}  // namespace sarf

using namespace sarf;

extern "C" int sarf_matched_filter(sarf_ctx *ctx, const sarf_mf_desc *d, const void *ph,
                                   const double *ant, const double *r0, const double *f0,
                                   const double *df, void *img, void *stream) {
    clear_error();
    SARF_TRY(use_device(ctx));
    StreamOrder order_(ctx, (hipStream_t)stream);
    if (!d || !ph || !ant || !r0 || !f0 || !df || !img)
        return fail(SARF_ERR_INVALID, "sarf_matched_filter: null argument");
    if (d->Nx < 2 || d->Ny < 2 || d->K < 1 || d->Np < 1)
        return fail(SARF_ERR_INVALID, "sarf_matched_filter: bad sizes Nx=%d Ny=%d K=%d Np=%d",
                    d->Nx, d->Ny, d->K, d->Np);
    if (d->K > kMfMaxK)
        return fail(SARF_ERR_UNSUPPORTED, "sarf_matched_filter: K=%d > %d", d->K, kMfMaxK);
    if (!(d->Wx > 0) || !(d->Wy > 0) || !std::isfinite(d->x0) || !std::isfinite(d->y0))
        return fail(SARF_ERR_INVALID, "sarf_matched_filter: bad geometry Wx=%g Wy=%g", d->Wx,
                    d->Wy);
    hipStream_t s = (hipStream_t)stream;
    // bins per period: a power of two >= 4 K, at most 16384 (above 4096
    // samples: between 2 K and 4 K, with two more terms)
    int L = 5;
    while (L < 14 && (1 << L) < 4 * d->K) L++;
    const int N = 1 << L, npl = (long)N >= 4L * d->K ? 3 : 4;
    const float *wts = nullptr;
    const float2 *tw = nullptr;
    SARF_TRY(mf_weights(ctx, d->K, N, 2 * npl, &wts));
    SARF_TRY(twiddles_f32(ctx, L, &tw));
    const size_t pulse_bytes = sizeof(float4) * (size_t)npl * N;
    const int slab = (int)std::min<long>(d->Np, std::max<long>(1, (long)(kMfSlabBytes / pulse_bytes)));
    void *tbuf = nullptr;
    SARF_TRY(scratch_get(ctx, "mf.table", pulse_bytes * slab, &tbuf));
    float4 *tab = (float4 *)tbuf;
    void *pbuf = nullptr;
    SARF_TRY(scratch_get(ctx, "mf.pulses", sizeof(MfPulse) * (size_t)slab, &pbuf));
    MfPulse *pulses = (MfPulse *)pbuf;
    MfArgs a{};
    a.Nx = d->Nx;
    a.Ny = d->Ny;
    a.Kc = d->K / 2;
    a.N = N;
    a.tiles_x = (d->Nx + kMfTX - 1) / kMfTX;
    a.tiles_y = (d->Ny + kMfTY - 1) / kMfTY;
    a.dx = d->Wx / (d->Nx - 1);
    a.dy = d->Wy / (d->Ny - 1);
    a.left = d->x0 - d->Wx / 2;
    a.bottom = d->y0 - d->Wy / 2;
    const int ntiles = a.tiles_x * a.tiles_y;
    // Pulse splits: groups of at least 4 pulses until there are 4 workgroups
    // per CU.
    int splits = d->pulse_split;
    if (splits <= 0) {
        splits = 1;
        const int want = 4 * (ctx->cu_count > 0 ? ctx->cu_count : 256);
        while (splits < 64 && ntiles * splits < want && slab / (2 * splits) >= 4) splits *= 2;
    }
    splits = std::max(1, std::min(splits, d->Np));
    const long npix = (long)d->Nx * d->Ny;
    float2 *out = (float2 *)img;
    a.splits = splits;
    if (splits > 1) {
        void *buf = nullptr;
        SARF_TRY(scratch_get(ctx, "mf.partials", sizeof(float2) * npix * splits, &buf));
        out = (float2 *)buf;
        a.split_stride = npix;
    }
    const int into = (d->flags & SARF_BP_ACCUMULATE) ? 1 : 0;
    const float2 *x = (const float2 *)ph;
    for (int n0 = 0; n0 < d->Np; n0 += slab) {
        const int np = std::min(slab, d->Np - n0);
        const float2 *xs = x + (size_t)n0 * d->K;
        const double *const geo[4] = {ant + 3 * (size_t)n0, r0 + n0, f0 + n0, df + n0};
        switch (L) {
            case 5: launch_table_t<5, 3>(xs, d->K, np, wts, tw, geo, tab, pulses, s); break;
            case 6: launch_table_t<6, 3>(xs, d->K, np, wts, tw, geo, tab, pulses, s); break;
            case 7: launch_table_t<7, 3>(xs, d->K, np, wts, tw, geo, tab, pulses, s); break;
            case 8: launch_table_t<8, 3>(xs, d->K, np, wts, tw, geo, tab, pulses, s); break;
            case 9: launch_table_t<9, 3>(xs, d->K, np, wts, tw, geo, tab, pulses, s); break;
            case 10: launch_table_t<10, 3>(xs, d->K, np, wts, tw, geo, tab, pulses, s); break;
            case 11: launch_table_t<11, 3>(xs, d->K, np, wts, tw, geo, tab, pulses, s); break;
            case 12: launch_table_t<12, 3>(xs, d->K, np, wts, tw, geo, tab, pulses, s); break;
            case 13: launch_table_t<13, 3>(xs, d->K, np, wts, tw, geo, tab, pulses, s); break;
            default:
                if (npl == 3) launch_table_t<14, 3>(xs, d->K, np, wts, tw, geo, tab, pulses, s);
                else launch_table_t<14, 4>(xs, d->K, np, wts, tw, geo, tab, pulses, s);
        }
        SARF_HIP(hipGetLastError());
        a.Np = np;
        // the first slab writes its (partial) image, later ones add to it
        a.accumulate = n0 > 0 || (splits == 1 && into) ? 1 : 0;
        if (npl == 3)
            hipLaunchKernelGGL(mf_interp<3>, dim3(ntiles * splits), dim3(kMfThreads), 0, s, a, tab,
                               pulses, out);
        else
            hipLaunchKernelGGL(mf_interp<4>, dim3(ntiles * splits), dim3(kMfThreads), 0, s, a, tab,
                               pulses, out);
        SARF_HIP(hipGetLastError());
    }
    if (splits > 1)
        SARF_TRY(launch_reduce_partials(out, npix, splits, npix, into, (float2 *)img, s));
    return SARF_OK;
}
