// sarf_bp_core.hpp -- the backprojection tile engine shared by every BP
// kernel (image formation, candidate batches, adjoint).
//
// Reference semantics (src/cpuBackProjection/cpuBackProjection.hpp:24-93):
// for every pulse n and pixel p,
//   dR  = |a_n - p| - R0_n                                   (:70-74)
//   if r_0 < dR < r_{N-1}, r_i = (i/N - 0.5) maxWr           (:76, :45)
//     pos = (dR/maxWr + 0.5) N, left bin i = floor(pos)      (:83, :28-29)
//     v   = s_i + (pos - i)(s_{i+1} - s_i)                   (:38-40)
//     img[x*Ny + y] += v * exp(j 4 pi f0_n dR / c)           (:78-79, :87)
// The interpolation rule is the CPU reference's (first bin with r > dR),
// not the GPU reference's roundf (cuda_BackProjectionKernels.cuh:68-69).
//
// Design for gfx950 (one workgroup = 256 lanes = 4 wave64 per pixel tile):
//   * Lanes run along y (contiguous stores, image is y fastest); each lane
//     owns PX pixels of one row; the tile is TX x TY.
//   * Pulses go in chunks of up to kBpChunk.  For each (tile, pulse) one lane
//     computes in FP64: u = a_n - p_c (p_c = tile centre), R_c = |u|,
//     dR_c = R_c - R0, the profile window the tile needs (from its corners,
//     exact for any geometry) and psi_c = frac(2 f0 dR_c / c) in revolutions.
//     Only these need more than FP32: at R ~ 12.5 km an FP32 range has a
//     1 mm ulp (0.4 rad at 9.6 GHz).
//   * Per pixel, FP32, q = p - p_c (a few metres), uh = u / R_c:
//         s = uh.q,  t = |q|^2 - s^2,
//         dR - dR_c = -s + t (g0 + g1 s),  g0 = 1/(2 R_c), g1 = 1/(2 R_c^2)
//     (expansion of (R_c - s) sqrt(1 + t/(R_c - s)^2) - R_c; remainder
//     t^2/(8 R^3)), so no square root per pixel.
//   * Lane orientation: lanes run along y (XL = false) or along x (XL =
//     true).  Lanes along the cross-range axis read nearly the same profile
//     bin, so the per-pixel window gathers are LDS broadcasts; lanes along
//     the line of sight spread over ~1.4 bins per lane and bank-conflict.
//   * XL tiles use the same expansion in separable form: with P the pixel-
//     axis and L the lane-axis coordinate (uh components u_p, u_l),
//         dR - dR_c = F_p(P) + F_l(L) + P C1(L) + P^2 C2(L),
//     F_p staged per (pulse, column) in LDS and F_l folded into the lane's
//     window-position and phase offsets, so a pixel needs two FMAs for its
//     local range instead of four.
//   * Profile windows are staged in LDS as intercept and slope in
//     window-local bin units, {s_i - i d_i, d_i} with d_i = s_{i+1} - s_i,
//     so the lerp at position p (i = floor p) is one 16-byte LDS read and
//     two FMAs on p itself: no fract.  The intercept's rounding is of the
//     order of ulp(p) |d_i|, the error p itself already carries.  A chunk's
//     windows are packed.
//   * Phase psi = psi_c + (2 f0/c)(dR - dR_c) in revolutions goes straight
//     into v_sin_f32 / v_cos_f32 (they take revolutions and reduce exactly
//     for |psi| <= 256; outside that range they are not valid).
//   * Fast pulses (uniform per (tile, pulse)): the window lies inside the
//     profile, so no per-pixel swath gate, and (2 f0/c)|dR - dR_c| <= 250
//     over the tile, so no phase reduction.  Other pulses take the gated
//     path, which also reduces the phase to one revolution.
#pragma once

#include "sarf_internal.hpp"

namespace sarf {

constexpr int kBpThreads = 256;
constexpr int kBpChunk = 32;  // max pulses staged per chunk (the 256-lane tile stages 64)
constexpr int kBpCap = 2048;  // LDS window capacity, in bins (16 B each)
// The same of kernels for geometries whose windows are never wider, so that
// five workgroups fit in a CU's LDS.
constexpr int kBpCapX = 1536;
static_assert(kBpChunk <= 64 && kBpCap % kBpThreads == 0, "staging layout");

// Waves per SIMD the tile kernels are compiled for: 4 (<= 128 VGPRs) up to
// 8 pixels per lane, except lanes-along-x tiles whose column terms take the
// LDS past 40 KiB (3 workgroups per CU); the 16-pixel tiles need more
// registers than that.  Tiles 5, 13, 15 and 16 with the smaller windows: 5 (2048^2
// at 0.05 m, 4096 pulses, tile 16 6.98 -> 6.74 ms, tile 13 7.23 -> 6.94; 343
// candidates at 512^2, 128 pulses, tile 15 4.52 -> 4.48 ms; 777 x 603, 1237 pulses,
// tile 5 with range compression 367 -> 352 us); which launches take them is
// bp_five_waves.
template <int TY, int PX, bool XL, int CAP = kBpCap>
constexpr int bp_waves_per_eu() {
    return CAP < kBpCap ? 5 : PX > 8 ? 1 : (XL && (kBpThreads / TY) * PX > 32) ? 3 : 4;
}
// The same for a tile described at run time (lanes tl, pixels per lane px).
constexpr int bp_waves_per_eu_rt(int tl, int px, bool xl) {
    return px > 8 ? 1 : (xl && (kBpThreads / tl) * px > 32) ? 3 : 4;
}
struct BpArgs {
    int Nx, Ny, Nfft, Np;
    int tiles_x, tiles_y;
    int accumulate;
    int splits;         // pulse groups per tile (> 1: partial images, reduced after)
    int tail;           // > 0 (with splits > 1): split 0 takes the first Np - tail
                        // pulses straight into the image, the other splits share
                        // the last tail pulses in partial images
    long split_stride;  // elements between partial images
    float2 *part;       // partial images (splits > 1)
    double left, bottom, dx, dy;  // pixel (i,j) = (left + i dx, bottom + j dy)
    double maxWr;
    float invbin;  // Nfft / maxWr (bins per metre)
    double binv;   // the same in FP64
    // Windows against kBpCapX: their bound but for the curvature term |q|^2 / R
    // (BpTileU, which has a form for wider ones), and with it for any antenna
    // no nearer than the tile's half diagonal (BpTile, which cuts them there).
    int narrow, five;
};

// Whether a launch of `groups` workgroups of tile 5, 13, 15 or 16 takes BpTile's
// kernel for five waves per SIMD.  That has fewer registers (it spills) and a
// smaller window buffer, so it pays only where the fifth wave has work: more
// than eight workgroups per CU.  Measured with four waves and five (us, 256 CUs):
// images of 1536 workgroups 137.6 / 140.2 (211 x 186, 1611 pulses, tile 5), 1728
// 61.2 / 62.5 (537 x 362, 263, tile 13), 2912 58.8 / 56.9 (415 x 410, 307, tile 5),
// 4248 83.7 / 79.6 (1095 x 931, 90); candidate batches of 750 workgroups 110.0 /
// 115.0, 1600 212 / 215, 2048 239 / 241, 2457 307 / 305, 6250 718 / 703, 43904
// 4518 / 4476 (128 pulses).
inline bool bp_five_waves(const BpArgs &a, long groups, int cus) {
    return a.five && groups > 8L * (cus > 0 ? cus : 256);
}

// Pulse range [nbeg, nend) of split s of a tile: even groups, or, with a
// tail, one head group of the first Np - tail pulses and the tail pulses in
// even groups over the remaining splits.  Split-major launch order runs every
// tile's head first, so the short tail groups fill in as CUs free up.
__device__ __forceinline__ void split_range(const BpArgs &a, int s, int &nbeg, int &nend) {
    if (a.tail > 0 && a.splits > 1) {
        const int head = a.Np - a.tail;
        if (s == 0) {
            nbeg = 0;
            nend = head;
            return;
        }
        const int per = (a.tail + a.splits - 2) / (a.splits - 1);
        nbeg = min(a.Np, head + (s - 1) * per);
        nend = min(a.Np, nbeg + per);
        return;
    }
    const int per = (a.Np + a.splits - 1) / a.splits;
    nbeg = min(a.Np, s * per);
    nend = min(a.Np, nbeg + per);
}

// Staged state of one chunk of up to CH pulses, CAP window bins.
template <int CH, int CAP>
struct BpLdsT {
    static_assert(CH <= 64, "one wave stages a chunk");
    float4 win[CAP];
    float4 pA[CH];  // uh_x, uh_y, g0, g1
    float4 pB[CH];  // pos_c (window-local), psi_c, kappa, W - 2
    int4 pI[CH];    // start bin, LDS offset (bins), W, interior
    float4 pC[CH];  // separable terms (lane axis): c2l, c3l, e1, e2
    float4 pD[CH];  // separable terms: e3, c2p, c3p (pixel axis), -
    int nc;   // pulses staged
    int tot;  // window bins staged
};

// Antenna positions as given.
struct PlainPos {
    const double *ant;
    __device__ __forceinline__ double3 operator()(int n) const {
        return make_double3(ant[3 * n], ant[3 * n + 1], ant[3 * n + 2]);
    }
};

// Candidate trajectory: a_n + (sum_k coef_k basis_k[n]) dir_n -- e.g. a
// polynomial line-of-sight error a t^2 + b t^3 + c t^4 along the unit LOS --
// or, with one direction field per basis (per_basis),
// a_n + sum_k coef_k basis_k[n] dir_k,n -- e.g. absolute positions that are
// polynomials in the pulse index along x, y and z.
struct LosPolyPos {
    const double *ant, *dir, *basis, *coef;
    int nbasis, Np, per_basis;
    __device__ __forceinline__ double3 operator()(int n) const {
        if (per_basis) {
            double x = ant[3 * n], y = ant[3 * n + 1], z = ant[3 * n + 2];
            for (int k = 0; k < nbasis; k++) {
                const double w = coef[k] * basis[(size_t)k * Np + n];
                const double *d = dir + 3 * ((size_t)k * Np + n);
                x = fma(w, d[0], x);
                y = fma(w, d[1], y);
                z = fma(w, d[2], z);
            }
            return make_double3(x, y, z);
        }
        double off = 0.0;
        for (int k = 0; k < nbasis; k++) off = fma(coef[k], basis[(size_t)k * Np + n], off);
        return make_double3(fma(off, dir[3 * n], ant[3 * n]), fma(off, dir[3 * n + 1], ant[3 * n + 1]),
                            fma(off, dir[3 * n + 2], ant[3 * n + 2]));
    }
};

// XCD-aware tile order: workgroup b runs on XCD b % 8 (round-robin
// dispatch); give each XCD a contiguous run of tiles.  Tiles are numbered
// x fastest, so a run is a band of image rows at similar range whose
// profile windows overlap in that XCD's L2.  Bijective on [0, ntiles).
__device__ __forceinline__ int swizzle_tile(int b, int ntiles) {
    const int full = ntiles & ~7;
    if (b >= full) return b;
    const int per = full >> 3;
    return (b & 7) * per + (b >> 3);
}

// LDS address of a position's bin without a conversion.  q = p - 1/32 (p: position
// in bins, p >= 0) added to 2^19 + the window's first bin rounds to sixteenths of
// a bin, the nearest sixteenth to p - 1/32 being floor(16 p) / 16, and the sum's
// low mantissa bits are sixteen times the bin plus four bits of fraction: with
// those masked off, the byte offset of the bin's 16 bytes.  The add and the mask
// issue in about 2.4 cycles each per wave, v_cvt_i32_f32 and v_lshl_add_u32 in 4
// (measured over 8 waves per SIMD: add, FMA, and 62-67 T lane operations/s, convert
// and shift-add 38): 2048^2 x 4096 pulses with range compression 5.99 -> 5.82 ms.
// At an integer p the sum may round to the bin below, whose line meets the next
// one's there.
constexpr float kBinShift = 0.03125f, kBinMagic = 524288.f;
__device__ __forceinline__ int bin_bytes(float q, float magic) {
    return __float_as_int(q + magic) & 0x7ff0;
}

// Bins of a tile's windows, staged by the whole workgroup: bin f of the
// packed windows belongs to the last pulse c with offset <= f (pI.y), profile
// bin pI.x + f - pI.y; the chunk's first profile is `base`.  In rounds of
// kSlots bins per thread whose loads are all issued before any is consumed.
// SHIFTED: intercepts for positions 1/32 bin below the true ones (kBinMagic).
template <int CH, bool SHIFTED = false>
__device__ __forceinline__ void fill_windows(float4 *win, const int4 *pI, int nc, int tot,
                                             const float2 *__restrict__ base, int Nfft) {
    const int tid = threadIdx.x;
    constexpr int kSlots = 4;
    for (int f0r = 0; f0r < tot; f0r += kSlots * kBpThreads) {
        float2 v0[kSlots], v1[kSlots];
        int wb[kSlots];
#pragma unroll
        for (int k = 0; k < kSlots; k++) {
            const int f = f0r + tid + k * kBpThreads;
            v0[k] = make_float2(0.f, 0.f);
            v1[k] = make_float2(0.f, 0.f);
            wb[k] = 0;
            if (f < tot) {
                int c = 0;
#pragma unroll
                for (int step = CH / 2; step >= 1; step >>= 1)
                    if (c + step < nc && pI[c + step].y <= f) c += step;
                const int4 I = pI[c];
                const int b = f - I.y;
                const int g = I.x + b;  // profile bin; |g| < 2 Nfft
                const unsigned o = (unsigned)(c * Nfft + g);  // < CH * Nfft
                if (g >= 0 && g < Nfft) v0[k] = base[o];
                if (g + 1 >= 0 && g + 1 < Nfft) v1[k] = base[o + 1];
                wb[k] = b;
            }
        }
#pragma unroll
        for (int k = 0; k < kSlots; k++) {
            const int f = f0r + tid + k * kBpThreads;
            if (f < tot) {
                const float dr = v1[k].x - v0[k].x, di = v1[k].y - v0[k].y;
                const float fb = (float)wb[k] - (SHIFTED ? kBinShift : 0.f);
                win[f] = make_float4(fmaf(-fb, dr, v0[k].x), fmaf(-fb, di, v0[k].y), dr, di);
            }
        }
    }
}

// XL = false: the TY lanes of a group run along y and each lane owns PX
// pixels along x (tile (256/TY * PX) x TY).  XL = true: the TY lanes run
// along x and each lane owns PX pixels along y (tile TY x (256/TY * PX)).
template <int TY, int PX, bool XL = false, int CAP = kBpCap>
struct BpTile {
    static constexpr int TL = TY;                  // lanes along the lane axis
    static constexpr int GX = kBpThreads / TL;     // lane groups along the pixel axis
    static constexpr int NP = GX * PX;             // tile extent along the pixel axis
    static constexpr int kPx = PX;                 // pixels per lane
    static constexpr int TX = XL ? TL : NP;        // tile extent along x
    static constexpr int TYE = XL ? NP : TL;       // tile extent along y
    static constexpr bool kSep = XL;               // separable local range
    // Pulses per chunk: 64 for the 256-lane tile, whose narrow windows and
    // 8-column F_p table leave room for them within four workgroups' LDS per
    // CU (fewer chunk rounds: 2048^2 x 4096 pulses 6.88 -> 6.71 ms), 32 else.
    static constexpr int CH = (XL && TL == 256 && PX <= 8) ? 64 : kBpChunk;
    using Lds = BpLdsT<CH, CAP>;
    static constexpr int kFx = kSep ? CH * NP : 4;  // LDS floats for F_p
    int ix0, iy0, ly, gx;
    double pcx, pcy, hx, hy;
    float qy;  // lane coordinate, tile-centred (y if !XL, x if XL)
    float qx[PX], q2[PX], x2[PX], accr[PX], acci[PX];  // pixel-axis coordinates

    // With 64 lanes or more along the lane axis a wave has one range of
    // pixel-axis coordinates: scalar registers instead of 2 PX vector registers.
    static __device__ __forceinline__ float uniform(float v) {
        return TL >= 64 ? __int_as_float(__builtin_amdgcn_readfirstlane(__float_as_int(v))) : v;
    }

    __device__ __forceinline__ void init(const BpArgs &a, int t) {
        const int ty = t / a.tiles_x, tx = t - ty * a.tiles_x;
        ix0 = tx * TX;
        iy0 = ty * TYE;
        pcx = a.left + (ix0 + 0.5 * (TX - 1)) * a.dx;
        pcy = a.bottom + (iy0 + 0.5 * (TYE - 1)) * a.dy;
        hx = 0.5 * (TX - 1) * a.dx;
        hy = 0.5 * (TYE - 1) * a.dy;
        const int tid = threadIdx.x;
        ly = tid % TL;
        gx = TL >= 64 ? __builtin_amdgcn_readfirstlane(tid / TL) : tid / TL;
        const double dl = XL ? a.dx : a.dy, dp = XL ? a.dy : a.dx;
        qy = (float)((ly - 0.5 * (TL - 1)) * dl);
#pragma unroll
        for (int j = 0; j < PX; j++) {
            qx[j] = uniform((float)((gx * PX + j - 0.5 * (NP - 1)) * dp));
            q2[j] = qx[j] * qx[j] + qy * qy;
            x2[j] = uniform(qx[j] * qx[j]);
            accr[j] = 0.f;
            acci[j] = 0.f;
        }
    }

    __device__ __forceinline__ bool pixel(int j, int &x, int &y, const BpArgs &a) const {
        if (XL) {
            x = ix0 + ly;
            y = iy0 + gx * PX + j;
        } else {
            x = ix0 + gx * PX + j;
            y = iy0 + ly;
        }
        return x < a.Nx && y < a.Ny;
    }

    // Per-(tile,pulse) FP64 set-up for pulses [n0, n0 + cmax): fills L.pA,
    // L.pB, L.pI, L.pC, L.pD, packs windows, sets L.nc; then stages the
    // windows and, for separable tiles given fx, F_p per (pulse, column).
    template <class Pos>
    __device__ __forceinline__ void stage(const BpArgs &a, Lds &L, const float2 *__restrict__ prof,
                                          const Pos &pos, const double *__restrict__ r0,
                                          const double *__restrict__ f0, int n0, int cmax,
                                          float *fx = nullptr) {
        const int tid = threadIdx.x;
        __syncthreads();  // previous users of L are done
        // Wave 0, one lane per pulse of the chunk (cmax <= CH <= 64).
        int W = 0, start = 0, interior = 0;
        if (tid < cmax) {
            const int n = n0 + tid;
            const double3 an = pos(n);
            const double ux = an.x - pcx, uy = an.y - pcy, uz = an.z;
            const double Rc = sqrt(ux * ux + uy * uy + uz * uz);
            const double iR = 1.0 / Rc;
            const double dRc = Rc - r0[n];
            const double posg = (dRc / a.maxWr + 0.5) * a.Nfft;
            // |dR - dR_c| over the tile <= |uh_x| hx + |uh_y| hy + |q|^2/(2 R_c)
            const double ext = fabs(ux * iR) * hx + fabs(uy * iR) * hy + (hx * hx + hy * hy) * 0.5 * iR;
            const double span = ext * a.Nfft / a.maxWr;
            const long st = (long)floor(posg - span) - 1;
            // Clamped so a pulse always fits; the host checks the worst case so
            // the clamp does not bind for valid geometry.
            W = min((int)((long)ceil(posg + span) - st) + 2, CAP);
            start = (int)st;
            const double kap = 2.0 * f0[n] / kClight;  // revolutions per metre
            double psi = kap * dRc;
            psi -= rint(psi);
            L.pA[tid] = make_float4((float)(ux * iR), (float)(uy * iR), (float)(0.5 * iR),
                                    (float)(0.5 * iR * iR));
            L.pB[tid] = make_float4((float)(posg - (double)st), (float)psi, (float)kap,
                                    (float)(W - 2));
            {
                // separable form of the same third-order expansion (u_p, u_l:
                // uh along the pixel and lane axes):
                //   F_p = -u_p P + g0 (1-u_p^2) P^2 + g1 u_p (1-u_p^2) P^3  (c2p, c3p)
                //   F_l = -u_l L + g0 (1-u_l^2) L^2 + g1 u_l (1-u_l^2) L^3  (c2l, c3l)
                //   C1  = -2 u_p u_l g0 L + g1 u_p (1-3u_l^2) L^2            (e1, e2)
                //   C2  = g1 u_l (1-3u_p^2) L                                (e3)
                const double ah = ux * iR, bh = uy * iR, g0 = 0.5 * iR, g1 = 0.5 * iR * iR;
                const double up = XL ? bh : ah, ul = XL ? ah : bh;
                const double mp = 1.0 - up * up, ml = 1.0 - ul * ul;
                L.pC[tid] = make_float4((float)(g0 * ml), (float)(g1 * ul * ml),
                                        (float)(-2.0 * up * ul * g0),
                                        (float)(g1 * up * (1.0 - 3.0 * ul * ul)));
                L.pD[tid] = make_float4((float)(g1 * ul * (1.0 - 3.0 * up * up)), (float)(g0 * mp),
                                        (float)(g1 * up * mp), 0.f);
            }
            // Fast path: the window lies inside the profile (no swath gate) and
            // |psi| <= 0.5 + |kap| * ext stays inside v_sin/v_cos's input range
            // (|x| <= 256 revolutions), so the phase needs no reduction.
            interior = (st >= 0 && st + W <= a.Nfft && fabs(kap) * ext <= 250.0) ? 1 : 0;
        }
        if (tid < 64) {
            // Windows are packed back to back: offsets are the exclusive
            // prefix sum of W over the chunk (a wave scan), and the pulses
            // whose windows fit in LDS are a prefix of the chunk.
            int incl = W;
#pragma unroll
            for (int d = 1; d < CH; d <<= 1) {
                const int t = __shfl_up(incl, d, 64);
                if (tid >= d) incl += t;
            }
            const int nc = __popcll(__ballot(tid < cmax && incl <= CAP));
            if (tid < cmax) L.pI[tid] = make_int4(start, incl - W, W, interior);
            if (tid == nc - 1) {
                L.nc = nc;
                L.tot = incl;
            }
        }
        __syncthreads();
        const int nc = L.nc, tot = L.tot;
        fill_windows<CH>(L.win, L.pI, nc, tot, prof + (size_t)n0 * a.Nfft, a.Nfft);
        if (kSep && fx != nullptr) {
            static_assert(kBpThreads % NP == 0, "a thread keeps one column");
            const int col = tid % NP;
            const double dp = XL ? a.dy : a.dx;
            const float P = (float)((col - 0.5 * (NP - 1)) * dp);  // == qx of that column
            for (int c = tid / NP; c < nc; c += kBpThreads / NP) {
                const float4 A = L.pA[c];
                const float up = XL ? A.y : A.x;
                const float4 D = L.pD[c];
                fx[c * NP + col] = P * fmaf(P, fmaf(P, D.z, D.y), -up);
            }
        }
        __syncthreads();
    }

    // Separable form (XL tiles): per pulse the lane forms F_l, C1, C2 and
    // folds F_l into its window-position and phase offsets; per pixel
    // dl = F_p + P C1 + P^2 C2 = dR - dR_c - F_l.
    __device__ __forceinline__ void accumulate_chunk_sep(const BpArgs &a, const Lds &L,
                                                         const float *__restrict__ fx) {
        const float invbin = a.invbin;
        const int nc = L.nc;
        for (int c = 0; c < nc; c++) {
            const float4 A = L.pA[c];
            const float4 B = L.pB[c];
            const int4 I = L.pI[c];
            const float4 C = L.pC[c];
            const float e3 = L.pD[c].x;
            const float ul = XL ? A.x : A.y;
            const float Fl = qy * fmaf(qy, fmaf(qy, C.y, C.x), -ul);
            const float C1 = qy * fmaf(qy, C.w, C.z);
            const float C2 = qy * e3;
            const float bx = fmaf(Fl, invbin, B.x);  // window position at dl = 0
            const float by = fmaf(Fl, B.z, B.y);     // phase (revolutions) at dl = 0
            float F[PX];
#pragma unroll
            for (int j = 0; j < PX; j += 4) {
                const float4 f4 = *reinterpret_cast<const float4 *>(fx + c * NP + gx * PX + j);
                F[j] = f4.x;
                F[j + 1] = f4.y;
                F[j + 2] = f4.z;
                F[j + 3] = f4.w;
            }
            const float wmax = B.w;
            if (I.w) {
                // interior: no gate, no clamp (as in accumulate_chunk); every
                // window read of the pulse is issued before the first is used
                float p[PX], ph[PX];
                float4 w[PX];
#pragma unroll
                for (int j = 0; j < PX; j++) {
                    const float dl = fmaf(x2[j], C2, fmaf(qx[j], C1, F[j]));
                    p[j] = fmaf(dl, invbin, bx);
                    ph[j] = fmaf(dl, B.z, by);  // revolutions
                    w[j] = L.win[I.y + (int)p[j]];
                }
                __builtin_amdgcn_sched_barrier(0);
#pragma unroll
                for (int j = 0; j < PX; j++) {
                    const float vr = fmaf(p[j], w[j].z, w[j].x);
                    const float vi = fmaf(p[j], w[j].w, w[j].y);
                    const float sn = __builtin_amdgcn_sinf(ph[j]);
                    const float cs = __builtin_amdgcn_cosf(ph[j]);
                    accr[j] = fmaf(vr, cs, fmaf(-vi, sn, accr[j]));
                    acci[j] = fmaf(vr, sn, fmaf(vi, cs, acci[j]));
                }
            } else {
                // swath gate and one-revolution phase (as in accumulate_chunk)
                const float glo = (float)(-I.x);
                const float ghi = (float)(a.Nfft - 1 - I.x);
#pragma unroll
                for (int j = 0; j < PX; j++) {
                    const float dl = fmaf(x2[j], C2, fmaf(qx[j], C1, F[j]));
                    const float p = fmaf(dl, invbin, bx);
                    const int i = (int)__builtin_amdgcn_fmed3f(p, 0.f, wmax);
                    const float4 w = L.win[I.y + i];
                    const bool ok = p > glo && p < ghi;
                    const float vr = ok ? fmaf(p, w.z, w.x) : 0.f;
                    const float vi = ok ? fmaf(p, w.w, w.y) : 0.f;
                    const float ph = __builtin_amdgcn_fractf(fmaf(dl, B.z, by));
                    const float sn = __builtin_amdgcn_sinf(ph);
                    const float cs = __builtin_amdgcn_cosf(ph);
                    accr[j] = fmaf(vr, cs, fmaf(-vi, sn, accr[j]));
                    acci[j] = fmaf(vr, sn, fmaf(vi, cs, acci[j]));
                }
            }
        }
    }

    // Accumulate the staged chunk into the lane's pixels.
    __device__ __forceinline__ void accumulate_chunk(const BpArgs &a, const Lds &L,
                                                     const float *__restrict__ fx) {
        if constexpr (kSep) {
            accumulate_chunk_sep(a, L, fx);
            return;
        }
        const float invbin = a.invbin;
        const int nc = L.nc;
        for (int c = 0; c < nc; c++) {
            const float4 A = L.pA[c];
            const float4 B = L.pB[c];
            const int4 I = L.pI[c];
            const float ul = XL ? A.x : A.y;  // uh along the lane axis
            const float up = XL ? A.y : A.x;  // uh along the pixel axis
            const float sy = ul * qy;
            const float wmax = B.w;
            if (I.w) {
                // Interior: the window has one bin of margin on each side of
                // [pos_c - span, pos_c + span] and span bounds |dl| * invbin,
                // so 1 <= p <= W - 2 up to FP32 rounding (< 0.01 bin) and the
                // truncating conversion needs no clamp.
#pragma unroll
                for (int j = 0; j < PX; j++) {
                    const float s = fmaf(up, qx[j], sy);
                    const float tq = fmaf(-s, s, q2[j]);
                    const float g = fmaf(s, A.w, A.z);
                    const float dl = fmaf(tq, g, -s);  // dR - dR_c
                    const float p = fmaf(dl, invbin, B.x);
                    const int i = (int)p;
                    const float4 w = L.win[I.y + i];
                    const float vr = fmaf(p, w.z, w.x);
                    const float vi = fmaf(p, w.w, w.y);
                    const float ph = fmaf(dl, B.z, B.y);  // revolutions
                    const float sn = __builtin_amdgcn_sinf(ph);
                    const float cs = __builtin_amdgcn_cosf(ph);
                    accr[j] = fmaf(vr, cs, fmaf(-vi, sn, accr[j]));
                    acci[j] = fmaf(vr, sn, fmaf(vi, cs, acci[j]));
                }
            } else {
                // swath gate r_0 < dR < r_{N-1}  <=>  0 < pos_global < N - 1;
                // the phase is reduced to one revolution (high carriers or
                // large tiles take it past the sine unit's range)
                const float glo = (float)(-I.x);
                const float ghi = (float)(a.Nfft - 1 - I.x);
#pragma unroll
                for (int j = 0; j < PX; j++) {
                    const float s = fmaf(up, qx[j], sy);
                    const float tq = fmaf(-s, s, q2[j]);
                    const float g = fmaf(s, A.w, A.z);
                    const float dl = fmaf(tq, g, -s);
                    const float p = fmaf(dl, invbin, B.x);
                    const int i = (int)__builtin_amdgcn_fmed3f(p, 0.f, wmax);
                    const float4 w = L.win[I.y + i];
                    const bool ok = p > glo && p < ghi;
                    const float vr = ok ? fmaf(p, w.z, w.x) : 0.f;
                    const float vi = ok ? fmaf(p, w.w, w.y) : 0.f;
                    const float ph = __builtin_amdgcn_fractf(fmaf(dl, B.z, B.y));
                    const float sn = __builtin_amdgcn_sinf(ph);
                    const float cs = __builtin_amdgcn_cosf(ph);
                    accr[j] = fmaf(vr, cs, fmaf(-vi, sn, accr[j]));
                    acci[j] = fmaf(vr, sn, fmaf(vi, cs, acci[j]));
                }
            }
        }
    }

    // All pulses in [nbeg, nend); fx: LDS of kFx floats.
    template <class Pos>
    __device__ __forceinline__ void run(const BpArgs &a, Lds &L, float *fx,
                                        const float2 *__restrict__ prof, const Pos &pos,
                                        const double *__restrict__ r0,
                                        const double *__restrict__ f0, int nbeg, int nend) {
        for (int n0 = nbeg; n0 < nend;) {
            stage(a, L, prof, pos, r0, f0, n0, min(CH, nend - n0), fx);
            accumulate_chunk(a, L, fx);
            n0 += L.nc;
        }
    }
};

// ---------------------------------------------------------------------------
// BpTileU: tile 15 (256 lanes along x, 8 pixels per lane along y, so that all lanes
// have the same pixel-axis coordinates) for image formation.  Same expansion of
// the range as BpTile, kept in revolutions and regrouped around the tile's middle
// row (P = d in pixel spacings, d = +-1/2, +-3/2, .., so instruction literals):
//   phase(d) = by + d^2 kB + d kA,
//   by = psi_c + rev(L), kA, kB its slope and half its curvature along P,
// per (pulse, lane) 11 instructions; then a pair of pixels +-d shares
// by + d^2 kB, and the window position follows from the phase,
//   p = phase * bins_per_revolution + bx,
// so a pixel takes 2.5 FMA for phase and position where the separable form of
// BpTile takes 4 and two LDS reads.  by is reduced to one revolution first,
// which leaves the phase a few revolutions at most: its rounding (the
// error of the image) is no larger than before.
// A carrier of few revolutions per bin would magnify that rounding in p
// (kBpPhaseBins); its pulses form p by itself, 3.5 FMA for both.  Pulses whose
// window or phase needs it take the gated form of that.  The
// direct expansion over the profile in memory remains for pulses whose window
// does not fit in LDS, that are so near that the cubic term along the pixel
// axis (left out here) would show, or that have no carrier to speak of.
// Bound by the LDS data path (0.86 of its rate at 2048^2) and VALU issue together:
// 96 instructions and 16 sines and cosines per 8 pixels and pulse where BpTile
// takes 109 and 16, and one 16-byte read per pixel and pulse.  It hides its LDS latencies only with
// five waves per SIMD (kBpCapX is what five workgroups' LDS leaves; 96 VGPRs):
// 2048^2 at 0.05 m, 4096 pulses, tile 15: BpTile 6.75 ms, this with four waves
// 6.25, with five 5.85 (six waves the same; 5.65 and 3.0 T pixel-pulses/s with the
// addresses of bin_bytes), and rel-L2
// against FP64 2.7e-6 -> 1.8e-6.  With 16 pixels per lane (107 instructions per
// 8 pixels, 128 VGPRs, four waves) 6.29.  Only tile 15: tiles 16 and 13 keep
// the rounding of BpTile, which is most of what their images are off by.
// ---------------------------------------------------------------------------
enum : int { kPulseFast = 0, kPulseCoarse = 1, kPulseGated = 2, kPulseDirect = 3 };
constexpr int kBpWavesU = 5;  // waves per SIMD (workgroups per CU)
// Most bins per revolution for which the position is taken from the phase: the
// phase's rounding, an ulp of a revolution or two (1.2e-7 to 2.4e-7), is then 2e-6 of
// a bin, an ulp of a position being 8e-6 to 1.2e-4.  rel-L2 of white samples, 300 x
// 200 at 0.05 m: 5.3 bins per revolution 1.05e-6 either way; 17.5 from the phase
// 1.23e-6, by itself 0.99e-6; 5250 1.9e-4 and 0.97e-6.
constexpr float kBpPhaseBins = 8.f;

struct BpLdsU {
    static constexpr int CH = 64;  // pulses per chunk: one wave stages them
    float4 win[kBpCapX];
    // (k: revolutions per metre; w: pixel spacing along the pixel axis)
    float4 qA[CH];  // -k u_l, k c2l, k c3l, psi_c
    float4 qB[CH];  // -k w u_p, k w e1, k w e2, k w^2 c2p
    float4 qC[CH];  // k w^2 e3, bins per revolution, pos_c - kBinShift, kBinMagic + LDS offset (bins)
    int4 pI[CH];    // start bin, LDS offset, W, kPulse*
    float4 pA[CH];  // direct form: uh_x, uh_y, g0, g1
    float4 pB[CH];  // slopes of the window position -b u_l, -b w u_p (b: bins per metre); k
    int nc, tot, fast;  // pulses staged, window bins staged, all of them kPulseFast
};

struct BpTileU {
    static constexpr int TX = kBpThreads, PX = 8;  // lanes along x, pixels per lane along y
    static constexpr int kPx = PX, CH = BpLdsU::CH;
    using Lds = BpLdsU;
    static_assert(kBpCapX * 16 <= 0x8000, "bin_bytes");
    static constexpr int kFx = 4;  // no per-column terms (BpTile's interface)
    int ix0, iy0;
    double pcx, pcy, hx, hy;
    float ql;  // lane coordinate, tile-centred
    float accr[PX], acci[PX];

    __device__ __forceinline__ void init(const BpArgs &a, int t) {
        const int ty = t / a.tiles_x, tx = t - ty * a.tiles_x;
        ix0 = tx * TX;
        iy0 = ty * PX;
        pcx = a.left + (ix0 + 0.5 * (TX - 1)) * a.dx;
        pcy = a.bottom + (iy0 + 0.5 * (PX - 1)) * a.dy;
        hx = 0.5 * (TX - 1) * a.dx;
        hy = 0.5 * (PX - 1) * a.dy;
        ql = (float)(((int)threadIdx.x - 0.5 * (TX - 1)) * a.dx);
#pragma unroll
        for (int j = 0; j < PX; j++) accr[j] = acci[j] = 0.f;
    }

    __device__ __forceinline__ bool pixel(int j, int &x, int &y, const BpArgs &a) const {
        x = ix0 + (int)threadIdx.x;
        y = iy0 + j;
        return x < a.Nx && y < a.Ny;
    }

    template <class Pos>
    __device__ __forceinline__ void stage(const BpArgs &a, Lds &L, const float2 *__restrict__ prof,
                                          const Pos &pos, const double *__restrict__ r0,
                                          const double *__restrict__ f0, int n0, int cmax) {
        const int tid = threadIdx.x;
        __syncthreads();  // previous users of L are done
        if (tid < 64) {
            // one lane per pulse of the chunk (cmax <= CH <= 64); the set-up,
            // window bound and packing of BpTile::stage
            int W = 0, start = 0, mode = kPulseFast;
            float4 C = make_float4(0.f, 0.f, 0.f, 0.f);
            if (tid < cmax) {
                const int n = n0 + tid;
                const double3 an = pos(n);
                const double ux = an.x - pcx, uy = an.y - pcy, uz = an.z;
                const double Rc = sqrt(ux * ux + uy * uy + uz * uz);
                const double iR = 1.0 / Rc;
                const double dRc = Rc - r0[n];
                const double posg = fma(dRc, a.binv, 0.5 * a.Nfft);
                const double ext = fabs(ux * iR) * hx + fabs(uy * iR) * hy + (hx * hx + hy * hy) * 0.5 * iR;
                const double span = ext * a.binv;
                const double st = floor(posg - span) - 1.0;
                const double wd = ceil(posg + span) - st + 2.0;
                start = (int)st;
                const double kap = f0[n] * (2.0 / kClight);
                double psi = kap * dRc;
                psi -= rint(psi);
                const double ah = ux * iR, bh = uy * iR, g0 = 0.5 * iR, g1 = 0.5 * iR * iR;
                const double up = bh, ul = ah;
                const double mp = 1.0 - up * up, ml = 1.0 - ul * ul;
                L.qA[tid] = make_float4((float)(-kap * ul), (float)(kap * g0 * ml),
                                        (float)(kap * g1 * ul * ml), (float)psi);
                const double w = a.dy, kw = kap * w;
                L.qB[tid] = make_float4((float)(-kw * up), (float)(-2.0 * kw * up * ul * g0),
                                        (float)(kw * g1 * up * (1.0 - 3.0 * ul * ul)),
                                        (float)(kw * w * g0 * mp));
                C = make_float4((float)(kw * w * g1 * ul * (1.0 - 3.0 * up * up)),
                                (float)(a.binv / kap), (float)(posg - st - kBinShift), 0.f);
                L.pA[tid] = make_float4((float)ah, (float)bh, (float)g0, (float)g1);
                L.pB[tid] = make_float4((float)(-a.binv * ul), (float)(-a.binv * w * up), (float)kap, 0.f);
                const bool inside = st >= 0.0 && st + wd <= a.Nfft && fabs(kap) * ext <= 250.0;
                mode = !inside ? kPulseGated : fabsf(C.y) <= kBpPhaseBins ? kPulseFast : kPulseCoarse;
                // half extent along the pixel axis; the cubic term there in
                // revolutions, and a carrier so low that the phase cannot
                // carry the position
                if (!(wd <= kBpCapX) || !(fabs(kap) * g1 * hy * hy * hy <= 1e-6) ||
                    !(fabsf(C.y) <= 1e4f))
                    mode = kPulseDirect;
                else
                    W = (int)wd;
            }
            int incl = W;
#pragma unroll
            for (int d = 1; d < CH; d <<= 1) {
                const int t = __shfl_up(incl, d, 64);
                if (tid >= d) incl += t;
            }
            const int nc = __popcll(__ballot(tid < cmax && incl <= kBpCapX));
            const bool slow = __ballot(tid < nc && mode != kPulseFast) != 0;
            if (tid < cmax) {
                C.w = kBinMagic + (float)(incl - W);
                L.qC[tid] = C;
                L.pI[tid] = make_int4(start, incl - W, W, mode);
            }
            if (tid == nc - 1) {
                L.nc = nc;
                L.tot = incl;
                L.fast = slow ? 0 : 1;
            }
        }
        __syncthreads();
        fill_windows<CH, true>(L.win, L.pI, L.nc, L.tot, prof + (size_t)n0 * a.Nfft, a.Nfft);
        __syncthreads();
    }

    // One staged pulse, kPulseFast, kPulseCoarse or kPulseGated.
    template <int MODE>
    __device__ __forceinline__ void pulse(const BpArgs &a, const Lds &L, int c) {
        constexpr bool GATED = MODE == kPulseGated;
        const float4 A = L.qA[c];
        const float4 B = L.qB[c];
        const float4 C = L.qC[c];
        const float kB = fmaf(ql, C.x, B.w);
        const float kA = fmaf(ql, fmaf(ql, B.z, B.y), B.x);
        const float rev = ql * fmaf(ql, fmaf(ql, A.z, A.y), A.x);
        const float by = __builtin_amdgcn_fractf(A.w + rev);
        // window position (less kBinShift): at phase 0 of the reduced phase, or by
        // itself at the middle row, with its slope and half its curvature
        float bx, pA = 0.f, pB = 0.f;
        if constexpr (MODE == kPulseFast) {
            bx = fmaf(C.y, rev - by, C.z);
        } else {
            const float4 b = L.pB[c];
            bx = fmaf(ql, fmaf(C.y * ql, fmaf(ql, A.z, A.y), b.x), C.z);
            pA = fmaf(C.y, ql * fmaf(ql, B.z, B.y), b.y);
            pB = C.y * kB;
        }
        const char *win = (const char *)L.win;
        float glo = 0.f, ghi = 0.f, wmax = 0.f;
        if constexpr (GATED) {
            const int4 I = L.pI[c];
            glo = (float)(-I.x) - kBinShift;
            ghi = (float)(a.Nfft - 1 - I.x) - kBinShift;
            wmax = (float)(I.z - 2);
        }
        // every window read of the pulse is issued before the first is used (left
        // alone the compiler waits for each in turn: 5.94 against 5.87 ms)
        float ph[PX], p[PX];
        float4 w[PX];
#pragma unroll
        for (int j = 0; j < PX; j++) {
            const float d = j - 0.5f * (PX - 1);
            ph[j] = fmaf(d, kA, fmaf(d * d, kB, by));
            p[j] = MODE == kPulseFast ? fmaf(ph[j], C.y, bx) : fmaf(d, fmaf(d, pB, pA), bx);
            // not gated: the window has a bin of margin on each side, 1 <= p <= W - 2
            w[j] = *(const float4 *)(win + bin_bytes(GATED ? __builtin_amdgcn_fmed3f(p[j], 0.f, wmax) : p[j], C.w));
        }
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int j = 0; j < PX; j++) {
            const bool ok = !GATED || (p[j] > glo && p[j] < ghi);
            const float vr = ok ? fmaf(p[j], w[j].z, w[j].x) : 0.f;
            const float vi = ok ? fmaf(p[j], w[j].w, w[j].y) : 0.f;
            const float rev = GATED ? __builtin_amdgcn_fractf(ph[j]) : ph[j];
            const float sn = __builtin_amdgcn_sinf(rev);
            const float cs = __builtin_amdgcn_cosf(rev);
            accr[j] = fmaf(vr, cs, fmaf(-vi, sn, accr[j]));
            acci[j] = fmaf(vr, sn, fmaf(vi, cs, acci[j]));
        }
    }

    // One pulse by the direct expansion from its profile in memory, gated.
    __device__ __forceinline__ void pulse_direct(const BpArgs &a, const Lds &L, int c,
                                                 const float2 *__restrict__ row) {
        const float4 A = L.pA[c];
        const int start = L.pI[c].x;
        const float kap = L.pB[c].z, psi = L.qA[c].w, pos = L.qC[c].z + kBinShift;
        const float ul = A.x, up = A.y;
        const float glo = (float)(-start), ghi = (float)(a.Nfft - 1 - start);
        // opaque, so that this path's per-pixel constants are not held in
        // registers through the others
        float dp = (float)a.dy;
        __asm__ volatile("" : "+v"(dp));
#pragma unroll
        for (int j = 0; j < PX; j++) {
            const float P = (j - 0.5f * (PX - 1)) * dp;
            const float s = fmaf(up, P, ul * ql);
            const float t = fmaf(-s, s, fmaf(P, P, ql * ql));
            const float dl = fmaf(t, fmaf(s, A.w, A.z), -s);
            const float p = fmaf(dl, a.invbin, pos);  // from bin `start`
            const bool ok = p > glo && p < ghi;
            const int i = (int)floorf(p);
            const int g = max(0, min(start + i, a.Nfft - 2));
            const float2 v0 = row[g], v1 = row[g + 1];
            const float f = p - (float)i;
            const float vr = ok ? fmaf(f, v1.x - v0.x, v0.x) : 0.f;
            const float vi = ok ? fmaf(f, v1.y - v0.y, v0.y) : 0.f;
            const float ph = __builtin_amdgcn_fractf(fmaf(dl, kap, psi));
            const float sn = __builtin_amdgcn_sinf(ph);
            const float cs = __builtin_amdgcn_cosf(ph);
            accr[j] = fmaf(vr, cs, fmaf(-vi, sn, accr[j]));
            acci[j] = fmaf(vr, sn, fmaf(vi, cs, acci[j]));
        }
    }

    // All pulses in [nbeg, nend).
    template <class Pos>
    __device__ __forceinline__ void run(const BpArgs &a, Lds &L, float *,
                                        const float2 *__restrict__ prof, const Pos &pos,
                                        const double *__restrict__ r0,
                                        const double *__restrict__ f0, int nbeg, int nend) {
        for (int n0 = nbeg; n0 < nend;) {
            stage(a, L, prof, pos, r0, f0, n0, min(CH, nend - n0));
            const int nc = L.nc;
            if (__builtin_amdgcn_readfirstlane(L.fast)) {
                for (int c = 0; c < nc; c++) pulse<kPulseFast>(a, L, c);
            } else {
                for (int c = 0; c < nc; c++) {
                    const int mode = __builtin_amdgcn_readfirstlane(L.pI[c].w);
                    if (mode == kPulseFast) pulse<kPulseFast>(a, L, c);
                    else if (mode == kPulseCoarse) pulse<kPulseCoarse>(a, L, c);
                    else if (mode == kPulseGated) pulse<kPulseGated>(a, L, c);
                    else pulse_direct(a, L, c, prof + (size_t)(n0 + c) * a.Nfft);
                }
            }
            n0 += nc;
        }
    }
};

// Wave64 + workgroup sum of two doubles; result valid on thread 0.
__device__ __forceinline__ double2 block_sum2(double a, double b, double2 *red /* [4] */) {
#pragma unroll
    for (int o = 32; o >= 1; o >>= 1) {
        a += __shfl_xor(a, o, 64);
        b += __shfl_xor(b, o, 64);
    }
    const int wave = threadIdx.x >> 6;
    __syncthreads();
    if ((threadIdx.x & 63) == 0) red[wave] = make_double2(a, b);
    __syncthreads();
    double2 r = make_double2(0.0, 0.0);
    if (threadIdx.x == 0) {
        for (int w = 0; w < (int)(blockDim.x >> 6); w++) {
            r.x += red[w].x;
            r.y += red[w].y;
        }
    }
    return r;
}

}  // namespace sarf
