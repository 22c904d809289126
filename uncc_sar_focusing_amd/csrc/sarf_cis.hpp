// sarf_cis.hpp -- e^{j 2 pi t} from polynomials, for kernels whose phases need
// more than the sine/cosine unit gives.  Host and device: the polynomials are
// checked against libm on the host.
#pragma once

#include <hip/hip_runtime.h>

namespace sarf {

// e^{j 2 pi t}, 0 <= t <= 1, within an ulp of FP32 (the sine/cosine unit's
// absolute error is about four times that): t - q/4 in [-1/8, 1/8] exactly, the
// Taylor polynomials of sin(2 pi x) and cos(2 pi x) there (the first terms left
// out are below 3e-9), 2 pi x in two parts, and a quarter turn's exchange and
// signs.
__host__ __device__ __forceinline__ float2 cis_rev(float t) {
    constexpr float kTwoPi = 6.28318548f, kTwoPiRest = -1.74845560e-7f;
    const float q = rintf(4.f * t);
    const float x = fmaf(-0.25f, q, t), z = x * x;
    const float s = fmaf(x, kTwoPi,
                         x * fmaf(z, fmaf(z, fmaf(z, fmaf(z, 42.058693944897658f, -76.705859753061383f),
                                                  81.605249276075054f), -41.341702240399755f),
                                  kTwoPiRest));
    const float c = fmaf(z, fmaf(z, fmaf(z, fmaf(z, fmaf(z, -26.426256783374398f,
                                                         60.244641371876663f), -85.456817206693725f),
                                         64.939394022668291f), -19.739208802178717f), 1.f);
    const int k = (int)q;
    const float a = (k & 1) ? s : c, b = (k & 1) ? c : s;  // |cos|, |sin| after the turns
    // turns 0..4: (c, s), (-s, c), (-c, -s), (s, -c), (c, s)
    return make_float2(((k + 1) & 2) ? -a : a, (k & 2) ? -b : b);
}

// e^{j 2 pi t}, |t| <= 1/2 and a little, to an ulp or so of FP64: t - q/4 in
// [-1/8, 1/8], the Taylor polynomials of sin(2 pi x) to x^15 and cos(2 pi x) to
// x^16 there (the first terms left out are below 6e-17) and a quarter turn's
// exchange and signs.
__host__ __device__ __forceinline__ double2 cis_rev64(double t) {
    const double q = rint(4.0 * t);
    const double x = fma(-0.25, q, t), z = x * x;
    double s = -0.71812230177850051223;
    s = fma(z, s, 3.8199525848482821277);
    s = fma(z, s, -15.094642576822990392);
    s = fma(z, s, 42.058693944897653145);
    s = fma(z, s, -76.705859753061385842);
    s = fma(z, s, 81.605249276075054203);
    s = fma(z, s, -41.341702240399760234);
    s = fma(z, s, 6.2831853071795864769);
    s *= x;
    double c = 0.28200596845579121507;
    c = fma(z, c, -1.7143907110886720654);
    c = fma(z, c, 7.9035363713184688042);
    c = fma(z, c, -26.426256783374397453);
    c = fma(z, c, 60.244641371876660363);
    c = fma(z, c, -85.456817206693727736);
    c = fma(z, c, 64.939394022668291491);
    c = fma(z, c, -19.739208802178717238);
    c = fma(z, c, 1.0);
    const int k = (int)q;
    const double a = (k & 1) ? s : c, b = (k & 1) ? c : s;
    return make_double2(((k + 1) & 2) ? -a : a, (k & 2) ? -b : b);
}

}  // namespace sarf
