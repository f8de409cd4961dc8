// Factors applied to half-spectrum points (kx, ky) of an N x N image: the CTF (ctf.cu:80-240) in double, and
// the projection preparation's band-pass, dose and WBP weights.  Shared by the Fourier filter kernels
// (fft2d.hip) and the ones over library transforms (spectral.hip, prep.hip), so that both give one value.
#pragma once

#include <hip/hip_runtime.h>

#include "artia_internal.hpp"

namespace artia {

struct CtfK {
    float cs_m;         // Cs * 0.001 (mm -> m)
    float lambda;       // electron wavelength (m), the reference's float constants
    float freq_step;    // (1 / (2 * pixelsize)) / (N / 2)
    float pc, ac;       // phase and amplitude contrast
    float halfN;        // c_pixelcount * 0.5
    float def0, def1, angle;   // metres, metres, radians
    float wiener;
    float beta[4];
    int forFP, phaseFlip, N;
    double cos2a, sin2a;       // of twice the angle
};

// A stack of slabs, each with its own defocus.
struct CtfStack {
    CtfK k;
    float def0[kFftBatchMax], def1[kFftBatchMax];
};

// The exact CTF factor of one spectrum point in two parts: what does not depend on the defocus
// (ctf_point), and the factor and its application for one defocus pair (ctf_apply_at).  The phase
// (hundreds of radians at Nyquist, where a float phase carries 1e-5) is computed in double:
// m = pi/2 (Cs lam^3 len^4 - 2 defocus lam len^2), with the kernel body's float pi/2 and
// defocus = def0 + (1 - cos 2 beta) (def1 - def0).  r^2 cos 2 beta, beta the angle to the astigmatism axis, is
// (x^2 - y^2) cos 2a + 2 x y sin 2a, so that neither an arc tangent nor a division is needed.
struct CtfPoint {
    double A, B0, B1;   // the phase, in quarter turns: A - B0 def0 - B1 (def1 - def0)
    double env;         // the envelope, clamped as the direction requires (used when damped)
    bool damped;        // outside the untouched low-frequency disk, and not phase flipping
};

// exp of the envelope's polynomial at spatial frequency len = sqrt(len2)
__device__ __forceinline__ double ctf_envelope(double len2, const CtfK& k) {
    double arg = -(double)k.beta[2] * (len2 * 1e-16);
    if (k.beta[1] != 0.0f || k.beta[3] != 0.0f) {   // uniform
        const double l = sqrt(len2) * 1e-8;
        arg += (-(double)k.beta[1] - (double)k.beta[3] * l * l) * l;
    }
    return exp(arg);
}

// env: ctf_envelope of the point (not used when phase flipping)
__device__ __forceinline__ CtfPoint ctf_point(int x, int y, const CtfK& k, double env) {
    CtfPoint p;
    const double xp = (double)x, yp = (double)(y + y > k.N ? y - k.N : y);
    const double x2 = xp * xp, y2 = yp * yp, r2 = x2 + y2, lam = k.lambda, fs2 = (double)k.freq_step * (double)k.freq_step;
    const double quarter = (double)(3.14159265358979323846f / 2.0f) * 0.63661977236758134308;
    const double Kb = quarter * 2.0 * lam * fs2;
    p.A = (quarter * (double)k.cs_m * lam * lam * lam * fs2 * fs2) * (r2 * r2);
    p.B0 = Kb * r2;
    p.B1 = Kb * (r2 - ((x2 - y2) * k.cos2a + (2.0 * xp * yp) * k.sin2a));
    p.damped = !k.phaseFlip && (k.beta[0] < 0.0f || r2 > (double)k.beta[0] * (double)k.beta[0]);
    p.env = k.phaseFlip ? 0.0 : fmax(env, k.forFP ? (double)0.01f : (double)k.wiener);
    return p;
}
__device__ __forceinline__ double ctf_len2(int x, int y, const CtfK& k) {
    const double xp = (double)x, yp = (double)(y + y > k.N ? y - k.N : y), fs = (double)k.freq_step;
    return (xp * xp + yp * yp) * (fs * fs);
}
__device__ __forceinline__ CtfPoint ctf_point(int x, int y, const CtfK& k) {
    return ctf_point(x, y, k, k.phaseFlip ? 0.0 : ctf_envelope(ctf_len2(x, y, k), k));
}

// The envelopes of column x at y = y0, y0 + step, .. without an exp for each (no odd powers): exp(a len^2)
// steps by a factor that itself steps by a constant one.  |y| grows along the run, so that with the usual a < 0 all
// three only decay and a steep envelope that underflows stays 0 as its exp does (towards y = 0 the product
// could not rise from 0 again, or would be 0 times infinity); with a > 0 the envelope overflows first.
struct CtfEnvelopeRun {
    double e, r, q;
    // yp: the signed frequency of the first point, step: away from 0
    __device__ __forceinline__ void start(int x, int yp, int step, const CtfK& k) {
        const double fs = (double)k.freq_step, a = -(double)k.beta[2] * 1e-16 * (fs * fs);
        const double y = (double)yp, s = (double)step, xp = (double)x;
        e = exp(a * (xp * xp + y * y));
        r = exp(a * (s * (2.0 * y + s)));
        q = exp(a * (2.0 * s * s));
    }
    __device__ __forceinline__ void next() {
        e *= r;
        r *= q;
    }
};

// sin and cos of t quarter turns: on [-pi/4, pi/4] the polynomials in x^2 that meet (sin x - x) / x^3 and
// (cos x - 1 + x^2 / 2) / x^4 at the six Chebyshev nodes of [0, (pi/4)^2]; they err by 1.4e-17 and 9e-19, below
// the rounding of the values (1.1e-16), which the Taylor polynomials need one term more each for.
__device__ __forceinline__ void sincos_quarters(double t, double& s, double& c) {
    const double n = rint(t), x = (t - n) * 1.57079632679489661923, x2 = x * x;
    const int q = (int)(long long)n;
    double a = __builtin_fma(x2, 1.5918129280835e-10, -2.5051131844808866e-08);
    a = __builtin_fma(x2, a, 2.7557316102551507e-06);
    a = __builtin_fma(x2, a, -0.00019841269836758574);
    a = __builtin_fma(x2, a, 0.008333333333330948);
    a = __builtin_fma(x2, a, -0.16666666666666666);
    a = __builtin_fma(x2 * x, a, x);
    double b = __builtin_fma(x2, -1.1382632416743667e-11, 2.087614626828136e-09);
    b = __builtin_fma(x2, b, -2.755731727172921e-07);
    b = __builtin_fma(x2, b, 2.4801587298765686e-05);
    b = __builtin_fma(x2, b, -0.0013888888888887398);
    b = __builtin_fma(x2, b, 0.041666666666666664);
    b = __builtin_fma(x2, b, -0.5);
    b = __builtin_fma(x2, b, 1.0);
    const double u = (q & 1) ? b : a, w = (q & 1) ? a : b;
    s = (q & 2) ? -u : u;
    c = ((q + 1) & 2) ? -w : w;
}

__device__ __forceinline__ float2 ctf_apply_at(float2 r, const CtfPoint& p, const CtfK& k, float def0f, float def1f) {
    const double def0 = def0f, def1 = def1f;
    double sm, cm;
    sincos_quarters(p.A - p.B0 * def0 - p.B1 * (def1 - def0), sm, cm);
    const double n = (double)k.pc * sm + (double)k.ac * cm;
    double f = 1.0;
    if (!k.phaseFlip) {   // uniform
        double val = n * p.env, g;
        if (k.forFP) {
            if (fabs(val) < (double)0.0001f) val = val >= 0 ? (double)0.0001f : -(double)0.0001f;
            g = -val;
        } else {
            g = -val / (val * val + (double)k.wiener);
        }
        f = p.damped ? g : 1.0;
    }
    if (k.phaseFlip && n >= 0) f = -f;
    r.x = (float)((double)r.x * f);
    r.y = (float)((double)r.y * f);
    return r;
}

// wbpWeighting.cu:48-144 in double; sn, cs: sine and cosine of the weighting's angle
__device__ __forceinline__ float2 wbp_weighted(float2 r, int x, int y, int N, double sn, double cs, int method) {
    const double xpos = (double)x, ypos = (double)(y + y > N ? y - N : y);
    const double len = (sn * xpos + cs * ypos) / (double)N / 2.0;
    double w = 1.0;
    if (method == 0) {
        w = fmin(fabs(len), 1.0);
    } else if (method >= 2 && method <= 4) {
        const double P[3][4] = {{1.000654227857550f, 0.006008581017124f, 0.004159659493151f, 0.000975903396538f},
                                {1.003784816598589f, 0.029016377161629f, 0.019582940715148f, 0.004559409669984f},
                                {0.999884616010943f, 0.000307646262566f, 0.004742915272196f, 0.004806551368900f}};
        const double* q = P[method - 2];
        if (len == 0) {
            w = 0;
        } else {
            const double L = log(fabs(len));
            w = ((q[0] + q[1] * L) + q[2] * L * L) + q[3] * L * L * L;
        }
        w = fmax(0.0, fmin(w, 1.0));
    }
    r.x = (float)((double)r.x * w);
    r.y = (float)((double)r.y * w);
    return r;
}

// Per-projection state of the preparation, on the device for the whole call.
struct PrepStat {
    double sq_mean;          // mean of the converted square (the bad-pixel reference)
    double mean, std;        // statistics of the normalisation region
    float mean_hf, std_hf;   // the normalisation's subtrahend and divisor magnitude
    float dose, cos_tilt;    // AccumulatedDose; cosf(|tilt| in radians) for DownWeightTiltsForWBP
    int bad;                 // bad pixels replaced
    int pad;
};

// The preparation's spectrum filters for the images of a chunk.
struct PrepFilter {
    int band;
    float lp, hp, lps, hps;
    int dose_on;
    float pixA;
    int wbp, method;                                  // exact-numerics WBP weighting (method as artia_wbp_weight)
    double sn[kFftBatchMax], cs[kFftBatchMax];        // of each image's angle
    const PrepStat* st;
    // out (or null): each wave's sum of the filtered spectrum's squares over both half planes, without frequency 0
    // (fft2d_col_waves(N) an image), and frequency 0 taken out
    double* power;
    float* dc;                                        // out (or null): image z's filtered value at frequency 0
};

// fourierFilter (wbpWeighting.cu:146-212), doseWeighting (:214-240) and wbpWeighting (:48-144), each a
// factor applied in the reference's order.
__device__ __forceinline__ float2 prep_factor(float2 e, int kx, int ky, int N, const PrepFilter& f, int z) {
    const float mx = (float)kx;
    float my = (float)ky;
    if (my > N * 0.5f) my = (N - my) * -1.0f;
    const float dist = sqrtf(mx * mx + my * my);
    if (f.band) {
        float fil = 0;
        const float lp = f.lp - f.lps, hp = f.hp + f.hps, lps = f.lps, hps = f.hps;
        if (lp > 0) {
            if (dist <= lp) fil = 1;
        } else {
            if (dist <= N / 2 - 1) fil = 1;
        }
        if (lps > 0) {
            const float fil2 = (-fil + 1.0f) * expf(-((dist - lp) * (dist - lp) / (2 * lps * lps)));
            if (fil2 > 0.001f) fil = fil2;
        }
        if (lps > 0 && lp == 0 && hp == 0 && hps == 0) fil = expf(-((dist - lp) * (dist - lp) / (2 * lps * lps)));
        if (hp > 0) {
            float fil2 = 0;
            if (dist >= hp) fil2 = 1;
            fil *= fil2;
            if (hps > 0) {
                const float fil3 = (-fil2 + 1) * expf(-((dist - hp) * (dist - hp) / (2 * hps * hps)));
                if (fil3 > 0.001f) fil = fil3;
            }
        }
        e.x *= fil;
        e.y *= fil;
    }
    if (f.dose_on) {
        const float d = dist / (N / 2 / f.pixA);
        const float fil = expf(-f.st[z].dose * d);
        e.x *= fil;
        e.y *= fil;
    }
    if (f.wbp) e = wbp_weighted(e, kx, ky, N, f.sn[z], f.cs[z], f.method);
    return e;
}

}  // namespace artia
