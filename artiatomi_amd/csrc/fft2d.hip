// The three-kernel 2D Fourier filter (fft2d.hpp).
//
// A complex transform of N points is Stockham's with its points in registers: thread t of T holds
// points t + T i (i < E), does radix-R butterflies on them and exchanges through LDS between passes.
// The last pass leaves point t + T i in register i again, so the inverse transform of a column starts
// without an exchange.  Twiddles come from a table of exp(-2 pi i k / N) in double rounded to float; a
// radix-16 butterfly loads six and multiplies the other nine from two of them.
//
// What bounds the kernels is memory: per filtered image the row and column kernels read and write the
// half spectrum once each (4 N^2 bytes) next to the image itself.  A library plan of the same filter
// made six to eight passes (transposes and real-transform pre- and post-passes among them) besides
// separate kernels for squaring, filtering and finishing.  Measured at 4096 x 4096 per image: a CTF slab of
// a shared spectrum 82 us (columns 40, rows back 42: 3.3 TB/s) against 168 us with library transforms; the
// preparation of a 16-bit image 175 us against 500 us.  Running one column block's images one after another
// on an XCD, so that its L2 holds the shared column, made the columns slower (44 us).
#include <cmath>

#include "device_common.hpp"
#include "fft2d.hpp"

namespace artia {
namespace {

struct C2 {
    float x, y;
};
__device__ __forceinline__ C2 operator+(C2 a, C2 b) { return C2{a.x + b.x, a.y + b.y}; }
__device__ __forceinline__ C2 operator-(C2 a, C2 b) { return C2{a.x - b.x, a.y - b.y}; }
__device__ __forceinline__ C2 cmul(C2 a, C2 w) {
    return C2{__builtin_fmaf(a.x, w.x, -(a.y * w.y)), __builtin_fmaf(a.x, w.y, a.y * w.x)};
}
// a times the twiddle w of the forward transform, conjugated for the inverse one
template <bool kInv>
__device__ __forceinline__ C2 ctw(C2 a, C2 w) {
    return kInv ? C2{__builtin_fmaf(a.x, w.x, a.y * w.y), __builtin_fmaf(a.y, w.x, -(a.x * w.y))} : cmul(a, w);
}
// a times -i (forward) or i (inverse)
template <bool kInv>
__device__ __forceinline__ C2 rot(C2 a) {
    return kInv ? C2{-a.y, a.x} : C2{a.y, -a.x};
}

// Values at 32-bit byte offsets from a uniform base: one address register per access instead of two
// (fft2d_fits: images and spectra stay below 4 GiB).
template <typename V>
__device__ __forceinline__ V load_at(const void* base, uint32_t off) {
    return *reinterpret_cast<const V*>(static_cast<const char*>(base) + off);
}
template <typename V>
__device__ __forceinline__ void store_at(void* base, uint32_t off, V v) {
    *reinterpret_cast<V*>(static_cast<char*>(base) + off) = v;
}

template <bool kInv>
__device__ __forceinline__ void dft2(C2& a, C2& b) {
    const C2 t = a - b;
    a = a + b;
    b = t;
}
template <bool kInv>
__device__ __forceinline__ void dft4(C2& a, C2& b, C2& c, C2& d) {
    const C2 s = a + c, t = a - c, u = b + d, w = rot<kInv>(b - d);
    a = s + u;
    b = t + w;
    c = s - u;
    d = t - w;
}
constexpr float kS8 = 0.70710678118654752440f;   // cos(pi / 4)
template <bool kInv>
__device__ __forceinline__ void dft8(C2 v[8]) {
    dft4<kInv>(v[0], v[2], v[4], v[6]);
    dft4<kInv>(v[1], v[3], v[5], v[7]);
    // odd outputs times w8^k
    const C2 o1 = v[3], o2 = v[5], o3 = v[7], o0 = v[1];
    const C2 r1 = rot<kInv>(o1), r3 = rot<kInv>(o3);
    const C2 t1 = C2{kS8 * (o1.x + r1.x), kS8 * (o1.y + r1.y)};       // w8 = (1 - i) / sqrt 2
    const C2 t2 = rot<kInv>(o2);
    const C2 t3 = C2{kS8 * (r3.x - o3.x), kS8 * (r3.y - o3.y)};       // w8^3 = (-1 - i) / sqrt 2
    const C2 e0 = v[0], e1 = v[2], e2 = v[4], e3 = v[6];
    v[0] = e0 + o0;
    v[4] = e0 - o0;
    v[1] = e1 + t1;
    v[5] = e1 - t1;
    v[2] = e2 + t2;
    v[6] = e2 - t2;
    v[3] = e3 + t3;
    v[7] = e3 - t3;
}
template <bool kInv>
__device__ __forceinline__ void dft16(C2 v[16]) {
    constexpr float c1 = 0.92387953251128675613f, s1 = 0.38268343236508977173f;   // cos, sin (pi / 8)
    // x[4 a + b]: transforms over a, twiddles w16^(b k), transforms over b; output k + 4 m at [4 k + m]
#pragma unroll
    for (int b = 0; b < 4; b++) dft4<kInv>(v[b], v[4 + b], v[8 + b], v[12 + b]);
    const C2 w1{c1, -s1}, w2{kS8, -kS8}, w3{s1, -c1}, w6{-kS8, -kS8}, w9{-c1, s1};
    v[4 + 1] = ctw<kInv>(v[4 + 1], w1);
    v[4 + 2] = ctw<kInv>(v[4 + 2], w2);
    v[4 + 3] = ctw<kInv>(v[4 + 3], w3);
    v[8 + 1] = ctw<kInv>(v[8 + 1], w2);
    v[8 + 2] = rot<kInv>(v[8 + 2]);
    v[8 + 3] = ctw<kInv>(v[8 + 3], w6);
    v[12 + 1] = ctw<kInv>(v[12 + 1], w3);
    v[12 + 2] = ctw<kInv>(v[12 + 2], w6);
    v[12 + 3] = ctw<kInv>(v[12 + 3], w9);
#pragma unroll
    for (int k = 0; k < 4; k++) dft4<kInv>(v[4 * k], v[4 * k + 1], v[4 * k + 2], v[4 * k + 3]);
    // natural order: output k + 4 m
    C2 t[16];
#pragma unroll
    for (int i = 0; i < 16; i++) t[i] = v[i];
#pragma unroll
    for (int k = 0; k < 4; k++)
#pragma unroll
        for (int m = 0; m < 4; m++) v[k + 4 * m] = t[4 * k + m];
}

__device__ __forceinline__ C2 tw_at(const float2* __restrict__ tw, int i) {
    const float2 w = tw[i];
    return C2{w.x, w.y};
}

// Radix-R butterflies of the pass whose sub-transforms have length Ns, on registers v[i] = point t + T i:
// butterfly b takes v[b + r E / R].
template <int N, int E, int R, int Ns, bool kInv>
__device__ __forceinline__ void fft_pass(C2 v[E], int t, const float2* __restrict__ tw) {
    constexpr int T = N / E, B = E / R;
#pragma unroll
    for (int b = 0; b < B; b++) {
        C2 u[R];
#pragma unroll
        for (int r = 0; r < R; r++) u[r] = v[b + r * B];
        if (Ns > 1) {
            const int k = ((t + b * T) & (Ns - 1)) * (N / (Ns * R));
            if (R == 16) {
                const C2 w1 = tw_at(tw, k), w2 = tw_at(tw, 2 * k), w3 = tw_at(tw, 3 * k);
                const C2 w4 = tw_at(tw, 4 * k), w8 = tw_at(tw, 8 * k), w12 = tw_at(tw, 12 * k);
                u[1] = ctw<kInv>(u[1], w1);
                u[2] = ctw<kInv>(u[2], w2);
                u[3] = ctw<kInv>(u[3], w3);
                u[4] = ctw<kInv>(u[4], w4);
                u[5 % R] = ctw<kInv>(u[5 % R], cmul(w4, w1));
                u[6 % R] = ctw<kInv>(u[6 % R], cmul(w4, w2));
                u[7 % R] = ctw<kInv>(u[7 % R], cmul(w4, w3));
                u[8 % R] = ctw<kInv>(u[8 % R], w8);
                u[9 % R] = ctw<kInv>(u[9 % R], cmul(w8, w1));
                u[10 % R] = ctw<kInv>(u[10 % R], cmul(w8, w2));
                u[11 % R] = ctw<kInv>(u[11 % R], cmul(w8, w3));
                u[12 % R] = ctw<kInv>(u[12 % R], w12);
                u[13 % R] = ctw<kInv>(u[13 % R], cmul(w12, w1));
                u[14 % R] = ctw<kInv>(u[14 % R], cmul(w12, w2));
                u[15 % R] = ctw<kInv>(u[15 % R], cmul(w12, w3));
            } else {
#pragma unroll
                for (int r = 1; r < R; r++) u[r] = ctw<kInv>(u[r], tw_at(tw, r * k));
            }
        }
        if (R == 2) dft2<kInv>(u[0], u[1]);
        else if (R == 4) dft4<kInv>(u[0], u[1], u[2 % R], u[3 % R]);
        else if (R == 8) dft8<kInv>(u);
        else dft16<kInv>(u);
#pragma unroll
        for (int r = 0; r < R; r++) v[b + r * B] = u[r];
    }
}

// LDS slot of point i of the transform whose points are kStep apart (one float2 of padding per 16)
template <int kStep>
__device__ __forceinline__ int slot(int i) {
    return (i + (i >> 4)) * kStep;
}
__host__ __device__ constexpr int padded(int n) { return n + n / 16; }

// The pass's outputs from registers to their places, and the next pass's inputs back.
template <int N, int E, int R, int Ns, int kStep>
__device__ __forceinline__ void fft_exchange(C2 v[E], int t, C2* __restrict__ lds) {
    constexpr int T = N / E, B = E / R;
#pragma unroll
    for (int b = 0; b < B; b++) {
        const int j = t + b * T, at = (j / Ns) * (Ns * R) + (j & (Ns - 1));
#pragma unroll
        for (int r = 0; r < R; r++) lds[slot<kStep>(at + r * Ns)] = v[b + r * B];
    }
    __syncthreads();
#pragma unroll
    for (int i = 0; i < E; i++) v[i] = lds[slot<kStep>(t + T * i)];
    __syncthreads();
}

// Points per thread and radices of each length.
template <int N>
struct Plan;
#define ARTIA_FFT_PLAN3(N_, E_, A_, B_, C_)                                                           \
    template <>                                                                                      \
    struct Plan<N_> {                                                                                \
        static constexpr int E = E_, T = N_ / E_;                                                    \
        template <bool kInv, int kStep>                                                              \
        __device__ __forceinline__ static void run(C2 v[E_], int t, const float2* tw, C2* lds) {     \
            fft_pass<N_, E_, A_, 1, kInv>(v, t, tw);                                                 \
            fft_exchange<N_, E_, A_, 1, kStep>(v, t, lds);                                           \
            fft_pass<N_, E_, B_, A_, kInv>(v, t, tw);                                                \
            if (C_ > 1) {                                                                            \
                fft_exchange<N_, E_, B_, A_, kStep>(v, t, lds);                                      \
                fft_pass<N_, E_, (C_ > 1 ? C_ : 2), (C_ > 1 ? A_ * B_ : 1), kInv>(v, t, tw);         \
            }                                                                                        \
        }                                                                                            \
    };
ARTIA_FFT_PLAN3(128, 8, 8, 8, 2)
ARTIA_FFT_PLAN3(256, 8, 8, 8, 4)
ARTIA_FFT_PLAN3(512, 8, 8, 8, 8)
ARTIA_FFT_PLAN3(1024, 16, 16, 16, 4)
ARTIA_FFT_PLAN3(2048, 16, 16, 16, 8)
ARTIA_FFT_PLAN3(4096, 16, 16, 16, 16)
#undef ARTIA_FFT_PLAN3

// Complex transforms (row pairs, or columns) per block: four, or two of 4096 (70 KB of LDS, two blocks on a compute
// unit).  Blocks of 512 threads left one small image a handful of them, each thread with its points' CTF factors
// in turn: a 256 x 256 slab filter took 45 us with five blocks of columns, 29.5 with 33 (and eight points a thread
// instead of 16; 31 with library transforms); 40 images of 1024 x 1024 prepared 466 -> 414 us.
template <int N>
struct Shape {
    static constexpr int E = Plan<N>::E, T = Plan<N>::T;
    static constexpr int F = 512 / T < 4 ? 512 / T : 4;   // row pairs
    static constexpr int threads = F * T;
    static constexpr int rows = 2 * F;
    static constexpr int pairs = F / 2;   // pairs of columns per column block
};

// ---------------------------------------------------------------- rows forward

enum { kSrcSquare = 0, kSrcPrep = 1 };

template <int N>
__device__ __forceinline__ float square_pixel(const RowSrc& s, int x, int y, int z) {
    const int xi = x - s.bx, yi = y - s.by;
    if (xi < 0 || xi >= s.W || yi < 0 || yi >= s.H) return 0.0f;
    float v = load_at<float>(s.src + (size_t)z * s.stride, ((uint32_t)yi * (uint32_t)s.pitch + (uint32_t)xi) * 4u);
    if (s.weight) {
        const float w = load_at<float>(s.weight, (uint32_t)(y * N + x) * 4u);
        const int rep = s.rep0 + s.rep_step * z;
        for (int r = 0; r < rep; r++) v = w * v;
    }
    return v;
}

// Rows y and y + 1 of the mirrored raw image of type V, pixels t + T i
template <int N, typename V>
__device__ __forceinline__ void load_raw_rows(const RowSrc& s, int t, int y, int z, C2 v[Shape<N>::E]) {
    constexpr int E = Shape<N>::E, T = Shape<N>::T;
    const V* img = static_cast<const V*>(s.raw) + (size_t)z * s.stride;
    uint32_t row[2];
#pragma unroll
    for (int q = 0; q < 2; q++) {
        int xi, yi;
        mirror_source(s.bx, y + q, s.W, s.H, s.bx, s.by, 0, xi, yi);
        row[q] = (uint32_t)(s.mirror_y ? s.H - yi - 1 : yi) * (uint32_t)s.pitch;
    }
#pragma unroll
    for (int i = 0; i < E; i++) {
        int xi, yi;
        mirror_source(t + T * i, s.by, s.W, s.H, s.bx, s.by, 0, xi, yi);
        v[i].x = (float)load_at<V>(img, (row[0] + (uint32_t)xi) * (uint32_t)sizeof(V));
        v[i].y = (float)load_at<V>(img, (row[1] + (uint32_t)xi) * (uint32_t)sizeof(V));
    }
}

template <int N, int kKind>
__global__ void __launch_bounds__(Shape<N>::threads, 4) rows_forward_kernel(const float2* __restrict__ tw, RowSrc s,
                                                                       float2* __restrict__ spec, size_t zstride) {
    constexpr int E = Shape<N>::E, T = Shape<N>::T, F = Shape<N>::F, R = Shape<N>::rows;
    __shared__ C2 lds[F * padded(N)];
    __shared__ int nbad;
    const int f = (int)threadIdx.x / T, t = (int)threadIdx.x % T, z = (int)blockIdx.y;
    const int y0 = (int)blockIdx.x * R;
    if (kKind == kSrcPrep && threadIdx.x == 0) nbad = 0;
    C2 v[E];
    int bad = 0;
    const int y = y0 + 2 * f;
    if (kKind == kSrcSquare) {
#pragma unroll
        for (int i = 0; i < E; i++) {
            v[i].x = square_pixel<N>(s, t + T * i, y, z);
            v[i].y = square_pixel<N>(s, t + T * i, y + 1, z);
        }
    } else {
        // (one branch on the type for all loads, which then run side by side: a branch for each pixel took
        // twice the time of the kernel)
        switch (s.dtype) {
            case ARTIA_DT_SHORT: load_raw_rows<N, short>(s, t, y, z, v); break;
            case ARTIA_DT_USHORT: load_raw_rows<N, unsigned short>(s, t, y, z, v); break;
            case ARTIA_DT_INT: load_raw_rows<N, int>(s, t, y, z, v); break;
            case ARTIA_DT_UINT: load_raw_rows<N, unsigned>(s, t, y, z, v); break;
            default: load_raw_rows<N, float>(s, t, y, z, v); break;
        }
        if (s.correct || s.norm) {
            const PrepStat st = s.st[z];
#pragma unroll
            for (int i = 0; i < E; i++) {
                v[i].x = prep_pixel(s, st, v[i].x, bad);
                v[i].y = prep_pixel(s, st, v[i].y, bad);
            }
        }
    }
    C2* mine = lds + f * padded(N);
    Plan<N>::template run<false, 1>(v, t, tw, mine);
#pragma unroll
    for (int i = 0; i < E; i++) mine[slot<1>(t + T * i)] = v[i];
    if (kKind == kSrcPrep && bad) atomicAdd(&nbad, bad);
    __syncthreads();
    if (kKind == kSrcPrep && threadIdx.x == 0 && nbad) atomicAdd(&s.st[z].bad, nbad);
    // the two real rows of a transform: X0 = (Z[k] + conj Z[-k]) / 2, X1 = (Z[k] - conj Z[-k]) / 2i; a lane
    // stores two columns of one row, neighbouring lanes the block's rows
    float4* __restrict__ out = reinterpret_cast<float4*>(spec + (size_t)z * zstride);
    for (int e = (int)threadIdx.x; e < (N / 4 + 1) * R; e += Shape<N>::threads) {
        const int r = e % R, p = e / R;
        const C2* Z = lds + (r >> 1) * padded(N);
        C2 X[2];
#pragma unroll
        for (int h = 0; h < 2; h++) {
            const int k = (2 * p + h) & (N - 1);
            const C2 a = Z[slot<1>(k)], b = Z[slot<1>((N - k) & (N - 1))];
            X[h] = (r & 1) ? C2{0.5f * (a.y + b.y), 0.5f * (b.x - a.x)} : C2{0.5f * (a.x + b.x), 0.5f * (a.y - b.y)};
        }
        out[(size_t)p * N + (size_t)(y0 + r)] = make_float4(X[0].x, X[0].y, X[1].x, X[1].y);
    }
}

// ---------------------------------------------------------------- columns

enum { kColForward = 0, kColCtf = 1, kColFan = 2, kColPrep = 3 };

template <int N, int kKind>
__global__ void __launch_bounds__(Shape<N>::threads, 4) cols_kernel(const float2* __restrict__ tw,
                                                               const float2* __restrict__ base,
                                                               float2* __restrict__ spec, size_t zstride, CtfStack ctf,
                                                               PrepFilter pf, const uint32_t* need, uint32_t wanted) {
    constexpr int E = Shape<N>::E, T = Shape<N>::T, P = Shape<N>::pairs;
    __shared__ C2 lds[2 * P * padded(N)];
    // lanes alternate between the two columns of a pair, whose values alternate in memory
    const int g = (int)threadIdx.x / (2 * T), u = (int)threadIdx.x % (2 * T), h = u & 1, t = u >> 1;
    const int z = (int)blockIdx.y;
    if (kKind == kColFan && !((wanted >> z) & 1u)) return;   // whole workgroup
    const int p = min((int)blockIdx.x * P + g, N / 4);   // (the last block repeats the last pair)
    const bool own = (int)blockIdx.x * P + g <= N / 4;
    const int kx = 2 * p + h;
    float2* out = spec + (size_t)z * zstride;
    const float2* in = kKind == kColFan ? base : out;
    const uint32_t off = (uint32_t)(p * N * 2 + 2 * t + h) * 8u;
    C2* mine = lds + g * (2 * padded(N)) + h;
    C2 v[E];
    if (kKind != kColFan) {
#pragma unroll
        for (int i = 0; i < E; i++) {
            const float2 a = load_at<float2>(in, off + (uint32_t)(16 * T * i));
            v[i] = C2{a.x, a.y};
        }
        Plan<N>::template run<false, 2>(v, t, tw, mine);
    }
    if (kKind != kColForward) {
        // the factors in a rolled loop over the thread's own points in LDS: unrolled over registers, the
        // double arithmetic of several points at once spilled up to 500 bytes per lane
        if (kKind != kColFan) {
#pragma unroll
            for (int i = 0; i < E; i++) mine[slot<2>(t + T * i)] = v[i];
        }
        const bool steps = kKind != kColPrep && !ctf.k.phaseFlip && ctf.k.beta[1] == 0.0f && ctf.k.beta[3] == 0.0f;
        double power = 0.0;
#pragma unroll 1
        for (int half = 0; half < 2; half++) {   // frequencies >= 0 and < 0, each outwards (see CtfEnvelopeRun)
            const int step = half ? -T : T;
            CtfEnvelopeRun env{0.0, 0.0, 0.0};
            if (steps) env.start(kx, half ? t - T : t, step, ctf.k);
            int ky = half ? t + T * (E - 1) : t;
#pragma unroll 1
            for (int i = 0; i < E / 2; i++, ky += step) {
                C2* at = mine + slot<2>(ky);
                float2 r;
                if (kKind == kColFan) {
                    r = load_at<float2>(in, (uint32_t)(p * N * 2 + 2 * ky + h) * 8u);
                } else {
                    r = make_float2(at->x, at->y);
                }
                if (kKind == kColPrep) {
                    r = prep_factor(r, kx, ky, N, pf, z);
                    if (pf.dc && kx == 0 && ky == 0) {
                        pf.dc[z] = r.x;
                        // with the statistics from the spectrum the mean leaves here
                        if (pf.power) r = make_float2(0.0f, 0.0f);
                    } else
                        power = __builtin_fma((double)r.x, (double)r.x, __builtin_fma((double)r.y, (double)r.y, power));
                } else {
                    const CtfPoint pt = steps ? ctf_point(kx, ky, ctf.k, env.e) : ctf_point(kx, ky, ctf.k);
                    r = ctf_apply_at(r, pt, ctf.k, ctf.def0[z], ctf.def1[z]);
                    env.next();
                }
                *at = C2{r.x, r.y};
            }
        }
        if (kKind == kColPrep && pf.power) {   // uniform
            // columns 1 .. N / 2 - 1 stand for their mirror images too; the last pair's second is not used
            power = own && kx <= N / 2 ? (kx == 0 || kx == N / 2 ? power : 2.0 * power) : 0.0;
            for (int o = 32; o > 0; o >>= 1) power += __shfl_down(power, o);
            constexpr int waves = Shape<N>::threads / 64;
            if ((threadIdx.x & 63) == 0)
                pf.power[((size_t)z * gridDim.x + blockIdx.x) * waves + (threadIdx.x >> 6)] = power;
        }
#pragma unroll
        for (int i = 0; i < E; i++) v[i] = mine[slot<2>(t + T * i)];
        __syncthreads();
    }
    if (kKind != kColForward) {
        // the table and the offsets behind other names: the forward transform's twiddles and addresses kept
        // for this one would spill
        const float2* tw2 = tw;
        int t2 = t;
        __asm__ volatile("" : "+s"(tw2), "+v"(t2));
        Plan<N>::template run<true, 2>(v, t2, tw2, mine);
    }
    if (own) {
        uint32_t off2 = off;
        __asm__ volatile("" : "+v"(off2));
#pragma unroll
        for (int i = 0; i < E; i++) {
            if (kKind == kColFan && need) {   // uniform
                const int ky = t + T * i;
                if (!((need[(size_t)z * (N / 32) + (ky >> 5)] >> (ky & 31)) & 1u)) continue;
            }
            store_at(out, off2 + (uint32_t)(16 * T * i), make_float2(v[i].x, v[i].y));
        }
    }
}

// ---------------------------------------------------------------- rows back

enum { kDstStore = 0, kDstPrep = 1 };

// Rows y0 .. y0 + rows - 1 of image z, two per transform: v[i] = pixels t + T i of rows y0 + 2 f (x) and
// y0 + 2 f + 1 (y).  Like the library's real transform, the imaginary parts of columns 0 and N / 2 do
// not enter.
template <int N>
__device__ __forceinline__ void rows_back(const float2* __restrict__ tw, const float2* __restrict__ spec, int y0, int f,
                                          int t, C2* __restrict__ lds, C2 v[Shape<N>::E]) {
    constexpr int E = Shape<N>::E, T = Shape<N>::T, R = Shape<N>::rows;
    // the rows' half spectra side by side, N / 2 + 1 each
    const float4* __restrict__ in = reinterpret_cast<const float4*>(spec);
    for (int e = (int)threadIdx.x; e < (N / 4) * R; e += Shape<N>::threads) {
        const int r = e % R, p = e / R;
        const float4 a = in[(size_t)p * N + (size_t)(y0 + r)];
        C2* row = lds + r * (N / 2 + 1) + 2 * p;
        row[0] = C2{a.x, a.y};
        row[1] = C2{a.z, a.w};
    }
    for (int r = (int)threadIdx.x; r < R; r += Shape<N>::threads) {
        const float2 a = spec[((size_t)(N / 4) * N + (size_t)(y0 + r)) * 2];
        lds[r * (N / 2 + 1) + N / 2] = C2{a.x, a.y};
    }
    __syncthreads();
    const C2 *A = lds + (2 * f) * (N / 2 + 1), *B = A + (N / 2 + 1);
#pragma unroll
    for (int i = 0; i < E; i++) {
        const int k = t + T * i;
        if (k <= N / 2) {
            const C2 a = A[k], b = B[k];
            v[i] = (k == 0 || k == N / 2) ? C2{a.x, b.x} : C2{a.x - b.y, a.y + b.x};
        } else {
            const C2 a = A[N - k], b = B[N - k];
            v[i] = C2{a.x + b.y, b.x - a.y};
        }
    }
    __syncthreads();
    Plan<N>::template run<true, 1>(v, t, tw, lds + f * padded(N));
}

template <int N, int kKind>
__global__ void __launch_bounds__(Shape<N>::threads, 4) rows_back_kernel(const float2* __restrict__ tw,
                                                                    const float2* __restrict__ spec, size_t zstride,
                                                                    RowDst d) {
    constexpr int E = Shape<N>::E, T = Shape<N>::T, F = Shape<N>::F;
    __shared__ C2 lds[F * padded(N)];
    const int f = (int)threadIdx.x / T, t = (int)threadIdx.x % T;
    const int y0 = (int)blockIdx.x * Shape<N>::rows, y = y0 + 2 * f - d.by;
    C2 v[E];
    const int z = (int)blockIdx.y;
    if (kKind == kDstStore && d.need) {   // uniform
        constexpr int R = Shape<N>::rows, step = R < 32 ? R : 32;
        uint32_t any = 0;
        for (int r = 0; r < R; r += step)
            any |= (d.need[(size_t)z * (N / 32) + ((y0 + r) >> 5)] >> ((y0 + r) & 31)) & (step == 32 ? ~0u : (1u << (step & 31)) - 1u);
        if (!any) return;   // whole workgroup
    }
    rows_back<N>(tw, spec + (size_t)z * zstride, y0, f, t, lds, v);
    float* out = d.out + (size_t)z * d.stride;
    double s1 = 0.0, s2 = 0.0;
    const double c = kKind == kDstPrep ? (double)(d.dc[z] * d.scale) : 0.0;
#pragma unroll
    for (int i = 0; i < E; i++) {
        const int x = t + T * i - d.bx;
#pragma unroll
        for (int q = 0; q < 2; q++) {
            if (!(x >= 0 && x < d.W && y + q >= 0 && y + q < d.H)) continue;
            float val = (q ? v[i].y : v[i].x) * d.scale;
            const uint32_t at = ((uint32_t)(y + q) * (uint32_t)d.pitch + (uint32_t)x) * 4u;
            if (kKind == kDstStore) {
                if (d.st) val = val / -d.st[z].std_hf;   // uniform
                if (d.weight)
                    val = load_at<float>(d.weight, (uint32_t)((y0 + 2 * f + q) * N + t + T * i) * 4u) * val;
                store_at(out, at, d.accumulate ? load_at<float>(out, at) + val : val);
            } else {
                store_at(out, at, val);
                if (x >= d.rx0 && x < d.rx0 + d.rw && y + q >= d.ry0 && y + q < d.ry0 + d.rh) {
                    const double e = (double)val - c;
                    s1 += e;
                    s2 = __builtin_fma(e, e, s2);
                }
            }
        }
    }
    if (kKind == kDstPrep) {
        for (int o = 32; o > 0; o >>= 1) {
            s1 += __shfl_down(s1, o);
            s2 += __shfl_down(s2, o);
        }
        double* part = reinterpret_cast<double*>(lds);
        const int wave = (int)threadIdx.x >> 6;
        if ((threadIdx.x & 63) == 0) {
            part[2 * wave] = s1;
            part[2 * wave + 1] = s2;
        }
        __syncthreads();
        if (threadIdx.x == 0) {
            for (int w = 1; w < Shape<N>::threads / 64; w++) {
                s1 += part[2 * w];
                s2 += part[2 * w + 1];
            }
            double* o = d.partial + 2 * ((size_t)z * gridDim.x + blockIdx.x);
            o[0] = s1;
            o[1] = s2;
        }
    }
}

// f(integral_constant<N>) for the supported length N
template <class Fn>
void with_length(int N, Fn&& f) {
    switch (N) {
        case 128: f(std::integral_constant<int, 128>()); break;
        case 256: f(std::integral_constant<int, 256>()); break;
        case 512: f(std::integral_constant<int, 512>()); break;
        case 1024: f(std::integral_constant<int, 1024>()); break;
        case 2048: f(std::integral_constant<int, 2048>()); break;
        default: f(std::integral_constant<int, 4096>()); break;
    }
}

template <int kKind>
void launch_rows_forward(artia_ctx* ctx, int N, const float2* tw, const RowSrc& s, float2* spec, int nz) {
    with_length(N, [&](auto n) {
        constexpr int L = decltype(n)::value;
        hipLaunchKernelGGL((rows_forward_kernel<L, kKind>), dim3(L / Shape<L>::rows, (unsigned)nz),
                           dim3(Shape<L>::threads), 0, ctx->stream, tw, s, spec, fft2d_spec_size(L));
    });
}
template <int kKind>
void launch_cols(artia_ctx* ctx, int N, const float2* tw, const float2* base, float2* spec, const CtfStack& c,
                 const PrepFilter& f, int nz, const uint32_t* need = nullptr, uint32_t wanted = ~0u) {
    with_length(N, [&](auto n) {
        constexpr int L = decltype(n)::value;
        hipLaunchKernelGGL((cols_kernel<L, kKind>), dim3((L / 4 + Shape<L>::pairs) / Shape<L>::pairs, (unsigned)nz),
                           dim3(Shape<L>::threads), 0, ctx->stream, tw, base, spec, fft2d_spec_size(L), c, f, need, wanted);
    });
}
template <int kKind>
void launch_rows_back(artia_ctx* ctx, int N, const float2* tw, const float2* spec, const RowDst& d, int nz) {
    with_length(N, [&](auto n) {
        constexpr int L = decltype(n)::value;
        hipLaunchKernelGGL((rows_back_kernel<L, kKind>), dim3(L / Shape<L>::rows, (unsigned)nz),
                           dim3(Shape<L>::threads), 0, ctx->stream, tw, spec, fft2d_spec_size(L), d);
    });
}

}  // namespace

bool fft2d_supports(int N) { return N >= 128 && N <= 4096 && (N & (N - 1)) == 0; }

int fft2d_row_blocks(int N) {
    int n = 0;
    with_length(N, [&](auto l) { n = decltype(l)::value / Shape<decltype(l)::value>::rows; });
    return n;
}

int fft2d_col_waves(int N) {
    int n = 0;
    with_length(N, [&](auto l) {
        constexpr int L = decltype(l)::value;
        n = (L / 4 + Shape<L>::pairs) / Shape<L>::pairs * (Shape<L>::threads / 64);
    });
    return n;
}

void fft2d_rows_square(artia_ctx* ctx, int N, const float2* tw, const RowSrc& s, float2* spec, int nz) {
    launch_rows_forward<kSrcSquare>(ctx, N, tw, s, spec, nz);
}
void fft2d_rows_prep(artia_ctx* ctx, int N, const float2* tw, const RowSrc& s, float2* spec, int nz) {
    launch_rows_forward<kSrcPrep>(ctx, N, tw, s, spec, nz);
}
void fft2d_cols_forward(artia_ctx* ctx, int N, const float2* tw, float2* spec, int nz) {
    launch_cols<kColForward>(ctx, N, tw, nullptr, spec, CtfStack{}, PrepFilter{}, nz);
}
void fft2d_cols_ctf(artia_ctx* ctx, int N, const float2* tw, float2* spec, const CtfStack& c, int nz) {
    launch_cols<kColCtf>(ctx, N, tw, nullptr, spec, c, PrepFilter{}, nz);
}
void fft2d_cols_fan(artia_ctx* ctx, int N, const float2* tw, const float2* base, float2* spec, const CtfStack& c,
                    int nz, const uint32_t* need, uint32_t wanted) {
    launch_cols<kColFan>(ctx, N, tw, base, spec, c, PrepFilter{}, nz, need, wanted);
}
void fft2d_cols_prep(artia_ctx* ctx, int N, const float2* tw, float2* spec, const PrepFilter& f, int nz) {
    launch_cols<kColPrep>(ctx, N, tw, nullptr, spec, CtfStack{}, f, nz);
}
void fft2d_rows_store(artia_ctx* ctx, int N, const float2* tw, const float2* spec, const RowDst& d, int nz) {
    launch_rows_back<kDstStore>(ctx, N, tw, spec, d, nz);
}
void fft2d_rows_prep_store(artia_ctx* ctx, int N, const float2* tw, const float2* spec, const RowDst& d, int nz) {
    launch_rows_back<kDstPrep>(ctx, N, tw, spec, d, nz);
}

}  // namespace artia
