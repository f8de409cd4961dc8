// Fourier-space operators on gfx950: the CTF multiply / Wiener inverse / phase flip (ctf.cu:80-240),
// the WBP weighting (wbpWeighting.cu:48-144), and the fused per-slab image filters that replace
// the reference's cuFFT/NPP glue (Reconstructor.cpp:557-583, 952-965, 1271-1319):
//   slab filter : cropBorder (in place) -> makeSquare (zero fill) -> R2C -> ctf -> C2R ->
//                 / N^2 with crop to W x H -> cropBorder -> store or accumulate
//   WBP filter  : makeSquare (reflect) -> R2C -> wbpWeighting -> C2R -> / N^2 with crop
// For N = 128 .. 4096 a power of two and exact numerics the filters run in three kernels (fft2d.hpp);
// otherwise the FFTs are hipFFT single-precision plans cached per size in the context, on the
// (N/2+1) x N half spectrum, rows of N/2+1 complex values.
#include <algorithm>
#include <cmath>

#include "device_common.hpp"
#include "fft2d.hpp"
#include "image_ops.hpp"
#include "spectral_factors.hpp"

namespace artia {
namespace {

constexpr float kPiF = 3.14159265358979323846f;

// Reference numerics: the kernel body's float operation order.
__global__ void __launch_bounds__(256) ctf_ref_kernel(float2* __restrict__ spec, size_t pitch, CtfK k) {
    const int x = (int)(blockIdx.x * blockDim.x + threadIdx.x);
    const int y = (int)(blockIdx.y * blockDim.y + threadIdx.y);
    if (x >= k.N / 2 + 1 || y >= k.N) return;
    float xpos = (float)x, ypos = (float)y;
    if (ypos > (float)k.N * 0.5f) ypos = ((float)k.N - ypos) * -1.0f;
    const float alpha = (xpos == 0) ? (kPiF * 0.5f) : atan2f(ypos, xpos);
    const float beta = alpha - k.angle;
    const float defocus = k.def0 + (1 - cosf(2 * beta)) * (k.def1 - k.def0);
    float len = sqrtf(xpos * xpos + ypos * ypos);
    len *= k.freq_step;
    const float lam = k.lambda, Cs = k.cs_m;
    const float m = (kPiF / 2.0f) * (Cs * lam * lam * lam * len * len * len * len - 2 * defocus * lam * len * len);
    const float n = k.pc * sinf(m) + k.ac * cosf(m);
    float2 r = spec[(size_t)y * pitch + x];
    const float radius = sqrtf(xpos * xpos + ypos * ypos);
    if (!k.phaseFlip && radius > k.beta[0]) {
        const float l = len / 100000000.0f;
        float e = expf((-k.beta[1] * l - k.beta[2] * l * l) - k.beta[3] * l * l * l);
        if (k.forFP) {
            e = fmaxf(e, 0.01f);
            float val = n * e;
            if (fabsf(val) < 0.0001f && val >= 0) val = 0.0001f;
            if (fabsf(val) < 0.0001f && val < 0) val = -0.0001f;
            r.x = r.x * -val;
            r.y = r.y * -val;
        } else {
            e = fmaxf(e, k.wiener);
            const float val = n * e;
            r.x = r.x * -val / (val * val + k.wiener);
            r.y = r.y * -val / (val * val + k.wiener);
        }
    }
    if (k.phaseFlip && n >= 0) {
        r.x = -r.x;
        r.y = -r.y;
    }
    spec[(size_t)y * pitch + x] = r;
}

// Exact numerics: the CTF factor in double (spectral_factors.hpp), applied to the float spectrum.
__device__ __forceinline__ void ctf_exact_at(float2* __restrict__ spec, size_t pitch, int x, int y, const CtfK& k) {
    const CtfPoint p = ctf_point(x, y, k);
    float2* q = spec + (size_t)y * pitch + x;
    *q = ctf_apply_at(*q, p, k, k.def0, k.def1);
}

__global__ void __launch_bounds__(256) ctf_exact_kernel(float2* __restrict__ spec, size_t pitch, CtfK k) {
    const int x = (int)(blockIdx.x * blockDim.x + threadIdx.x);
    const int y = (int)(blockIdx.y * blockDim.y + threadIdx.y);
    if (x >= k.N / 2 + 1 || y >= k.N) return;
    ctf_exact_at(spec, pitch, x, y, k);
}

// The same over a stack of half spectra (stride N * (N/2+1)), each slab with its own defocus.
__global__ void __launch_bounds__(256) ctf_exact_stack_kernel(float2* __restrict__ spec, size_t pitch, CtfStack b,
                                                              int ns) {
    const int x = (int)(blockIdx.x * blockDim.x + threadIdx.x);
    const int y = (int)(blockIdx.y * blockDim.y + threadIdx.y);
    if (x >= b.k.N / 2 + 1 || y >= b.k.N) return;
    const CtfPoint p = ctf_point(x, y, b.k);   // once for the stack's ns spectra
    float2* q = spec + (size_t)y * pitch + x;
    const size_t plane = pitch * (size_t)b.k.N;
    for (int s = 0; s < ns; s++) q[(size_t)s * plane] = ctf_apply_at(q[(size_t)s * plane], p, b.k, b.def0[s], b.def1[s]);
}

// ns slabs of ONE image: spectrum s = base * CTF(slab s's defocus) * scale.  scale is 1, or 1 / N^2
// (a power of two, so the product is exact) when the inverse transform writes the slab images
// straight into their destination: C2R(scale X) = scale C2R(X) bit for bit, which is the
// division by N^2 of the finishing pass.
__global__ void __launch_bounds__(256) ctf_exact_fan_kernel(const float2* __restrict__ base,
                                                            float2* __restrict__ spec, size_t pitch, CtfStack b,
                                                            int ns, float scale) {
    const int x = (int)(blockIdx.x * blockDim.x + threadIdx.x);
    const int y = (int)(blockIdx.y * blockDim.y + threadIdx.y);
    if (x >= b.k.N / 2 + 1 || y >= b.k.N) return;
    const CtfPoint p = ctf_point(x, y, b.k);
    const size_t i = (size_t)y * pitch + x, plane = pitch * (size_t)b.k.N;
    const float2 r0 = base[i];
    for (int s = 0; s < ns; s++) {
        float2 r = ctf_apply_at(r0, p, b.k, b.def0[s], b.def1[s]);
        r.x = r.x * scale;
        r.y = r.y * scale;
        spec[(size_t)s * plane + i] = r;
    }
}

// wbpWeighting.cu:48-144 over a stack of spectra (sin/cos of the angles as IEEE functions rather than
// __sinf/__cosf)
struct WbpStack {
    float ang[kFftBatchMax];
    double sn[kFftBatchMax], cs[kFftBatchMax];
};

__global__ void __launch_bounds__(256) wbp_weight_kernel(float2* __restrict__ spec, size_t pitch, int N, WbpStack a,
                                                         int method, int exact) {
    const int x = (int)(blockIdx.x * blockDim.x + threadIdx.x);
    const int y = (int)(blockIdx.y * blockDim.y + threadIdx.y);
    if (x >= N / 2 + 1 || y >= N) return;
    spec += (size_t)blockIdx.z * pitch * (size_t)N;
    if (exact) {
        spec[(size_t)y * pitch + x] =
            wbp_weighted(spec[(size_t)y * pitch + x], x, y, N, a.sn[blockIdx.z], a.cs[blockIdx.z], method);
        return;
    }
    const unsigned pc = (unsigned)N;
    const float ang = a.ang[blockIdx.z];
    float w = 1.0f;
    float xpos = (float)x, ypos = (float)y;
    if (ypos > (float)pc * 0.5f) ypos = ((float)pc - ypos) * -1.0f;
    const float temp = xpos;
    const float sn = sinf(ang), cs = cosf(ang);
    xpos = cs * xpos - sn * ypos;
    ypos = sn * temp + cs * ypos;
    const float len = ypos / (float)pc / 2.0f;
    if (method == 0) {
        w = fminf(fabsf(len), 1.0f);
    } else if (method >= 2 && method <= 4) {
        const float P[3][4] = {{1.000654227857550f, 0.006008581017124f, 0.004159659493151f, 0.000975903396538f},
                               {1.003784816598589f, 0.029016377161629f, 0.019582940715148f, 0.004559409669984f},
                               {0.999884616010943f, 0.000307646262566f, 0.004742915272196f, 0.004806551368900f}};
        const float* q = P[method - 2];
        if (len == 0) {
            w = 0;
        } else {
            const float L = logf(fabsf(len));
            w = ((q[0] + q[1] * L) + q[2] * L * L) + q[3] * L * L * L;
        }
        w = fmaxf(0.0f, fminf(w, 1.0f));
    }
    float2 r = spec[(size_t)y * pitch + x];
    r.x *= w;
    r.y *= w;
    spec[(size_t)y * pitch + x] = r;
}

// out (+)= crop(x, y) * (square[by + y][bx + x] / N^2)  (nppiDivC + cropBorder + nppiAdd); over a
// stack of ns squares, square s into out + s * out_stride
__global__ void __launch_bounds__(256) finish_kernel(const float* __restrict__ sq, int ns, int N, int bx, int by, int W,
                                                     int H, float* __restrict__ out, size_t pitch, float norm,
                                                     int accumulate, int crop, CropParams cp, size_t out_stride) {
    const int x = (int)(blockIdx.x * blockDim.x + threadIdx.x);
    const int y = (int)(blockIdx.y * blockDim.y + threadIdx.y);
    if (x >= W || y >= H) return;
    // the crop weight depends on the pixel only: evaluated once for the ns squares
    const float w = crop ? crop_weight(x, y, W, H, cp) : 1.0f;
    const size_t j = (size_t)(by + y) * N + (bx + x), plane = (size_t)N * (size_t)N;
    const size_t i = (size_t)y * pitch + x;
    for (int s = 0; s < ns; s++) {
        float v = sq[(size_t)s * plane + j] / norm;
        if (crop) v = w * v;
        float* o = out + (size_t)s * out_stride;
        o[i] = accumulate ? o[i] + v : v;
    }
}

// out += crop(x, y) * (square_s[by + y][bx + x] / N^2) for s = 0 .. ns-1 in turn: the sum, rounded
// after every slab, of ns accumulating finish_kernel calls
__global__ void __launch_bounds__(256) finish_sum_kernel(const float* __restrict__ sq, int ns, int N, int bx, int by,
                                                         int W, int H, float* __restrict__ out, size_t pitch,
                                                         float norm, int crop, CropParams cp) {
    const int x = (int)(blockIdx.x * blockDim.x + threadIdx.x);
    const int y = (int)(blockIdx.y * blockDim.y + threadIdx.y);
    if (x >= W || y >= H) return;
    const float w = crop ? crop_weight(x, y, W, H, cp) : 1.0f;
    const size_t i = (size_t)y * pitch + x;
    const size_t j = (size_t)(by + y) * N + (bx + x), plane = (size_t)N * (size_t)N;
    float acc = out[i];
    for (int s = 0; s < ns; s++) {
        float v = sq[(size_t)s * plane + j] / norm;
        if (crop) v = w * v;
        acc = acc + v;
    }
    out[i] = acc;
}

// Zero-filled centred squares of a stack of ns slab images: square_s = makeSquare(cropBorder^r(src_s))
// with r = rep0 + rep_step * s crops applied in turn (rep_step 1: the repeated in-place crop of one
// image, src_stride 0, carried from slab to slab with one multiplication each)
__global__ void __launch_bounds__(256) slab_square_kernel(const float* __restrict__ src, size_t src_stride, int W,
                                                          int H, size_t pitch, int N, int bx, int by,
                                                          float* __restrict__ sq, CropParams cp, int rep0,
                                                          int rep_step, int ns) {
    const int x = (int)(blockIdx.x * blockDim.x + threadIdx.x);
    const int y = (int)(blockIdx.y * blockDim.y + threadIdx.y);
    if (x >= N || y >= N) return;
    const size_t plane = (size_t)N * (size_t)N;
    float* o = sq + (size_t)y * N + x;
    const int xi = x - bx, yi = y - by;
    if (!(xi >= 0 && xi < W && yi >= 0 && yi < H)) {
        for (int s = 0; s < ns; s++) o[(size_t)s * plane] = 0.0f;
        return;
    }
    const float* in = src + (size_t)yi * pitch + xi;
    const float w = (rep0 > 0 || rep_step > 0) ? crop_weight(xi, yi, W, H, cp) : 1.0f;
    if (rep_step == 0) {
        for (int s = 0; s < ns; s++) {
            float val = in[(size_t)s * src_stride];
            for (int r = 0; r < rep0; r++) val = w * val;
            o[(size_t)s * plane] = val;
        }
    } else {
        float val = in[0];
        for (int r = 0; r < rep0; r++) val = w * val;
        for (int s = 0; s < ns; s++) {
            o[(size_t)s * plane] = val;
            val = w * val;
        }
    }
}

dim3 grid2d(int w, int h) { return dim3((unsigned)((w + 63) / 64), (unsigned)((h + 3) / 4)); }

CtfK make_ctf(int N, const artia_ctf_params& p, float dmin_nm, float dmax_nm, float angle_deg, int forFP) {
    CtfK k;
    k.cs_m = p.cs_mm * 0.001f;
    k.lambda = ctf_wavelength(p.voltage_kV);
    const float ps = p.pixelsize_nm * powf(10.0f, -9.0f);
    const float maxFreq = (float)(1.0 / (double)(ps * 2.0f));
    k.freq_step = maxFreq / ((float)N / 2.0f);
    k.ac = p.amp_contrast;
    k.pc = sqrtf(1 - p.amp_contrast * p.amp_contrast);
    k.halfN = (float)N * 0.5f;
    k.def0 = dmin_nm * 0.000000001f;
    k.def1 = dmax_nm * 0.000000001f;
    k.angle = angle_deg / 180.0f * kPiF;
    k.wiener = p.wiener;
    for (int i = 0; i < 4; i++) k.beta[i] = p.beta_fac[i];
    k.forFP = forFP;
    k.phaseFlip = p.phase_flip_only;
    k.N = N;
    k.cos2a = cos(2.0 * (double)k.angle);
    k.sin2a = sin(2.0 * (double)k.angle);
    return k;
}

// Defocus pairs of slabs 0 .. b - 1.
CtfStack make_ctf_stack(int N, const artia_ctf_params& p, const float* dmin_nm, const float* dmax_nm, float angle_deg,
                        int forFP, int b) {
    CtfStack cs{};
    cs.k = make_ctf(N, p, dmin_nm[0], dmax_nm[0], angle_deg, forFP);
    for (int s = 0; s < b; s++) {
        const CtfK ks = make_ctf(N, p, dmin_nm[s], dmax_nm[s], angle_deg, forFP);
        cs.def0[s] = ks.def0;
        cs.def1[s] = ks.def1;
    }
    return cs;
}

// cropBorder's weights at the places of the image in its square, 0 around them
__global__ void __launch_bounds__(256) square_weight_kernel(float* __restrict__ out, int N, int W, int H, int bx, int by,
                                                            CropParams cp) {
    const int x = (int)(blockIdx.x * blockDim.x + threadIdx.x);
    const int y = (int)(blockIdx.y * blockDim.y + threadIdx.y);
    if (x >= N || y >= N) return;
    const int xi = x - bx, yi = y - by;
    out[(size_t)y * N + x] = xi >= 0 && xi < W && yi >= 0 && yi < H ? crop_weight(xi, yi, W, H, cp) : 0.0f;
}

// out += img_s for s = 0 .. ns - 1 in turn, rounded after every image
__global__ void __launch_bounds__(256) sum_images_kernel(const float* __restrict__ img, size_t stride, int ns, int W, int H,
                                                         float* __restrict__ out, size_t pitch) {
    const int x = (int)(blockIdx.x * blockDim.x + threadIdx.x);
    const int y = (int)(blockIdx.y * blockDim.y + threadIdx.y);
    if (x >= W || y >= H) return;
    const float* p = img + ((size_t)y * W + x);
    float* o = out + ((size_t)y * pitch + x);
    float acc = *o;
    for (int s0 = 0; s0 < ns; s0 += 8) {
        float v[8];
#pragma unroll
        for (int s = 0; s < 8; s++) v[s] = p[(size_t)min(s0 + s, ns - 1) * stride];
#pragma unroll
        for (int s = 0; s < 8; s++)
            if (s0 + s < ns) acc = acc + v[s];
    }
    *o = acc;
}

RowSrc square_source(const float* src, size_t stride, int W, int H, size_t pitch, int N) {
    RowSrc s{};
    s.W = W;
    s.H = H;
    s.bx = (N - W) / 2;
    s.by = (N - H) / 2;
    s.src = src;
    s.pitch = pitch;
    s.stride = stride;
    return s;
}
RowDst square_target(float* out, size_t stride, int W, int H, size_t pitch, int N, const float* weight, int accumulate) {
    RowDst d{};
    d.W = W;
    d.H = H;
    d.bx = (N - W) / 2;
    d.by = (N - H) / 2;
    d.scale = 1.0f / ((float)N * (float)N);
    d.out = out;
    d.pitch = pitch;
    d.stride = stride;
    d.weight = weight;
    d.accumulate = accumulate;
    return d;
}

// ctf_filter_slabs over the three-kernel filter (fft2d.hpp)
artia_status ctf_filter_slabs_own(artia_ctx* ctx, const float* src, size_t src_stride, int n, int W, int H, size_t pitch,
                                  float* out, size_t out_stride, const int corners[8], const float cut[2],
                                  const float dim[2], const artia_ctf_params& p, const float* dmin_nm,
                                  const float* dmax_nm, float angle_deg, int forFP, const uint32_t* need,
                                  const unsigned char* wanted) {
    const int N = W > H ? W : H;
    FftOwn& f = ctx->ffto;
    artia_status st = f.ensure(ctx, N, FftOwn::kStack | (corners ? FftOwn::kWeight : 0) | (forFP ? FftOwn::kImages : 0));
    if (st != ARTIA_OK) return st;
    const float* weight = nullptr;
    if (corners) {
        weight = f.weight;
        hipLaunchKernelGGL(square_weight_kernel, grid2d(N, N), dim3(64, 4), 0, ctx->stream, f.weight, N, W, H, (N - W) / 2,
                           (N - H) / 2, make_crop_params(cut, dim, corners));
    }
    // every slab filtering the same uncropped image (the sub-volume WBP): one forward transform, kept in
    // the spare slot, serves all slabs
    const bool shared = src_stride == 0 && !corners;
    float2* base = f.spec + (size_t)f.cap * fft2d_spec_size(N);
    RowSrc s = square_source(src, src_stride, W, H, pitch, N);
    if (shared) {
        fft2d_rows_square(ctx, N, f.tw, s, base, 1);
        fft2d_cols_forward(ctx, N, f.tw, base, 1);
    }
    for (int k0 = 0; k0 < n; k0 += f.cap) {
        const int b = std::min(f.cap, n - k0);
        const CtfStack cs = make_ctf_stack(N, p, dmin_nm + k0, dmax_nm + k0, angle_deg, forFP, b);
        if (shared) {
            uint32_t use = ~0u;
            if (need && wanted) {
                use = 0;
                for (int i = 0; i < b; i++) use |= wanted[k0 + i] ? 1u << i : 0u;
                if (!use) {
                    need += (size_t)b * (size_t)(N / 32);
                    continue;
                }
            }
            fft2d_cols_fan(ctx, N, f.tw, base, f.spec, cs, b, need, use);
        } else {
            s.src = src + (size_t)k0 * src_stride;
            s.weight = weight;
            s.rep0 = !corners ? 0 : (forFP ? 1 : k0 + 1);
            s.rep_step = corners && !forFP ? 1 : 0;
            fft2d_rows_square(ctx, N, f.tw, s, f.spec, b);
            fft2d_cols_ctf(ctx, N, f.tw, f.spec, cs, b);
        }
        if (forFP) {
            const size_t plane = (size_t)W * (size_t)H;
            fft2d_rows_store(ctx, N, f.tw, f.spec, square_target(f.images, plane, W, H, (size_t)W, N, weight, 0), b);
            hipLaunchKernelGGL(sum_images_kernel, grid2d(W, H), dim3(64, 4), 0, ctx->stream, f.images, plane, b, W, H, out,
                               pitch);
        } else {
            RowDst d = square_target(out + (size_t)k0 * out_stride, out_stride, W, H, pitch, N, weight, 0);
            d.need = shared ? need : nullptr;
            fft2d_rows_store(ctx, N, f.tw, f.spec, d, b);
            if (need) need += (size_t)b * (size_t)(N / 32);
        }
        if ((st = check_hip(ctx, hipGetLastError(), "stacked slab filter")) != ARTIA_OK) return st;
    }
    return ARTIA_OK;
}

}  // namespace

// ctf.cu:47-63 with the kernel's float constants (h = 6.63e-34, c = 3e8, E0 = 511 keV)
float ctf_wavelength(float voltage_kV) {
    const float h = (float)6.63E-34, c = (float)3.00E+08;
    const int E0 = 511;
    const float a = (2 * E0 * voltage_kV * 1000.0f * 1000.0f) + (voltage_kV * voltage_kV * 1000.0f * 1000.0f);
    const double arg = (double)a * 1.602E-19 * 1.602E-19;
    return (h * c) / sqrtf((float)arg);
}

artia_status FftPlans::ensure(artia_ctx* ctx, int n) {
    if (N == n && r2c && c2r) return ARTIA_OK;
    release();
    if (hipfftPlan2d(&r2c, n, n, HIPFFT_R2C) != HIPFFT_SUCCESS ||
        hipfftPlan2d(&c2r, n, n, HIPFFT_C2R) != HIPFFT_SUCCESS) {
        release();
        return fail(ctx, ARTIA_ERR_FFT, "hipfftPlan2d(%d x %d) failed", n, n);
    }
    artia_status st = check_hip(ctx, hipMalloc(&square, (size_t)n * n * sizeof(float)), "hipMalloc(square)");
    if (st != ARTIA_OK) {
        release();
        return st;
    }
    st = check_hip(ctx, hipMalloc(&spec, (size_t)(n / 2 + 1) * n * sizeof(float2)), "hipMalloc(spectrum)");
    if (st != ARTIA_OK) {
        release();
        return st;
    }
    N = n;
    return ARTIA_OK;
}

void FftPlans::release() {
    if (r2c) hipfftDestroy(r2c);
    if (c2r) hipfftDestroy(c2r);
    if (square) (void)hipFree(square);
    if (spec) (void)hipFree(spec);
    r2c = c2r = 0;
    square = nullptr;
    spec = nullptr;
    N = 0;
}

artia_status FftBatch::ensure(artia_ctx* ctx, int n) {
    if (N == n && cap > 0) return ARTIA_OK;
    release();
    const double per_slab = (double)n * n * sizeof(float) + (double)(n / 2 + 1) * n * sizeof(float2);
    int c = kFftBatchMax;
    while (c > 1 && (double)c * per_slab > 2147483648.0) c /= 2;
    size_t work_bytes = 0;
    int dims[2] = {n, n};
    for (int i = 0, b = 1; b <= c; i++, b *= 2) {
        size_t w1 = 0, w2 = 0;
        if (hipfftCreate(&r2c[i]) != HIPFFT_SUCCESS || hipfftCreate(&c2r[i]) != HIPFFT_SUCCESS ||
            hipfftSetAutoAllocation(r2c[i], 0) != HIPFFT_SUCCESS ||
            hipfftSetAutoAllocation(c2r[i], 0) != HIPFFT_SUCCESS ||
            hipfftMakePlanMany(r2c[i], 2, dims, nullptr, 1, n * n, nullptr, 1, n * (n / 2 + 1), HIPFFT_R2C, b,
                               &w1) != HIPFFT_SUCCESS ||
            hipfftMakePlanMany(c2r[i], 2, dims, nullptr, 1, n * (n / 2 + 1), nullptr, 1, n * n, HIPFFT_C2R, b,
                               &w2) != HIPFFT_SUCCESS) {
            release();
            return fail(ctx, ARTIA_ERR_FFT, "hipfftMakePlanMany(%d x %d, batch %d) failed", n, n, b);
        }
        work_bytes = std::max(work_bytes, std::max(w1, w2));
    }
    artia_status st = check_hip(ctx, hipMalloc(&square, (size_t)c * n * n * sizeof(float)), "hipMalloc(squares)");
    if (st == ARTIA_OK)
        st = check_hip(ctx, hipMalloc(&spec, (size_t)(c + 1) * (n / 2 + 1) * n * sizeof(float2)), "hipMalloc(spectra)");
    if (st == ARTIA_OK && work_bytes > 0)
        st = check_hip(ctx, hipMalloc(&work, work_bytes), "hipMalloc(fft work area)");
    if (st != ARTIA_OK) {
        release();
        return st;
    }
    for (int i = 0, b = 1; b <= c; i++, b *= 2) {
        if (hipfftSetWorkArea(r2c[i], work) != HIPFFT_SUCCESS || hipfftSetWorkArea(c2r[i], work) != HIPFFT_SUCCESS) {
            release();
            return fail(ctx, ARTIA_ERR_FFT, "hipfftSetWorkArea failed");
        }
    }
    N = n;
    cap = c;
    return ARTIA_OK;
}

void FftBatch::release() {
    for (int i = 0; i < kFftBatchPlans; i++) {
        if (r2c[i]) hipfftDestroy(r2c[i]);
        if (c2r[i]) hipfftDestroy(c2r[i]);
        r2c[i] = c2r[i] = 0;
    }
    if (square) (void)hipFree(square);
    if (spec) (void)hipFree(spec);
    if (work) (void)hipFree(work);
    square = nullptr;
    spec = nullptr;
    work = nullptr;
    N = cap = 0;
}

artia_status FftOwn::ensure(artia_ctx* ctx, int n, int buffers) {
    const size_t image = (size_t)n * n * sizeof(float), spectrum = fft2d_spec_size(n) * sizeof(float2);
    artia_status st = ARTIA_OK;
    if (N != n) {
        release();
        std::vector<float2> t((size_t)n);
        for (int k = 0; k < n; k++) {
            const double a = -2.0 * 3.14159265358979323846 * (double)k / (double)n;
            t[(size_t)k] = make_float2((float)std::cos(a), (float)std::sin(a));
        }
        st = check_hip(ctx, hipMalloc(&tw, (size_t)n * sizeof(float2)), "hipMalloc(twiddles)");
        if (st == ARTIA_OK)
            st = check_hip(ctx, hipMemcpy(tw, t.data(), (size_t)n * sizeof(float2), hipMemcpyHostToDevice),
                           "hipMemcpy(twiddles)");
        if (st != ARTIA_OK) {
            release();
            return st;
        }
        N = n;
        // up to eight spectra of 4096 (540 MB) at a time: a 4096 x 4096 image takes 95.5 us of column and row
        // kernels alone, 86 us in pairs or fours and 81.5 us among eight (fewer nearly empty last waves of blocks)
        cap = (int)std::min<size_t>((size_t)kFftBatchMax, std::max<size_t>(1, ((size_t)544 << 20) / spectrum));
    }
    if ((buffers & kOne) && !one) st = check_hip(ctx, hipMalloc(&one, spectrum), "hipMalloc(spectrum)");
    if (buffers & kOne) buffers |= kWeight;
    if (st == ARTIA_OK && (buffers & kStack) && !spec)
        st = check_hip(ctx, hipMalloc(&spec, (size_t)(cap + 1) * spectrum), "hipMalloc(spectra)");
    if (st == ARTIA_OK && (buffers & kWeight) && !weight)
        st = check_hip(ctx, hipMalloc(&weight, image), "hipMalloc(crop weights)");
    if (st == ARTIA_OK && (buffers & kImages) && !images)
        st = check_hip(ctx, hipMalloc(&images, (size_t)cap * image), "hipMalloc(slab images)");
    return st;
}

void FftOwn::release() {
    for (void* p : {(void*)tw, (void*)one, (void*)spec, (void*)weight, (void*)images})
        if (p) (void)hipFree(p);
    tw = one = spec = nullptr;
    weight = images = nullptr;
    N = cap = 0;
}

artia_status run_ctf(artia_ctx* ctx, float2* spec, int N, size_t pitch, const artia_ctf_params& p, float dmin_nm,
                     float dmax_nm, float angle_deg, int forFP) {
    const CtfK k = make_ctf(N, p, dmin_nm, dmax_nm, angle_deg, forFP);
    if (ctx->numerics == ARTIA_NUMERICS_REFERENCE)
        hipLaunchKernelGGL(ctf_ref_kernel, grid2d(N / 2 + 1, N), dim3(64, 4), 0, ctx->stream, spec, pitch, k);
    else
        hipLaunchKernelGGL(ctf_exact_kernel, grid2d(N / 2 + 1, N), dim3(64, 4), 0, ctx->stream, spec, pitch, k);
    return check_hip(ctx, hipGetLastError(), "ctf launch");
}

artia_status run_wbp_weight(artia_ctx* ctx, float2* spec, int N, size_t pitch, const float* psi_deg, int n, int method) {
    for (int k0 = 0; k0 < n; k0 += kFftBatchMax) {
        const int b = std::min(kFftBatchMax, n - k0);
        WbpStack a{};
        for (int i = 0; i < b; i++) {
            a.ang[i] = -psi_deg[k0 + i] / 180.0f * kPiF;
            a.sn[i] = sin((double)a.ang[i]);
            a.cs[i] = cos((double)a.ang[i]);
        }
        dim3 g = grid2d(N / 2 + 1, N);
        g.z = (unsigned)b;
        hipLaunchKernelGGL(wbp_weight_kernel, g, dim3(64, 4), 0, ctx->stream, spec + (size_t)k0 * pitch * (size_t)N, pitch,
                           N, a, method, ctx->numerics == ARTIA_NUMERICS_EXACT ? 1 : 0);
    }
    return check_hip(ctx, hipGetLastError(), "wbpWeighting launch");
}

artia_status ctf_slab_filter(artia_ctx* ctx, float* img, int W, int H, size_t pitch, float* out, size_t out_pitch,
                             int accumulate, const int corners[8], const float cut[2], const float dim[2],
                             const artia_ctf_params& p, float dmin_nm, float dmax_nm, float angle_deg, int forFP) {
    const int N = W > H ? W : H;
    if (fft2d_supports(N) && fft2d_fits(H, pitch) && fft2d_fits(H, out_pitch) && ctx->numerics == ARTIA_NUMERICS_EXACT) {
        FftOwn& f = ctx->ffto;
        const artia_status so = f.ensure(ctx, N, FftOwn::kOne);
        if (so != ARTIA_OK) return so;
        if (corners) {
            launch_crop_border(ctx, W, H, pitch, img, cut, dim, corners);
            hipLaunchKernelGGL(square_weight_kernel, grid2d(N, N), dim3(64, 4), 0, ctx->stream, f.weight, N, W, H,
                               (N - W) / 2, (N - H) / 2, make_crop_params(cut, dim, corners));
        }
        fft2d_rows_square(ctx, N, f.tw, square_source(img, 0, W, H, pitch, N), f.one, 1);
        fft2d_cols_ctf(ctx, N, f.tw, f.one, make_ctf_stack(N, p, &dmin_nm, &dmax_nm, angle_deg, forFP, 1), 1);
        fft2d_rows_store(ctx, N, f.tw, f.one,
                         square_target(out, 0, W, H, out_pitch, N, corners ? f.weight : nullptr, accumulate), 1);
        return check_hip(ctx, hipGetLastError(), "slab filter");
    }
    artia_status st = ctx->fft.ensure(ctx, N);
    if (st != ARTIA_OK) return st;
    if (corners) launch_crop_border(ctx, W, H, pitch, img, cut, dim, corners);
    launch_make_square(ctx, W, H, pitch, img, N, ctx->fft.square, (N - W) / 2, (N - H) / 2, 0, 1);
    if (hipfftSetStream(ctx->fft.r2c, ctx->stream) != HIPFFT_SUCCESS ||
        hipfftSetStream(ctx->fft.c2r, ctx->stream) != HIPFFT_SUCCESS)
        return fail(ctx, ARTIA_ERR_FFT, "hipfftSetStream failed");
    if (hipfftExecR2C(ctx->fft.r2c, ctx->fft.square, (hipfftComplex*)ctx->fft.spec) != HIPFFT_SUCCESS)
        return fail(ctx, ARTIA_ERR_FFT, "hipfftExecR2C failed");
    st = run_ctf(ctx, ctx->fft.spec, N, (size_t)(N / 2 + 1), p, dmin_nm, dmax_nm, angle_deg, forFP);
    if (st != ARTIA_OK) return st;
    if (hipfftExecC2R(ctx->fft.c2r, (hipfftComplex*)ctx->fft.spec, ctx->fft.square) != HIPFFT_SUCCESS)
        return fail(ctx, ARTIA_ERR_FFT, "hipfftExecC2R failed");
    const CropParams cp = corners ? make_crop_params(cut, dim, corners) : CropParams{};
    hipLaunchKernelGGL(finish_kernel, grid2d(W, H), dim3(64, 4), 0, ctx->stream, ctx->fft.square, 1, N, (N - W) / 2,
                       (N - H) / 2, W, H, out, out_pitch, (float)(N * N), accumulate, corners ? 1 : 0, cp, (size_t)0);
    return check_hip(ctx, hipGetLastError(), "slab filter");
}

int slab_row_block(int W, int H) {
    const int N = W > H ? W : H;
    return fft2d_supports(N) ? N / fft2d_row_blocks(N) : 0;
}

artia_status ctf_filter_slabs(artia_ctx* ctx, const float* src, size_t src_stride, int n, int W, int H, size_t pitch,
                              float* out, size_t out_stride, const int corners[8], const float cut[2],
                              const float dim[2], const artia_ctf_params& p, const float* dmin_nm,
                              const float* dmax_nm, float angle_deg, int forFP, const uint32_t* need,
                              const unsigned char* wanted) {
    if (n <= 0) return ARTIA_OK;
    const int N = W > H ? W : H;
    if (fft2d_supports(N) && fft2d_fits(H, pitch))
        return ctf_filter_slabs_own(ctx, src, src_stride, n, W, H, pitch, out, out_stride, corners, cut, dim, p, dmin_nm,
                                    dmax_nm, angle_deg, forFP, need, wanted);
    FftBatch& fb = ctx->fftb;
    artia_status st = fb.ensure(ctx, N);
    if (st != ARTIA_OK) return st;
    const int crop = corners ? 1 : 0;
    const CropParams cp = crop ? make_crop_params(cut, dim, corners) : CropParams{};
    const int bx = (N - W) / 2, by = (N - H) / 2;
    const size_t half = (size_t)(N / 2 + 1);
    // Every slab filtering the same uncropped image (the sub-volume WBP): one forward transform,
    // kept in the spare spectrum slot, serves all slabs.  When the slab images are whole squares
    // of a power-of-two edge stored back to back, the inverse transform writes them in place with
    // 1 / N^2 folded into the CTF factor.
    const bool shared = src_stride == 0 && !crop;
    const bool direct = shared && !forFP && W == N && H == N && pitch == (size_t)N &&
                        out_stride == (size_t)N * (size_t)N && (N & (N - 1)) == 0;
    float2* base = fb.spec + (size_t)fb.cap * half * (size_t)N;
    if (shared) {
        hipLaunchKernelGGL(slab_square_kernel, dim3((unsigned)((N + 63) / 64), (unsigned)((N + 3) / 4)), dim3(64, 4), 0,
                           ctx->stream, src, (size_t)0, W, H, pitch, N, bx, by, fb.square, cp, 0, 0, 1);
        if (hipfftSetStream(fb.r2c[0], ctx->stream) != HIPFFT_SUCCESS)
            return fail(ctx, ARTIA_ERR_FFT, "hipfftSetStream failed");
        if (hipfftExecR2C(fb.r2c[0], fb.square, (hipfftComplex*)base) != HIPFFT_SUCCESS)
            return fail(ctx, ARTIA_ERR_FFT, "hipfftExecR2C failed");
    }
    for (int k0 = 0; k0 < n;) {
        // the largest power-of-two batch that fits: at most log2(cap) + 1 chunks past the full ones
        int b = fb.cap, pi = 0;
        while (b > n - k0) b /= 2;
        for (int t = b; t > 1; t /= 2) pi++;
        if (hipfftSetStream(fb.r2c[pi], ctx->stream) != HIPFFT_SUCCESS ||
            hipfftSetStream(fb.c2r[pi], ctx->stream) != HIPFFT_SUCCESS)
            return fail(ctx, ARTIA_ERR_FFT, "hipfftSetStream failed");
        if (!shared) {
            hipLaunchKernelGGL(slab_square_kernel, dim3((unsigned)((N + 63) / 64), (unsigned)((N + 3) / 4)),
                               dim3(64, 4), 0, ctx->stream, src + (size_t)k0 * src_stride, src_stride, W, H, pitch, N,
                               bx, by, fb.square, cp, !crop ? 0 : (forFP ? 1 : k0 + 1), crop && !forFP ? 1 : 0, b);
            if (hipfftExecR2C(fb.r2c[pi], fb.square, (hipfftComplex*)fb.spec) != HIPFFT_SUCCESS)
                return fail(ctx, ARTIA_ERR_FFT, "hipfftExecR2C (batch %d) failed", b);
        }
        const CtfStack cs = make_ctf_stack(N, p, dmin_nm + k0, dmax_nm + k0, angle_deg, forFP, b);
        const dim3 sgrid((unsigned)((N / 2 + 1 + 63) / 64), (unsigned)((N + 3) / 4));
        if (shared)
            hipLaunchKernelGGL(ctf_exact_fan_kernel, sgrid, dim3(64, 4), 0, ctx->stream, base, fb.spec, half, cs, b,
                               direct ? 1.0f / ((float)N * (float)N) : 1.0f);
        else
            hipLaunchKernelGGL(ctf_exact_stack_kernel, sgrid, dim3(64, 4), 0, ctx->stream, fb.spec, half, cs, b);
        float* inv = direct ? out + (size_t)k0 * out_stride : fb.square;
        if (hipfftExecC2R(fb.c2r[pi], (hipfftComplex*)fb.spec, inv) != HIPFFT_SUCCESS)
            return fail(ctx, ARTIA_ERR_FFT, "hipfftExecC2R (batch %d) failed", b);
        if (direct) {
            // the slab images are written
        } else if (forFP)
            hipLaunchKernelGGL(finish_sum_kernel, grid2d(W, H), dim3(64, 4), 0, ctx->stream, fb.square, b, N, bx, by, W,
                               H, out, pitch, (float)(N * N), crop, cp);
        else
            hipLaunchKernelGGL(finish_kernel, grid2d(W, H), dim3(64, 4), 0, ctx->stream, fb.square, b, N, bx, by, W, H,
                               out + (size_t)k0 * out_stride, pitch, (float)(N * N), 0, crop, cp, out_stride);
        st = check_hip(ctx, hipGetLastError(), "stacked slab filter");
        if (st != ARTIA_OK) return st;
        k0 += b;
    }
    return ARTIA_OK;
}

artia_status wbp_filter(artia_ctx* ctx, const float* img, int W, int H, size_t pitch, float* out, size_t out_pitch,
                        float psi_deg, int method) {
    const int N = W > H ? W : H;
    if (fft2d_supports(N) && fft2d_fits(H, pitch) && fft2d_fits(H, out_pitch) && ctx->numerics == ARTIA_NUMERICS_EXACT) {
        FftOwn& f = ctx->ffto;
        const artia_status so = f.ensure(ctx, N, FftOwn::kOne);
        if (so != ARTIA_OK) return so;
        RowSrc s = square_source(nullptr, 0, W, H, pitch, N);
        s.raw = img;
        s.dtype = ARTIA_DT_FLOAT;
        PrepFilter pf{};
        pf.wbp = 1;
        pf.method = method;
        const float ang = -psi_deg / 180.0f * kPiF;
        pf.sn[0] = sin((double)ang);
        pf.cs[0] = cos((double)ang);
        fft2d_rows_prep(ctx, N, f.tw, s, f.one, 1);
        fft2d_cols_prep(ctx, N, f.tw, f.one, pf, 1);
        fft2d_rows_store(ctx, N, f.tw, f.one, square_target(out, 0, W, H, out_pitch, N, nullptr, 0), 1);
        return check_hip(ctx, hipGetLastError(), "wbp filter");
    }
    artia_status st = ctx->fft.ensure(ctx, N);
    if (st != ARTIA_OK) return st;
    launch_make_square(ctx, W, H, pitch, img, N, ctx->fft.square, (N - W) / 2, (N - H) / 2, 0, 0);
    if (hipfftSetStream(ctx->fft.r2c, ctx->stream) != HIPFFT_SUCCESS ||
        hipfftSetStream(ctx->fft.c2r, ctx->stream) != HIPFFT_SUCCESS)
        return fail(ctx, ARTIA_ERR_FFT, "hipfftSetStream failed");
    if (hipfftExecR2C(ctx->fft.r2c, ctx->fft.square, (hipfftComplex*)ctx->fft.spec) != HIPFFT_SUCCESS)
        return fail(ctx, ARTIA_ERR_FFT, "hipfftExecR2C failed");
    st = run_wbp_weight(ctx, ctx->fft.spec, N, (size_t)(N / 2 + 1), &psi_deg, 1, method);
    if (st != ARTIA_OK) return st;
    if (hipfftExecC2R(ctx->fft.c2r, (hipfftComplex*)ctx->fft.spec, ctx->fft.square) != HIPFFT_SUCCESS)
        return fail(ctx, ARTIA_ERR_FFT, "hipfftExecC2R failed");
    const CropParams cp{};
    hipLaunchKernelGGL(finish_kernel, grid2d(W, H), dim3(64, 4), 0, ctx->stream, ctx->fft.square, 1, N, (N - W) / 2,
                       (N - H) / 2, W, H, out, out_pitch, (float)(N * N), 0, 0, cp, (size_t)0);
    return check_hip(ctx, hipGetLastError(), "wbp filter");
}

}  // namespace artia

using namespace artia;

namespace {
bool valid_ctf(const artia_ctf_params* p) {
    return p && p->voltage_kV > 0.0f && p->pixelsize_nm > 0.0f && p->wiener >= 0.0f;
}
}  // namespace

extern "C" {

artia_status artia_ctf_apply(artia_ctx* ctx, void* spectrum, int n, size_t pitch, const artia_ctf_params* p,
                             float defocus_min_nm, float defocus_max_nm, float angle_deg, int for_fp, float* ms) {
    if (!ctx) return ARTIA_ERR_INVALID_ARGUMENT;
    if (!spectrum || n <= 1 || pitch < (size_t)(n / 2 + 1) || !valid_ctf(p))
        return fail(ctx, ARTIA_ERR_INVALID_ARGUMENT, "artia_ctf_apply: invalid arguments");
    Timing t(ctx, ms);
    artia_status st = run_ctf(ctx, (float2*)spectrum, n, pitch, *p, defocus_min_nm, defocus_max_nm, angle_deg, for_fp);
    if (st != ARTIA_OK) return st;
    return t.finish();
}

artia_status artia_wbp_weight(artia_ctx* ctx, void* spectrum, int n, size_t pitch, float psi_deg, int method,
                              float* ms) {
    if (!ctx) return ARTIA_ERR_INVALID_ARGUMENT;
    if (!spectrum || n <= 1 || pitch < (size_t)(n / 2 + 1) || method < 0 || method > 4)
        return fail(ctx, ARTIA_ERR_INVALID_ARGUMENT, "artia_wbp_weight: invalid arguments");
    Timing t(ctx, ms);
    artia_status st = run_wbp_weight(ctx, (float2*)spectrum, n, pitch, &psi_deg, 1, method);
    if (st != ARTIA_OK) return st;
    return t.finish();
}

artia_status artia_ctf_slab_filter(artia_ctx* ctx, float* img, int width, int height, size_t pitch, float* out,
                                   size_t out_pitch, int accumulate, const int corners[8], const float cut_length[2],
                                   const float dim_length[2], const artia_ctf_params* p, float defocus_min_nm,
                                   float defocus_max_nm, float angle_deg, int for_fp, float* ms) {
    if (!ctx) return ARTIA_ERR_INVALID_ARGUMENT;
    if (!img || !out || (corners && (!cut_length || !dim_length)) || !valid_ctf(p) || width <= 0 || height <= 0 ||
        pitch < (size_t)width || out_pitch < (size_t)width)
        return fail(ctx, ARTIA_ERR_INVALID_ARGUMENT, "artia_ctf_slab_filter: invalid arguments");
    Timing t(ctx, ms);
    artia_status st = ctf_slab_filter(ctx, img, width, height, pitch, out, out_pitch, accumulate, corners, cut_length,
                                      dim_length, *p, defocus_min_nm, defocus_max_nm, angle_deg, for_fp);
    if (st != ARTIA_OK) return st;
    return t.finish();
}

artia_status artia_wbp_filter(artia_ctx* ctx, const float* img, int width, int height, size_t pitch, float* out,
                              size_t out_pitch, float psi_deg, int method, float* ms) {
    if (!ctx) return ARTIA_ERR_INVALID_ARGUMENT;
    if (!img || !out || width <= 0 || height <= 0 || pitch < (size_t)width || out_pitch < (size_t)width ||
        method < 0 || method > 4)
        return fail(ctx, ARTIA_ERR_INVALID_ARGUMENT, "artia_wbp_filter: invalid arguments");
    Timing t(ctx, ms);
    artia_status st = wbp_filter(ctx, img, width, height, pitch, out, out_pitch, psi_deg, method);
    if (st != ARTIA_OK) return st;
    return t.finish();
}

}  // extern "C"
