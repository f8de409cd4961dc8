// Projection preparation on gfx950: PrepareProjection (Reconstructor.cpp:1158-1383) over a stack of
// projections.  The reference prepares one projection at a time with NPP statistics copied to the
// host between steps; here a chunk of projections goes through every step together, and the per-projection
// statistics stay on the device until the end of the call.  For squares of 128 .. 4096 (a power of two)
// the steps between the raw pixels and the filtered image are the three filter kernels' own loads,
// factors and stores (fft2d.hpp); other sizes take batched hipFFT plans with one launch per step.
//
// Steps per projection (see artia_prepare_projections in artia.h):
//   convert + mirror square -> mean of the square -> bad pixels -> [WBP: crop, statistics,
//   normalise, mirror square] -> [R2C -> fourierFilter -> doseWeighting -> wbpWeighting -> C2R]
//   -> crop / n^2 -> [SART: statistics, normalise].
// Sums are in double, in a fixed order (block partials, then one block per projection), so a
// projection's statistics do not depend on the chunk it is in.
#include <algorithm>
#include <cmath>
#include <vector>

#include "artia_internal.hpp"
#include "device_common.hpp"
#include "fft2d.hpp"
#include "image_ops.hpp"
#include "spectral_factors.hpp"

namespace artia {
namespace {

constexpr int kRedBlocks = 256;   // partial sums per image and reduction

dim3 grid2(int w, int h, int z) { return dim3((unsigned)((w + 63) / 64), (unsigned)((h + 3) / 4), (unsigned)z); }

// nppiConvert_*32f + CopyToSquare (mirror padding) of image z of the chunk, its bad pixels replaced and counted
// (nppiCompareC (> bad_value * mean) + nppiSum_8u / 255 + nppiSet_32f_C1MR(mean)) and, for WBP, normalised, in
// one pass: a pass for each read and wrote the squares three times more (41 images in squares of 960: 1.37 -> 1.14 ms)
template <class T>
__global__ void __launch_bounds__(256) prep_square_kernel(RowSrc s, int N, float* __restrict__ sq) {
    __shared__ int nbad;
    const bool first = threadIdx.x == 0 && threadIdx.y == 0;
    const int x = (int)(blockIdx.x * blockDim.x + threadIdx.x);
    const int y = (int)(blockIdx.y * blockDim.y + threadIdx.y), z = (int)blockIdx.z;
    if (first) nbad = 0;
    __syncthreads();
    int bad = 0;
    if (x < N && y < N) {
        int xi, yi;
        mirror_source(x, y, s.W, s.H, s.bx, s.by, 0, xi, yi);
        if (s.mirror_y) yi = s.H - yi - 1;
        const float v = (float)static_cast<const T*>(s.raw)[(size_t)z * s.stride + (size_t)yi * s.pitch + (size_t)xi];
        sq[(size_t)z * (size_t)N * (size_t)N + (size_t)y * N + x] = prep_pixel(s, s.st[z], v, bad);
    }
    if (bad) atomicAdd(&nbad, bad);
    __syncthreads();
    if (first && nbad) atomicAdd(&s.st[z].bad, nbad);
}

__device__ __forceinline__ double block_sum(double v, double* sh) {
    sh[threadIdx.x] = v;
    __syncthreads();
    for (int s = 128; s > 0; s >>= 1) {
        if ((int)threadIdx.x < s) sh[threadIdx.x] += sh[threadIdx.x + s];
        __syncthreads();
    }
    const double r = sh[0];
    __syncthreads();
    return r;
}

// Partial sums over the w x h region at (x0, y0) of image z: pass 0 sums the values, pass 1 the
// squared deviations from st[z].mean.  Block b takes rows b, b + kRedBlocks, ..
__global__ void __launch_bounds__(256) region_sums_kernel(const float* __restrict__ img, size_t istride, size_t pitch,
                                                          int x0, int y0, int w, int h, const PrepStat* __restrict__ st,
                                                          int pass, double* __restrict__ partial) {
    __shared__ double sh[256];
    const int z = (int)blockIdx.y;
    const float* base = img + (size_t)z * istride;
    const double m = pass ? st[z].mean : 0.0;
    double acc = 0.0;
    for (int r = (int)blockIdx.x; r < h; r += kRedBlocks) {
        const float* row = base + (size_t)(y0 + r) * pitch + x0;
        for (int c = (int)threadIdx.x; c < w; c += 256) {
            const double v = (double)row[c];
            acc += pass ? (v - m) * (v - m) : v;
        }
    }
    const double s = block_sum(acc, sh);
    if (threadIdx.x == 0) partial[(size_t)z * kRedBlocks + blockIdx.x] = s;
}

// which: 0 -> sq_mean = sum / count, 1 -> mean = sum / count, 2 -> std = sqrt(sum / count)
__global__ void __launch_bounds__(256) region_finish_kernel(const double* __restrict__ partial, double count, int which,
                                                            PrepStat* __restrict__ st) {
    __shared__ double sh[256];
    const int z = (int)blockIdx.x;
    const double s = block_sum(partial[(size_t)z * kRedBlocks + threadIdx.x], sh);
    if (threadIdx.x == 0) {
        if (which == 0) st[z].sq_mean = s / count;
        else if (which == 1) st[z].mean = s / count;
        else st[z].std = sqrt(s / count);
    }
}

// The normalisation's m and s (Reconstructor.cpp:1232-1260 for WBP, :1346-1368 for SART)
__global__ void norm_params_kernel(PrepStat* __restrict__ st, int nz, int wbp, int norm, int down_weight) {
    const int z = (int)(blockIdx.x * blockDim.x + threadIdx.x);
    if (z >= nz) return;
    PrepStat& s = st[z];
    float std_hf = (float)s.std;
    const float meanValue = (float)s.mean;
    float mean_hf = meanValue;
    if (norm == ARTIA_NORM_MEAN) std_hf = meanValue;
    if (norm == ARTIA_NORM_NONE) {
        std_hf = 1.0f;
        if (wbp) mean_hf = 0.0f;
    }
    if (wbp && down_weight) std_hf = std_hf / s.cos_tilt;
    s.mean_hf = mean_hf;
    s.std_hf = std_hf;
}

// out = square[by + y][bx + x] / norm (nppiDivC from the square's inner region)
__global__ void __launch_bounds__(256) crop_div_kernel(const float* __restrict__ sq, int N, int bx, int by, int W, int H,
                                                       float norm, float* __restrict__ out, size_t pitch,
                                                       size_t ostride) {
    const int x = (int)(blockIdx.x * blockDim.x + threadIdx.x);
    const int y = (int)(blockIdx.y * blockDim.y + threadIdx.y);
    if (x >= W || y >= H) return;
    out[(size_t)blockIdx.z * ostride + (size_t)y * pitch + x] =
        sq[(size_t)blockIdx.z * (size_t)N * (size_t)N + (size_t)(by + y) * N + (bx + x)] / norm;
}

// nppiSubC(m) then nppiDivC(-s), in place
__global__ void __launch_bounds__(256) normalise_kernel(float* __restrict__ img, int W, int H, size_t pitch,
                                                        size_t istride, const PrepStat* __restrict__ st) {
    const int x = (int)(blockIdx.x * blockDim.x + threadIdx.x);
    const int y = (int)(blockIdx.y * blockDim.y + threadIdx.y);
    if (x >= W || y >= H) return;
    const PrepStat& s = st[blockIdx.z];
    float* p = img + (size_t)blockIdx.z * istride + (size_t)y * pitch + x;
    float v = *p - s.mean_hf;
    v = v / -s.std_hf;
    *p = v;
}

// The filters' factors (prep_factor) on the half spectra of the chunk
__global__ void __launch_bounds__(256) prep_spectrum_kernel(float2* __restrict__ spec, size_t pitch, int N,
                                                            PrepFilter f) {
    const int x = (int)(blockIdx.x * blockDim.x + threadIdx.x);
    const int y = (int)(blockIdx.y * blockDim.y + threadIdx.y);
    if (x >= N / 2 + 1 || y >= N) return;
    float2* p = spec + (size_t)blockIdx.z * pitch * (size_t)N + (size_t)y * pitch + x;
    *p = prep_factor(*p, x, y, N, f, (int)blockIdx.z);
}

// The square's or the image's sums over raw pixels of type T, in the order of region_sums_kernel: pass 0
// over the mirrored N x N square (its mean, the bad-pixel reference), pass 1 and 2 over the W x H image
// with its bad pixels replaced (mean, squared deviations).
template <class T>
__global__ void __launch_bounds__(256) raw_sums_kernel(const T* __restrict__ in, size_t pitch, size_t istride, int W,
                                                       int H, int N, int bx, int by, int mirror_y, int correct,
                                                       float bad_value, const PrepStat* __restrict__ st, int pass,
                                                       double* __restrict__ partial) {
    __shared__ double sh[256];
    const int z = (int)blockIdx.y, w = pass ? W : N, h = pass ? H : N;
    const T* base = in + (size_t)z * istride;
    const double m = pass == 2 ? st[z].mean : 0.0;
    const float mean = pass && correct ? (float)st[z].sq_mean : 0.0f;
    double acc = 0.0;
    for (int r = (int)blockIdx.x; r < h; r += kRedBlocks) {
        int x0 = 0, yi = r;
        if (!pass) mirror_source(bx, r, W, H, bx, by, 0, x0, yi);
        const T* row = base + (size_t)(mirror_y ? H - yi - 1 : yi) * pitch;
        // eight loads in flight (one at a time read 0.5 TB/s)
        for (int c = (int)threadIdx.x; c < w; c += 8 * 256) {
            float f[8];
#pragma unroll
            for (int j = 0; j < 8; j++) {
                int xi = min(c + 256 * j, w - 1), y2;
                if (!pass) mirror_source(xi, by, W, H, bx, by, 0, xi, y2);
                f[j] = (float)row[xi];
            }
#pragma unroll
            for (int j = 0; j < 8; j++) {
                if (pass && correct && f[j] > bad_value * mean) f[j] = mean;
                const double v = (double)f[j];
                if (c + 256 * j < w) acc += pass == 2 ? (v - m) * (v - m) : v;
            }
        }
    }
    const double s = block_sum(acc, sh);
    if (threadIdx.x == 0) partial[(size_t)z * kRedBlocks + blockIdx.x] = s;
}

// The statistics of a filtered image from its row blocks' sums of v - c and (v - c)^2
__global__ void __launch_bounds__(256) row_stats_finish_kernel(const double* __restrict__ partial, int blocks, double count,
                                                               const float* __restrict__ dc, float scale,
                                                               PrepStat* __restrict__ st) {
    __shared__ double sh[256];
    const int z = (int)blockIdx.x;
    double a1 = 0.0, a2 = 0.0;
    for (int b = (int)threadIdx.x; b < blocks; b += 256) {
        a1 += partial[2 * ((size_t)z * blocks + b)];
        a2 += partial[2 * ((size_t)z * blocks + b) + 1];
    }
    const double s1 = block_sum(a1, sh), s2 = block_sum(a2, sh);
    if (threadIdx.x == 0) {
        const double d = s1 / count, var = s2 / count - d * d;
        st[z].mean = (double)(dc[z] * scale) + d;
        st[z].std = sqrt(var < 0.0 ? 0.0 : var);
    }
}

// The statistics of a filtered N x N image from its spectrum: the mean from frequency 0 and the variance from
// the other squares (Parseval).
__global__ void __launch_bounds__(256) spectrum_stats_kernel(const double* __restrict__ power, int waves, int N,
                                                             const float* __restrict__ dc, float scale,
                                                             PrepStat* __restrict__ st) {
    __shared__ double sh[256];
    const int z = (int)blockIdx.x;
    double a = 0.0;
    for (int w = (int)threadIdx.x; w < waves; w += 256) a += power[(size_t)z * waves + w];
    const double s = block_sum(a, sh);
    if (threadIdx.x == 0) {
        st[z].mean = (double)(dc[z] * scale);
        st[z].std = sqrt(s) * (double)scale;
    }
}

template <class T>
void launch_raw_sums(artia_ctx* ctx, const RowSrc& s, int N, int pass, double* partial, int b) {
    hipLaunchKernelGGL(raw_sums_kernel<T>, dim3(kRedBlocks, (unsigned)b), dim3(256), 0, ctx->stream,
                       static_cast<const T*>(s.raw), s.pitch, s.stride, s.W, s.H, N, s.bx, s.by, s.mirror_y, s.correct,
                       s.bad_value, s.st, pass, partial);
}
// pass 0 -> sq_mean, 1 -> mean, 2 -> std
void raw_stat(artia_ctx* ctx, const RowSrc& s, int N, int pass, double* partial, int b) {
    switch (s.dtype) {
        case ARTIA_DT_SHORT: launch_raw_sums<short>(ctx, s, N, pass, partial, b); break;
        case ARTIA_DT_USHORT: launch_raw_sums<unsigned short>(ctx, s, N, pass, partial, b); break;
        case ARTIA_DT_INT: launch_raw_sums<int>(ctx, s, N, pass, partial, b); break;
        case ARTIA_DT_UINT: launch_raw_sums<unsigned>(ctx, s, N, pass, partial, b); break;
        default: launch_raw_sums<float>(ctx, s, N, pass, partial, b); break;
    }
    const double count = pass ? (double)s.W * (double)s.H : (double)N * (double)N;
    hipLaunchKernelGGL(region_finish_kernel, dim3((unsigned)b), dim3(256), 0, ctx->stream, partial, count, pass, s.st);
}

template <class T>
void launch_square(artia_ctx* ctx, const RowSrc& s, int N, float* sq, int b) {
    hipLaunchKernelGGL(prep_square_kernel<T>, grid2(N, N, b), dim3(64, 4), 0, ctx->stream, s, N, sq);
}

void square_of(artia_ctx* ctx, const RowSrc& s, int N, float* sq, int b) {
    switch (s.dtype) {
        case ARTIA_DT_SHORT: launch_square<short>(ctx, s, N, sq, b); break;
        case ARTIA_DT_USHORT: launch_square<unsigned short>(ctx, s, N, sq, b); break;
        case ARTIA_DT_INT: launch_square<int>(ctx, s, N, sq, b); break;
        case ARTIA_DT_UINT: launch_square<unsigned>(ctx, s, N, sq, b); break;
        default: launch_square<float>(ctx, s, N, sq, b); break;
    }
}

size_t dtype_size(int dtype) {
    return dtype == ARTIA_DT_SHORT || dtype == ARTIA_DT_USHORT ? 2 : 4;
}

// mean (which 1) or sq_mean (which 0), or std (which 2, needs mean), of a region of b images
void region_stat(artia_ctx* ctx, const float* img, size_t istride, size_t pitch, int x0, int y0, int w, int h,
                 PrepStat* st, int which, double* partial, int b) {
    hipLaunchKernelGGL(region_sums_kernel, dim3(kRedBlocks, (unsigned)b), dim3(256), 0, ctx->stream, img, istride,
                       pitch, x0, y0, w, h, st, which == 2 ? 1 : 0, partial);
    hipLaunchKernelGGL(region_finish_kernel, dim3((unsigned)b), dim3(256), 0, ctx->stream, partial,
                       (double)w * (double)h, which, st);
}

}  // namespace
}  // namespace artia

using namespace artia;

extern "C" {

artia_status artia_prepare_projections(artia_ctx* ctx, const artia_prep_params* pp, const void* images, int n,
                                       int width, int height, size_t pitch, const float* tilt_deg,
                                       const float* psi_deg, const float* dose, float* out, size_t out_pitch,
                                       float* mean, float* std, int* bad_pixels, float* ms) {
    if (!ctx) return ARTIA_ERR_INVALID_ARGUMENT;
    if (!pp || !images || !out || n <= 0 || width <= 0 || height <= 0 || pitch < (size_t)width ||
        out_pitch < (size_t)width || !mean || !std || !bad_pixels)
        return fail(ctx, ARTIA_ERR_INVALID_ARGUMENT, "artia_prepare_projections: invalid arguments");
    if (pp->dtype < ARTIA_DT_SHORT || pp->dtype > ARTIA_DT_FLOAT)
        return fail(ctx, ARTIA_ERR_INVALID_ARGUMENT, "artia_prepare_projections: unsupported data type %d", pp->dtype);
    if (pp->normalization < ARTIA_NORM_MEAN || pp->normalization > ARTIA_NORM_NONE)
        return fail(ctx, ARTIA_ERR_INVALID_ARGUMENT, "artia_prepare_projections: unknown normalisation %d",
                    pp->normalization);
    if (pp->wbp && (pp->wbp_method < 0 || pp->wbp_method > 4 || !psi_deg || (pp->down_weight_tilts && !tilt_deg)))
        return fail(ctx, ARTIA_ERR_INVALID_ARGUMENT,
                    "artia_prepare_projections: WBP needs a method 0..4, psi angles and, to down-weight, tilt angles");
    if (pp->dose_weighting && (!dose || !(pp->pixelsize_nm > 0.0f)))
        return fail(ctx, ARTIA_ERR_INVALID_ARGUMENT,
                    "artia_prepare_projections: dose weighting needs doses and a pixel size");
    const int N = width > height ? width : height;
    const bool fft = !pp->skip_filter || pp->wbp;
    // the three-kernel filter (fft2d.hpp), or library transforms of the chunk's squares
    const bool own = fft && fft2d_supports(N) && fft2d_fits(height, pitch) && fft2d_fits(height, out_pitch) &&
                     ctx->numerics == ARTIA_NUMERICS_EXACT;
    FftBatch& fb = ctx->fftb;
    FftOwn& fo = ctx->ffto;
    artia_status st = own ? fo.ensure(ctx, N, FftOwn::kStack) : fb.ensure(ctx, N);
    if (st != ARTIA_OK) return st;
    const int cap = own ? fo.cap : fb.cap, rowBlocks = own ? fft2d_row_blocks(N) : 0;
    // The normalisation of a whole square's mean and deviation needs no pass over the image: both come from the
    // spectrum, whose frequency 0 is then taken out so that a high mean rounds no pixel, and the pixels are
    // divided as they are stored (31 images of 4096 x 4096: 5.4 -> 4.7 ms).
    // Not with a high pass and the mean as divisor, where a frequency 0 filtered to nothing would be divided by.
    const bool fromSpectrum = own && !pp->wbp && width == N && height == N &&
                              (pp->normalization == ARTIA_NORM_STD ||
                               (pp->normalization == ARTIA_NORM_MEAN && !(pp->hp > 0.0f)));
    const int waves = fromSpectrum ? fft2d_col_waves(N) : 0;
    // workspace: partial sums of a chunk, then the per-projection state and, behind it, the squares' means
    const size_t partFloats = (size_t)cap * (size_t)std::max(kRedBlocks, std::max(2 * rowBlocks, waves)) * 2;
    const size_t statFloats = ((size_t)n * sizeof(PrepStat) + sizeof(float) - 1) / sizeof(float);
    if ((st = ensure_workspace(ctx, partFloats + statFloats + 2 + kFftBatchMax)) != ARTIA_OK) return st;
    double* partial = reinterpret_cast<double*>(ctx->ws);
    PrepStat* d_stat = reinterpret_cast<PrepStat*>(ctx->ws + partFloats);
    float* d_dc = ctx->ws + partFloats + statFloats + 2;
    std::vector<PrepStat> hs((size_t)n);
    for (int i = 0; i < n; i++) {
        PrepStat& s = hs[(size_t)i];
        s = PrepStat{};
        s.dose = pp->dose_weighting ? dose[i] : 0.0f;
        // Reconstructor.cpp:1250: cosf(abs(tilt) / 180.0f * M_PI), the product in double
        s.cos_tilt = (pp->wbp && pp->down_weight_tilts)
                         ? cosf((float)((double)(std::fabs(tilt_deg[i]) / 180.0f) * 3.14159265358979323846))
                         : 1.0f;
    }
    Timing t(ctx, ms);
    st = check_hip(ctx, hipMemcpyAsync(d_stat, hs.data(), hs.size() * sizeof(PrepStat), hipMemcpyHostToDevice,
                                       ctx->stream),
                   "hipMemcpyAsync(projection state)");
    if (st != ARTIA_OK) return st;
    const size_t half = (size_t)(N / 2 + 1);
    const size_t istride = (size_t)height * pitch, ostride = (size_t)height * out_pitch;
    const int bx = (N - width) / 2, by = (N - height) / 2;
    const float pixA = pp->pixelsize_nm * 10.0f;
    const bool centre = !pp->wbp && pp->normalization == ARTIA_NORM_NONE;
    const int rx0 = centre ? width / 4 : 0, ry0 = centre ? height / 4 : 0;
    const int rw = centre ? width / 2 : width, rh = centre ? height / 2 : height;
    for (int k0 = 0; k0 < n;) {
        int b = cap, pi = 0;
        if (own) b = std::min(b, n - k0);
        while (b > n - k0) b /= 2;
        for (int q = b; q > 1; q /= 2) pi++;
        PrepStat* s = d_stat + k0;
        float* o = out + (size_t)k0 * ostride;
        const void* raw = static_cast<const char*>(images) + (size_t)k0 * istride * dtype_size(pp->dtype);
        PrepFilter f{};
        f.band = pp->skip_filter ? 0 : 1;
        f.lp = pp->lp;
        f.hp = pp->hp;
        f.lps = pp->lps;
        f.hps = pp->hps;
        f.dose_on = pp->dose_weighting;
        f.pixA = pixA;
        f.st = s;
        RowSrc r{};
        r.W = width;
        r.H = height;
        r.bx = bx;
        r.by = by;
        r.raw = raw;
        r.pitch = pitch;
        r.stride = istride;
        r.dtype = pp->dtype;
        r.mirror_y = pp->mirror_y;
        r.correct = pp->correct_bad_pixels;
        r.bad_value = pp->bad_pixel_value;
        r.st = s;
        if (r.correct) raw_stat(ctx, r, N, 0, partial, b);
        if (pp->wbp) {
            // the raw image's statistics; its pixels are normalised as they are loaded
            raw_stat(ctx, r, N, 1, partial, b);
            raw_stat(ctx, r, N, 2, partial, b);
            hipLaunchKernelGGL(norm_params_kernel, dim3((unsigned)((b + 63) / 64)), dim3(64), 0, ctx->stream, s, b, 1,
                               pp->normalization, pp->down_weight_tilts);
            r.norm = 1;
        }
        if (own) {
            if (pp->wbp) {
                f.wbp = 1;
                f.method = pp->wbp_method;
                for (int i = 0; i < b; i++) {
                    const float ang = -psi_deg[k0 + i] / 180.0f * 3.14159265358979323846f;
                    f.sn[i] = sin((double)ang);
                    f.cs[i] = cos((double)ang);
                }
            }
            f.dc = d_dc;
            f.power = fromSpectrum ? partial : nullptr;
            fft2d_rows_prep(ctx, N, fo.tw, r, fo.spec, b);
            fft2d_cols_prep(ctx, N, fo.tw, fo.spec, f, b);
            RowDst d{};
            d.W = width;
            d.H = height;
            d.bx = bx;
            d.by = by;
            d.scale = 1.0f / ((float)N * (float)N);
            d.out = o;
            d.pitch = out_pitch;
            d.stride = ostride;
            if (pp->wbp) {
                fft2d_rows_store(ctx, N, fo.tw, fo.spec, d, b);
            } else if (fromSpectrum) {
                hipLaunchKernelGGL(spectrum_stats_kernel, dim3((unsigned)b), dim3(256), 0, ctx->stream, partial, waves, N,
                                   d_dc, d.scale, s);
                hipLaunchKernelGGL(norm_params_kernel, dim3((unsigned)((b + 63) / 64)), dim3(64), 0, ctx->stream, s, b, 0,
                                   pp->normalization, 0);
                d.st = s;
                fft2d_rows_store(ctx, N, fo.tw, fo.spec, d, b);
            } else {
                d.rx0 = rx0;
                d.ry0 = ry0;
                d.rw = rw;
                d.rh = rh;
                d.dc = d_dc;
                d.partial = partial;
                fft2d_rows_prep_store(ctx, N, fo.tw, fo.spec, d, b);
                hipLaunchKernelGGL(row_stats_finish_kernel, dim3((unsigned)b), dim3(256), 0, ctx->stream, partial,
                                   rowBlocks, (double)rw * (double)rh, d_dc, d.scale, s);
                hipLaunchKernelGGL(norm_params_kernel, dim3((unsigned)((b + 63) / 64)), dim3(64), 0, ctx->stream, s, b, 0,
                                   pp->normalization, 0);
                hipLaunchKernelGGL(normalise_kernel, grid2(width, height, b), dim3(64, 4), 0, ctx->stream, o, width,
                                   height, out_pitch, ostride, s);
            }
            if ((st = check_hip(ctx, hipGetLastError(), "projection preparation launch")) != ARTIA_OK) return st;
            k0 += b;
            continue;
        }
        square_of(ctx, r, N, fb.square, b);
        if (fft) {
            if (hipfftSetStream(fb.r2c[pi], ctx->stream) != HIPFFT_SUCCESS ||
                hipfftSetStream(fb.c2r[pi], ctx->stream) != HIPFFT_SUCCESS)
                return fail(ctx, ARTIA_ERR_FFT, "hipfftSetStream failed");
            if (hipfftExecR2C(fb.r2c[pi], fb.square, (hipfftComplex*)fb.spec) != HIPFFT_SUCCESS)
                return fail(ctx, ARTIA_ERR_FFT, "hipfftExecR2C (batch %d) failed", b);
            if (f.band || f.dose_on)
                hipLaunchKernelGGL(prep_spectrum_kernel, grid2(N / 2 + 1, N, b), dim3(64, 4), 0, ctx->stream, fb.spec,
                                   half, N, f);
            if (pp->wbp &&
                (st = run_wbp_weight(ctx, fb.spec, N, half, psi_deg + k0, b, pp->wbp_method)) != ARTIA_OK)
                return st;
            if (hipfftExecC2R(fb.c2r[pi], (hipfftComplex*)fb.spec, fb.square) != HIPFFT_SUCCESS)
                return fail(ctx, ARTIA_ERR_FFT, "hipfftExecC2R (batch %d) failed", b);
        }
        hipLaunchKernelGGL(crop_div_kernel, grid2(width, height, b), dim3(64, 4), 0, ctx->stream, fb.square, N, bx, by,
                           width, height, fft ? (float)N * (float)N : 1.0f, o, out_pitch, ostride);
        if (!pp->wbp) {
            // SART: statistics of the filtered image (its centre for IMOD-aligned stacks), normalised
            region_stat(ctx, o, ostride, out_pitch, rx0, ry0, rw, rh, s, 1, partial, b);
            region_stat(ctx, o, ostride, out_pitch, rx0, ry0, rw, rh, s, 2, partial, b);
            hipLaunchKernelGGL(norm_params_kernel, dim3((unsigned)((b + 63) / 64)), dim3(64), 0, ctx->stream, s, b, 0,
                               pp->normalization, 0);
            hipLaunchKernelGGL(normalise_kernel, grid2(width, height, b), dim3(64, 4), 0, ctx->stream, o, width, height,
                               out_pitch, ostride, s);
        }
        if ((st = check_hip(ctx, hipGetLastError(), "projection preparation launch")) != ARTIA_OK) return st;
        k0 += b;
    }
    st = check_hip(ctx, hipMemcpyAsync(hs.data(), d_stat, hs.size() * sizeof(PrepStat), hipMemcpyDeviceToHost,
                                       ctx->stream),
                   "hipMemcpyAsync(projection statistics)");
    if (st == ARTIA_OK) st = check_hip(ctx, hipStreamSynchronize(ctx->stream), "hipStreamSynchronize");
    if (st != ARTIA_OK) return st;
    for (int i = 0; i < n; i++) {
        mean[i] = (float)hs[(size_t)i].mean;
        std[i] = (float)hs[(size_t)i].std;
        bad_pixels[i] = hs[(size_t)i].bad;
    }
    return t.finish();
}

}  // extern "C"
