// Image filters through the 2D Fourier domain in three kernels: rows (two real rows per complex
// transform) -> columns forward, filter, columns back -> rows.  Everything that comes before and
// after the transforms (squaring, mirroring, crop weights, bad pixels; normalisation, slab sums,
// statistics) is part of the row kernels' loads and stores, and the filter is applied to a column
// while it is in registers.  For N x N squares with N = 128 .. 4096 a power of two (fft2d_supports),
// the lengths with register butterflies of at most 16 points and two passes of exchange through 70 KB of
// LDS, at exact numerics; other sizes take the hipFFT plans of spectral.hip and prep.hip.
//
// Layout of the half spectra: [pair of columns kx / 2][ky][kx & 1], N / 4 + 1 pairs, so that a row
// block stores and a column block loads contiguous memory without a transpose.
#pragma once

#include "artia_internal.hpp"
#include "image_ops.hpp"
#include "spectral_factors.hpp"

namespace artia {

bool fft2d_supports(int N);
// whether an image of this height, pitch (elements) is within the row kernels' 32-bit byte offsets
inline bool fft2d_fits(int H, size_t pitch) { return pitch < ((size_t)1 << 30) && (size_t)H * pitch < ((size_t)1 << 30); }
// float2 values of one half spectrum
inline size_t fft2d_spec_size(int N) { return (size_t)(N / 4 + 1) * (size_t)N * 2; }

// What the forward row kernel reads for square pixel (x, y) of image z.
struct RowSrc {
    int W, H, bx, by;       // the image centred in the square
    // kSquare: zero fill outside; src + z * stride, times the crop weight rep0 + z * rep_step times over
    const float* src;
    size_t pitch, stride;
    const float* weight;    // crop weights of the square (N x N, 0 outside the image), or null
    int rep0, rep_step;
    // kPrep: mirror padding of raw pixels of type dtype (artia_dtype); values above bad_value * mean are
    // set to the mean and counted; then (norm != 0) the WBP normalisation
    const void* raw;
    int dtype, mirror_y, correct, norm;
    float bad_value;
    PrepStat* st;
};

// a raw pixel's bad value replaced, and its normalisation
__device__ __forceinline__ float prep_pixel(const RowSrc& s, const PrepStat& st, float v, int& bad) {
    if (s.correct) {
        const float mean = (float)st.sq_mean;
        if (v > s.bad_value * mean) {
            v = mean;
            bad++;
        }
    }
    if (s.norm) {
        v = v - st.mean_hf;
        v = v / -st.std_hf;
    }
    return v;
}

// What the backward row kernel does with image pixel (x, y) of image z: v = value * scale, then
struct RowDst {
    int W, H, bx, by;
    float scale;           // 1 / N^2 (a power of two: the product is the division's result)
    float* out;
    size_t pitch, stride;
    const float* weight;   // as RowSrc's
    // kStore: out[z * stride] = w v (accumulate: += ), rows in need; with st divided by the preparation's
    // deviation (its mean has left with frequency 0)
    int accumulate;
    const PrepStat* st;
    const uint32_t* need;
    // kPrep: out = v, and the double sums of v - c and (v - c)^2 over the region [rx0, rx0 + rw) x
    // [ry0, ry0 + rh), c = dc[z] * scale (the square's mean), per block: partial[2 * (z * blocks + block)]
    int rx0, ry0, rw, rh;
    const float* dc;
    double* partial;
};

int fft2d_row_blocks(int N);   // blocks per image of the row kernels
int fft2d_col_waves(int N);    // waves per image of the column kernels

// spec[z] = half spectrum rows of image z (not yet transformed along the columns)
void fft2d_rows_square(artia_ctx* ctx, int N, const float2* tw, const RowSrc& s, float2* spec, int nz);
void fft2d_rows_prep(artia_ctx* ctx, int N, const float2* tw, const RowSrc& s, float2* spec, int nz);
// Rows of the stack's images that are wanted: bit y % 32 of word y / 32 of image z at need + z * N / 32, whole
// row blocks (fft2d_row_blocks) at a time; null: all.  The others are neither written by the columns nor
// transformed.  wanted: bit z 0 where image z has none (its columns are left out too).
// columns: forward only (in place)
void fft2d_cols_forward(artia_ctx* ctx, int N, const float2* tw, float2* spec, int nz);
// forward, CTF of slab z, back (in place)
void fft2d_cols_ctf(artia_ctx* ctx, int N, const float2* tw, float2* spec, const CtfStack& c, int nz);
// spec[z] = back(base * CTF of slab z), base transformed along the columns
void fft2d_cols_fan(artia_ctx* ctx, int N, const float2* tw, const float2* base, float2* spec, const CtfStack& c,
                    int nz, const uint32_t* need = nullptr, uint32_t wanted = ~0u);
// forward, projection preparation's filters, back (in place)
void fft2d_cols_prep(artia_ctx* ctx, int N, const float2* tw, float2* spec, const PrepFilter& f, int nz);
// rows back: each image stored (or added), or the preparation's store
void fft2d_rows_store(artia_ctx* ctx, int N, const float2* tw, const float2* spec, const RowDst& d, int nz);
void fft2d_rows_prep_store(artia_ctx* ctx, int N, const float2* tw, const float2* spec, const RowDst& d, int nz);

}  // namespace artia
