// Adjoint and shift gradient of the forward projector (exact numerics), for gradient-based
// refinement.  No reference counterpart: the reference's backprojector (BackProjectionSquareOS.cu)
// is SART's normalised update, not the transpose of its ray marcher.  Here
//   P x [pixel] = 0.25 * step * sum over the pixel's 4 sub-rays and their samples q_k of trilinear(x, q_k)
// is the forward projector of fp.hip (march_exact_kernel), and
//   fp_adjoint:    vol_grad += scale * P^T r, the transpose of the forward projector's per-cell
//                  closed form along the same sub-rays and cells (recomputed, never stored);
//   fp_shift_grad: out += sum_pixels g[pixel] * dP[pixel]/d(shift_x, shift_y), where the tilt's 2D
//                  shift moves the detector origin by -shift_x*u - shift_y*v (Projection.cpp:183-195)
//                  and with it every sample: dq_k/ds = scale * (-u + (dt_in/ds) n) per sub-ray.
#include "artia_internal.hpp"
#include "flat_walk.hpp"
#include "fp_common.hpp"
#include "tube_walk.hpp"

namespace artia {
namespace {

struct Roi {
    int x0, y0, x1, y1;
};

// One lane per sub-ray, the forward projector's mapping (8x8 pixels per 256-thread block).  The
// lane walks the same cells as the forward projector's march_sum and scatters the transpose of its
// per-cell closed form (cell_weights) with one set of eight atomics per cell.
template <bool kBig>
__global__ void __launch_bounds__(256) fp_adjoint_kernel(VolG v, TiltG g, const float* __restrict__ resid,
                                                         size_t pitch, Roi roi, float scale,
                                                         float* __restrict__ grad) {
    const int lane = (int)(threadIdx.x & 63), wave = (int)(threadIdx.x >> 6);
    const int sub = lane & 3, pix = lane >> 2;
    const int x = roi.x0 + (int)blockIdx.x * 8 + (wave & 1) * 4 + (pix & 3);
    const int y = roi.y0 + (int)blockIdx.y * 8 + (wave >> 1) * 4 + (pix >> 2);
    if (x >= roi.x1 || y >= roi.y1) return;
    const double step = (double)v.vs[0] * 0.15;
    // proj = (float)(0.25 * step * sum): the same factor per sample
    const double r = (double)resid[(size_t)y * pitch + (size_t)x] * (double)scale * (step * 0.25);
    if (r == 0.0) return;
    SubraySamples s;
    const double px = (double)x + ((sub & 2) ? 0.75 : 0.25);
    const double py = (double)y + ((sub & 1) ? 0.75 : 0.25);
    if (!subray_samples(v, g, px, py, step, s)) return;
    if (g.n[1] == 0.0f) {   // uniform
        const FlatDir d = flat_dir(s.dq);
        FlatWalker w;
        w.init(d, s.q0, s.count);
        flat_scatter_direct(v, grad, d, s.q0, r, w, []() { return true; });
        return;
    }
    for_each_cell(s.q0, s.dq, s.count, [&](const int cell[3], int k, int mi) {
        size_t o[8];
        cell_corners<kBig>(v, cell, o);
        double W[8];
        cell_weights(cell_moments(s.q0, s.dq, cell, k, mi), W);
#pragma unroll
        for (int i = 0; i < 8; i++) {
            const float add = (float)(r * W[i]);
            if (add != 0.0f) unsafeAtomicAdd(grad + o[i], add);
        }
    });
}

// The same transpose with each tile's rays walked through LDS-staged slabs (tube_walk.hpp): the
// weights are summed per slab in a box of shared memory and added to grad with one atomic per box
// voxel, not eight per cell.  The box is in double: its float additions in LDS took 3.5 of 3.9 ms per
// 512x512x128 tilt, a wave's ds_add_f32 194 cycles of a compute unit against 9 of a ds_add_f64; 0.51 ms so, where
// 0.36 ms are the walk and the weights.  tp.box values of LDS: the tilt's largest slab box.  Tiles are dealt to the XCDs in groups, as in the forward projector.  A wave
// takes one sub-ray of every pixel of the tile, so that its lanes are a pixel apart and rarely add to the
// same voxel at once.
template <bool kFlat>
__global__ void __launch_bounds__(256) fp_adjoint_lds_kernel(VolG v, TiltG g, const float* __restrict__ resid,
                                                             size_t pitch, Roi roi, float scale,
                                                             float* __restrict__ grad, TubePlan tp) {
    extern __shared__ double chunk[];   // tp.box values
    __shared__ int zr[2];
    const int pix = (int)(threadIdx.x & 63), sub = (int)(threadIdx.x >> 6);
    const int xcd = (int)(blockIdx.x & 7u), slot = (int)(blockIdx.x >> 3);
    const int grp = (slot / (kXcdGroup * kXcdGroup)) * 8 + xcd, mem = slot % (kXcdGroup * kXcdGroup);
    const int gtx = (grp % tp.groups_x) * kXcdGroup + mem % kXcdGroup;
    const int gty = (grp / tp.groups_x) * kXcdGroup + mem / kXcdGroup;
    if (gtx >= tp.tiles_x || gty >= tp.tiles_y) return;   // whole workgroup
    const int tx0 = roi.x0 + gtx * 8, ty0 = roi.y0 + gty * 8;
    const int x = tx0 + (pix & 7), y = ty0 + (pix >> 3);
    const double step = (double)v.vs[0] * 0.15;
    double r = 0.0;
    SubraySamples s;
    s.count = 0;
#pragma unroll
    for (int c = 0; c < 3; c++) s.q0[c] = s.dq[c] = 0.0f;
    if (x < roi.x1 && y < roi.y1) {
        // proj = (float)(0.25 * step * sum): the same factor per sample
        r = (double)resid[(size_t)y * pitch + (size_t)x] * (double)scale * (step * 0.25);
        const double px = (double)x + ((sub & 2) ? 0.75 : 0.25);
        const double py = (double)y + ((sub & 1) ? 0.75 : 0.25);
        if (r == 0.0 || !subray_samples(v, g, px, py, step, s)) s.count = 0;
    }
    const TubeBox tb = tube_box(v, g, tp, (double)tx0 + 0.25, (double)tx0 + 7.75, (double)ty0 + 0.25,
                                (double)ty0 + 7.75, 0.0, 0.0);
    if (kFlat) {
        float dq[3];
        tube_step(v, g, step, dq);
        flat_tube_scatter(v, grad, chunk, zr, tp, tb, dq, s.q0, s.count, r);
        return;
    }
    const TubeDir td = tube_dir(v, g, step);
    tube_scatter(v, grad, chunk, zr, tp, tb, td, s.q0, s.count, [&](double wgt[8], const int cell[3], int k, int mi) {
        double W[8];
        cell_weights(cell_moments(s.q0, td.dq, cell, k, mi), W);
#pragma unroll
        for (int i = 0; i < 8; i++) wgt[i] = r * W[i];
    });
}

// d projection / d (shift_x, shift_y) of a lane's sub-ray, weighted by its pixel's gradient go: G holds the
// summed gradients of its samples with respect to the texel coordinates (zero along an axis where the
// coordinate is clamped).  d p_k / d shift = -u (-v) + (d t_in / d shift) n, d t_in / d shift = u_a / n_a (v_a / n_a)
// with a the entry axis.  Added over the block into out.
__device__ __forceinline__ void shift_grad_store(const VolG& v, const TiltG& g, const SubraySamples& s,
                                                 const double G[3], double go, double step, double* __restrict__ out) {
    __shared__ double part[2][4];
    double gsx = 0.0, gsy = 0.0;
    if (s.count > 0) {
        // entry-axis components by select (a dynamic index would put the geometry in scratch)
        const int a = s.entry_axis;
        const float ua = a == 0 ? g.u[0] : (a == 1 ? g.u[1] : g.u[2]);
        const float va = a == 0 ? g.v[0] : (a == 1 ? g.v[1] : g.v[2]);
        const float na = a == 0 ? g.n[0] : (a == 1 ? g.n[1] : g.n[2]);
        const double tu = (double)ua / (double)na, tv = (double)va / (double)na;
        double dx = 0.0, dy = 0.0;
#pragma unroll
        for (int i = 0; i < 3; i++) {
            const double scale = (double)v.rcp[i] * (double)v.dim[i];
            dx += G[i] * scale * (-(double)g.u[i] + tu * (double)g.n[i]);
            dy += G[i] * scale * (-(double)g.v[i] + tv * (double)g.n[i]);
        }
        const double w = go * step * 0.25;
        gsx = w * dx;
        gsy = w * dy;
    }
    for (int o = 32; o > 0; o >>= 1) {
        gsx += __shfl_down(gsx, o);
        gsy += __shfl_down(gsy, o);
    }
    const int lane = (int)(threadIdx.x & 63), wave = (int)(threadIdx.x >> 6);
    if (lane == 0) {
        part[0][wave] = gsx;
        part[1][wave] = gsy;
    }
    __syncthreads();
    if (threadIdx.x == 0) {
        unsafeAtomicAdd(out, ((part[0][0] + part[0][1]) + part[0][2]) + part[0][3]);
        unsafeAtomicAdd(out + 1, ((part[1][0] + part[1][1]) + part[1][2]) + part[1][3]);
    }
}

// The lane's sub-ray of pixel (x, y), without samples outside the region or where the gradient is 0.
__device__ __forceinline__ double shift_grad_lane(const VolG& v, const TiltG& g, const float* __restrict__ gout,
                                                  size_t pitch, const Roi& roi, int x, int y, int sub, double step,
                                                  SubraySamples& s) {
    const double px = (double)x + ((sub & 2) ? 0.75 : 0.25);
    const double py = (double)y + ((sub & 1) ? 0.75 : 0.25);
    const float go = x < roi.x1 && y < roi.y1 ? gout[(size_t)y * pitch + (size_t)x] : 0.0f;
    if (go == 0.0f || !subray_samples(v, g, px, py, step, s)) {
        s.count = 0;
#pragma unroll
        for (int c = 0; c < 3; c++) s.q0[c] = s.dq[c] = 0.0f;
    }
    return (double)go;
}

// One lane per sub-ray.  A cell of the lattice contributes the closed-form sum of its samples' gradients, so
// the walk reads a cell once where a sum over samples reads eight voxels for each (about six per cell).
// This form reads the volume directly; the next one through LDS-staged slabs.
__global__ void __launch_bounds__(256) fp_shift_grad_kernel(VolG v, TiltG g, const float* __restrict__ vol,
                                                            const float* __restrict__ gout, size_t pitch, Roi roi,
                                                            double* __restrict__ out) {
    const int lane = (int)(threadIdx.x & 63), wave = (int)(threadIdx.x >> 6);
    const int sub = lane & 3, pix = lane >> 2;
    const int x = roi.x0 + (int)blockIdx.x * 8 + (wave & 1) * 4 + (pix & 3);
    const int y = roi.y0 + (int)blockIdx.y * 8 + (wave >> 1) * 4 + (pix >> 2);
    const double step = (double)v.vs[0] * 0.15;
    SubraySamples s;
    const double go = shift_grad_lane(v, g, gout, pitch, roi, x, y, sub, step, s);
    double G[3] = {0.0, 0.0, 0.0};
    if (g.n[1] == 0.0f) {   // uniform
        if (s.count > 0) {
            const FlatDir d = flat_dir(s.dq);
            FlatWalker w;
            w.init(d, s.q0, s.count);
            flat_walk_direct<true>(v, vol, d, s.q0, w, []() { return true; },
                                   [&](float A, float B, float C, float D, float yA, float yB, float yC, float yD, float a,
                                       float c, float m) { flat_grad_sum(A, B, C, D, yA, yB, yC, yD, a, c, m, d.K, G); });
            G[0] *= (double)d.sgn[0];
            G[2] *= (double)d.sgn[1];
        }
    } else {
        for_each_cell(s.q0, s.dq, s.count, [&](const int cell[3], int k, int mi) {
            size_t o[8];
            cell_corners<true>(v, cell, o);
            float val[8];
#pragma unroll
            for (int i = 0; i < 8; i++) val[i] = vol[o[i]];
            cell_grad_sum(val, cell_moments(s.q0, s.dq, cell, k, mi), G);
        });
    }
    shift_grad_store(v, g, s, G, go, step, out);
}

// The forward projector's tiles and slabs (march_lds_kernel); bound by the walk's VALU work.  512x512x128 to 512^2
// pixels: 2.33 ms with eight global reads per sample, 0.33 ms so (five waves per SIMD; four 0.35, six 0.36).
template <bool kFlat>
__global__ void __launch_bounds__(256, 5) fp_shift_grad_lds_kernel(VolG v, TiltG g, const float* __restrict__ vol,
                                                                   const float* __restrict__ gout, size_t pitch, Roi roi,
                                                                   double* __restrict__ out, TubePlan tp) {
    __shared__ float chunk[kChunkFloats];
    __shared__ int zr[2];
    const int lane = (int)(threadIdx.x & 63), wave = (int)(threadIdx.x >> 6);
    const int sub = lane & 3, pix = lane >> 2;
    const int xcd = (int)(blockIdx.x & 7u), slot = (int)(blockIdx.x >> 3);
    const int grp = (slot / (kXcdGroup * kXcdGroup)) * 8 + xcd, mem = slot % (kXcdGroup * kXcdGroup);
    const int gtx = (grp % tp.groups_x) * kXcdGroup + mem % kXcdGroup;
    const int gty = (grp / tp.groups_x) * kXcdGroup + mem / kXcdGroup;
    if (gtx >= tp.tiles_x || gty >= tp.tiles_y) return;   // whole workgroup
    const int tx0 = roi.x0 + gtx * 8, ty0 = roi.y0 + gty * 8;
    const int x = tx0 + (wave & 1) * 4 + (pix & 3), y = ty0 + (wave >> 1) * 4 + (pix >> 2);
    const double step = (double)v.vs[0] * 0.15;
    SubraySamples s;
    const double go = shift_grad_lane(v, g, gout, pitch, roi, x, y, sub, step, s);
    const TubeBox tb = tube_box(v, g, tp, (double)tx0 + 0.25, (double)tx0 + 7.75, (double)ty0 + 0.25,
                                (double)ty0 + 7.75, 0.0, 0.0);
    double G[3] = {0.0, 0.0, 0.0};
    if (kFlat) {
        float dq[3];
        tube_step(v, g, step, dq);
        const FlatDir d = flat_dir(dq);
        flat_tube_walk<true, true>(v, vol, chunk, zr, tp, tb, dq, s.q0, s.count,
                                   [&](float A, float B, float C, float D, float yA, float yB, float yC, float yD, float a,
                                       float c, float m) { flat_grad_sum(A, B, C, D, yA, yB, yC, yD, a, c, m, d.K, G); });
        G[0] *= (double)d.sgn[0];
        G[2] *= (double)d.sgn[1];
    } else {
        const TubeDir td = tube_dir(v, g, step);
        tube_walk<true>(v, vol, chunk, zr, tp, tb, td, s.q0, s.count,
                        [&](const float val[8], const int* cell, int k, int mi) {
                            cell_grad_sum(val, cell_moments(s.q0, td.dq, cell, k, mi), G);
                        });
    }
    shift_grad_store(v, g, s, G, go, step, out);
}

Roi clip_roi(const int* roi, int W, int H) {
    Roi r{0, 0, W, H};
    if (roi) {
        r.x0 = roi[0] < 0 ? 0 : roi[0];
        r.y0 = roi[1] < 0 ? 0 : roi[1];
        r.x1 = roi[2] > W ? W : roi[2];
        r.y1 = roi[3] > H ? H : roi[3];
    }
    return r;
}

dim3 grid_of(const Roi& r) {
    return dim3((unsigned)((r.x1 - r.x0 + 7) / 8), (unsigned)((r.y1 - r.y0 + 7) / 8));
}

// The staged kernels' 1D grid over the region's tiles, in groups (tp's tiles and groups are set).
dim3 tile_grid(const Roi& r, TubePlan& tp) {
    const dim3 grid = grid_of(r);
    tp.tiles_x = (int)grid.x;
    tp.tiles_y = (int)grid.y;
    tp.groups_x = (tp.tiles_x + kXcdGroup - 1) / kXcdGroup;
    const int groups = tp.groups_x * ((tp.tiles_y + kXcdGroup - 1) / kXcdGroup);
    return dim3((unsigned)(((groups + 7) / 8) * 8 * kXcdGroup * kXcdGroup));
}

artia_status check_args(artia_ctx* ctx, const char* fn, const artia_vol_geom* vg, const artia_tilt_geom* tg, int W,
                        int H, size_t pitch) {
    if (!valid_geometry(vg, tg))
        return fail(ctx, ARTIA_ERR_INVALID_ARGUMENT, "%s: null pointer or invalid geometry", fn);
    if (vg->nx < 2 || vg->ny < 2 || vg->nz < 2)
        return fail(ctx, ARTIA_ERR_UNSUPPORTED, "%s: volumes need at least 2 voxels per axis", fn);
    if (W <= 0 || H <= 0 || pitch < (size_t)W)
        return fail(ctx, ARTIA_ERR_INVALID_ARGUMENT, "%s: bad image size %d x %d (pitch %zu)", fn, W, H, pitch);
    return ARTIA_OK;
}

}  // namespace
}  // namespace artia

using namespace artia;

extern "C" {

artia_status artia_fp_adjoint(artia_ctx* ctx, const artia_vol_geom* vg, const artia_tilt_geom* tg,
                              const float* resid, int width, int height, size_t pitch, float* vol_grad,
                              const int* roi, float scale, float* ms) {
    if (!ctx) return ARTIA_ERR_INVALID_ARGUMENT;
    artia_status st = check_args(ctx, "artia_fp_adjoint", vg, tg, width, height, pitch);
    if (st != ARTIA_OK) return st;
    if (!resid || !vol_grad) return fail(ctx, ARTIA_ERR_INVALID_ARGUMENT, "artia_fp_adjoint: null pointer");
    const Roi r = clip_roi(roi, width, height);
    Timing t(ctx, ms);
    const VolG vd = to_device(*vg);
    const TiltG gd = flat_beam(to_device(*tg));
    TubePlan tp;
    if (r.x1 > r.x0 && r.y1 > r.y0 && ctx->march_lds && tube_plan(vd, gd, tp)) {
        const dim3 grid1 = tile_grid(r, tp);
        if (gd.n[1] == 0.0f)
            hipLaunchKernelGGL(fp_adjoint_lds_kernel<true>, grid1, dim3(256), tp.box * sizeof(double), ctx->stream, vd, gd, resid, pitch, r,
                               scale, vol_grad, tp);
        else
            hipLaunchKernelGGL(fp_adjoint_lds_kernel<false>, grid1, dim3(256), tp.box * sizeof(double), ctx->stream, vd, gd, resid, pitch, r,
                               scale, vol_grad, tp);
    } else if (r.x1 > r.x0 && r.y1 > r.y0)
    {
        const bool big = (double)vg->nx * (double)vg->ny * (double)vg->nz >= 1073741824.0;
        if (big)
            hipLaunchKernelGGL(fp_adjoint_kernel<true>, grid_of(r), dim3(256), 0, ctx->stream, vd,
                               gd, resid, pitch, r, scale, vol_grad);
        else
            hipLaunchKernelGGL(fp_adjoint_kernel<false>, grid_of(r), dim3(256), 0, ctx->stream, vd,
                               gd, resid, pitch, r, scale, vol_grad);
    }
    st = check_hip(ctx, hipGetLastError(), "artia_fp_adjoint launch");
    if (st != ARTIA_OK) return st;
    return t.finish();
}

artia_status artia_fp_shift_grad(artia_ctx* ctx, const artia_vol_geom* vg, const artia_tilt_geom* tg,
                                 const float* vol, const float* grad_proj, int width, int height, size_t pitch,
                                 const int* roi, double* out, float* ms) {
    if (!ctx) return ARTIA_ERR_INVALID_ARGUMENT;
    artia_status st = check_args(ctx, "artia_fp_shift_grad", vg, tg, width, height, pitch);
    if (st != ARTIA_OK) return st;
    if (!vol || !grad_proj || !out) return fail(ctx, ARTIA_ERR_INVALID_ARGUMENT, "artia_fp_shift_grad: null pointer");
    const Roi r = clip_roi(roi, width, height);
    Timing t(ctx, ms);
    const VolG vd = to_device(*vg);
    const TiltG gd = flat_beam(to_device(*tg));
    TubePlan tp;
    if (r.x1 > r.x0 && r.y1 > r.y0) {
        if (ctx->march_lds && tube_plan(vd, gd, tp)) {
            const dim3 grid = tile_grid(r, tp);
            if (gd.n[1] == 0.0f)
                hipLaunchKernelGGL(fp_shift_grad_lds_kernel<true>, grid, dim3(256), 0, ctx->stream, vd, gd, vol, grad_proj,
                                   pitch, r, out, tp);
            else
                hipLaunchKernelGGL(fp_shift_grad_lds_kernel<false>, grid, dim3(256), 0, ctx->stream, vd, gd, vol, grad_proj,
                                   pitch, r, out, tp);
        } else {
            hipLaunchKernelGGL(fp_shift_grad_kernel, grid_of(r), dim3(256), 0, ctx->stream, vd, gd, vol, grad_proj, pitch,
                               r, out);
        }
    }
    st = check_hip(ctx, hipGetLastError(), "artia_fp_shift_grad launch");
    if (st != ARTIA_OK) return st;
    return t.finish();
}

}  // extern "C"
