// Batched refinement over (sub-volume, tilt) pairs: the forward projector, its shift derivative
// and its transpose restricted to each pair's detector window, and EmSARTRefine's
// cross-correlation shift search (GetDisplacement, Reconstructor.cpp:1746-1959), each over all
// pairs of a refinement step in one launch.
//
// One 256-thread workgroup per pair walks its window in 8x8-pixel tiles with one lane per sub-ray
// (the forward projector's mapping), so per-pair sums need no atomics and come out in a fixed
// order.  Workgroup b is dispatched to XCD b mod 8; pairs are ordered by sub-volume and dealt to
// XCDs in contiguous runs, so the tilts of one sub-volume share one XCD's L2.
//
// Per sub-ray the samples are summed cell by cell in closed form (fp_common.hpp); the shift
// derivative of the sub-ray is (sum of the interpolant's gradients over its samples) . dq0/ds,
// because a detector shift translates all samples of a sub-ray alike: dq0/ds = scale * (-u +
// (u_a / n_a) n) with a the axis whose face sets the entry point (likewise v).
#include <algorithm>
#include <climits>
#include <numeric>
#include <vector>

#include "artia_internal.hpp"
#include "flat_walk.hpp"
#include "fp_common.hpp"
#include "tube_walk.hpp"

namespace artia {
namespace {

struct PairDev {
    TiltG g;
    VolG v;
    TubePlan tp;            // LDS-staged walk of the window's tiles (staged != 0)
    int staged;
    long long vol_offset;   // floats into the volume buffer
    long long img_offset;   // floats into image buffers
    int x0, y0, w, h;
};

enum { kProject = 0, kLossGrad = 1, kShiftGrad = 2 };

struct PairArgs {
    const PairDev* pairs;
    const int* order;        // slot -> pair, grouped by sub-volume
    int npairs, per_xcd;
    const float* vols;
    const double* shifts;    // 2 per pair or null
    const float* in;         // targets (kLossGrad), weights (kShiftGrad), residuals (adjoint)
    float* out;              // images (kProject), residuals (kLossGrad, may be null)
    double* loss;
    double* grad;
    double* normal;          // J^T J per pair (kLossGrad, may be null)
};

// Slot of workgroup b: XCD b % 8 takes slots [xcd * per_xcd, (xcd + 1) * per_xcd).
__device__ __forceinline__ int slot_of_block(int per_xcd) {
    return (int)(blockIdx.x & 7u) * per_xcd + (int)(blockIdx.x >> 3);
}

__device__ __forceinline__ void load_cell(const __amdgpu_buffer_rsrc_t rs, const VolG& v, const int cell[3],
                                          float val[8], uint32_t o[8]) {
    cell_corners_bytes(v, cell, o);
#pragma unroll
    for (int i = 0; i < 8; i++)   // the b32 load returns the word's bits
        val[i] = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(rs, (int)o[i], 0, 0));
}

// Block sum of three doubles in a fixed order; the result is valid in thread 0.  Ends with a
// barrier, so it can be called again right away.
__device__ __forceinline__ void block_sum3(double& a, double& b, double& c) {
    __shared__ double part[3][4];
    for (int o = 32; o > 0; o >>= 1) {
        a += __shfl_down(a, o);
        b += __shfl_down(b, o);
        c += __shfl_down(c, o);
    }
    const int lane = (int)(threadIdx.x & 63), wave = (int)(threadIdx.x >> 6);
    if (lane == 0) {
        part[0][wave] = a;
        part[1][wave] = b;
        part[2][wave] = c;
    }
    __syncthreads();
    if (threadIdx.x == 0) {
        a = ((part[0][0] + part[0][1]) + part[0][2]) + part[0][3];
        b = ((part[1][0] + part[1][1]) + part[1][2]) + part[1][3];
        c = ((part[2][0] + part[2][1]) + part[2][2]) + part[2][3];
    }
    __syncthreads();
}

// Five waves per SIMD (96 registers, a few spilled): measured faster than the unconstrained
// allocation (3-4 waves) for the LDS-staged walk.  The flat walk with gradients takes four (128 registers): at five
// it spilled 200 to 320 bytes a lane (40 cubes of 64^3 by 21 tilts, loss and gradient 7.26 -> 5.32 ms, shift gradient
// 5.47 -> 4.61; 200 of 16^3 by 11 1.23 -> 0.80 and 0.91 -> 0.54).
// Projections alone (kProject) split a pair's tiles over kPairParts workgroups: shorter ones fill the chip's
// last round (4100 windows of 80 x 94: 15.3 -> 14.0 ms, and 12.3 in a kernel of its own; two parts 14.4, eight
// 13.9) and a short list of pairs.  The other modes sum over the pair's pixels in one workgroup.
constexpr int kPairParts = 4;
// kFlat: the pairs whose rays have no y component (n_y == 0 after flat_beam), otherwise the others.  A kernel for
// each, because one with both walks spills the registers of the longer one in the other too (4 cubes of 128^3 by
// 11 tilts with a y component, loss and gradient: 36.5 ms alone, 44.2 together with the flat walk).
template <int kMode, bool kFlat>
__global__ void __launch_bounds__(256, kMode != kProject && kFlat ? 4 : 5) pair_march_kernel(PairArgs a) {
    __shared__ float chunk[kChunkFloats];
    __shared__ int zr[2];
    constexpr int kParts = kMode == kProject ? kPairParts : 1;
    const int block = (int)(blockIdx.x >> 3), slot = (int)(blockIdx.x & 7u) * a.per_xcd + block / kParts;
    if (slot >= a.npairs) return;   // whole workgroup
    const int p = a.order[slot];
    const PairDev& P = a.pairs[p];
    if ((P.g.n[1] == 0.0f) != kFlat) return;   // whole workgroup: the other kernel's pair
    const int x0 = P.x0, y0 = P.y0, w = P.w, h = P.h;
    const long long io = P.img_offset;
    const int lane = (int)(threadIdx.x & 63), wave = (int)(threadIdx.x >> 6);
    const int sub = lane & 3, pix = lane >> 2;
    const int tx = (wave & 1) * 4 + (pix & 3), ty = (wave >> 1) * 4 + (pix >> 2);
    const int ntx = (w + 7) >> 3, ntiles = ntx * ((h + 7) >> 3);
    double lsum = 0.0, gx = 0.0, gy = 0.0, jxx = 0.0, jxy = 0.0, jyy = 0.0;
    for (int t = block % kParts; t < ntiles; t += kParts) {
        // The geometry is re-read (scalar loads) per tile: hoisted out of the loop, its double
        // conversions would stay live in vector registers and halve the occupancy.
        __asm__ volatile("" ::: "memory");
        const VolG v = P.v;
        const TiltG g = P.g;
        const __amdgpu_buffer_rsrc_t rs = volume_rsrc(a.vols + P.vol_offset, v);
        const double sx = a.shifts ? a.shifts[2 * p] : 0.0, sy = a.shifts ? a.shifts[2 * p + 1] : 0.0;
        const double step = (double)v.vs[0] * 0.15;
        const int i = (t % ntx) * 8 + tx, j = (t / ntx) * 8 + ty;
        const bool active = i < w && j < h;
        const long long pofs = io + (long long)j * w + i;
        float win = 0.0f;
        if (kMode != kProject && active) win = a.in[pofs];
        double acc = 0.0, dxs = 0.0, dys = 0.0;
        SubraySamples s;
        const double px = (double)(x0 + i) + ((sub & 2) ? 0.75 : 0.25);
        const double py = (double)(y0 + j) + ((sub & 1) ? 0.75 : 0.25);
        const bool ok = active && (kMode != kShiftGrad || win != 0.0f) && subray_samples(v, g, px, py, step, s, sx, sy);
        if (!ok) {
            s.count = 0;
#pragma unroll
            for (int c = 0; c < 3; c++) s.q0[c] = s.dq[c] = 0.0f;
        }
        double G[3] = {0.0, 0.0, 0.0};
        auto cell_fn = [&](const float val[8], const int* cell, int k, int mi) {
            const CellMoments cm = cell_moments(s.q0, s.dq, cell, k, mi);
            if (kMode != kShiftGrad) acc += cell_sum_values(val, cm);
            if (kMode != kProject) cell_grad_sum(val, cm, G);
        };
        const double pi0 = (double)(x0 + (t % ntx) * 8), pj0 = (double)(y0 + (t / ntx) * 8);
        if constexpr (kFlat) {
            float dq[3];
            tube_step(v, g, step, dq);
            const FlatDir d = flat_dir(dq);
            auto flat_fn = [&](float A, float B, float C, float D, float yA, float yB, float yC, float yD, float ca,
                               float cc, float m) {
                if (kMode != kShiftGrad) acc += (double)flat_cell_sum(A, B, C, D, ca, cc, m, d.K);
                if (kMode != kProject) flat_grad_sum(A, B, C, D, yA, yB, yC, yD, ca, cc, m, d.K, G);
            };
            if (P.staged) {   // uniform: the whole block walks the tile's tube through LDS
                const TubeBox tb = tube_box(v, g, P.tp, pi0 + 0.25, pi0 + 7.75, pj0 + 0.25, pj0 + 7.75, sx, sy);
                flat_tube_walk<kMode != kProject, kMode == kLossGrad>(v, a.vols + P.vol_offset, chunk, zr, P.tp, tb, dq,
                                                                      s.q0, s.count, flat_fn);
            } else if (ok) {
                FlatWalker fw;
                fw.init(d, s.q0, s.count);
                flat_walk_direct<false>(v, a.vols + P.vol_offset, d, s.q0, fw, []() { return true; }, flat_fn);
            }
            G[0] *= (double)d.sgn[0];
            G[2] *= (double)d.sgn[1];
        } else if (P.staged) {
            const TubeDir td = tube_dir(v, g, step);
            const TubeBox tb = tube_box(v, g, P.tp, pi0 + 0.25, pi0 + 7.75, pj0 + 0.25, pj0 + 7.75, sx, sy);
            tube_walk<false>(v, a.vols + P.vol_offset, chunk, zr, P.tp, tb, td, s.q0, s.count, cell_fn);
        } else if (ok) {
            for_each_cell(s.q0, s.dq, s.count, [&](const int cell[3], int k, int mi) {
                float val[8];
                uint32_t o[8];
                load_cell(rs, v, cell, val, o);
                cell_fn(val, cell, k, mi);
            });
        }
        if (ok) {
            if (kMode != kProject) {
                // entry-axis components by select (a dynamic index would put the geometry in scratch)
                const int ax = s.entry_axis;
                const float ua = ax == 0 ? g.u[0] : (ax == 1 ? g.u[1] : g.u[2]);
                const float va = ax == 0 ? g.v[0] : (ax == 1 ? g.v[1] : g.v[2]);
                const float na = ax == 0 ? g.n[0] : (ax == 1 ? g.n[1] : g.n[2]);
                const double tu = (double)ua / (double)na, tv = (double)va / (double)na;
#pragma unroll
                for (int c = 0; c < 3; c++) {
                    const double scale = (double)v.rcp[c] * (double)v.dim[c];
                    dxs += G[c] * scale * (-(double)g.u[c] + tu * (double)g.n[c]);
                    dys += G[c] * scale * (-(double)g.v[c] + tv * (double)g.n[c]);
                }
            }
        }
        // the four sub-rays of a pixel are lanes 4q .. 4q+3
        if (kMode != kShiftGrad) {
            acc += __shfl_xor(acc, 1);
            acc += __shfl_xor(acc, 2);
        }
        if (kMode != kProject) {
            dxs += __shfl_xor(dxs, 1);
            dxs += __shfl_xor(dxs, 2);
            dys += __shfl_xor(dys, 1);
            dys += __shfl_xor(dys, 2);
        }
        if (active && sub == 0) {
            const double dpx = dxs * step * 0.25, dpy = dys * step * 0.25;
            if (kMode == kProject) {
                a.out[pofs] = (float)(acc * step * 0.25);
            } else if (kMode == kLossGrad) {
                const float pv = (float)(acc * step * 0.25);
                const double r = (double)pv - (double)win;
                if (a.out) a.out[pofs] = (float)r;
                lsum += r * r;
                gx += 2.0 * r * dpx;
                gy += 2.0 * r * dpy;
                jxx += dpx * dpx;
                jxy += dpx * dpy;
                jyy += dpy * dpy;
            } else {
                gx += (double)win * dpx;
                gy += (double)win * dpy;
            }
        }
    }
    if (kMode == kProject) return;
    block_sum3(lsum, gx, gy);
    if (threadIdx.x == 0) {
        if (kMode == kLossGrad) a.loss[p] = lsum;
        a.grad[2 * p] = gx;
        a.grad[2 * p + 1] = gy;
    }
    if (kMode == kLossGrad && a.normal) {   // uniform branch
        block_sum3(jxx, jxy, jyy);
        if (threadIdx.x == 0) {
            a.normal[3 * p] = jxx;
            a.normal[3 * p + 1] = jxy;
            a.normal[3 * p + 2] = jyy;
        }
    }
}

// The transpose summed per sub-volume slab in LDS.  A workgroup owns cell layers [zs, zs + L) of
// one sub-volume (voxel layers max(zs, 0) .. min(zs + L, nz - 1) in LDS) and walks every sub-ray
// of every tilt of that sub-volume through them only: the samples between the sub-ray's crossings
// of the slab's two z faces (the walker's own face-crossing formula, so neighbouring slabs split
// each sub-ray's samples without overlap or gap).  The tilts' weights meet in LDS (shared-memory
// atomics) and reach the gradient with one atomic per voxel and slab, instead of one per box voxel
// and tube slab of every pair.  A corner outside the layers (a sample rounded across a slab face)
// goes to global memory directly.  The layers accumulate in double: a voxel receives the weights of
// every sub-ray of every tilt near it (hundreds of terms of both signs for a signed image), whose
// float sum would carry about 1e-6 of rounding and depend on the atomics' order.
constexpr int kAdjSlabDoubles = 8192;   // 64 KiB of LDS: the x-y layers of a slab

// Cell layers per slab of a sub-volume (0: its x-y layer pair does not fit).
__host__ __device__ __forceinline__ int adj_slab_layers(int nx, int ny) {
    const long long nxy = (long long)nx * (long long)ny;
    const long long layers = (long long)kAdjSlabDoubles / (nxy > 0 ? nxy : 1);
    return layers >= 2 ? (int)(layers - 1) : 0;
}

struct AdjSlabArgs {
    const int2* items;      // (sub-volume, first cell layer zs), per XCD in runs of per_xcd; x < 0: none
    int per_xcd;
    const int* vfirst;      // per sub-volume: first slot of its pairs in `order`, and their count
    const int* vcount;
};

__global__ void __launch_bounds__(256) pair_adjoint_slab_kernel(PairArgs a, AdjSlabArgs sa, float scale,
                                                                float* __restrict__ grads) {
    __shared__ double box[kAdjSlabDoubles];
    const int pos = (int)(blockIdx.x >> 3);
    if (pos >= sa.per_xcd) return;   // whole workgroup
    const int2 it = sa.items[(int)(blockIdx.x & 7u) * sa.per_xcd + pos];
    if (it.x < 0) return;   // whole workgroup
    const int first = sa.vfirst[it.x], npair = sa.vcount[it.x];
    const VolG v0 = a.pairs[a.order[first]].v;
    const int L = adj_slab_layers(v0.nx, v0.ny);
    const int zs = it.y, ze = min(zs + L, v0.nz);   // cell layers [zs, ze); layer c spans q_z in [c, c + 1)
    const int bz0 = max(zs, 0), bz1 = min(ze, v0.nz - 1);
    const int nxy = v0.nx * v0.ny, nbox = nxy * (bz1 - bz0 + 1);
    for (int e = (int)threadIdx.x; e < nbox; e += 256) box[e] = 0.0;
    __syncthreads();
    const int lane = (int)(threadIdx.x & 63), wave = (int)(threadIdx.x >> 6);
    const int sub = lane & 3, pix = lane >> 2;
    const int tx = (wave & 1) * 4 + (pix & 3), ty = (wave >> 1) * 4 + (pix >> 2);
    for (int q = 0; q < npair; q++) {
        const int p = a.order[first + q];
        const PairDev& P = a.pairs[p];
        const int x0 = P.x0, y0 = P.y0, w = P.w, h = P.h;
        const long long io = P.img_offset;
        const int ntx = (w + 7) >> 3, ntiles = ntx * ((h + 7) >> 3);
        for (int t = 0; t < ntiles; t++) {
            __asm__ volatile("" ::: "memory");   // geometry re-read per tile, as in pair_march_kernel
            const VolG v = P.v;
            const TiltG g = P.g;
            float* __restrict__ gv = grads + P.vol_offset;
            const double sx = a.shifts ? a.shifts[2 * p] : 0.0, sy = a.shifts ? a.shifts[2 * p + 1] : 0.0;
            const double step = (double)v.vs[0] * 0.15;
            const int i = (t % ntx) * 8 + tx, j = (t / ntx) * 8 + ty;
            if (!(i < w && j < h)) continue;
            // proj = (float)(0.25 * step * sum): the same factor per sample
            const double r = (double)a.in[io + (long long)j * w + i] * (double)scale * (step * 0.25);
            if (r == 0.0) continue;
            SubraySamples s;
            const double px = (double)(x0 + i) + ((sub & 2) ? 0.75 : 0.25);
            const double py = (double)(y0 + j) + ((sub & 1) ? 0.75 : 0.25);
            if (!subray_samples(v, g, px, py, step, s, sx, sy)) continue;
            int sgn[3];
            float inv[3];
#pragma unroll
            for (int c = 0; c < 3; c++) walk_dir(s.dq[c], sgn[c], inv[c]);
            // samples of this slab: from the crossing of its entry face to that of its exit face, as
            // the walker computes face crossings (CellWalker::step), clamped to the sub-ray
            const float offz = -s.q0[2] * inv[2];
            const float fin = (float)(sgn[2] > 0 ? zs : ze), fout = (float)(sgn[2] > 0 ? ze : zs);
            // (the first and last slabs also take what a volume stored in part is sampled at beyond its layers)
            const bool bottom = zs <= -1, top = ze >= v.nz;
            const int kin = max(0, min(s.count, (int)ceilf(__builtin_fmaf(fin, inv[2], offz))));
            const int kout = max(0, min(s.count, (int)ceilf(__builtin_fmaf(fout, inv[2], offz))));
            const int kA = (sgn[2] > 0 ? bottom : top) ? 0 : kin, kB = (sgn[2] > 0 ? top : bottom) ? s.count : kout;
            if (kB <= kA) continue;
            CellWalker wk;
            wk.init_from(s.q0, s.dq, sgn, inv, kA, kB);
            while (wk.active()) {
                wk.step([&](const int cell[3], int k, int mi) {
                    double W[8];
                    cell_weights(cell_moments(s.q0, s.dq, cell, k, mi), W);
                    // clamp-addressed corners (cell_corners): 0 step where an index is clamped
                    const int xa = clampi(cell[0], 0, v.nx - 1), ya = clampi(cell[1], 0, v.ny - 1);
                    const int za = clampi(cell[2], 0, v.nz - 1);
                    const int dx = (cell[0] + 1 > xa && xa + 1 < v.nx) ? 1 : 0;
                    const int dy = (cell[1] + 1 > ya && ya + 1 < v.ny) ? v.nx : 0;
                    const int zb = (cell[2] + 1 > za && za + 1 < v.nz) ? za + 1 : za;
                    const int o0 = ya * v.nx + xa;
#pragma unroll
                    for (int c = 0; c < 8; c++) {
                        const double wc = r * W[c];
                        if (wc == 0.0) continue;
                        const int zc = (c & 4) ? zb : za;
                        const int o = o0 + ((c & 1) ? dx : 0) + ((c & 2) ? dy : 0);
                        if (zc >= bz0 && zc <= bz1)
                            unsafeAtomicAdd(box + (zc - bz0) * nxy + o, wc);
                        else
                            unsafeAtomicAdd(gv + (size_t)zc * (size_t)nxy + (size_t)o, (float)wc);
                    }
                });
            }
        }
    }
    __syncthreads();
    float* __restrict__ gv = grads + a.pairs[a.order[first]].vol_offset + (size_t)bz0 * (size_t)nxy;
    for (int e = (int)threadIdx.x; e < nbox; e += 256)
        if (box[e] != 0.0) unsafeAtomicAdd(gv + e, (float)box[e]);
}

// The transpose for flat rays, summed per sub-volume and run of y rows: a flat ray stays in one cell
// row (the voxel rows y and y + 1), so a workgroup that owns rows [ys, ys + L) of a sub-volume sets up
// and walks exactly the sub-rays of its tilts that lie there, each once and over its whole length (a z
// slab sets every sub-ray of every tilt up again for each slab, 65 times for 64 layers).  The rows'
// voxel planes are in LDS in double, padded by the clamp border, and reach the gradient with one atomic
// per voxel and run.  Lanes run along the detector axis on which y changes less, over the pixels of the
// run, and on along the other: a wave's rays lie a pixel apart and rarely add to one voxel at once.  The
// planes leave room for one workgroup on a compute unit, so it has sixteen waves to cover the LDS
// additions (a wave's ds_add_f64 takes nine cycles).
// 100 cubes of 64^3 by 41 tilts: 19.5 ms (22.2 with eight waves), against 156 ms with z slabs and eight
// additions per cell.
constexpr int kAdjFlatThreads = 1024;
constexpr int kAdjFlatBytes = 144 << 10;   // LDS for the padded planes
constexpr int kAdjFlatPlanes = 8;          // at most

// Voxel planes a workgroup holds (one more than its cell rows), or 0 when two do not fit.
__host__ __device__ __forceinline__ int adj_flat_planes(int nx, int nz) {
    const long long plane = (long long)(nx + 2) * (long long)(nz + 2) * (long long)sizeof(double);
    const long long n = (long long)kAdjFlatBytes / plane;
    return n < 2 ? 0 : (n > kAdjFlatPlanes ? kAdjFlatPlanes : (int)n);
}

__global__ void __launch_bounds__(kAdjFlatThreads) pair_adjoint_flat_kernel(PairArgs a, AdjSlabArgs sa, float scale,
                                                                           float* __restrict__ grads) {
    extern __shared__ double rows[];
    const int pos = (int)(blockIdx.x >> 3);
    if (pos >= sa.per_xcd) return;   // whole workgroup
    const int2 it = sa.items[(int)(blockIdx.x & 7u) * sa.per_xcd + pos];
    if (it.x < 0) return;   // whole workgroup
    const int first = sa.vfirst[it.x], npair = sa.vcount[it.x];
    const VolG v0 = a.pairs[a.order[first]].v;
    const int L = adj_flat_planes(v0.nx, v0.nz) - 1, ys = it.y;
    const int px = v0.nx + 2, pz = v0.nz + 2, plane = px * pz, nbox = plane * (L + 1);
    for (int e = (int)threadIdx.x; e < nbox; e += kAdjFlatThreads) rows[e] = 0.0;
    __syncthreads();
    for (int q = 0; q < npair; q++) {
        __asm__ volatile("" ::: "memory");   // geometry re-read per pair, as in pair_march_kernel
        const int p = a.order[first + q];
        const PairDev& P = a.pairs[p];
        const VolG v = P.v;
        const TiltG g = P.g;
        float* __restrict__ gv = grads + P.vol_offset;
        const double sx = a.shifts ? a.shifts[2 * p] : 0.0, sy = a.shifts ? a.shifts[2 * p + 1] : 0.0;
        const double step = (double)v.vs[0] * 0.15;
        // texel y of the sub-ray at (px, py) (subray_samples' q0[1]): affine, gx per pixel in x, gy in y
        const double ysc = (double)v.rcp[1] * (double)v.dim[1];
        auto texel_y = [&](double pxd, double pyd) {
            const double xa = (((double)g.A[0] * pxd + (double)g.A[1] * pyd) + (double)g.A[2]) - sx;
            const double ya = (((double)g.A[3] * pxd + (double)g.A[4] * pyd) + (double)g.A[5]) - sy;
            const double c = ((double)g.d[1] + xa * (double)g.u[1]) + ya * (double)g.v[1];
            return (float)((c - (double)v.bbMin[1]) * ysc - 0.5);
        };
        const double y00 = (double)texel_y((double)P.x0, (double)P.y0);
        const double gx = ((double)g.A[0] * g.u[1] + (double)g.A[3] * g.v[1]) * ysc;
        const double gy = ((double)g.A[1] * g.u[1] + (double)g.A[4] * g.v[1]) * ysc;
        const bool along_x = fabs(gx) <= fabs(gy);
        const int ni = along_x ? P.w : P.h, nj = along_x ? P.h : P.w;   // lanes along i
        const double gi = along_x ? gx : gy, gj = along_x ? gy : gx;
        // y of the run's sub-rays: [ys, ys + L), the first and last rows to the volume's faces (a ray beyond them
        // misses it); tol is far above the rounding of texel_y and of the row's first pixel
        constexpr double tol = 1e-2;
        const double lo = (ys <= -1 ? -0.5 : (double)ys) - tol - y00;
        const double face = ((double)v.bbMax[1] - (double)v.bbMin[1]) * ysc - 0.5;
        const double hi = (ys + L >= v.ny ? face : (double)(ys + L)) + tol - y00;
        // a sub-ray's y is i gi + j gj and its offset in the pixel, om .. oM: the j with such sub-rays for some i,
        const double om = fmin(0.25 * gx, 0.75 * gx) + fmin(0.25 * gy, 0.75 * gy);
        const double oM = fmax(0.25 * gx, 0.75 * gx) + fmax(0.25 * gy, 0.75 * gy);
        int j0 = 0, j1 = nj - 1;
        if (fabs(gj) > 1e-3) {
            const double l = lo - oM - fmax(0.0, gi * (ni - 1)), h = hi - om - fmin(0.0, gi * (ni - 1));
            const double a0 = fmin(l / gj, h / gj), a1 = fmax(l / gj, h / gj);
            j0 = (int)fmax(0.0, fmin((double)nj, ceil(a0)));
            j1 = (int)fmin((double)(nj - 1), fmax(-1.0, floor(a1)));
        }
        // and of each j the `row` pixels i from the first with sub-rays in the run, so that a wave's lanes are rays
        // of the run also where the detector's axes are oblique to y (all ni pixels of a row kept a few of 64
        // lanes busy at 45 degrees: 12 cubes of 94^3 by 21 tilts 122 ms, 11.6 so; by z slabs 59 ms); all ni where
        // the run is as wide
        const double inv = fabs(gi) > 1e-3 ? 1.0 / gi : 0.0, wide = floor((hi - lo + (oM - om)) * fabs(inv)) + 1.0;
        const bool part = inv != 0.0 && wide < (double)ni;
        const double edge = part ? (gi > 0.0 ? lo - oM : hi - om) * inv : 0.0, step_j = part ? gj * inv : 0.0;
        const int row = wave_uniform(part ? (int)fmax(0.0, wide) : ni);
        const int nrow = wave_uniform(j1 - j0 + 1), total = row * nrow * 4;
        const float start = wave_uniform((float)(edge - step_j * j0)), slope = wave_uniform((float)step_j);
        j0 = wave_uniform(j0);
        for (int idx = (int)threadIdx.x; idx < total; idx += kAdjFlatThreads) {
            const int rest = idx / row, sub = rest / nrow, jj = rest - sub * nrow, j = j0 + jj;
            const int i = idx - rest * row + (int)ceilf(start - slope * (float)jj);   // (+ 0 without part)
            if (i < 0 || i >= ni) continue;
            const int wx = along_x ? i : j, wy = along_x ? j : i;
            const double pxd = (double)(P.x0 + wx) + ((sub & 2) ? 0.75 : 0.25);
            const double pyd = (double)(P.y0 + wy) + ((sub & 1) ? 0.75 : 0.25);
            const float qy = texel_y(pxd, pyd);
            const int yc = clampi((int)floorf(qy), -1, v.ny - 1);   // beyond the volume: both rows clamp alike
            if (yc < ys || yc >= ys + L) continue;
            // proj = (float)(0.25 * step * sum): the same factor per sample
            const double r = (double)a.in[P.img_offset + (long long)wy * P.w + wx] * (double)scale * (step * 0.25);
            if (r == 0.0) continue;
            SubraySamples s;
            if (!subray_samples(v, g, pxd, pyd, step, s, sx, sy)) continue;
            const FlatDir d = flat_dir(s.dq);
            FlatWalker w;
            w.init(d, s.q0, s.count);
            // the walk's cells in the padded planes (-1 .. n): the first sample's as it is, the last with a
            // quarter of a cell for the walk's rounding, half as far as a whole volume's last sample is from the
            // border (a volume stored in part, with a z shift, is sampled beyond it)
            const float last = (float)(s.count - 1);
            const int xf = (int)floorf(s.q0[0]), zf = (int)floorf(s.q0[2]);
            const float xl = __builtin_fmaf(last, s.dq[0], s.q0[0]), zl = __builtin_fmaf(last, s.dq[2], s.q0[2]);
            if (xf < -1 || xf > v.nx - 1 || zf < -1 || zf > v.nz - 1 ||
                !(xl >= -0.75f && xl < (float)v.nx - 0.25f && zl >= -0.75f && zl < (float)v.nz - 0.25f)) {
                flat_scatter_direct(v, gv, d, s.q0, r, w, []() { return true; });
                continue;
            }
            const double b = (double)(s.q0[1] - floorf(s.q0[1]));
            const int ox = d.sgn[0], oz = d.sgn[1] * px;
            int o = (yc - ys) * plane + (d.sgn[1] * w.near(d, s.q0, 1) + 1) * px + (d.sgn[0] * w.near(d, s.q0, 0) + 1);
            FlatEdgeSums e;
            e.clear();
            for (;;) {
                const bool ax = w.kb[0] < w.kb[1];
                float ca, cc;
                const float m = w.samples(d, ax ? w.kb[0] : w.kb[1], ca, cc);
                e.add(r, ca, cc, m, d.K);
                w.advance(d, ax);
                auto put = [&](int dx, int dz, double val) {
                    const int at = o + (dx ? ox : 0) + (dz ? oz : 0);
                    const double v1 = val * b;
                    unsafeAtomicAdd(rows + at, val - v1);
                    unsafeAtomicAdd(rows + at + plane, v1);
                };
                if (!w.active()) {
                    e.flush(put);
                    break;
                }
                e.step(ax, put);
                o += ax ? ox : oz;
            }
        }
    }
    __syncthreads();
    float* __restrict__ gv = grads + a.pairs[a.order[first]].vol_offset;
    for (int e = (int)threadIdx.x; e < nbox; e += kAdjFlatThreads) {
        const double add = rows[e];
        if (add == 0.0) continue;
        const int yp = e / plane, rem = e - yp * plane, z = rem / px, x = rem - z * px;
        const int gy = clampi(ys + yp, 0, v0.ny - 1), gz = clampi(z - 1, 0, v0.nz - 1), gx = clampi(x - 1, 0, v0.nx - 1);
        unsafeAtomicAdd(gv + ((size_t)gz * (size_t)v0.ny + (size_t)gy) * (size_t)v0.nx + gx, (float)add);
    }
}

// vol_grads += scale * P_s^T in: the transpose of the per-cell closed form, one set of eight
// atomics per cell a sub-ray crosses (as fp_adjoint_kernel).
__global__ void __launch_bounds__(256) pair_adjoint_kernel(PairArgs a, float scale, float* __restrict__ grads) {
    __shared__ double chunk[kChunkFloats];
    __shared__ int zr[2];
    const int slot = slot_of_block(a.per_xcd);
    if (slot >= a.npairs) return;
    const int p = a.order[slot];
    const PairDev& P = a.pairs[p];
    const int x0 = P.x0, y0 = P.y0, w = P.w, h = P.h;
    const long long io = P.img_offset;
    const int lane = (int)(threadIdx.x & 63), wave = (int)(threadIdx.x >> 6);
    const int sub = lane & 3, pix = lane >> 2;
    const int tx = (wave & 1) * 4 + (pix & 3), ty = (wave >> 1) * 4 + (pix >> 2);
    const int ntx = (w + 7) >> 3, ntiles = ntx * ((h + 7) >> 3);
    for (int t = 0; t < ntiles; t++) {
        __asm__ volatile("" ::: "memory");   // geometry re-read per tile, as in pair_march_kernel
        const VolG v = P.v;
        const TiltG g = P.g;
        float* __restrict__ gv = grads + P.vol_offset;
        const double sx = a.shifts ? a.shifts[2 * p] : 0.0, sy = a.shifts ? a.shifts[2 * p + 1] : 0.0;
        const double step = (double)v.vs[0] * 0.15;
        const int i = (t % ntx) * 8 + tx, j = (t / ntx) * 8 + ty;
        double r = 0.0;
        SubraySamples s;
        s.count = 0;
#pragma unroll
        for (int c = 0; c < 3; c++) s.q0[c] = s.dq[c] = 0.0f;
        if (i < w && j < h) {
            // proj = (float)(0.25 * step * sum): the same factor per sample
            r = (double)a.in[io + (long long)j * w + i] * (double)scale * (step * 0.25);
            const double px = (double)(x0 + i) + ((sub & 2) ? 0.75 : 0.25);
            const double py = (double)(y0 + j) + ((sub & 1) ? 0.75 : 0.25);
            if (r == 0.0 || !subray_samples(v, g, px, py, step, s, sx, sy)) s.count = 0;
        }
        auto weights = [&](double wgt[8], const int cell[3], int k, int mi) {
            double W[8];
            cell_weights(cell_moments(s.q0, s.dq, cell, k, mi), W);
#pragma unroll
            for (int c = 0; c < 8; c++) wgt[c] = r * W[c];
        };
        if (g.n[1] == 0.0f) {   // uniform: flat rays (flat_walk.hpp)
            float dq[3];
            tube_step(v, g, step, dq);
            if (P.staged) {
                const double pi0 = (double)(x0 + (t % ntx) * 8), pj0 = (double)(y0 + (t / ntx) * 8);
                const TubeBox tb = tube_box(v, g, P.tp, pi0 + 0.25, pi0 + 7.75, pj0 + 0.25, pj0 + 7.75, sx, sy);
                flat_tube_scatter(v, gv, chunk, zr, P.tp, tb, dq, s.q0, s.count, r);
            } else if (s.count > 0) {
                const FlatDir d = flat_dir(dq);
                FlatWalker w;
                w.init(d, s.q0, s.count);
                flat_scatter_direct(v, gv, d, s.q0, r, w, []() { return true; });
            }
        } else if (P.staged) {   // uniform: per-slab sums in LDS, one atomic per box voxel
            const TubeDir td = tube_dir(v, g, step);
            const double pi0 = (double)(x0 + (t % ntx) * 8), pj0 = (double)(y0 + (t / ntx) * 8);
            const TubeBox tb = tube_box(v, g, P.tp, pi0 + 0.25, pi0 + 7.75, pj0 + 0.25, pj0 + 7.75, sx, sy);
            tube_scatter(v, gv, chunk, zr, P.tp, tb, td, s.q0, s.count, weights);
        } else if (s.count > 0) {
            for_each_cell(s.q0, s.dq, s.count, [&](const int cell[3], int k, int mi) {
                uint32_t o[8];
                cell_corners_bytes(v, cell, o);
                double wgt[8];
                weights(wgt, cell, k, mi);
#pragma unroll
                for (int c = 0; c < 8; c++)
                    if (wgt[c] != 0.0) unsafeAtomicAdd(gv + (o[c] >> 2), (float)wgt[c]);
            });
        }
    }
}

constexpr int kMaxCcShift = 32;

// GetDisplacement per pair (Reconstructor.cpp:1746-1959) as a direct sum over the window: the
// raw correlation C(r) = sum_y B(y) A(y - r) for every integer r in the disk, then the square's
// mean and energy terms, the maxShift disk (wbpWeighting.cu:265-294) and nppiMaxIndx's first
// maximum in the square's row-major order.
//
// The sum is bound by double multiply-adds (the products of floats are exact in double), so the work is
// tiled for registers: a thread owns one row shift ry, every S-th window row and kCcR column shifts in
// double accumulators, and for each 8 window columns takes 8 values of B and 16 of A from LDS for 72
// multiply-adds.  Neighbouring lanes have neighbouring ry: odd row pitches keep their reads of A apart.
// Windows are staged in tiles of at most kCcTile columns and as many rows as fit, zero outside the image.
// 4100 windows of about 76 x 76 with shifts to 12: 22.3 ms with one wave per candidate and two loads per
// multiply-add, 1.4 ms so.
// multi != 0: MultiPeakDetection (Reconstructor.cpp:1887-1935): among the peaks of the float map
// (findPeak, wbpWeighting.cu:329-386: above the 8 neighbours, the two upper diagonal ones or equal,
// and at least 0.9f of the maximum) the one nearest to zero shift (maxShiftWeighted,
// wbpWeighting.cu:295-327: weight 1 / (dist + 0.0001f)), first in row-major order; the CC value and
// the failure test keep the first search's maximum.  Candidates outside the disk are 0 in the map.
constexpr int kCcR = 9, kCcTile = 80;
constexpr int kCcStageBytes = 35 << 10;   // four blocks per compute unit at small max_shift

__host__ __device__ inline int cc_side(int M) { return 2 * M + 1; }
// window rows taken side by side: 256 threads over the row shifts
__host__ __device__ inline int cc_slices(int M) { return 256 / cc_side(M) < 32 ? 256 / cc_side(M) : 32; }
// bytes of the staged tiles: less where the candidates' sums leave less of 60 KB, always enough for one
// row per slice and 256 * kCcR doubles (cc_slices * (pa + pb) + 2 M pa floats: 24.9 KB at M = 32, where
// 27.6 KB are left)
__host__ __device__ inline int cc_stage_bytes(int M) {
    const int rest = (60 << 10) - cc_side(M) * cc_side(M) * 8;
    return rest < kCcStageBytes ? rest : kCcStageBytes;
}
__device__ __forceinline__ bool cc_in_disk(int rx, int ry, int M) {
    return sqrtf((float)(rx * rx + ry * ry)) <= (float)M;
}

// The first maximum of val over the block's order keys k (each thread's own first): its key in *key on
// all threads, and its value.
__device__ __forceinline__ double block_first_max(double val, int k, int* key) {
    __shared__ double bv[256];
    __shared__ int bk[256];
    bv[threadIdx.x] = val;
    bk[threadIdx.x] = k;
    __syncthreads();
    for (int o = 128; o > 0; o >>= 1) {
        if ((int)threadIdx.x < o) {
            const double v = bv[threadIdx.x + o];
            const int q = bk[threadIdx.x + o];
            // a thread without candidates has key INT_MAX
            if (q != INT_MAX && (bk[threadIdx.x] == INT_MAX || v > bv[threadIdx.x] ||
                                 (v == bv[threadIdx.x] && q < bk[threadIdx.x]))) {
                bv[threadIdx.x] = v;
                bk[threadIdx.x] = q;
            }
        }
        __syncthreads();
    }
    const double r = bv[0];
    *key = bk[0];
    __syncthreads();
    return r;
}

__global__ void __launch_bounds__(256) pair_cc_kernel(const PairDev* __restrict__ pairs, int npairs,
                                                      const float* __restrict__ models,
                                                      const float* __restrict__ targets, int N, int M,
                                                      int multi, int* __restrict__ peak, float* __restrict__ ccv,
                                                      float* __restrict__ ccmap) {
    extern __shared__ double cc_lds[];   // the candidates' sums, then the staged tiles
    const int p = (int)blockIdx.x;
    if (p >= npairs) return;
    const PairDev& P = pairs[p];
    const int w = P.w, h = P.h;
    const float* __restrict__ A = targets + P.img_offset;
    const float* __restrict__ B = models + P.img_offset;
    const int lane = (int)(threadIdx.x & 63), wave = (int)(threadIdx.x >> 6), tid = (int)threadIdx.x;
    // window sums of A, A^2, B, B^2 (the square is zero outside the window)
    double sa = 0.0, saa = 0.0, sb = 0.0;
    double sbb = 0.0;
    for (long long q = threadIdx.x; q < (long long)w * h; q += 256) {
        const double av = (double)A[q], bv = (double)B[q];
        sa += av;
        saa += av * av;
        sb += bv;
        sbb += bv * bv;
    }
    block_sum3(sa, saa, sb);
    __shared__ double tot[4];
    if (threadIdx.x == 0) {
        tot[0] = sa;
        tot[1] = saa;
        tot[2] = sb;
    }
    double d = 0.0, e = 0.0;
    block_sum3(sbb, d, e);
    if (threadIdx.x == 0) tot[3] = sbb;
    const int side = cc_side(M), ncand = side * side, S = cc_slices(M);
    double* const craw = cc_lds;
    float* const stage = reinterpret_cast<float*>(cc_lds + ncand);
    const int ry = tid % side - M, slice = tid / side;
    const int ntx = (w + kCcTile - 1) / kCcTile, xt = ((w + ntx - 1) / ntx + 7) / 8 * 8;
    const int pa = (xt + 8) | 1, pb = xt | 1;   // row pitches of the tiles of A and B
    const int fit = (cc_stage_bytes(M) / 4 - 2 * M * pa) / (S * (pa + pb));
    const int nty = (h + fit * S - 1) / (fit * S);
    const int nb = S * ((h + S * nty - 1) / (S * nty));   // window rows per tile
    float* const At = stage;
    float* const Bt = stage + (nb + 2 * M) * pa;
    for (int rx0 = -M; rx0 <= M; rx0 += kCcR) {
        double acc[kCcR];
#pragma unroll
        for (int r = 0; r < kCcR; r++) acc[r] = 0.0;
        for (int y0 = 0; y0 < h; y0 += nb) {
            for (int x0 = 0; x0 < w; x0 += xt) {
                __syncthreads();
                for (int r = wave; r < nb + 2 * M; r += 4) {
                    const int y = y0 - M + r;
                    for (int c = lane; c < xt + 8; c += 64) {
                        const int x = x0 - rx0 - 8 + c;
                        At[r * pa + c] = y >= 0 && y < h && x >= 0 && x < w ? A[(long long)y * w + x] : 0.0f;
                    }
                }
                for (int r = wave; r < nb; r += 4) {
                    const int y = y0 + r;
                    for (int c = lane; c < xt; c += 64) {
                        const int x = x0 + c;
                        Bt[r * pb + c] = y < h && x < w ? B[(long long)y * w + x] : 0.0f;
                    }
                }
                __syncthreads();
                if (slice < S) {
                    for (int y = slice; y < nb && y0 + y < h; y += S) {
                        const float* arow = At + (y - ry + M) * pa;
                        const float* brow = Bt + y * pb;
                        for (int x = 0; x < xt; x += 8) {
                            double a[16], b[8];
#pragma unroll
                            for (int q = 0; q < 16; q++) a[q] = (double)arow[x + q];
#pragma unroll
                            for (int q = 0; q < 8; q++) b[q] = (double)brow[x + q];
#pragma unroll
                            for (int q = 0; q < 8; q++)
#pragma unroll
                                for (int r = 0; r < kCcR; r++) acc[r] = __builtin_fma(b[q], a[q - r + 8], acc[r]);
                        }
                    }
                }
            }
        }
        __syncthreads();
        double* const part = reinterpret_cast<double*>(stage);
#pragma unroll
        for (int r = 0; r < kCcR; r++) part[r * 256 + tid] = acc[r];
        __syncthreads();
        for (int q = tid; q < kCcR * side; q += 256) {
            const int r = q / side, row = q % side;
            double sum = 0.0;
            for (int k = 0; k < S; k++) sum += part[r * 256 + k * side + row];
            if (rx0 + r <= M) craw[row * side + rx0 + r + M] = sum;
        }
    }
    __syncthreads();
    const double SA = tot[0], SB = tot[2], n2 = (double)N * (double)N;
    const double sumA = tot[1] - SA * SA / n2, sumB = tot[3] - SB * SB / n2;
    const double den = sqrt(sumA * sumB), off = SA * SB / n2;
    const bool ok = sumA * sumB > 0.0;
    // candidates in the square's row-major order k: rows ry = 0..M, then -M..-1; likewise columns
    const auto shift_of = [&](int k, int& rx, int& ry) {
        const int yy = k / side, xx = k % side;
        ry = yy <= M ? yy : yy - side;
        rx = xx <= M ? xx : xx - side;
    };
    double best = 0.0;
    int bestk = INT_MAX;
    for (int k = tid; k < ncand; k += 256) {
        int rx, ry;
        shift_of(k, rx, ry);
        const int c = (ry + M) * side + (rx + M);
        const bool in = cc_in_disk(rx, ry, M);
        const double cc = in && ok ? (craw[c] - off) / den : 0.0;
        craw[c] = cc;
        if (ccmap) ccmap[(long long)p * ncand + c] = (float)cc;
        if (in && (bestk == INT_MAX || cc > best)) {
            best = cc;
            bestk = k;
        }
    }
    best = block_first_max(best, bestk, &bestk);
    int bx, by;
    if (multi) {
        // the float map value at shift (rx, ry), wrapped around the N x N square as findPeak's
        // neighbours are: 0 outside the disk (maxShift)
        auto map = [&](int rx, int ry) -> float {
            rx = ((rx % N) + N) % N;
            ry = ((ry % N) + N) % N;
            rx = rx > N / 2 ? rx - N : rx;
            ry = ry > N / 2 ? ry - N : ry;
            if (rx < -M || rx > M || ry < -M || ry > M) return 0.0f;
            return (float)craw[(ry + M) * side + (rx + M)];
        };
        const float thr = (float)best * 0.9f;
        float bestw = 0.0f;
        bestk = INT_MAX;
        for (int k = tid; k < ncand; k += 256) {
            int rx, ry;
            shift_of(k, rx, ry);
            const float d = sqrtf((float)(rx * rx + ry * ry));
            float wv = 0.0f;
            if (d <= (float)M) {
                const float val = map(rx, ry);
                const bool pk = map(rx - 1, ry) < val && map(rx + 1, ry) < val && map(rx, ry - 1) < val &&
                                map(rx, ry + 1) < val && map(rx - 1, ry - 1) <= val && map(rx - 1, ry + 1) < val &&
                                map(rx + 1, ry - 1) <= val && map(rx + 1, ry + 1) < val && val >= thr;
                wv = pk ? 1.0f / (d + 0.0001f) : 0.0f;
            }
            if (bestk == INT_MAX || wv > bestw) {
                bestw = wv;
                bestk = k;
            }
        }
        (void)block_first_max((double)bestw, bestk, &bestk);
    }
    if (tid != 0) return;
    shift_of(bestk, bx, by);
    const bool fail = !ok || !(best > 0.0);
    peak[2 * p] = fail ? -1000 : bx;
    peak[2 * p + 1] = fail ? -1000 : by;
    ccv[p] = ok ? (float)best : 0.0f;
}

}  // namespace
}  // namespace artia

using namespace artia;

struct artia_pairs {
    artia_ctx* ctx = nullptr;
    PairDev* pairs = nullptr;
    int* order = nullptr;
    int npairs = 0, per_xcd = 0;
    bool any_flat = false, any_other = false;   // pairs with and without n_y == 0
    // the summed adjoint (pair_adjoint_flat_kernel when every pair's rays are flat, otherwise
    // pair_adjoint_slab_kernel): work items and per-volume slot ranges, or none when a sub-volume's
    // planes do not fit or a tilt runs parallel to its z layers
    int2* slab_items = nullptr;
    int* vfirst = nullptr;
    int* vcount = nullptr;
    int slab_per_xcd = 0;
    bool flat = false;       // the items are runs of y rows (flat rays), not z slabs
    size_t flat_lds = 0;     // LDS bytes of the largest run's planes
};

namespace {

artia_status pairs_fail(artia_pairs* ps, artia_status code, const char* what) {
    return fail(ps->ctx, code, "%s", what);
}

PairArgs base_args(const artia_pairs* ps) {
    PairArgs a{};
    a.pairs = ps->pairs;
    a.order = ps->order;
    a.npairs = ps->npairs;
    a.per_xcd = ps->per_xcd;
    return a;
}

dim3 pair_grid(const artia_pairs* ps, int parts = 1) { return dim3((unsigned)(8 * ps->per_xcd * parts)); }

template <int kMode>
void launch_march(const artia_pairs* ps, const PairArgs& a) {
    const dim3 grid = pair_grid(ps, kMode == kProject ? kPairParts : 1);
    if (ps->any_flat) hipLaunchKernelGGL((pair_march_kernel<kMode, true>), grid, dim3(256), 0, ps->ctx->stream, a);
    if (ps->any_other) hipLaunchKernelGGL((pair_march_kernel<kMode, false>), grid, dim3(256), 0, ps->ctx->stream, a);
}

}  // namespace

extern "C" {

artia_status artia_pairs_create(artia_ctx* ctx, const artia_pair_volume* volumes, int nvol, const artia_pair* pairs,
                                const artia_tilt_geom* geoms, int npairs, artia_pairs** out) {
    if (!ctx) return ARTIA_ERR_INVALID_ARGUMENT;
    if (!out || !volumes || !pairs || !geoms || nvol <= 0 || npairs <= 0)
        return fail(ctx, ARTIA_ERR_INVALID_ARGUMENT, "artia_pairs_create: null pointer or empty set");
    *out = nullptr;
    for (int i = 0; i < nvol; i++) {
        const artia_vol_geom& g = volumes[i].geom;
        if (!valid_geometry(&g, &geoms[0]) || volumes[i].offset < 0)
            return fail(ctx, ARTIA_ERR_INVALID_ARGUMENT, "artia_pairs_create: invalid sub-volume %d", i);
        if (g.nx < 2 || g.ny < 2 || g.nz < 2 || g.nx >= (1 << 24) || (double)g.ny * g.nz >= 16777216.0 ||
            (double)g.nx * g.ny * g.nz >= 1073741824.0)
            return fail(ctx, ARTIA_ERR_UNSUPPORTED,
                        "artia_pairs_create: sub-volume %d is %d x %d x %d (needs 2 .. 2^24-1 voxels per axis, "
                        "ny*nz < 2^24, fewer than 2^30 voxels)",
                        i, g.nx, g.ny, g.nz);
    }
    std::vector<PairDev> host((size_t)npairs);
    for (int p = 0; p < npairs; p++) {
        const artia_pair& q = pairs[p];
        if (q.volume < 0 || q.volume >= nvol || q.w <= 0 || q.h <= 0 || q.offset < 0)
            return fail(ctx, ARTIA_ERR_INVALID_ARGUMENT, "artia_pairs_create: pair %d has a bad volume or window", p);
        if (!valid_geometry(&volumes[q.volume].geom, &geoms[p]))
            return fail(ctx, ARTIA_ERR_INVALID_ARGUMENT, "artia_pairs_create: invalid geometry of pair %d", p);
        PairDev& d = host[(size_t)p];
        d.g = flat_beam(to_device(geoms[p]));   // as the exact forward projector takes it
        d.v = to_device(volumes[q.volume].geom);
        d.staged = ctx->march_lds && tube_plan(d.v, d.g, d.tp) ? 1 : 0;
        d.vol_offset = volumes[q.volume].offset;
        d.img_offset = q.offset;
        d.x0 = q.x0;
        d.y0 = q.y0;
        d.w = q.w;
        d.h = q.h;
    }
    // slots grouped by sub-volume (stable), dealt to the 8 XCDs in contiguous runs
    std::vector<int> order((size_t)npairs);
    std::iota(order.begin(), order.end(), 0);
    std::stable_sort(order.begin(), order.end(), [&](int a, int b) { return pairs[a].volume < pairs[b].volume; });
    artia_pairs* ps = new artia_pairs();
    ps->ctx = ctx;
    ps->npairs = npairs;
    ps->per_xcd = (npairs + 7) / 8;
    // slab work items of the summed adjoint: every sub-volume's cell layers -1 .. nz - 1 in runs of
    // its slab depth, all on the XCD of the sub-volume (volume index mod 8), so the pairs' windows
    // are read through one L2
    std::vector<int> vfirst((size_t)nvol, 0), vcount((size_t)nvol, 0);
    for (int s = 0; s < npairs; s++) {
        const int vi = pairs[order[(size_t)s]].volume;
        if (vcount[(size_t)vi]++ == 0) vfirst[(size_t)vi] = s;
    }
    // (the staging switch off keeps the per-pair scatter, as it keeps the per-pair walks direct)
    bool slab_ok = ctx->march_lds, flat = ctx->march_lds;
    for (int p = 0; p < npairs; p++) {
        slab_ok = slab_ok && std::fabs(host[(size_t)p].g.n[2]) > 1e-3f;   // rays cross the z layers
        (host[(size_t)p].g.n[1] == 0.0f ? ps->any_flat : ps->any_other) = true;
    }
    flat = flat && !ps->any_other;
    for (int vi = 0; vi < nvol && flat; vi++)
        flat = vcount[(size_t)vi] == 0 || adj_flat_planes(volumes[vi].geom.nx, volumes[vi].geom.nz) > 0;
    slab_ok = slab_ok || flat;
    std::vector<std::vector<int2>> per((size_t)8);
    for (int vi = 0; vi < nvol && slab_ok; vi++) {
        if (vcount[(size_t)vi] == 0) continue;
        const artia_vol_geom& g = volumes[vi].geom;
        if (flat) {
            const int planes = adj_flat_planes(g.nx, g.nz);
            ps->flat_lds = std::max(ps->flat_lds, (size_t)planes * (size_t)(g.nx + 2) * (size_t)(g.nz + 2) * sizeof(double));
            for (int y = -1; y < g.ny; y += planes - 1) per[(size_t)(vi % 8)].push_back(make_int2(vi, y));
            continue;
        }
        const int L = adj_slab_layers(g.nx, g.ny);
        if (L <= 0) {
            slab_ok = false;
            break;
        }
        for (int zs = -1; zs < g.nz; zs += L) per[(size_t)(vi % 8)].push_back(make_int2(vi, zs));
    }
    ps->flat = flat;
    std::vector<int2> items;
    if (slab_ok) {
        size_t longest = 0;
        for (const auto& l : per) longest = std::max(longest, l.size());
        ps->slab_per_xcd = (int)longest;
        items.assign(8 * longest, make_int2(-1, 0));
        for (size_t x = 0; x < 8; x++)
            for (size_t k = 0; k < per[x].size(); k++) items[x * longest + k] = per[x][k];
    }
    hipError_t e = hipSetDevice(ctx->device);
    if (e == hipSuccess && flat)
        e = hipFuncSetAttribute(reinterpret_cast<const void*>(pair_adjoint_flat_kernel),
                                hipFuncAttributeMaxDynamicSharedMemorySize, kAdjFlatBytes);
    if (e == hipSuccess) e = hipMalloc(&ps->pairs, sizeof(PairDev) * (size_t)npairs);
    if (e == hipSuccess) e = hipMalloc(&ps->order, sizeof(int) * (size_t)npairs);
    if (e == hipSuccess)
        e = hipMemcpyAsync(ps->pairs, host.data(), sizeof(PairDev) * (size_t)npairs, hipMemcpyHostToDevice,
                           ctx->stream);
    if (e == hipSuccess)
        e = hipMemcpyAsync(ps->order, order.data(), sizeof(int) * (size_t)npairs, hipMemcpyHostToDevice, ctx->stream);
    if (e == hipSuccess && !items.empty()) {
        e = hipMalloc(&ps->slab_items, sizeof(int2) * items.size());
        if (e == hipSuccess) e = hipMalloc(&ps->vfirst, sizeof(int) * (size_t)nvol);
        if (e == hipSuccess) e = hipMalloc(&ps->vcount, sizeof(int) * (size_t)nvol);
        if (e == hipSuccess)
            e = hipMemcpyAsync(ps->slab_items, items.data(), sizeof(int2) * items.size(), hipMemcpyHostToDevice,
                               ctx->stream);
        if (e == hipSuccess)
            e = hipMemcpyAsync(ps->vfirst, vfirst.data(), sizeof(int) * (size_t)nvol, hipMemcpyHostToDevice,
                               ctx->stream);
        if (e == hipSuccess)
            e = hipMemcpyAsync(ps->vcount, vcount.data(), sizeof(int) * (size_t)nvol, hipMemcpyHostToDevice,
                               ctx->stream);
    }
    if (e == hipSuccess) e = hipStreamSynchronize(ctx->stream);
    if (e != hipSuccess) {
        artia_pairs_destroy(ps);
        return check_hip(ctx, e, "artia_pairs_create");
    }
    *out = ps;
    return ARTIA_OK;
}

artia_status artia_pairs_destroy(artia_pairs* ps) {
    if (!ps) return ARTIA_OK;
    if (ps->pairs) (void)hipFree(ps->pairs);
    if (ps->order) (void)hipFree(ps->order);
    if (ps->slab_items) (void)hipFree(ps->slab_items);
    if (ps->vfirst) (void)hipFree(ps->vfirst);
    if (ps->vcount) (void)hipFree(ps->vcount);
    delete ps;
    return ARTIA_OK;
}

artia_status artia_pairs_project(artia_pairs* ps, const float* volumes, const double* shifts, float* images,
                                 float* ms) {
    if (!ps) return ARTIA_ERR_INVALID_ARGUMENT;
    if (!volumes || !images) return pairs_fail(ps, ARTIA_ERR_INVALID_ARGUMENT, "artia_pairs_project: null pointer");
    artia_ctx* ctx = ps->ctx;
    PairArgs a = base_args(ps);
    a.vols = volumes;
    a.shifts = shifts;
    a.out = images;
    Timing t(ctx, ms);
    launch_march<kProject>(ps, a);
    artia_status st = check_hip(ctx, hipGetLastError(), "artia_pairs_project launch");
    if (st != ARTIA_OK) return st;
    return t.finish();
}

artia_status artia_pairs_loss_grad(artia_pairs* ps, const float* volumes, const double* shifts, const float* targets,
                                   double* loss, double* grad, double* normal, float* resid, float* ms) {
    if (!ps) return ARTIA_ERR_INVALID_ARGUMENT;
    if (!volumes || !targets || !loss || !grad)
        return pairs_fail(ps, ARTIA_ERR_INVALID_ARGUMENT, "artia_pairs_loss_grad: null pointer");
    artia_ctx* ctx = ps->ctx;
    PairArgs a = base_args(ps);
    a.vols = volumes;
    a.shifts = shifts;
    a.in = targets;
    a.out = resid;
    a.loss = loss;
    a.grad = grad;
    a.normal = normal;
    Timing t(ctx, ms);
    launch_march<kLossGrad>(ps, a);
    artia_status st = check_hip(ctx, hipGetLastError(), "artia_pairs_loss_grad launch");
    if (st != ARTIA_OK) return st;
    return t.finish();
}

artia_status artia_pairs_shift_grad(artia_pairs* ps, const float* volumes, const double* shifts,
                                    const float* weights, double* grad, float* ms) {
    if (!ps) return ARTIA_ERR_INVALID_ARGUMENT;
    if (!volumes || !weights || !grad)
        return pairs_fail(ps, ARTIA_ERR_INVALID_ARGUMENT, "artia_pairs_shift_grad: null pointer");
    artia_ctx* ctx = ps->ctx;
    PairArgs a = base_args(ps);
    a.vols = volumes;
    a.shifts = shifts;
    a.in = weights;
    a.grad = grad;
    Timing t(ctx, ms);
    launch_march<kShiftGrad>(ps, a);
    artia_status st = check_hip(ctx, hipGetLastError(), "artia_pairs_shift_grad launch");
    if (st != ARTIA_OK) return st;
    return t.finish();
}

artia_status artia_pairs_adjoint(artia_pairs* ps, const double* shifts, const float* images, float scale,
                                 float* vol_grads, float* ms) {
    if (!ps) return ARTIA_ERR_INVALID_ARGUMENT;
    if (!images || !vol_grads) return pairs_fail(ps, ARTIA_ERR_INVALID_ARGUMENT, "artia_pairs_adjoint: null pointer");
    artia_ctx* ctx = ps->ctx;
    PairArgs a = base_args(ps);
    a.shifts = shifts;
    a.in = images;
    Timing t(ctx, ms);
    if (ps->slab_items) {
        const AdjSlabArgs sa{ps->slab_items, ps->slab_per_xcd, ps->vfirst, ps->vcount};
        if (ps->flat)
            hipLaunchKernelGGL(pair_adjoint_flat_kernel, dim3((unsigned)(8 * ps->slab_per_xcd)), dim3(kAdjFlatThreads),
                               ps->flat_lds, ctx->stream, a, sa, scale, vol_grads);
        else
            hipLaunchKernelGGL(pair_adjoint_slab_kernel, dim3((unsigned)(8 * ps->slab_per_xcd)), dim3(256), 0,
                               ctx->stream, a, sa, scale, vol_grads);
    } else {
        hipLaunchKernelGGL(pair_adjoint_kernel, pair_grid(ps), dim3(256), 0, ctx->stream, a, scale, vol_grads);
    }
    artia_status st = check_hip(ctx, hipGetLastError(), "artia_pairs_adjoint launch");
    if (st != ARTIA_OK) return st;
    return t.finish();
}

artia_status artia_pairs_cc_search(artia_pairs* ps, const float* models, const float* targets, int square,
                                   int max_shift, int multi_peak, int* peak, float* cc_value, float* cc_map,
                                   float* ms) {
    if (!ps) return ARTIA_ERR_INVALID_ARGUMENT;
    if (!models || !targets || !peak || !cc_value)
        return pairs_fail(ps, ARTIA_ERR_INVALID_ARGUMENT, "artia_pairs_cc_search: null pointer");
    if (max_shift < 0 || max_shift > kMaxCcShift || square < 2 * max_shift + 1)
        return fail(ps->ctx, ARTIA_ERR_INVALID_ARGUMENT,
                    "artia_pairs_cc_search: max_shift %d must be in 0..%d and square %d at least 2 max_shift + 1",
                    max_shift, kMaxCcShift, square);
    artia_ctx* ctx = ps->ctx;
    Timing t(ctx, ms);
    const size_t lds = (size_t)cc_side(max_shift) * cc_side(max_shift) * sizeof(double) + (size_t)cc_stage_bytes(max_shift);
    hipLaunchKernelGGL(pair_cc_kernel, dim3((unsigned)ps->npairs), dim3(256), lds, ctx->stream, ps->pairs, ps->npairs,
                       models, targets, square, max_shift, multi_peak ? 1 : 0, peak, cc_value,
                       cc_map);
    artia_status st = check_hip(ctx, hipGetLastError(), "artia_pairs_cc_search launch");
    if (st != ARTIA_OK) return st;
    return t.finish();
}

}  // extern "C"
