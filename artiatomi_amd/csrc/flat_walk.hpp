// The cell walk of rays without a y component (n_y == 0: every tilt about the y axis once flat_beam
// has snapped its residue), used by every exact forward kernel for such tilts.
//
// Along such a ray the y interpolation weight b is constant, so a cell of the x-z lattice is the
// bilinear interpolant of its four edges blended in y, w = lerp(v(y0), v(y0 + 1), b).  The axes are
// oriented along the ray (X = sgn x), which leaves one case: the ray enters a cell at its near edges
// and leaves it towards +X or +Z.  A step then shares two edges with the one before it and needs two
// new ones.
//
// What bounds the walk on gfx950 is VALU issue: plain 32-bit adds, multiplies and fmacs with vector
// operands issue every two cycles per SIMD, most other instructions every four, and a scalar operand
// makes an add or an fma one of the latter (measured: 964 G adds/s with vector operands, 563 G with a
// scalar one).  So the walk keeps positions relative to the current cell (r, which a step changes by
// an exact -1), advances one axis per step, and holds its direction constants in vector registers.
// Staged in LDS with y fastest, an edge is one ds_read2_b32, two per step instead of four.  Forward
// projection per tilt, against the walk with cell indices, eight corner reads and scalar constants:
// 1024x1024x256 to 1024^2 pixels 2.44 -> 1.94 ms, 256x256x64 to 256^2 0.102 -> 0.062 ms; with the boxes by
// columns and loaded ahead, and the position in two parts, 1.65 and 0.057 ms.
#pragma once

#include <climits>
#include <cmath>

#include "tube_walk.hpp"

namespace artia {

// Direction of a flat ray's samples (equal for all sub-rays of a tilt), x and z axes.
struct FlatDir {
    float inv[2];   // samples per cell, |1 / dq|; 0 on an axis without crossings
    float hd[2];    // |dq| / 2
    float c1[2];    // crossing index of the near cell's far face for r = 0: (1 - hd) * inv, or infinity
    float K;        // |dq_x| |dq_z| / 12
    int sgn[2];     // orientation: -1 where dq < 0
};

__device__ __forceinline__ FlatDir flat_dir(const float dq[3]) {
    FlatDir d;
#pragma unroll
    for (int i = 0; i < 2; i++) {
        int s;
        float inv;
        walk_dir(dq[2 * i], s, inv);
        d.sgn[i] = s < 0 ? -1 : 1;
        d.inv[i] = fabsf(inv);
        d.hd[i] = 0.5f * fabsf(dq[2 * i]);
        d.c1[i] = s != 0 ? (1.0f - d.hd[i]) * d.inv[i] : INFINITY;
    }
    d.K = fabsf(dq[0]) * fabsf(dq[2]) * (1.0f / 12.0f);
    return d;
}

// Samples k .. count - 1 of one sub-ray, cell by cell.  With R = (start - near edge) - hd in oriented
// coordinates the middle of samples k .. k + m - 1 lies (2 k + m) hd + R into the cell, and sample index
// kb = (1 - hd - R) inv crosses the cell's far face.  A step lowers R by 1 and takes the axis that is crossed
// first (z on a tie; the cell in between holds no samples).
//
// R is kept as r + lo, r a multiple of 2^-8 (exact down to -65536, so that steps do not round) and lo the rest,
// which stays.  R in one float rounds every time it passes a power of two, alike for all rays that enter through
// one face: at 256 layers a shift of 1e-5 of a cell that no averaging takes out.
struct FlatWalker {
    float r[2], lo[2], c1[2], kb[2];
    float k, count;

    __device__ __forceinline__ void crossings(const FlatDir& d) {
#pragma unroll
        for (int i = 0; i < 2; i++) kb[i] = __builtin_fmaf(-r[i], d.inv[i], c1[i]);
    }
    __device__ __forceinline__ void init(const FlatDir& d, const float q0[3], int n) {
#pragma unroll
        for (int i = 0; i < 2; i++) {
            const float q = q0[2 * i], fl = floorf(q), at = d.sgn[i] > 0 ? q - fl : (fl + 1.0f) - q;   // exact
            r[i] = rintf((at - d.hd[i]) * 256.0f) * 0.00390625f;
            lo[i] = (at - r[i]) - d.hd[i];
            c1[i] = __builtin_fmaf(-lo[i], d.inv[i], d.c1[i]);
        }
        crossings(d);
        k = 0.0f;
        count = (float)n;
    }
    __device__ __forceinline__ bool active() const { return k < count; }
    // near lattice index of the current cell on oriented axis i (r is start - near - hd up to lo, below 2^-9)
    __device__ __forceinline__ int near(const FlatDir& d, const float q0[3], int i) const {
        const float X = d.sgn[i] > 0 ? q0[2 * i] : -q0[2 * i];
        return (int)rintf((X - d.hd[i]) - r[i]);
    }
    // the current cell's samples: their number, and the coordinates of their middle from the near edges
    __device__ __forceinline__ float samples(const FlatDir& d, float kn, float& a, float& c) {
        const float kend = __builtin_amdgcn_fmed3f(ceilf(kn), k, count);
        const float m = kend - k, s = k + kend;
        a = __builtin_fmaf(s, d.hd[0], r[0]) + lo[0];
        c = __builtin_fmaf(s, d.hd[1], r[1]) + lo[1];
        k = kend;
        return m;
    }
    __device__ __forceinline__ void advance(const FlatDir& d, bool ax) {
        const float dx = ax ? -1.0f : 0.0f;
        r[0] += dx;
        r[1] += -1.0f - dx;
        crossings(d);
    }
};

// Sum of a cell's m samples from its y-blended edges A (near x, near z), B (far x), C (far z), D:
// m g(middle) + m (m^2 - 1) / 12 (D - C - B + A) |dq_x dq_z|, the sum rounded once to float (the ray adds
// the cells in double).  m = 0 gives +-0.
__host__ __device__ __forceinline__ float flat_cell_sum(float A, float B, float C, float D, float a, float c, float m,
                                                        float K) {
    const float d0 = B - A, d1 = D - C;
    const float e0 = __builtin_fmaf(a, d0, A), e1 = __builtin_fmaf(a, d1, C);
    const float g = __builtin_fmaf(c, e1 - e0, e0);
    return __builtin_fmaf(m, g, ((d1 - d0) * K) * (m * __builtin_fmaf(m, m, -1.0f)));
}

// Gradient of the cell's interpolant summed over its samples, in oriented texel coordinates, added to
// G: the x and z derivatives of the bilinear edges, and the y differences yA .. yD interpolated like
// the edges.
__device__ __forceinline__ void flat_grad_sum(float A, float B, float C, float D, float yA, float yB, float yC,
                                              float yD, float a, float c, float m, float K, double G[3]) {
    const float ga = lerpf(B - A, D - C, c), gc = lerpf(C - A, D - B, a);
    G[0] += (double)(m * ga);
    G[1] += (double)flat_cell_sum(yA, yB, yC, yD, a, c, m, K);
    G[2] += (double)(m * gc);
}

// One y-blended edge, and the y difference it is blended with.
__device__ __forceinline__ float flat_edge(float v0, float v1, float b, float& dy) {
    dy = v1 - v0;
    return __builtin_fmaf(b, dy, v0);
}

// The walk with its edges read from the volume (clamp addressing): all steps while go(), the path of
// unstaged volumes and of lanes whose cells leave a staged box.  f(A, B, C, D, yA, yB, yC, yD, a, c, m).
// A step keeps the two edges it shares with the one before and reads the other two.
// kBig: 64-bit addresses; otherwise buffer loads at 32-bit offsets (below 2^30 voxels, z * ny + y and x
// below 2^24).
template <bool kBig, typename T, class Go, class F>
__device__ __forceinline__ void flat_walk_direct(const VolG& v, const T* __restrict__ vol, const FlatDir& d,
                                                 const float q0[3], FlatWalker& w, Go&& go, F&& f) {
    if (!(w.active() && go())) return;
    const float yf = floorf(q0[1]), b = q0[1] - yf;
    const int y0 = clampi((int)yf, 0, v.ny - 1), y1 = clampi((int)yf + 1, 0, v.ny - 1);
    auto edge = [&](int xo, int zo, float& dy) {   // oriented lattice indices
        const int x = clampi(d.sgn[0] * xo, 0, v.nx - 1), z = clampi(d.sgn[1] * zo, 0, v.nz - 1);
        if (kBig) {
            const size_t o = ((size_t)z * (size_t)v.ny + (size_t)y0) * (size_t)v.nx + (size_t)x;
            return flat_edge(vox(vol, o), vox(vol, o + (size_t)(y1 - y0) * (size_t)v.nx), b, dy);
        }
        const __amdgpu_buffer_rsrc_t rs = volume_rsrc(vol, v);
        const uint32_t e = (uint32_t)sizeof(T);
        const uint32_t o = __umul24(__umul24((uint32_t)z, (uint32_t)v.ny) + (uint32_t)y0, (uint32_t)v.nx) + (uint32_t)x;
        return flat_edge(buffer_vox(rs, o * e, vol), buffer_vox(rs, (o + (uint32_t)(y1 - y0) * (uint32_t)v.nx) * e, vol),
                         b, dy);
    };
    int xf = w.near(d, q0, 0) + 1, zf = w.near(d, q0, 1) + 1;   // the current cell's far indices
    float yA, yB, yC, yD;
    float A = edge(xf - 1, zf - 1, yA), B = edge(xf, zf - 1, yB), C = edge(xf - 1, zf, yC), D = edge(xf, zf, yD);
    const int most = 4 * (int)w.count + 64;   // every step takes samples or advances an axis
    for (int guard = 1;; guard++) {
        const bool ax = w.kb[0] < w.kb[1];
        float a, c;
        const float m = w.samples(d, ax ? w.kb[0] : w.kb[1], a, c);
        if (m > 0.0f) f(A, B, C, D, yA, yB, yC, yD, a, c, m);   // (0 times an infinite voxel would be NaN)
        w.advance(d, ax);
        if (!(guard < most && w.active() && go())) break;
        xf += ax ? 1 : 0;
        zf += ax ? 0 : 1;
        float yN, yE = yD;
        const float N = edge(ax ? xf : xf - 1, ax ? zf - 1 : zf, yN), E = D;
        D = edge(xf, zf, yD);
        A = ax ? B : C;
        B = ax ? N : E;
        C = ax ? E : N;
        yA = ax ? yB : yC;
        yB = ax ? yN : yE;
        yC = ax ? yE : yN;
    }
}

// A box of the padded volume in LDS, y fastest: voxel (x, y, z) at ((z - Z0) CX + (x - X0)) SY + (y - Y0).
struct FlatBox {
    int X0, Y0, Z0, X1, Y1, Z1;   // inclusive
    int CX, CY, CZ, SY;
    bool staged;
};

// The box of cell layers [zs, ze] for the rays of a tile (see tube_slabs); x is padded by two
// clamp-addressed columns, so that a lane at the volume's faces keeps a column of margin.  SY is odd
// where that fits (lanes of neighbouring columns in different banks).
__device__ __forceinline__ FlatBox flat_box(const VolG& v, const TubePlan& tp, const TubeBox& tb, int zs, int ze,
                                            int cap = kChunkFloats) {
    FlatBox q;
    const float z0 = (float)zs, z1 = (float)(ze + 1);
    q.X0 = wave_uniform(max((int)floorf(tb.axl + fminf(tp.bx * z0, tp.bx * z1)) - 1, -2));
    q.X1 = min((int)floorf(tb.axh + fmaxf(tp.bx * z0, tp.bx * z1)) + 2, v.nx + 1);
    q.Y0 = wave_uniform(max((int)floorf(tb.ayl) - 1, -1));
    q.Y1 = min((int)floorf(tb.ayh) + 2, v.ny);
    q.Z0 = zs;
    q.Z1 = ze + 1;
    q.CX = wave_uniform(q.X1 - q.X0 + 1);
    q.CY = wave_uniform(q.Y1 - q.Y0 + 1);
    q.CZ = q.Z1 - q.Z0 + 1;
    const bool some = q.CX > 1 && q.CX <= 256 && q.CY > 1 && q.CZ > 1;
    q.SY = some && q.CX * (q.CY | 1) * q.CZ <= cap ? (q.CY | 1) : q.CY;
    q.staged = some && q.CX * q.SY * q.CZ <= cap;
    return q;
}

// A box is staged by columns along z: a thread keeps (x, y) columns t, t + 256, .. (one for most tilts) and
// loads their layers, whose base addresses are uniform: a lane offset that stays fixed and one LDS
// address step per voxel, with the clamps once per column (x, y) or in scalar registers (z).
template <typename T>
struct FlatColumn {
    uint32_t off;   // byte offset of the column within a layer
    int o;          // its first entry in the box
    __device__ __forceinline__ FlatColumn(const VolG& v, const FlatBox& q, int t) {
        const int y = small_div(t, q.CX), x = t - y * q.CX;
        // (nx ny < 2^30: tube_plan)
        off = ((uint32_t)clampi(q.Y0 + y, 0, v.ny - 1) * (uint32_t)v.nx + (uint32_t)clampi(q.X0 + x, 0, v.nx - 1)) *
              (uint32_t)sizeof(T);
        o = x * q.SY + y;
    }
    __device__ __forceinline__ T layer(const VolG& v, const T* __restrict__ vol, int z) const {
        const char* p = reinterpret_cast<const char*>(vol + (size_t)clampi(z, 0, v.nz - 1) * ((size_t)v.nx * (size_t)v.ny));
        return *reinterpret_cast<const T*>(p + off);
    }
};

template <typename T>
__device__ __forceinline__ void stage_flat_box(const VolG& v, const T* __restrict__ vol, float* __restrict__ chunk,
                                               const FlatBox& q, int first = 0) {
    const int cols = q.CX * q.CY, plane = q.CX * q.SY;
    for (int t = first + (int)threadIdx.x; t < cols; t += 256) {
        const FlatColumn<T> c(v, q, t);
        float* __restrict__ o = chunk + c.o;
        int z = 0;
        for (; z + 4 < q.CZ; z += 5) {
            T val[5];
#pragma unroll
            for (int k = 0; k < 5; k++) val[k] = c.layer(v, vol, q.Z0 + z + k);
#pragma unroll
            for (int k = 0; k < 5; k++) o[k * plane] = (float)val[k];
            o += 5 * plane;
        }
        for (; z < q.CZ; z++, o += plane) *o = (float)c.layer(v, vol, q.Z0 + z);
    }
}

// The layers of the thread's first column, loaded ahead: while the slab before is walked.
template <typename T>
struct FlatAhead {
    T val[kSlabCells + 2];
    __device__ __forceinline__ void load(const VolG& v, const T* __restrict__ vol, const FlatBox& q) {
        if (!q.staged || (int)threadIdx.x >= q.CX * q.CY) return;
        const FlatColumn<T> c(v, q, (int)threadIdx.x);
#pragma unroll
        for (int k = 0; k < kSlabCells + 2; k++)
            if (k < q.CZ) val[k] = c.layer(v, vol, q.Z0 + k);
    }
    // the box: the first columns from the registers, the others (steep tilts) from the volume
    __device__ __forceinline__ void store(const VolG& v, const T* __restrict__ vol, float* __restrict__ chunk,
                                          const FlatBox& q) const {
        if (!q.staged) return;
        if ((int)threadIdx.x < q.CX * q.CY) {
            const FlatColumn<T> c(v, q, (int)threadIdx.x);
#pragma unroll
            for (int k = 0; k < kSlabCells + 2; k++)
                if (k < q.CZ) chunk[c.o + k * q.CX * q.SY] = (float)val[k];
        }
        stage_flat_box(v, vol, chunk, q, 256);
    }
};

// Whether the cells the lane crosses in layers [zs, ze] lie in the box with a column of margin: from its
// current cell (xn, zn) to its last sample or the slab's exit, whose layer the box holds.
__device__ __forceinline__ bool flat_lane_in_box(const VolG& v, const FlatBox& q, const FlatDir& d, const float q0[3],
                                                 const float dq[3], const FlatWalker& w, int zs, int ze, int xn,
                                                 int zn) {
    if (!q.staged) return false;
    const float zx = d.sgn[1] > 0 ? (float)(ze + 1) : (float)zs;
    const float ke = fminf(fmaxf(fabsf(zx - q0[2]) * d.inv[1], w.k), w.count - 1.0f);
    const int xb = (int)floorf(__builtin_fmaf(ke, dq[0], q0[0])), yc = (int)floorf(q0[1]);
    const int xa = d.sgn[0] > 0 ? xn : -(xn + 1), za = d.sgn[1] > 0 ? zn : -(zn + 1);
    return min(xa, xb) - 1 >= q.X0 && max(xa, xb) + 2 <= q.X1 && yc >= q.Y0 && yc + 1 <= q.Y1 &&
           (d.sgn[1] > 0 ? za >= q.Z0 : za + 1 <= q.Z1);
}

// The lane's samples in cell layers [zs, ze] of a slab, from the staged box where the cells they cross
// provably lie in it with a column of margin, otherwise from the volume.
template <bool kGrad, typename T, class F>
__device__ __forceinline__ void flat_walk_slab(const VolG& v, const T* __restrict__ vol,
                                               const float* __restrict__ chunk, const FlatBox& q, const FlatDir& d,
                                               const float q0[3], const float dq[3], FlatWalker& w, int zs, int ze,
                                               F&& f) {
    const int zlast = d.sgn[1] > 0 ? ze : -(zs + 1);   // near index of the slab's last layer, oriented
    const int xn = w.near(d, q0, 0), zn = w.near(d, q0, 1);
    if (zn > zlast) return;   // resumes in a later slab
    const int yc = (int)floorf(q0[1]);
    const bool fast = flat_lane_in_box(v, q, d, q0, dq, w, zs, ze, xn, zn);
    if (!fast) {
        flat_walk_direct<true>(v, vol, d, q0, w, [&]() { return w.near(d, q0, 1) <= zlast; }, f);
        return;
    }
    const float b = q0[1] - floorf(q0[1]);
    const float rstop = (w.r[1] - (float)(zlast - zn)) - 0.5f;   // r_z below it: past the last layer
    // byte offsets: the far-far edge of the current cell, and its steps along the oriented axes
    int sx = 4 * d.sgn[0] * q.SY, sz = 4 * d.sgn[1] * q.CX * q.SY;
    __asm__("" : "+v"(sx), "+v"(sz));   // (selects of scalar operands would copy them every step)
    int o = 4 * (((d.sgn[1] * (zn + 1) - q.Z0) * q.CX + (d.sgn[0] * (xn + 1) - q.X0)) * q.SY + (yc - q.Y0));
    const char* __restrict__ base = reinterpret_cast<const char*>(chunk);
    auto edge = [&](int at, float& dy) {
        const float* p = reinterpret_cast<const float*>(base + at);
        return flat_edge(p[0], p[1], b, dy);
    };
    // entered as by a step along x: the near edges are the far ones of the cell before
    float yA, yB, yC, yD, A, B = edge(o - sx - sz, yB), C, D = edge(o - sx, yD);
    bool ax = true;
    for (;;) {
        float yN, yE = yD;
        const float N = edge(ax ? o - sz : o - sx, yN), E = D;
        D = edge(o, yD);
        A = ax ? B : C;
        B = ax ? N : E;
        C = ax ? E : N;
        if (kGrad) {
            yA = ax ? yB : yC;
            yB = ax ? yN : yE;
            yC = ax ? yE : yN;
        }
        ax = w.kb[0] < w.kb[1];
        float a, c;
        const float m = w.samples(d, ax ? w.kb[0] : w.kb[1], a, c);
        f(A, B, C, D, yA, yB, yC, yD, a, c, m);
        w.advance(d, ax);
        if (!(w.r[1] > rstop && w.k < w.count)) break;
        o += ax ? sx : sz;
    }
}

// The cell layers the block's lanes cross: za .. zb per lane (za > zb: none), widened by one.
__device__ __forceinline__ void flat_layers(const VolG& v, int* zr, int za, int zb, int& zlo, int& zhi) {
    __syncthreads();   // a previous walk's readers are done with zr and the chunk
    if (threadIdx.x == 0) {
        zr[0] = INT_MAX;
        zr[1] = INT_MIN;
    }
    __syncthreads();
    if (za <= zb) {
        atomicMin(&zr[0], za - 1);
        atomicMax(&zr[1], zb + 1);
    }
    __syncthreads();
    zlo = max(zr[0], -1);
    zhi = min(zr[1], v.nz - 1);
}

// Walks every lane's samples q0 + k dq (k < count, dq[1] == 0) cell by cell, slab by slab through LDS.
// Called by all 256 threads of the block; chunk holds kChunkFloats floats and zr two ints of shared
// memory.  The steps and values are flat_walk_direct's, so sums are bit-identical to it.  kGrad: f uses
// the y differences.  kAhead: the next slab's voxels are loaded into
// registers during the walk (the march: 1.80 -> 1.63 ms per 1024x1024x256 tilt; the segments, the pair
// projection and the pairs' shift gradient lose by it).
template <bool kGrad, bool kAhead, typename T, class F>
__device__ __forceinline__ void flat_tube_walk(const VolG& v, const T* __restrict__ vol, float* __restrict__ chunk,
                                               int* zr, const TubePlan& tp, const TubeBox& tb, const float dq[3],
                                               const float q0[3], int count, F&& f) {
    const FlatDir d = flat_dir(dq);
    int za = 1, zb = 0, zlo, zhi;
    if (count > 0) {
        const int z0 = (int)floorf(q0[2]), z1 = (int)floorf(__builtin_fmaf((float)(count - 1), dq[2], q0[2]));
        za = min(z0, z1);
        zb = max(z0, z1);
    }
    flat_layers(v, zr, za, zb, zlo, zhi);
    FlatWalker w;
    w.init(d, q0, count);
    const int nslab = zlo <= zhi ? (zhi - zlo) / kSlabCells + 1 : 0;
    FlatAhead<T> ahead;
    FlatBox next{};
    int zs, ze;
    if (kAhead && nslab > 0) {
        slab_layers(v, tp.zdir, zlo, zhi, 0, zs, ze);
        next = flat_box(v, tp, tb, zs, ze);
        ahead.load(v, vol, next);
    }
    for (int j = 0; j < nslab; j++) {
        slab_layers(v, tp.zdir, zlo, zhi, j, zs, ze);
        const FlatBox q = kAhead ? next : flat_box(v, tp, tb, zs, ze);
        __syncthreads();   // the previous slab's reads are done
        if (kAhead) ahead.store(v, vol, chunk, q);
        else if (q.staged) stage_flat_box(v, vol, chunk, q);
        __syncthreads();
        if (kAhead && j + 1 < nslab) {
            int ns, ne;
            slab_layers(v, tp.zdir, zlo, zhi, j + 1, ns, ne);
            next = flat_box(v, tp, tb, ns, ne);
            ahead.load(v, vol, next);
        }
        if (w.active()) flat_walk_slab<kGrad>(v, vol, chunk, q, d, q0, dq, w, zs, ze, f);
    }
    // cells beyond the slabs
    flat_walk_direct<true>(v, vol, d, q0, w, []() { return true; }, f);
}

// The walk over a run of segments per lane: consecutive sample sets along the lane's ray, each with its
// own start seg.q0 and seg.count (a slicer sample lattice per CTF slab).  seg.next() finishes the
// lane's current segment, if any, and loads the next, returning false when none is left.  One pass over
// the slabs of cell layers serves all segments; each is walked as flat_tube_walk walks it alone.
template <typename T, class Seg, class F>
__device__ __forceinline__ void flat_tube_segments(const VolG& v, const T* __restrict__ vol, float* __restrict__ chunk,
                                                   int* zr, const TubePlan& tp, const TubeBox& tb, const float dq[3],
                                                   int za, int zb, Seg& seg, F&& f) {
    const FlatDir d = flat_dir(dq);
    int zlo, zhi;
    flat_layers(v, zr, za, zb, zlo, zhi);
    FlatWalker w;
    w.init(d, seg.q0, 0);   // no segment yet: the first pass below loads one
    bool more = true;
    const int nslab = zlo <= zhi ? (zhi - zlo) / kSlabCells + 1 : 0;
    // slabs of cell layers, then (j == nslab) the cells beyond them from the volume
    for (int j = 0; j <= nslab; j++) {
        const bool tail = j == nslab;
        int zs, ze;
        slab_layers(v, tp.zdir, zlo, zhi, j, zs, ze);
        FlatBox q{};
        if (!tail) {
            q = flat_box(v, tp, tb, zs, ze);
            __syncthreads();
            if (q.staged) stage_flat_box(v, vol, chunk, q);
            __syncthreads();
        }
        const int zlast = d.sgn[1] > 0 ? ze : -(zs + 1);
        for (;;) {
            if (!w.active()) {
                if (!more) break;
                more = seg.next();
                w.init(d, seg.q0, more ? seg.count : 0);
                continue;
            }
            if (tail) {
                flat_walk_direct<true>(v, vol, d, seg.q0, w, []() { return true; }, f);
                if (w.active()) break;   // (the walk's step bound)
                continue;
            }
            if (w.near(d, seg.q0, 1) > zlast) break;   // resumes in a later slab
            flat_walk_slab<false>(v, vol, chunk, q, d, seg.q0, dq, w, zs, ze, f);
        }
    }
}

// ---------------------------------------------------------------- the transpose
//
// Weights of a cell's four edges for a ray of residual rd, in double: flat_cell_sum is
// m ((1 - a)(1 - c) A + a (1 - c) B + (1 - a) c C + a c D) + s (A - B - C + D) with s = m (m^2 - 1) K,
// and an edge splits over its two voxels as 1 - b and b.  Consecutive cells share two edges, so a lane
// keeps the four edge sums in registers and a step hands two of them on (put), four voxel additions
// instead of eight.
struct FlatEdgeSums {
    double A, B, C, D;
    __device__ __forceinline__ void clear() { A = B = C = D = 0.0; }
    __device__ __forceinline__ void add(double rd, float a, float c, float m, float K) {
        const double md = rd * (double)m, ta = md * (double)a, tc = md * (double)c;
        const double wD = __builtin_fma(ta, (double)c, md * (double)(__builtin_fmaf(m, m, -1.0f) * K));
        const double wC = tc - wD;
        D += wD;
        C += wC;
        B += ta - wD;
        A += (md - ta) - wC;
    }
    // the edges a step along x (ax) or z leaves behind: A, and C or B
    template <class P>
    __device__ __forceinline__ void step(bool ax, P&& put) {
        put(0, 0, A);
        put(ax ? 0 : 1, ax ? 1 : 0, ax ? C : B);
        A = ax ? B : C;
        B = ax ? 0.0 : D;
        C = ax ? D : 0.0;
        D = 0.0;
    }
    template <class P>
    __device__ __forceinline__ void flush(P&& put) {
        put(0, 0, A);
        put(1, 0, B);
        put(0, 1, C);
        put(1, 1, D);
    }
};

// The transposed walk straight into the volume while go(): grad += the weights, clamp-addressed.
template <class Go>
__device__ __forceinline__ void flat_scatter_direct(const VolG& v, float* __restrict__ grad, const FlatDir& d,
                                                    const float q0[3], double rd, FlatWalker& w, Go&& go) {
    const float yf = floorf(q0[1]);
    const double b = (double)(q0[1] - yf);
    const int y0 = clampi((int)yf, 0, v.ny - 1), y1 = clampi((int)yf + 1, 0, v.ny - 1);
    const int most = 4 * (int)w.count + 64;
    FlatEdgeSums e;
    e.clear();
    for (int guard = 0; guard < most && w.active() && go(); guard++) {
        const int xn = w.near(d, q0, 0), zn = w.near(d, q0, 1);
        const bool ax = w.kb[0] < w.kb[1];
        float a, c;
        const float m = w.samples(d, ax ? w.kb[0] : w.kb[1], a, c);
        e.add(rd, a, c, m, d.K);
        w.advance(d, ax);
        auto put = [&](int dx, int dz, double s) {
            if (s == 0.0) return;
            const size_t x = (size_t)clampi(d.sgn[0] * (xn + dx), 0, v.nx - 1);
            const size_t z = (size_t)clampi(d.sgn[1] * (zn + dz), 0, v.nz - 1);
            const double s1 = s * b;
            unsafeAtomicAdd(grad + ((z * (size_t)v.ny + (size_t)y0) * (size_t)v.nx + x), (float)(s - s1));
            unsafeAtomicAdd(grad + ((z * (size_t)v.ny + (size_t)y1) * (size_t)v.nx + x), (float)s1);
        };
        if (w.active() && guard + 1 < most && go()) {
            e.step(ax, put);
        } else {
            e.flush(put);
            e.clear();
        }
    }
}

// The lane's samples in cell layers [zs, ze] of a slab, into the slab's box (zeroed before, added to
// the volume after) where its cells provably lie in it, otherwise straight into the volume.
__device__ __forceinline__ void flat_scatter_slab(const VolG& v, float* __restrict__ grad, double* __restrict__ chunk,
                                                  const FlatBox& q, const FlatDir& d, const float q0[3],
                                                  const float dq[3], double rd, FlatWalker& w, int zs, int ze) {
    const int zlast = d.sgn[1] > 0 ? ze : -(zs + 1);
    const int xn = w.near(d, q0, 0), zn = w.near(d, q0, 1);
    if (zn > zlast) return;
    if (!flat_lane_in_box(v, q, d, q0, dq, w, zs, ze, xn, zn)) {
        flat_scatter_direct(v, grad, d, q0, rd, w, [&]() { return w.near(d, q0, 1) <= zlast; });
        return;
    }
    const float yf = floorf(q0[1]);
    const double b = (double)(q0[1] - yf);
    const float rstop = (w.r[1] - (float)(zlast - zn)) - 0.5f;
    const int sx = d.sgn[0] * q.SY, sz = d.sgn[1] * q.CX * q.SY;
    int o = ((d.sgn[1] * zn - q.Z0) * q.CX + (d.sgn[0] * xn - q.X0)) * q.SY + ((int)yf - q.Y0);   // near-near edge
    FlatEdgeSums e;
    e.clear();
    for (;;) {
        const bool ax = w.kb[0] < w.kb[1];
        float a, c;
        const float m = w.samples(d, ax ? w.kb[0] : w.kb[1], a, c);
        e.add(rd, a, c, m, d.K);
        w.advance(d, ax);
        auto put = [&](int dx, int dz, double s) {
            const int at = o + (dx ? sx : 0) + (dz ? sz : 0);
            const double s1 = s * b;
            unsafeAtomicAdd(chunk + at, s - s1);
            unsafeAtomicAdd(chunk + at + 1, s1);
        };
        if (!(w.r[1] > rstop && w.k < w.count)) {
            e.flush(put);
            break;
        }
        e.step(ax, put);
        o += ax ? sx : sz;
    }
}

// grad += rd times the transpose of flat_tube_walk's sum over the lane's samples.
__device__ __forceinline__ void flat_tube_scatter(const VolG& v, float* __restrict__ grad, double* __restrict__ chunk,
                                                  int* zr, const TubePlan& tp, const TubeBox& tb, const float dq[3],
                                                  const float q0[3], int count, double rd) {
    const FlatDir d = flat_dir(dq);
    int za = 1, zb = 0, zlo, zhi;
    if (count > 0) {
        const int z0 = (int)floorf(q0[2]), z1 = (int)floorf(__builtin_fmaf((float)(count - 1), dq[2], q0[2]));
        za = min(z0, z1);
        zb = max(z0, z1);
    }
    flat_layers(v, zr, za, zb, zlo, zhi);
    FlatWalker w;
    w.init(d, q0, count);
    const int nslab = zlo <= zhi ? (zhi - zlo) / kSlabCells + 1 : 0;
    for (int j = 0; j < nslab; j++) {
        int zs, ze;
        slab_layers(v, tp.zdir, zlo, zhi, j, zs, ze);
        const FlatBox q = flat_box(v, tp, tb, zs, ze, tp.box);
        const int n = q.CX * q.SY * q.CZ;
        __syncthreads();   // the previous slab's box is in the volume
        if (q.staged)
            for (int e = (int)threadIdx.x; e < n; e += 256) chunk[e] = 0.0;
        __syncthreads();
        if (w.active()) flat_scatter_slab(v, grad, chunk, q, d, q0, dq, rd, w, zs, ze);
        if (q.staged) {
            __syncthreads();   // the box is complete
            // by rows along x (coalesced atomics), thread t on column t mod CX
            const int P = small_div(256, q.CX), t = (int)threadIdx.x, r0 = small_div(t, q.CX), x = t - r0 * q.CX;
            const int rows = q.CY * q.CZ;
            if (r0 < P) {
                const size_t gx = (size_t)clampi(q.X0 + x, 0, v.nx - 1);
                for (int r = r0; r < rows; r += P) {
                    const int zz = small_div(r, q.CY), yy = r - zz * q.CY;
                    const float add = (float)chunk[(zz * q.CX + x) * q.SY + yy];
                    const size_t row = (size_t)clampi(q.Z0 + zz, 0, v.nz - 1) * (size_t)v.ny +
                                       (size_t)clampi(q.Y0 + yy, 0, v.ny - 1);
                    if (add != 0.0f) unsafeAtomicAdd(grad + row * (size_t)v.nx + gx, add);
                }
            }
        }
    }
    // cells beyond the slabs
    flat_scatter_direct(v, grad, d, q0, rd, w, []() { return true; });
}

}  // namespace artia
