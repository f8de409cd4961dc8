// Fixed-window form of the exact backprojection (BackProjectionSquareOS.cu:263-782) for tilts
// whose beam has no y component (every tilt about the y axis: n_y is zero or a float residue of
// the rotation), POINT sampling, no magnification anisotropy.
//
// A voxel's sub-rays are the OS lattice points (i + 0.5) / OS of the detector inside the voxel's
// projected box.  The box holds at most kNI x kNJ lattice points for every voxel of a tilt, so the
// window starting at the box's first lattice point is walked fully unrolled, without per-voxel
// bounds; lattice points of the window outside the voxel's projection get a chord <= 0 and add
// nothing, as in the per-box loop.  With the sub-ray offset (a, b) from the projection of the
// voxel's min corner (detector pixels along u and v), the chord through the voxel is
//     chord = max(0, min(m, P, SP - P, Y, SY - Y))
// with P and Y affine in (a, b).  Only the ratio of two chord-weighted sums is used, so chords are taken in
// units of m, as the product of clamp01(min(P, SP - P) / m) = clamp01(SP/2 - |P - SP/2|) in those units and
// the y slab's inside test, itself the clamp of a huge coordinate:
//   - n_x != 0: the x and z slabs' entries e_x, e_z are affine in (a, b) and the chord
//     min(e_x + S_x, e_z + S_z) - max(e_x, e_z) equals min(min(S_x, S_z), S_x - d, S_z + d) for
//     d = e_z - e_x; P = S_x - d, SP = S_x + S_z, m = min(S_x, S_z);
//   - n_x == 0 (tilt 0): the ray runs inside the x slab when 0 < w_x < s_x (w_x the sub-ray's x
//     offset a u_x + b v_x); P = B w_x, SP = B s_x, m = S_z, with B = 2^100;
//   - y (parallel): Y = B w_y, SY = B s_y; min(Y, SY - Y) > 0 exactly when 0 < w_y < s_y, and
//     B is large enough that a sub-ray inside the slab by more than 1e-30 voxels is not clipped.
// For a float-residue n_y (~1e-9) the sub-ray's y offset drifts by less than 1e-8 voxels across a
// voxel, so the parallel form differs from the slab form only for sub-rays within rounding of a y
// face, where any evaluation is decided by rounding.
#pragma once

#include <cmath>
#include <type_traits>

#include "bp_common.hpp"
#include "device_common.hpp"

namespace artia {

constexpr float kWinBig = 1.2676506002282294e30f;   // 2^100
// A y coordinate beyond every slab (|Y| - SY/2 stays above 1e35 for |Y| moved by any window step):
// a row placed there has every chord 0.
constexpr float kWinFar = 1e36f;

// Per-tilt constants of the window form, prepared on the host in double.
struct BPWin {
    float PU, PV, PC;        // Pc = (P - SP/2) / m = a PU + b PV + PC
    float YU, YV, YC;        // Yc = Y - SY/2 = a YU + b YV + YC
    float PUd, PVd, YUd, YVd;   // the same per lattice step (times 1/OS)
    float SPh, SYh;          // SP/2 / m, SY/2
    float uMin, vMin;        // the voxel's projected box starts (with guard) relative to its corner
    double pu0, pui, puj, puk, pv0, pvi, pvj, pvk;   // corner projection (detector pixels)
    double G[2][3], lo[2], hi[2], tlo[2], thi[2];     // quad and block footprints (see BPExact)
    double gn[3], g0;                                 // dist gate: |gn . q + g0|
    int ni, nj;              // window size in lattice points
    // The reference sums only the sub-rays inside a quad's footprint, the box spanned by two
    // projected corners of its macro-cell (BackProjectionSquareOS.cu:365-509, x bounds swapped
    // when n_x <= 0), which need not cover a voxel's projected box.  covers != 0: it covers the
    // projected boxes of all four voxels of every quad of the volume, so a quad whose footprint
    // the image edges do not clamp may walk its windows without the per-point footprint test.
    int covers;
    // masked != 0: the voxel boxes stick out of the quad footprints by less than 1 - 1/os pixels,
    // so every window of a block lies in its footprint tile with a one-pixel margin, and a block
    // away from the image edges can apply the footprint test as a per-point chord cap (0 outside).
    int masked;
};

// Whether the window form applies to a tilt and its constants, for oversampling os and a window of
// at most maxN lattice points per axis.  Requires the affine footprint of prepare_exact (passed in).
inline bool prepare_window(const VolG& v, const TiltG& g, const BPExact& e, int os, int maxN, BPWin& w) {
    if (!e.affine || !e.identityAniso || os <= 0) return false;
    const double nf[3] = {g.n[0], g.n[1], g.n[2]};
    const double nl = std::sqrt(nf[0] * nf[0] + nf[1] * nf[1] + nf[2] * nf[2]);
    const double n[3] = {nf[0] / nl, nf[1] / nl, nf[2] / nl};
    if (!(std::fabs(n[1]) <= 1e-6) || !(std::fabs(n[2]) > 1e-3)) return false;
    const double u[3] = {g.u[0], g.u[1], g.u[2]}, wv[3] = {g.v[0], g.v[1], g.v[2]};
    const double vs[3] = {v.vs[0], v.vs[1], v.vs[2]};
    const double B = (double)kWinBig;
    auto slab = [&](int c, double& U, double& V, double& Smin, double& Sabs) {
        U = -u[c] / n[c];
        V = -wv[c] / n[c];
        const double S = vs[c] / n[c];
        Smin = std::fmin(0.0, S);
        Sabs = std::fabs(S);
    };
    double Uz, Vz, Sminz, Sabsz;
    slab(2, Uz, Vz, Sminz, Sabsz);
    double PU, PV, PC, SP, m;
    if (std::fabs(n[0]) > 1e-6) {
        double Ux, Vx, Sminx, Sabsx;
        slab(0, Ux, Vx, Sminx, Sabsx);
        // P = S_x - d, d = e_z - e_x
        PU = -(Uz - Ux);
        PV = -(Vz - Vx);
        PC = (Sabsx - (Sminz - Sminx)) - 0.5 * (Sabsx + Sabsz);
        SP = 0.5 * (Sabsx + Sabsz);
        m = std::fmin(Sabsx, Sabsz);
    } else {
        PU = B * u[0];
        PV = B * wv[0];
        PC = -0.5 * B * vs[0];
        SP = 0.5 * B * vs[0];
        m = 1.0;   // (the clamp gives 0 or 1 whatever the unit)
    }
    if (!(m > 0.0)) return false;
    w.PU = (float)(PU / m);
    w.PV = (float)(PV / m);
    w.PC = (float)(PC / m);
    w.SPh = (float)(SP / m);
    w.YU = (float)(B * u[1]);
    w.YV = (float)(B * wv[1]);
    w.YC = (float)(-0.5 * B * vs[1]);
    w.SYh = (float)(0.5 * B * vs[1]);
    w.PUd = (float)((double)w.PU / os);
    w.PVd = (float)((double)w.PV / os);
    w.YUd = (float)((double)w.YU / os);
    w.YVd = (float)((double)w.YV / os);
    w.uMin = e.uMin;
    w.vMin = e.vMin;
    w.pu0 = e.pu0;
    w.pui = e.pui;
    w.puj = e.puj;
    w.puk = e.puk;
    w.pv0 = e.pv0;
    w.pvi = e.pvi;
    w.pvj = e.pvj;
    w.pvk = e.pvk;
    for (int r = 0; r < 2; r++) {
        for (int k = 0; k < 3; k++) w.G[r][k] = e.G[r][k];
        w.lo[r] = e.lo[r];
        w.hi[r] = e.hi[r];
        w.tlo[r] = e.tlo[r];
        w.thi[r] = e.thi[r];
    }
    for (int k = 0; k < 3; k++) w.gn[k] = e.gn[k];
    w.g0 = e.g0;
    // lattice points in a box of length L: at most floor(L * os) + 1 (the box's float rounding is
    // far inside the 1e-4 guard already in uMin/uMax)
    w.ni = (int)std::floor(((double)e.uMax - (double)e.uMin) * os) + 1;
    w.nj = (int)std::floor(((double)e.vMax - (double)e.vMin) * os) + 1;
    // Footprint [G_r . q + lo_r, G_r . q + hi_r] against the union of the quad's voxel boxes
    // [p_r(q) + min(0, 3 p_ri) + min_r, p_r(q) + max(0, 3 p_ri) + max_r] (guarded, so conservative):
    // both ends are affine in the quad origin q, so the volume's corner quads decide.  A lattice
    // point inside a box then lies in [floor(lower) * os, ceil(upper) * os) as the clamp requires.
    // The window of a voxel ends less than 1/os past its box, so with boxes sticking out of the
    // footprint by less than 1 - 1/os pixels its pixels lie within one pixel of the footprint's
    // floor and ceiling: the block tile's margin.
    w.covers = 1;
    double stick = 0.0;   // largest distance a voxel box sticks out of its quad footprint
    const double qx[2] = {0.0, (double)std::max(0, v.nx - 4)}, qy[2] = {0.0, (double)(v.ny - 1)},
                 qz[2] = {0.0, (double)(v.nz - 1)};
    for (int c = 0; c < 8; c++) {
        const double q[3] = {qx[c & 1], qy[(c >> 1) & 1], qz[(c >> 2) & 1]};
        for (int r = 0; r < 2; r++) {
            const double gq = e.G[r][0] * q[0] + e.G[r][1] * q[1] + e.G[r][2] * q[2];
            const double p = r == 0 ? e.pu0 + e.pui * q[0] + e.puj * q[1] + e.puk * q[2]
                                    : e.pv0 + e.pvi * q[0] + e.pvj * q[1] + e.pvk * q[2];
            const double pi = r == 0 ? e.pui : e.pvi;
            const double boxLo = p + std::fmin(0.0, 3.0 * pi) + (double)(r == 0 ? e.uMin : e.vMin);
            const double boxHi = p + std::fmax(0.0, 3.0 * pi) + (double)(r == 0 ? e.uMax : e.vMax);
            if (!(gq + e.lo[r] <= boxLo && boxHi <= gq + e.hi[r])) w.covers = 0;
            stick = std::fmax(stick, std::fmax((gq + e.lo[r]) - boxLo, boxHi - (gq + e.hi[r])));
        }
    }
    w.masked = stick + 1.0 / os < 0.95 ? 1 : 0;
    return w.ni >= 1 && w.nj >= 1 && w.ni <= maxN && w.nj <= maxN;
}

// Whether the dist gate [distMin, distMax) passes every quad of the volume: |gn . q + g0| is the
// absolute value of an affine form of one sign over the volume (the affine footprint), so its
// extremes lie at the corner quads.
inline bool gate_passes_all(const VolG& v, const BPWin& w, double distMin, double distMax) {
    const double qx[2] = {0.0, (double)std::max(0, v.nx - 4)}, qy[2] = {0.0, (double)(v.ny - 1)},
                 qz[2] = {0.0, (double)(v.nz - 1)};
    for (int c = 0; c < 8; c++) {
        const double q[3] = {qx[c & 1], qy[(c >> 1) & 1], qz[(c >> 2) & 1]};
        const double t = std::fabs(std::fma(w.gn[0], q[0], std::fma(w.gn[1], q[1], std::fma(w.gn[2], q[2], w.g0))));
        if (!(t >= distMin && t < distMax)) return false;
    }
    return true;
}

// The constants of a window in vector registers: a scalar operand halves the rate of an add or a multiply-add.
struct WinRegs {
    float SPh, SYh, PUd, PVd, YUd, YVd, PUd2, YUd2;
    __device__ __forceinline__ explicit WinRegs(const BPWin& w)
        : SPh(w.SPh), SYh(w.SYh), PUd(w.PUd), PVd(w.PVd), YUd(w.YUd), YVd(w.YVd), PUd2(2.0f * w.PUd), YUd2(2.0f * w.YUd) {
        __asm__("" : "+v"(SPh), "+v"(SYh), "+v"(PUd), "+v"(PVd), "+v"(YUd), "+v"(YVd), "+v"(PUd2), "+v"(YUd2));
    }
    // x + d step, rounded once (step2: twice the step, which is exact)
    __device__ __forceinline__ static float at(float x, int d, float step, float step2) {
        return d == 0 ? x : (d == 1 ? x + step : (d == 2 ? x + step2 : __builtin_fmaf((float)d, step, x)));
    }
    __device__ __forceinline__ float px(float x, int d) const { return at(x, d, PUd, PUd2); }
    __device__ __forceinline__ float yx(float x, int d) const { return at(x, d, YUd, YUd2); }
    __device__ __forceinline__ float py(float x, int d) const { return d == 2 ? __builtin_fmaf(2.0f, PVd, x) : at(x, d, PVd, 0.0f); }
    __device__ __forceinline__ float yy(float x, int d) const { return d == 2 ? __builtin_fmaf(2.0f, YVd, x) : at(x, d, YVd, 0.0f); }
};

__device__ __forceinline__ float clamp01(float x) { return __builtin_amdgcn_fmed3f(x, 0.0f, 1.0f); }

// The chord-weighted sums of one voxel over its kNI x kNJ window, read from the block's LDS tile
// of image pixels (row pitch tw).  P0, Y0: Pc and Yc at the window's first lattice point, which lies in
// tile pixel `base`, in its ph-th column and qh-th row of lattice points.  Only lattice points in the quad
// footprint count: columns di with il + di < iw (unsigned), rows dj with jl + dj < jh, which kMode applies as:
//   kWinOpen:   not at all (the footprint covers every voxel box: w.covers);
//   kWinMasked: by moving the point out of its slabs (every window pixel lies in the tile);
//   kWinClamp:  by skipping the point and its read (blocks at the image edges).
// The three give the same sums for finite images: a point outside adds fma(val, 0, n) = n.
// kYCol: the y slab term does not change down a window column (YVd == 0: every tilt about y whose
// detector v axis has no y component, the u axis being the volume's y axis), so it is evaluated
// once per column, and the points whose chord is 0 for a whole column (outside the voxel's y slab,
// or outside the footprint's columns) or a whole row (outside the footprint's rows) are skipped
// with their reads.  The sums start at -0, the additive identity, so that the first point taken
// adds what the window's first point would.
//
// VALU issue bounds the sums: a lattice point takes seven instructions of full rate (two coordinates,
// two clamped differences, their product, the two sums) and its read; min and med3 in their place run at half.
// 1024x1024x256 from 1024^2 pixels, 3 x 3 points: 0.96 -> 0.82 ms per tilt, 300 sub-volumes by 41 tilts 20.4 ->
// 17.8 ms (with the four voxels of a quad in one branch and the tile's rows without integer division).
constexpr int kWinOpen = 0, kWinMasked = 1, kWinClamp = 2;
template <int kOS, int kNI, int kNJ, int kMode, bool kYCol = false>
__device__ __forceinline__ void window_sums(const WinRegs& w, const float* __restrict__ tile, int tw, int base,
                                            int ph, int qh, float P0, float Y0, int il, unsigned iw, int jl, unsigned jh,
                                            float& num, float& den) {
    const int qtw = qh ? tw : 0;
    // the window's columns: whether they count (in the footprint, and for kYCol in the y slab)
    bool live[kNI];
#pragma unroll
    for (int di = 0; di < kNI; di++)
        live[di] = (kMode == kWinOpen || (unsigned)(il + di) < iw) && (!kYCol || w.SYh - fabsf(w.yx(Y0, di)) > 0.0f);
    // masked: SP/2 of a column outside the footprint is below every |Pc|
    float SPcol[kNI];
#pragma unroll
    for (int di = 0; di < kNI; di++) SPcol[di] = kMode == kWinMasked && !live[di] ? -1.0f : w.SPh;
    float n = kYCol ? -0.0f : 0.0f, d = kYCol ? -0.0f : 0.0f;
#pragma unroll
    for (int dj = 0; dj < kNJ; dj++) {
        const bool rowOk = kMode == kWinOpen || (unsigned)(jl + dj) < jh;
        if (kYCol && !rowOk) continue;
        const float Pr = w.py(P0, dj);
        float Yr = w.yy(Y0, dj);
        // masked: a row outside the footprint moves beyond every y slab
        if (kMode == kWinMasked && !kYCol) Yr = rowOk ? Yr : kWinFar;
        const int rowBase = base + (kOS == 1 ? dj * tw : (dj >> 1) * tw + ((dj & 1) ? qtw : 0));
        const int rowOdd = rowBase + ph;   // odd di of the 2x lattice: pixel c0 + ph + (di - 1) / 2
#pragma unroll
        for (int di = 0; di < kNI; di++) {
            if (kYCol && !live[di]) continue;
            const float A = clamp01((kMode == kWinMasked && !kYCol ? SPcol[di] : w.SPh) - fabsf(w.px(Pr, di)));
            float chord = kYCol ? A : A * clamp01(w.SYh - fabsf(w.yx(Yr, di)));
            int addr = kOS == 1 ? rowBase + di : ((di & 1) ? rowOdd + (di >> 1) : rowBase + (di >> 1));
            if (kMode == kWinClamp && !kYCol) {
                const bool ok = rowOk && live[di];
                chord = ok ? chord : 0.0f;
                addr = ok ? addr : 0;
            }
            const float val = tile[addr];
            if (!kYCol && di == 0 && dj == 0) {
                n = val * chord;
                d = chord;
            } else {
                n = __builtin_fmaf(val, chord, n);
                d += chord;
            }
        }
    }
    num = n;
    den = d;
}

// The window form's plan for one tilt: the form applies, the footprint of a 64 x 4 x 8-voxel block
// fits the LDS tile and the window size has a compiled instance (OS 1: 1-3, OS 2: 2-4 lattice
// points per axis).  The per-call and the batched sub-volume backprojections take the same decision,
// so they stay bit-identical.
constexpr int kWinBlockZ = 8;   // slices per block of the per-call kernel (two quads per thread)
inline bool window_plan(const VolG& v, const TiltG& g, int os, BPWin& w) {
    if (os != 1 && os != 2) return false;
    const BPExact e = prepare_exact(v, g, 64, 4, kWinBlockZ);
    if ((long long)(e.tileW + 2) * (long long)(e.tileH + 2) > kTileFloats) return false;
    if (!prepare_window(v, g, e, os, os == 1 ? 3 : 4, w)) return false;
    return os == 1 ? true : (w.ni >= 2 && w.nj >= 2);
}

// The update of one quad (voxels x .. x+3 of row y, slice z) for one tilt: out[k] += lambda *
// num / den over each voxel's window, from an image tile of row pitch tw whose pixel (tx0, ty0) is
// tile[0] (the whole image with tw = pitch and tx0 = ty0 = 0).  Only lattice points in the quad's
// footprint clamped to [0, W-1] x [0, H-1] count, as in the per-box loop.  interior: the block's
// footprint lies in the image with a pixel to spare and the tile holds it with a one-pixel margin;
// then the footprint test is skipped (w.covers) or applied as a chord cap (w.masked), otherwise
// each point outside is skipped with its read.  Returns whether a voxel changed.
template <int kOS, int kNI, int kNJ, bool kYCol = false>
__device__ __forceinline__ bool window_quad(const BPWin& w, const float* __restrict__ tile, int tw, int tx0, int ty0,
                                            bool interior, int W, int H, unsigned x, unsigned y, unsigned z,
                                            float lambda, float out[4]) {
    constexpr float kDelta = 1.0f / (float)kOS;
    const double qx = (double)x, qy = (double)y, qz = (double)z;
    int li0 = 0, li1 = 0, lj0 = 0, lj1 = 0;
    const int mode = interior && w.covers ? kWinOpen : (interior && w.masked ? kWinMasked : kWinClamp);
    if (mode != kWinOpen) {
        // the quad's footprint clamped to [0, W-1] x [0, H-1] (footprint_affine): lattice points
        // [px0 * OS, px1 * OS) x [py0 * OS, py1 * OS); in an interior block the clamps are no-ops
        const double a0 = fma(w.G[0][0], qx, fma(w.G[0][1], qy, w.G[0][2] * qz));
        const double a1 = fma(w.G[1][0], qx, fma(w.G[1][1], qy, w.G[1][2] * qz));
        if (mode == kWinMasked) {
            li0 = kOS * (int)floor(a0 + w.lo[0]);
            li1 = kOS * (int)ceil(a0 + w.hi[0]);
            lj0 = kOS * (int)floor(a1 + w.lo[1]);
            lj1 = kOS * (int)ceil(a1 + w.hi[1]);
        } else {
            li0 = kOS * (int)fmin(fmax(floor(a0 + w.lo[0]), 0.0), (double)(W - 1));
            li1 = kOS * (int)fmin(fmax(ceil(a0 + w.hi[0]), 0.0), (double)(W - 1));
            lj0 = kOS * (int)fmin(fmax(floor(a1 + w.lo[1]), 0.0), (double)(H - 1));
            lj1 = kOS * (int)fmin(fmax(ceil(a1 + w.hi[1]), 0.0), (double)(H - 1));
        }
        if (li1 <= li0 || lj1 <= lj0) return false;
    }
    // corner projection of the quad's first voxel, split into an integer pixel and a float offset
    const double Uq = fma(w.pui, qx, fma(w.puj, qy, fma(w.puk, qz, w.pu0)));
    const double Vq = fma(w.pvi, qx, fma(w.pvj, qy, fma(w.pvk, qz, w.pv0)));
    const double fUq = floor(Uq), fVq = floor(Vq);
    const int iq = (int)fUq, jq = (int)fVq;
    const float fu = (float)(Uq - fUq), fv = (float)(Vq - fVq);
    const float dui = (float)w.pui, dvi = (float)w.pvi;
    const WinRegs r(w);
    // tile rows are small: 24-bit multiplies (full rate; the 32-bit one is a quarter)
    const int baseq = __mul24(jq - ty0, tw) + (iq - tx0);
    const int ilq = iq * kOS - li0, jlq = jq * kOS - lj0;
    bool any = false;
    const auto voxels = [&](auto mode_c) {
        constexpr int kMode = decltype(mode_c)::value;
#pragma unroll
        for (int k = 0; k < 4; k++) {
            const float du = __builtin_fmaf((float)k, dui, fu);
            const float dv = __builtin_fmaf((float)k, dvi, fv);
            // the window's first lattice point, as a float (an integer) and an int
            const float fi0 = ceilf((du + w.uMin) * (float)kOS - 0.5f), fj0 = ceilf((dv + w.vMin) * (float)kOS - 0.5f);
            const int i0 = (int)fi0, j0 = (int)fj0;
            const float a0 = __builtin_fmaf(fi0 + 0.5f, kDelta, -du), b0 = __builtin_fmaf(fj0 + 0.5f, kDelta, -dv);
            const float P0 = __builtin_fmaf(a0, w.PU, __builtin_fmaf(b0, w.PV, w.PC));
            const float Y0 = __builtin_fmaf(a0, w.YU, __builtin_fmaf(b0, w.YV, w.YC));
            // pixel of lattice point i: floor(i / kOS)
            const int base = kOS == 1 ? __mul24(j0, tw) + i0 + baseq : __mul24(j0 >> 1, tw) + (i0 >> 1) + baseq;
            const int ph = kOS == 1 ? 0 : (i0 & 1), qh = kOS == 1 ? 0 : (j0 & 1);
            float num, den;
            window_sums<kOS, kNI, kNJ, kMode, kYCol>(r, tile, tw, base, ph, qh, P0, Y0, ilq + i0, (unsigned)(li1 - li0),
                                                     jlq + j0, (unsigned)(lj1 - lj0), num, den);
            if (den > 0.0f) {
                out[k] += (lambda * num) * __builtin_amdgcn_rcpf(den);
                any = true;
            }
        }
    };
    // (the branch around the four voxels, so that their reads overlap)
    if (mode == kWinOpen) voxels(std::integral_constant<int, kWinOpen>());
    else if (mode == kWinMasked) voxels(std::integral_constant<int, kWinMasked>());
    else voxels(std::integral_constant<int, kWinClamp>());
    return any;
}

// window_quad with the window size chosen at run time (w.ni, w.nj) among the compiled instances.
template <int kOS>
__device__ __forceinline__ bool window_quad_any(const BPWin& w, const float* __restrict__ tile, int tw, int tx0,
                                                int ty0, bool interior, int W, int H, unsigned x, unsigned y,
                                                unsigned z, float lambda, float out[4]) {
    constexpr int kLo = kOS == 1 ? 1 : 2;
#define ARTIA_WIN_CASE(NI, NJ)                                                                                   \
    if (w.ni == (NI) && w.nj == (NJ))                                                                           \
        return window_quad<kOS, (NI), (NJ)>(w, tile, tw, tx0, ty0, interior, W, H, x, y, z, lambda, out);
    ARTIA_WIN_CASE(kLo + 1, kLo + 1)
    ARTIA_WIN_CASE(kLo, kLo)
    ARTIA_WIN_CASE(kLo, kLo + 1)
    ARTIA_WIN_CASE(kLo + 1, kLo)
    ARTIA_WIN_CASE(kLo + 2, kLo + 1)
    ARTIA_WIN_CASE(kLo + 1, kLo + 2)
    ARTIA_WIN_CASE(kLo + 2, kLo + 2)
    ARTIA_WIN_CASE(kLo, kLo + 2)
    ARTIA_WIN_CASE(kLo + 2, kLo)
#undef ARTIA_WIN_CASE
    return false;
}

}  // namespace artia
