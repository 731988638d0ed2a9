// Tiled steps for structured rectangles on gfx950: one kernel per step, for a
// tile of kTileJ cells along j (the fast index) by TI rows along i.
//
// MUSCL step (k_tile_step): the limited LSM gradient, the predictor's half
// state and the half state's values at the cell's four faces are computed for
// the tile and its one-cell halo; every face of the tile's cells is then
// evaluated once, for both of its cells (zfv_pair.hpp), and the next step's CFL
// candidate is fused at the end.  The first-order step (k_tile_flux1) is the
// same without the gradient and the predictor.
//
// What bounds it: FP64 instruction issue (a step is some 2,000 FP64
// instructions per cell against 118 B), so the split serves the instruction
// count.  A wavefront is one row of 64 consecutive cells: its row index is
// uniform, so everything of a column is scalar; neighbours along j come by
// lane shifts, those along i (other wavefronts) through LDS.  A cell's thread
// evaluates its right and top faces and hands each neighbour its share, which
// leaves one halo row and one halo lane of faces per tile in place of every
// face twice.  Ghost cells (copied or reflected states, written where the
// neighbour would be) replace the boundary choices of each face.
//
// Every per-cell value is computed by the same operations in the same order
// as the mesh-array kernels (zfv_kernels.hip), with two kinds of exceptions
// that change no value: terms whose factor is an exact zero on a canonical
// normal (the off-diagonal LSM matrix, dr across the normal) are left out, and
// 2 x - y and 0.5 (1 + x) are one rounding either way.  The slot geometry
// comes from per-column and per-row tables that the host checked, cell by
// cell, against the slot arrays.
//
// Layout of a workgroup of (TI + 2) wavefronts: wavefront r takes row
// i = i0 - 1 + r and lane l the cell j = j0 - 1 + l; the outputs are rows
// 1..TI and lanes 1..kTileJ.  Cell index c = off + i * ny + j.
#pragma once

#include <algorithm>

#include "zfv_internal.hpp"
#include "zfv_pair.hpp"
#include "zfv_step_common.hpp"

namespace zfv {

namespace {

constexpr int kBJ = kTileJ + 4;   // state box row: the tile's cells and a two-cell halo on each side

// min of v and its value a DPP move away (lanes without a source keep v).
template <int CTRL, int ROWS>
__device__ __forceinline__ double min_dpp(double v) {
    const int lo = __double2loint(v), hi = __double2hiint(v);
    const double o = __hiloint2double(__builtin_amdgcn_update_dpp(hi, hi, CTRL, ROWS, 0xF, false),
                                      __builtin_amdgcn_update_dpp(lo, lo, CTRL, ROWS, 0xF, false));
    return __builtin_fmin(v, o);
}

// min over the workgroup of the CFL candidates, then one 64-bit atomicMin on
// the bit pattern (block_min_atomic for workgroups of up to 16 wavefronts).
// A wavefront's minimum gathers in its last lane: shifts inside each row of
// 16 lanes, then row 0 into 1 and 2 into 3, then rows 0-1 into 2-3.
template <int NW>
__device__ __forceinline__ void tile_min_atomic(unsigned long long* slot, double v, double* red) {
    if (!(v < INFINITY)) v = INFINITY;   // NaN and +inf never win
    v = min_dpp<0x111, 0xF>(v);   // row_shr:1
    v = min_dpp<0x112, 0xF>(v);   // row_shr:2
    v = min_dpp<0x114, 0xF>(v);   // row_shr:4
    v = min_dpp<0x118, 0xF>(v);   // row_shr:8
    v = min_dpp<0x142, 0xA>(v);   // row_bcast:15
    v = min_dpp<0x143, 0xC>(v);   // row_bcast:31
    const int lane = threadIdx.x & 63, wid = threadIdx.x >> 6;
    if (lane == 63) red[wid] = v;
    __syncthreads();
    if (threadIdx.x == 0) {
        double m = red[0];
        for (int i = 1; i < NW; ++i) m = (red[i] < m) ? red[i] : m;
        if (m < INFINITY) atomicMin(slot, (unsigned long long)__double_as_longlong(m));
    }
}

__device__ __forceinline__ int wrap(int g, int n) {
    const int m = g % n;
    return m < 0 ? m + n : m;
}

// Problem of tile b: the last problem whose first tile is <= b.
template <int V>
__device__ __forceinline__ int problem_of(const TileMesh& T, int b) {
    int lo = 0, hi = T.n_probs - 1;
    while (lo < hi) {
        const int mid = (lo + hi + 1) >> 1;
        if (T.prob[mid].tile0[V] <= b) lo = mid;
        else hi = mid - 1;
    }
    return lo;
}

// By value: both sources end in scalar registers, where a selected reference
// would have to be one kind of memory.
__device__ __forceinline__ TileProb problem(const TileMesh& T, int pid) {
    TileProb P = T.one;
    if (T.n_probs != 1) P = T.prob[pid];
    return P;
}

// The value of lane l + 1 / lane l - 1 (DPP wave_shl:1 / wave_shr:1; the end
// lane gets 0).  Every lane of the wavefront must be active.
__device__ __forceinline__ double from_next(double v) {
    const int lo = __builtin_amdgcn_update_dpp(0, __double2loint(v), 0x130, 0xF, 0xF, true);
    const int hi = __builtin_amdgcn_update_dpp(0, __double2hiint(v), 0x130, 0xF, 0xF, true);
    return __hiloint2double(hi, lo);
}
__device__ __forceinline__ double from_prev(double v) {
    const int lo = __builtin_amdgcn_update_dpp(0, __double2loint(v), 0x138, 0xF, 0xF, true);
    const int hi = __builtin_amdgcn_update_dpp(0, __double2hiint(v), 0x138, 0xF, 0xF, true);
    return __hiloint2double(hi, lo);
}
__device__ __forceinline__ Z from_next(const Z& z) {
    return Z{from_next(z.r), from_next(z.u), from_next(z.v), from_next(z.p), from_next(z.e)};
}
__device__ __forceinline__ Q from_prev(const Q& q) {
    return Q{from_prev(q.r), from_prev(q.mx), from_prev(q.my), from_prev(q.E)};
}

__device__ __forceinline__ void put5(double* ex, int stride, int k, const Z& z) {
    ex[k] = z.r;
    ex[stride + k] = z.u;
    ex[2 * stride + k] = z.v;
    ex[3 * stride + k] = z.p;
    ex[4 * stride + k] = z.e;
}
__device__ __forceinline__ Z get5(const double* ex, int stride, int k) {
    return Z{ex[k], ex[stride + k], ex[2 * stride + k], ex[3 * stride + k], ex[4 * stride + k]};
}

// boundary_value of a face state at the left / right and the bottom / top side.
__device__ __forceinline__ Z bnd_x(Z z, int t) {
    if (t == SC_WALL) z.u = z.u - 2.0 * z.u;
    return z;
}
__device__ __forceinline__ Z bnd_y(Z z, int t) {
    if (t == SC_WALL) z.v = z.v - 2.0 * z.v;
    return z;
}

// To the frame of the top side and back (frame_local / frame_global).
__device__ __forceinline__ Z top_local(const Z& z) { return Z{z.r, z.v, -z.u, z.p, z.e}; }
__device__ __forceinline__ Q top_global(const Q& f) { return Q{f.r, -f.my, f.mx, f.E}; }

__device__ __forceinline__ Q scaled(const Q& f, double a) { return Q{f.r * a, f.mx * a, f.my * a, f.E * a}; }

// limiter2(a, b) * b.  The ratio limiters take v_min / v_max: their operands
// are not NaN where the result is used.
template <int LIM>
__device__ __forceinline__ double limited(double a, double b) {
    if constexpr (LIM == 3 || LIM == 10 || LIM == 11 || LIM == 12) {
        const double r = a / b, r2 = 2.0 * r;
        double m;
        if constexpr (LIM == 3) m = __builtin_fmin(__builtin_fma(0.5, r, 0.5), 2.0);
        else if constexpr (LIM == 10) m = __builtin_fmin(2.0, (1.0 + r2) / 3.0);
        else if constexpr (LIM == 11) m = __builtin_fmin(0.25 + 0.75 * r, 4.0);
        else m = __builtin_fmin(r, 2.0);
        if constexpr (LIM == 12) m = __builtin_fmax(0.0, __builtin_fmin(__builtin_fmin(r2, 1.0), m));
        else m = __builtin_fmax(0.0, __builtin_fmin(r2, m));
        return (isnan(r) ? 0.0 : m) * b;
    } else {
        return limiter2<LIM>(a, b) * b;
    }
}

// A face state moved from z, with its energy; z itself where that is no
// state (rare, so the choice is made only where some lane needs it).
__device__ __forceinline__ Z face_state(const Z& z, const double* d, const Eos& eos) {
    Z f{z.r + d[0], z.u + d[1], z.v + d[2], z.p + d[3], 0.0};
    f.e = eos_e(eos, f.r, f.p);
    const bool bad = is_bad(f, eos);
    if (__builtin_expect(__any(bad), 0)) {
        if (bad) f = z;
    }
    return f;
}

// The x and y fluxes of a face state (phys_flux between frame_local and
// frame_global of the right and the top side; the left and bottom sides'
// values are the exact negatives).
__device__ __forceinline__ Q flux_x(const Z& z) {
    const double m = z.r * z.u;
    return Q{m, m * z.u + z.p, m * z.v, (z.r * (z.e + 0.5 * vsq(z)) + z.p) * z.u};
}
__device__ __forceinline__ Q flux_y(const Z& z) {
    const double m = z.r * z.v;
    return Q{m, m * z.u, m * z.v + z.p, (z.r * (z.e + 0.5 * vsq(z)) + z.p) * z.v};
}

// A tile's place in its problem, and a thread's in the tile.
struct Place {
    int pid, nx, ny, off;
    int i0, j0;        // first output row and cell
    int w, l;          // wavefront and lane
    int gu, gv;        // this thread's row and cell, before wrapping
    int gi, gj;        // ... wrapped, or clamped to the domain
    bool perx, pery;
    bool first;        // the problem's first tile

    __device__ __forceinline__ int row(int g) const {
        return perx ? wrap(g, nx) : (g < 0 ? 0 : (g < nx ? g : nx - 1));
    }
    __device__ __forceinline__ int cell(int g) const {
        return pery ? wrap(g, ny) : (g < 0 ? 0 : (g < ny ? g : ny - 1));
    }
};

template <int V, int TI>
__device__ __forceinline__ Place place_of(const TileMesh& T, int b) {
    Place p;
    p.pid = T.n_probs == 1 ? 0 : problem_of<V>(T, b);
    const TileProb P = problem(T, p.pid);
    const int t = b - P.tile0[V];
    const int ti = t / P.tiles_j, tj = t - ti * P.tiles_j;
    p.nx = P.nx;
    p.ny = P.ny;
    p.off = P.off;
    p.first = t == 0;
    p.i0 = ti * TI;
    p.j0 = tj * kTileJ;
    p.w = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6);
    p.l = (int)threadIdx.x & 63;
    p.perx = P.per[0] != 0;
    p.pery = P.per[1] != 0;
    p.gu = p.i0 - 1 + p.w;
    p.gv = p.j0 - 1 + p.l;
    p.gi = p.row(p.gu);
    p.gj = p.cell(p.gv);
    return p;
}

// Whether this lane has a top face: from_next gives the last one no state.
__device__ __forceinline__ bool top_lane(const Place& p) { return p.l < 63; }

__device__ __forceinline__ void tile_prologue(const StepCtl& ctl, const Place& p, double dt) {
    if (p.first && threadIdx.x == 0) {
        ctl.dt_out[p.pid] = dt;
        ctl.dtmin[3 * p.pid + ctl.clr] = kInfBits;
    }
}

}  // namespace

// The workgroup's LDS, as separate arrays: the state box zs (rho, u, v, p),
// the exchange ex between neighbouring rows (first the left-face state of
// each row's cells, with ghosts, then the flux each row's cells take through
// their left face), the tile's row table rt, the isolation counters ws of the
// halo box, the CFL reduction red.
#define ZFV_TILE_LDS(TI)                                  \
    __shared__ double zs[4 * ((TI) + 4) * kBJ];           \
    __shared__ double ex[5 * ((TI) + 2) * 64];            \
    __shared__ double rt[kTileRowQ * 64];                 \
    __shared__ int ws[((TI) + 2) * 64];                   \
    __shared__ double red[(TI) + 2]

// SmFluid::update with acc 2 (sm_fluid.cpp:81-102) on one tile b of shape V:
// compute_grad (sm_fluid.cpp:116-125, gradient.h:226-282, 412-474),
// fluxes_stage1 (:176-253) and fluxes_stage2 (:255-366), plus the next step's
// CFL candidate (:104-114).
template <int FLUX, int LIM, int V, int TI>
__device__ __forceinline__ void tile_body(const TileMesh& T, const DevState& in, const DevState& out,
                                          const int* __restrict__ wait_in, int* __restrict__ wait_out,
                                          const Eos& eos, const StepCtl& ctl, int b, double* zs, double* ex,
                                          double* rt, int* ws, double* red) {
    constexpr int NW = TI + 2, XS = NW * 64, ZS = (TI + 4) * kBJ;
    const Place p = place_of<V, TI>(T, b);
    const TileProb P = problem(T, p.pid);
    const double dt = step_dt(ctl, p.pid);
    tile_prologue(ctl, p, dt);

    // ---- state box: each wavefront loads its own row, its two end lanes the
    // outer columns, the end wavefronts the outer rows.  Cells outside the
    // domain get the boundary value of the cell next to them.
    const int c = p.off + p.gi * p.ny + p.gj;
    const int o = (p.w + 1) * kBJ + p.l + 1;   // this thread's cell in the state box
    auto box_load = [&](int g, int h, int k) {
        const int cc = p.off + p.row(g) * p.ny + p.cell(h);
        Z z{in.r[cc], in.u[cc], in.v[cc], in.p[cc], 0.0};
        if (!p.perx && (g < 0 || g >= p.nx)) z = bnd_x(z, g < 0 ? P.t[0] : P.t[1]);
        if (!p.pery && (h < 0 || h >= p.ny)) z = bnd_y(z, h < 0 ? P.t[2] : P.t[3]);
        zs[k] = z.r;
        zs[ZS + k] = z.u;
        zs[2 * ZS + k] = z.v;
        zs[3 * ZS + k] = z.p;
        return z;
    };
    Z zc = box_load(p.gu, p.gv, o);
    zc.e = in.e[c];
    const int wc = wait_in[c];
    const double vol = T.vol[c];
    if (p.l == 0 || p.l == 63) box_load(p.gu, p.l == 0 ? p.j0 - 2 : p.j0 + 63, (p.w + 1) * kBJ + (p.l == 0 ? 0 : 65));
    if (p.w == 0) box_load(p.i0 - 2, p.gv, p.l + 1);
    if (p.w == TI + 1) box_load(p.i0 + TI + 1, p.gv, (TI + 3) * kBJ + p.l + 1);
    for (int q = p.w; q < kTileRowQ; q += NW) rt[q * 64 + p.l] = T.row[(size_t)q * T.row_stride + P.row + p.gj];
    const int x = p.w * 64 + p.l;   // this thread's place in the exchange
    ws[x] = wc;
    __syncthreads();

    // rows of the domain (and of the periodic halo) are computed
    const bool act = p.perx ? p.gu <= p.nx : (p.gu >= 0 && p.gu < p.nx);
    const bool out_row = p.w >= 1 && p.w <= TI && p.gu < p.nx;
    const bool out_lane = p.l >= 1 && p.l <= kTileJ && p.gv < p.ny;
    const TileCol& C = T.col[P.col + p.gi];
    const double* R = rt + p.l;
    bool bad = false;
    Z sR{};                 // the state at the right face
    Q fB{}, fT{};           // flux * area through the bottom and the top face
    bool robR = false;
    if (act) {
        // ---- gradient and limiting: the LSM system of a canonical cell is
        // diagonal (A01 = A10 = 0)
        const double A00 = C.A00, A11 = R[kRowA11 * 64];
        const double invdet = 1.0 / (A11 * A00);
        const double B00 = A11 * invdet, B11 = A00 * invdet;
        const double drL = C.drL, drR = C.drR, wL = C.wL, wR = C.wR;
        const double drB = R[kRowDrB * 64], drT = R[kRowDrT * 64], wB = R[kRowWB * 64], wT = R[kRowWT * 64];
        // the increments to the four faces, L, R, B, T
        double dL[4], dR[4], dB[4], dT[4], gx[4], gy[4];
        const double oxL = C.oxL, oxR = C.oxR, ox = C.ox;
        const double oy = R[kRowOy * 64], oyB = R[kRowOyB * 64], oyT = R[kRowOyT * 64];
#pragma unroll
        for (int k = 0; k < 4; ++k) {
            const double* z = zs + k * ZS + o;
            const double zk = z[0];
            const double a = z[-kBJ] - zk, d = z[kBJ] - zk, e = z[-1] - zk, f = z[1] - zk;
            double g = B00 * ((wL * a) * drL + (wR * d) * drR);
            double h = B11 * ((wB * e) * drB + (wT * f) * drT);
            const double la = limited<LIM>(__builtin_fma(2.0, g * drL, -a), a);
            const double ld = limited<LIM>(__builtin_fma(2.0, g * drR, -d), d);
            const double le = limited<LIM>(__builtin_fma(2.0, h * drB, -e), e);
            const double lf = limited<LIM>(__builtin_fma(2.0, h * drT, -f), f);
            g = B00 * ((wL * la) * drL + (wR * ld) * drR);
            h = B11 * ((wB * le) * drB + (wT * lf) * drT);
            gx[k] = g;
            gy[k] = h;
            const double hy = h * oy, gX = g * ox;
            dL[k] = g * oxL + hy;
            dR[k] = g * oxR + hy;
            dB[k] = gX + h * oyB;
            dT[k] = gX + h * oyT;
        }
        // ---- predictor
        Z zh;
        {
            const double aL = R[kRowAL * 64], aR = R[kRowAR * 64], aB = C.aB, aT = C.aT;
            Q F = scaled(flux_x(face_state(zc, dL, eos)), -aL);
            Q f = scaled(flux_x(face_state(zc, dR, eos)), aR);
            F = Q{F.r + f.r, F.mx + f.mx, F.my + f.my, F.E + f.E};
            f = scaled(flux_y(face_state(zc, dB, eos)), aB);
            F = Q{F.r - f.r, F.mx - f.mx, F.my - f.my, F.E - f.E};
            f = scaled(flux_y(face_state(zc, dT, eos)), aT);
            F = Q{F.r + f.r, F.mx + f.mx, F.my + f.my, F.E + f.E};
            Q q = to_q(zc);
            const double coef = 0.5 * dt / vol;
            q.r = q.r - coef * F.r;
            q.mx = q.mx - coef * F.mx;
            q.my = q.my - coef * F.my;
            q.E = q.E - coef * F.E;
            zh = to_z(q, eos);
            const bool keep = wc > 0 || is_bad(zh, eos);
            if (__builtin_expect(__any(keep), 0)) {
                if (keep) zh = zc;
            }
        }
        // The increments again, rather than held across the predictor (32
        // registers, which would spill).
#pragma unroll
        for (int k = 0; k < 4; ++k) {
            asm volatile("" : "+v"(gx[k]), "+v"(gy[k]));
            const double hy = gy[k] * oy, gX = gx[k] * ox;
            dL[k] = gx[k] * oxL + hy;
            dR[k] = gx[k] * oxR + hy;
            dB[k] = gX + gy[k] * oyB;
            dT[k] = gX + gy[k] * oyT;
        }
        // ---- the half state at the four faces.  A face of a cell in the
        // isolation mode, on either side, takes the half states themselves.
        // The halo cell beyond a periodic side is seen at its mirror image,
        // as its neighbour sees it.
        if (p.gu == p.nx) {
            const double n = T.col[P.col + p.nx - 1].nR;
#pragma unroll
            for (int k = 0; k < 4; ++k) dL[k] = gx[k] * n + gy[k] * oy;
        }
        if (p.gu == -1) {
            const double n = T.col[P.col].nL;
#pragma unroll
            for (int k = 0; k < 4; ++k) dR[k] = gx[k] * n + gy[k] * oy;
        }
        if (p.pery && (p.j0 == 0 || p.j0 + 63 > p.ny)) {
            const double nT = T.row[(size_t)kRowNT * T.row_stride + P.row + p.ny - 1];
            const double nB = T.row[(size_t)kRowNB * T.row_stride + P.row];
#pragma unroll
            for (int k = 0; k < 4; ++k) {
                if (p.gv == p.ny) dB[k] = gx[k] * ox + gy[k] * nT;
                if (p.gv == -1) dT[k] = gx[k] * ox + gy[k] * nB;
            }
        }
        Z sL = face_state(zh, dL, eos), sB = face_state(zh, dB, eos), sT = face_state(zh, dT, eos);
        sR = face_state(zh, dR, eos);
        const bool iso = wc > 0;
        const bool robL = iso || ws[p.w > 0 ? x - 64 : x] > 0, robB = iso || ws[p.l > 0 ? x - 1 : x] > 0;
        const bool robT = iso || ws[p.l < 63 ? x + 1 : x] > 0;
        robR = iso || ws[p.w <= TI ? x + 64 : x] > 0;
        if (__builtin_expect(__any(robL || robR || robB || robT), 0)) {
            if (robL) sL = zh;
            if (robR) sR = zh;
            if (robB) sB = zh;
            if (robT) sT = zh;
        }
        put5(ex, XS, x, sL);
        // ghosts beyond the left and right sides: the boundary value of the
        // face state; behind a one-sided periodic side (whose neighbour is
        // the cell itself) the state seen from the mirror image
        auto one_sided = [&](double dx, double dy, bool rob) {
            double d[4];
#pragma unroll
            for (int k = 0; k < 4; ++k) d[k] = gx[k] * dx + gy[k] * dy;
            const Z z = face_state(zh, d, eos);
            return rob ? zh : z;
        };
        if (!p.perx) {
            if (p.gu == 0 && p.w == 1)
                put5(ex, XS, p.l, P.t[0] == SC_PERIODIC ? one_sided(C.nL, oy, robL) : bnd_x(sL, P.t[0]));
            if (p.gu == p.nx - 1 && p.w <= TI)
                put5(ex, XS, x + 64, P.t[1] == SC_PERIODIC ? one_sided(C.nR, oy, robR) : bnd_x(sR, P.t[1]));
        }
        // ---- the faces along j: the thread's top face
        if (out_row) {
            Z A = sT, B = from_next(sB);
            bool rob = robT;
            if (!p.pery) {
                if (p.j0 + 63 >= p.ny) {   // the tile holds the top side
                    const Z g = P.t[3] == SC_PERIODIC
                                    ? one_sided(ox, T.row[(size_t)kRowNT * T.row_stride + P.row + p.ny - 1], robT)
                                    : bnd_y(sT, P.t[3]);
                    if (p.gv == p.ny - 1) B = g;
                }
                if (p.j0 == 0) {   // the bottom side, seen by the ghost in lane 0
                    const Z g = from_next(P.t[2] == SC_PERIODIC
                                              ? one_sided(ox, T.row[(size_t)kRowNB * T.row_stride + P.row], robB)
                                              : bnd_y(sB, P.t[2]));
                    if (p.l == 0) A = g;
                }
            }
            bool nanA = false, nanB = false;
            Q FA, GB;
            flux_pair_robust<FLUX>(top_local(A), top_local(B), rob, eos, top_lane(p), nanA, nanB, FA, GB);
            fT = scaled(top_global(FA), C.aT);
            fB = from_prev(scaled(top_global(GB), C.aB));
            bad |= (nanA && out_lane) || (nanB && p.l < kTileJ && p.gv + 1 < p.ny);
        }
    }
    __syncthreads();

    // ---- the faces along i: the face between this row and the next
    Q fR{};
    if (p.w <= TI && p.gu < p.nx) {
        const Z A = (p.gu == -1 && !p.perx) ? get5(ex, XS, p.l) : sR;
        const Z B = get5(ex, XS, x + 64);
        if (p.gu == -1 && !p.perx) robR = wc > 0;
        bool nanA = false, nanB = false;
        Q FA, GB;
        flux_pair_robust<FLUX>(A, B, robR, eos, true, nanA, nanB, FA, GB);
        fR = scaled(FA, R[kRowAR * 64]);
        const Q g = scaled(GB, R[kRowAL * 64]);
        ex[x + 64] = g.r;
        ex[XS + x + 64] = g.mx;
        ex[2 * XS + x + 64] = g.my;
        ex[3 * XS + x + 64] = g.E;
        bad |= out_lane && ((nanA && p.w >= 1) || (nanB && p.w < TI && p.gu + 1 < p.nx));
    }
    __syncthreads();

    // ---- update of the tile's cells, fluxes summed in slot order
    double cand = INFINITY;
    if (out_row && out_lane) {
        Q F{0.0 - ex[x], 0.0 - ex[XS + x], 0.0 - ex[2 * XS + x], 0.0 - ex[3 * XS + x]};
        F = Q{F.r + fR.r, F.mx + fR.mx, F.my + fR.my, F.E + fR.E};
        F = Q{F.r - fB.r, F.mx - fB.mx, F.my - fB.my, F.E - fB.E};
        F = Q{F.r + fT.r, F.mx + fT.mx, F.my + fT.my, F.E + fT.E};
        const Z z0{zs[o], zs[ZS + o], zs[2 * ZS + o], zs[3 * ZS + o], zc.e};
        Q q = to_q(z0);
        const double coef = dt / vol;
        q.r = q.r - coef * F.r;
        q.mx = q.mx - coef * F.mx;
        q.my = q.my - coef * F.my;
        q.E = q.E - coef * F.E;
        Z zn = to_z(q, eos);
        int wn;
        if (is_bad(zn, eos)) {
            zn = z0;
            wn = 3;
            atomicOr(ctl.err, kErrIsolated);
        } else {
            wn = wc > 0 ? wc - 1 : wc;
        }
        store_z(out, c, zn);
        wait_out[c] = wn;
        cand = cell_dt(zn, T.h[c], eos);
    }
    if (bad) *ctl.err = 1;
    tile_min_atomic<NW>(&ctl.dtmin[3 * p.pid + ctl.wr], cand, red);
}

// SmFluid::fluxes, first order (sm_fluid.cpp:127-174), on one tile, plus the
// next step's CFL candidate.
template <int FLUX, int V, int TI>
__device__ __forceinline__ void tile_flux1_body(const TileMesh& T, const DevState& in, const DevState& out,
                                                const Eos& eos, const StepCtl& ctl, int b, double* ex, double* red) {
    constexpr int NW = TI + 2, XS = NW * 64;
    const Place p = place_of<V, TI>(T, b);
    const TileProb P = problem(T, p.pid);
    const double dt = step_dt(ctl, p.pid);
    tile_prologue(ctl, p, dt);
    const int c = p.off + p.gi * p.ny + p.gj;
    const int x = p.w * 64 + p.l;
    const Z zc = load_z(in, c);
    const bool out_row = p.w >= 1 && p.w <= TI && p.gu < p.nx;
    const bool out_lane = p.l >= 1 && p.l <= kTileJ && p.gv < p.ny;
    const TileCol& C = T.col[P.col + p.gi];
    const double vol = T.vol[c];
    const double aL = T.row[(size_t)kRowAL * T.row_stride + P.row + p.gj];
    const double aR = T.row[(size_t)kRowAR * T.row_stride + P.row + p.gj];
    put5(ex, XS, x, zc);
    bool bad = false;
    Q fB{}, fT{}, fR{};
    if (out_row) {   // the top face
        Z A = zc, B = from_next(zc);
        if (!p.pery) {
            if (p.gv == p.ny - 1) B = bnd_y(zc, P.t[3]);
            if (p.gv == -1) A = bnd_y(B, P.t[2]);
        }
        bool nanA = false, nanB = false;
        Q FA, GB;
        flux_pair<FLUX>(top_local(A), top_local(B), eos, top_lane(p), nanA, nanB, FA, GB);
        fT = scaled(top_global(FA), C.aT);
        fB = from_prev(scaled(top_global(GB), C.aB));
        bad |= (nanA && out_lane) || (nanB && p.l < kTileJ && p.gv + 1 < p.ny);
    }
    __syncthreads();
    if (p.w <= TI && p.gu < p.nx) {   // the face between this row and the next
        Z A = zc, B = get5(ex, XS, x + 64);
        if (!p.perx) {
            if (p.gu == p.nx - 1) B = bnd_x(zc, P.t[1]);
            if (p.gu == -1) A = bnd_x(B, P.t[0]);
        }
        bool nanA = false, nanB = false;
        Q FA, GB;
        flux_pair<FLUX>(A, B, eos, true, nanA, nanB, FA, GB);
        fR = scaled(FA, aR);
        const Q g = scaled(GB, aL);
        ex[x + 64] = g.r;
        ex[XS + x + 64] = g.mx;
        ex[2 * XS + x + 64] = g.my;
        ex[3 * XS + x + 64] = g.E;
        bad |= out_lane && ((nanA && p.w >= 1) || (nanB && p.w < TI && p.gu + 1 < p.nx));
    }
    __syncthreads();
    double cand = INFINITY;
    if (out_row && out_lane) {
        Q F{0.0 - ex[x], 0.0 - ex[XS + x], 0.0 - ex[2 * XS + x], 0.0 - ex[3 * XS + x]};
        F = Q{F.r + fR.r, F.mx + fR.mx, F.my + fR.my, F.E + fR.E};
        F = Q{F.r - fB.r, F.mx - fB.mx, F.my - fB.my, F.E - fB.E};
        F = Q{F.r + fT.r, F.mx + fT.mx, F.my + fT.my, F.E + fT.E};
        Q q = to_q(zc);
        const double coef = dt / vol;
        q.r = q.r - coef * F.r;
        q.mx = q.mx - coef * F.mx;
        q.my = q.my - coef * F.my;
        q.E = q.E - coef * F.E;
        const Z zn = to_z(q, eos);
        store_z(out, c, zn);
        cand = cell_dt(zn, T.h[c], eos);
    }
    if (bad) *ctl.err = 1;
    tile_min_atomic<NW>(&ctl.dtmin[3 * p.pid + ctl.wr], cand, red);
}

// Workgroups of (TI + 2) wavefronts; WAVES = the resident waves per SIMD the
// register allocation is sized for.  One workgroup per tile, dealt to the
// XCDs in contiguous ranges of tiles (xcd_block).
template <int FLUX, int LIM, int V, int TI, int WAVES>
__global__ void __launch_bounds__((TI + 2) * 64) __attribute__((amdgpu_waves_per_eu(WAVES)))
k_tile_step(TileMesh T, DevState in, DevState out, const int* __restrict__ wait_in, int* __restrict__ wait_out,
            Eos eos, StepCtl ctl) {
    ZFV_TILE_LDS(TI);
    tile_body<FLUX, LIM, V, TI>(T, in, out, wait_in, wait_out, eos, ctl,
                                xcd_block((int)blockIdx.x, (int)gridDim.x), zs, ex, rt, ws, red);
}

// The same step by persistent workgroups: the grid is the number of
// workgroups the GPU holds at once (a multiple of 8), and workgroup g, on
// XCD g % 8 (workgroups are dealt to the XCDs round-robin), walks the tiles
// of that XCD's contiguous range (the ranges of xcd_block) with a stride of
// the XCD's workgroup count.  Every workgroup leaves after its last tile.
template <int FLUX, int LIM, int V, int TI, int WAVES>
__global__ void __launch_bounds__((TI + 2) * 64) __attribute__((amdgpu_waves_per_eu(WAVES)))
k_tile_step_p(TileMesh T, DevState in, DevState out, const int* __restrict__ wait_in, int* __restrict__ wait_out,
              Eos eos, StepCtl ctl) {
    ZFV_TILE_LDS(TI);
    const int n = T.n_tiles[V];
    const int g = (int)blockIdx.x, x = g & 7, wgs = (int)gridDim.x >> 3;
    const int q = n >> 3, rem = n & 7;
    const int begin = x * q + (x < rem ? x : rem), end = begin + q + (x < rem ? 1 : 0);
    for (int b = begin + (g >> 3); b < end; b += wgs) {
        tile_body<FLUX, LIM, V, TI>(T, in, out, wait_in, wait_out, eos, ctl, b, zs, ex, rt, ws, red);
        __syncthreads();   // the next tile's loads overwrite the LDS boxes
    }
}

template <int FLUX, int V, int TI>
__global__ void __launch_bounds__((TI + 2) * 64) __attribute__((amdgpu_waves_per_eu(4))) k_tile_flux1(TileMesh T, DevState in, DevState out, Eos eos,
                                                             StepCtl ctl) {
    __shared__ double ex[5 * (TI + 2) * 64];
    __shared__ double red[TI + 2];
    tile_flux1_body<FLUX, V, TI>(T, in, out, eos, ctl, xcd_block((int)blockIdx.x, (int)gridDim.x), ex, red);
}

// Workgroups the GPU holds at once for a persistent tiled-step kernel
// (a multiple of 8, at least 8).
template <int FLUX, int LIM, int V, int TI, int WAVES>
static hipError_t resident_grid(int* grid) {
    static int per_cu = 0;   // one value per kernel instance
    if (per_cu == 0) {
        int nb = 0;
        hipError_t e = hipOccupancyMaxActiveBlocksPerMultiprocessor(&nb, k_tile_step_p<FLUX, LIM, V, TI, WAVES>,
                                                                    (TI + 2) * 64, 0);
        if (e != hipSuccess) return e;
        per_cu = nb > 0 ? nb : 1;
    }
    int dev = 0, cus = 0;
    hipError_t e = hipGetDevice(&dev);
    if (e == hipSuccess) e = hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev);
    if (e != hipSuccess) return e;
    *grid = std::max(8, (per_cu * cus) / 8 * 8);
    return hipSuccess;
}

template <int FLUX, int V, int TI, int WAVES>
static hipError_t launch_tile_t(int limiter, bool persistent, const TileMesh& T, const DevState& in,
                                const DevState& out, const int* wait_in, int* wait_out, const Eos& eos,
                                const StepCtl& ctl, hipStream_t s) {
    const dim3 b((TI + 2) * 64);
    dim3 g(T.n_tiles[V]);
#define ZFV_TILE(L)                                                                                              \
    do {                                                                                                         \
        if constexpr (FLUX == 3) {                                                                               \
            if (persistent) {                                                                                    \
                int grid = 0;                                                                                    \
                const hipError_t e = resident_grid<FLUX, L, V, TI, WAVES>(&grid);                                \
                if (e != hipSuccess) return e;                                                                   \
                hipLaunchKernelGGL((k_tile_step_p<FLUX, L, V, TI, WAVES>), dim3(grid), b, 0, s, T, in, out,      \
                                   wait_in, wait_out, eos, ctl);                                                 \
                break;                                                                                           \
            }                                                                                                    \
        }                                                                                                        \
        hipLaunchKernelGGL((k_tile_step<FLUX, L, V, TI, WAVES>), g, b, 0, s, T, in, out, wait_in, wait_out, eos, \
                           ctl);                                                                                 \
    } while (0)
    switch (limiter) {
        case 0: ZFV_TILE(0); break;
        case 1: ZFV_TILE(1); break;
        case 2: ZFV_TILE(2); break;
        case 3: ZFV_TILE(3); break;
        case 4: ZFV_TILE(4); break;
        case 5: ZFV_TILE(5); break;
        case 6: ZFV_TILE(6); break;
        case 7: ZFV_TILE(7); break;
        case 8: ZFV_TILE(8); break;
        case 9: ZFV_TILE(9); break;
        case 10: ZFV_TILE(10); break;
        case 11: ZFV_TILE(11); break;
        default: ZFV_TILE(12); break;
    }
#undef ZFV_TILE
    return hipGetLastError();
}

// Tile shapes: 6 rows at 4 waves per SIMD (two workgroups per CU), 10 rows
// at 3 (one workgroup), 14 rows at 4 (one workgroup), 2 rows at 4.
template <int FLUX>
static hipError_t launch_tile_flux(int limiter, int variant, bool persistent, const TileMesh& T, const DevState& in,
                                   const DevState& out, const int* wait_in, int* wait_out, const Eos& eos,
                                   const StepCtl& ctl, hipStream_t s) {
    static_assert(kTileRows[0] == 6 && kTileRows[1] == 10 && kTileRows[2] == 14 && kTileRows[3] == 2, "tile shapes");
    switch (variant) {
        case 0: return launch_tile_t<FLUX, 0, 6, 4>(limiter, persistent, T, in, out, wait_in, wait_out, eos, ctl, s);
        case 1: return launch_tile_t<FLUX, 1, 10, 3>(limiter, persistent, T, in, out, wait_in, wait_out, eos, ctl, s);
        case 2: return launch_tile_t<FLUX, 2, 14, 4>(limiter, persistent, T, in, out, wait_in, wait_out, eos, ctl, s);
        default: return launch_tile_t<FLUX, 3, 2, 4>(limiter, persistent, T, in, out, wait_in, wait_out, eos, ctl, s);
    }
}

}  // namespace zfv
