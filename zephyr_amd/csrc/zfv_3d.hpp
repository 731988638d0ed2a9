// Device views of a three-dimensional Cuboid mesh and its SmFluid state,
// shared by the 3D kernels (zfv_3d.hip) and their host side (zfv_3d.cpp).
#pragma once

#include <hip/hip_runtime.h>

#include "zfv_physics.hpp"

namespace zfv {

// n cells; six face slots per cell (sides L, R, B, T, Z, F), slot s of cell
// c at s * stride + c.  type: SlotCode; adj: the neighbour (the cell itself
// on a non-periodic boundary); w: the least-squares weight of the slot.
struct Dev3Mesh {
    int n, stride;
    // A Cuboid's geometry as 1D tables (tnx > 0): every offset between cell and
    // face centres and every least-squares weight depends on one index only,
    // so the kernels read tables of nx + ny + nz entries instead of the slot
    // arrays (which the host compared with them bit for bit).  Six rows of
    // L = tnx + tny + tnz pairs, lower and upper side; entry base(a) + index_a,
    // base = 0, tnx, tnx + tny.  Row m < 3: component a of the centres of sides
    // 2 m and 2 m + 1 less the cell's.  For sides 2 a and 2 a + 1, row 3: the same
    // less the centre across (the cell's own on a boundary, its mirror point
    // on a periodic side); row 4: the centre across (the mirror point on any
    // edge) less the cell's; row 5: the weights.  area1, vol1: of every cell.
    // bcodes: the slot code of side s at the edge in bits 4 s to 4 s + 3 (an
    // array would go through scratch where s is a loop's index); per: bit a,
    // a periodic direction.
    int tnx, tny, tnz;
    const double2* tab;
    double area1[6], vol1;
    int bcodes, per;
    const double *cx, *cy, *cz, *vol, *h;
    const int *type, *adj;
    const double *fcx, *fcy, *fcz, *area, *w;
};

// Primitive state: the pairs (rho, u), (v, w) and (p, e), one array of n pairs
// each.  A load of 16 bytes a lane takes the L1 cache no longer than one of 8, and
// the step kernels are bound by it: 96^3 cells, HLLC and MC, 174 us with one array
// of doubles a field.
struct Dev3State {
    double2* q;
    int n;
};

// The predictor's record of a cell, kRecPairs arrays of n pairs: doubles 0 to 5
// hold the half state, 6 + 5 a + k the derivative of field k along axis a, 21
// the isolation counter.
constexpr int kRecPairs = 11;

// Step control, three rotating CFL slots of kSlotWords words (the bits of
// positive doubles, reduced with atomicMin): dtmin is the slot this step reads; the stage
// that ends a step reduces the new state's h / (|v| + c) into `next`, the
// slot the following step reads, and sets `reset`, the slot the previous
// step read, back to the largest finite double.
struct Dev3Ctl {
    unsigned long long* dtmin;
    unsigned long long* next;
    unsigned long long* reset;
    double cfl, max_dt;
    double* dt_out;
    int* err;
};

constexpr unsigned long long kDblMaxBits = 0x7fefffffffffffffULL;
// A CFL slot is kSubSlots partial minima, kSubStride words (128 bytes) apart,
// so that the workgroups' atomics spread over as many cache lines; the
// slot's value is their least.
constexpr int kSubSlots = 64;
constexpr int kSubStride = 16;
constexpr int kSlotWords = kSubSlots * kSubStride;

// The number of pairs of a Cuboid's geometry tables.
inline size_t tab3_size(int nx, int ny, int nz) { return 6 * (size_t)(nx + ny + nz); }

hipError_t launch3_dt(const Dev3Mesh& M, const Dev3State& z, const Eos& eos, unsigned long long* slot,
                      hipStream_t s);
hipError_t launch3_flux1(int flux, const Dev3Mesh& M, const Dev3State& in, const Dev3State& out, const Eos& eos,
                         const Dev3Ctl& ctl, hipStream_t s);
hipError_t launch3_grad_pred(int limiter, const Dev3Mesh& M, const Dev3State& in, double2* R, const int* wait,
                             const Eos& eos, const Dev3Ctl& ctl, hipStream_t s);
hipError_t launch3_corr(int flux, const Dev3Mesh& M, const Dev3State& init, const double2* R, int* wait_out,
                        const Dev3State& next, const Eos& eos, const Dev3Ctl& ctl, hipStream_t s);
hipError_t launch3_rows(const double2* q, int n, int c0, int len, int m0, int count, double* out, hipStream_t s);
hipError_t launch3_pack(const double* in, const Dev3State& z, int c0, int len, hipStream_t s);
hipError_t launch3_totals(const Dev3Mesh& M, const Dev3State& z, double* partial, int nblocks, hipStream_t s);

}  // namespace zfv
