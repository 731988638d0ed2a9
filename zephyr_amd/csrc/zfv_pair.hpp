// A face's numerical flux seen from both of its cells, for the tiled kernels:
// the reference evaluates every inner face twice, from cell A with the normal
// towards B and from B with the opposite normal (sm_fluid.cpp:137-161), and
// the two results differ in the last bits (HLLC's S_C numerator and its star
// terms are summed in another order), so one flux with both signs would not
// give the reference's values.  Reversing the normal negates both velocity
// components of the face frame; negation is exact, so of the second
// evaluation only the sums whose order changes have to be made again: the
// sound speeds, energies, physical fluxes, wave-speed bounds and p / a of the
// two sides are shared.  An HLLC face is then 12 divisions and square roots
// instead of 18.
#pragma once

#include "zfv_physics.hpp"

namespace zfv {

__device__ __forceinline__ Z mirrored(const Z& z) { return Z{z.r, -z.u, -z.v, z.p, z.e}; }
__device__ __forceinline__ Q mirrored(const Q& f) { return Q{-f.r, f.mx, f.my, -f.E}; }

// A and B in the frame of A's side.  FA: A's flux, as flux(A, B).  GB: B's
// flux, flux(mirrored(B), mirrored(A)), mirrored back into A's frame, so that
// B's sum takes -GB where A's takes +FA.  odd: a wave-speed bound is NaN; min
// and max keep their first argument, which is the other cell's for B, so its
// bounds are not A's negated ones and GB does not hold.
__device__ __forceinline__ void flux_hllc_both(const Z& A, const Z& B, const Eos& eos, bool& nanA, bool& nanB, Q& FA,
                                               Q& GB, bool& odd) {
    const double cA = eos_c(eos, A.r, A.p);
    const double cB = eos_c(eos, B.r, B.p);
    const double lA = A.u - cA, lB = B.u - cB, hA = A.u + cA, hB = B.u + cB;
    const double SL = smin(lA, lB);
    const double SR = smax(hA, hB);
    odd = __builtin_isunordered(lA, lB) | __builtin_isunordered(hA, hB);
    const double eA = A.e + 0.5 * vsq(A), eB = B.e + 0.5 * vsq(B);
    const double ruA = A.r * A.u, ruB = B.r * B.u;
    const double EA = A.r * eA, EB = B.r * eB;
    const Q fA{ruA, ruA * A.u + A.p, ruA * A.v, (EA + A.p) * A.u};
    const Q fB{ruB, ruB * B.u + B.p, ruB * B.v, (EB + B.p) * B.u};
    if (!(SL >= 0.0) && !(SR <= 0.0)) {
        const double aL = A.r * (SL - A.u);
        const double aR = B.r * (SR - B.u);
        const double den = aR - aL;
        const double pa = A.p / aL, pb = B.p / aR;
        const double rvA = A.r * A.v, rvB = B.r * B.v;
        const Q f{fA.r + fB.r, fA.mx + fB.mx, fA.my + fB.my, fA.E + fB.E};
        {
            const double SC = (A.p - B.p + aR * B.u - aL * A.u) / den;
            const double rsL = aL / (SL - SC);
            const double rsR = aR / (SR - SC);
            const double EsL = eA + (SC - A.u) * (SC + pa);
            const double EsR = eB + (SC - B.u) * (SC + pb);
            const double a = fabs(SC);
            auto sum = [&](double t, double sL, double qL, double sR, double qR) {
                t = t + SL * (sL - qL);
                t = t + a * (sL - sR);
                t = t + SR * (sR - qR);
                return 0.5 * t;
            };
            FA.r = sum(f.r, rsL, A.r, rsR, B.r);
            FA.mx = sum(f.mx, rsL * SC, ruA, rsR * SC, ruB);
            FA.my = sum(f.my, rsL * A.v, rvA, rsR * B.v, rvB);
            FA.E = sum(f.E, rsL * EsL, EA, rsR * EsR, EB);
            nanA |= isnan(FA.r) | isnan(FA.mx) | isnan(FA.my) | isnan(FA.E);
        }
        {
            // B's frame: left state B with velocity -u, bounds -SR and -SL,
            // a_L = -aR, a_R = -aL; the stars keep their side's letter
            const double SC = (B.p - A.p + aL * A.u - aR * B.u) / den;
            const double rsR = aR / (SR + SC);
            const double rsL = aL / (SL + SC);
            const double EsR = eB + (SC + B.u) * (SC - pb);
            const double EsL = eA + (SC + A.u) * (SC - pa);
            const double a = fabs(SC);
            auto sum = [&](double t, double sR, double qR, double sL, double qL) {
                t = t + SR * (sR - qR);
                t = t - a * (sR - sL);
                t = t + SL * (sL - qL);
                return 0.5 * t;
            };
            GB.r = sum(f.r, rsR, B.r, rsL, A.r);
            GB.my = sum(f.my, rsR * B.v, rvB, rsL * A.v, rvA);
            GB.E = sum(f.E, rsR * EsR, EB, rsL * EsL, EA);
            const double mR = rsR * SC, mL = rsL * SC;
            double t = f.mx - SR * (mR + ruB);
            t = t + a * (mR - mL);
            t = t - SL * (mL + ruA);
            GB.mx = 0.5 * t;
            nanB |= isnan(GB.r) | isnan(GB.mx) | isnan(GB.my) | isnan(GB.E);
        }
    } else {   // B's bounds are -SR and -SL; it tests its own left bound (-SR) first
        FA = SL >= 0.0 ? fA : fB;
        GB = SR <= 0.0 ? fB : fA;
    }
}

// flux_hllc_both, and where GB does not hold the evaluation from B's side, by
// the same code once more with the sides exchanged.  live: the lane's face is
// used.  A lane without a face may hold no state (lane shifts leave zeros, whose
// sound speed is NaN); were it asked, every wavefront would evaluate twice
// (1361 x 1023, HLLC and MC 162 us for 153; HLL, first order, 63 for 58).
__device__ __forceinline__ void flux_hllc_pair(const Z& A, const Z& B, const Eos& eos, bool live, bool& nanA,
                                               bool& nanB, Q& FA, Q& GB) {
    Z L = A, R = B;
    bool odd = false;
    for (int side = 0; side < 2; ++side) {
        Q fa, gb;
        bool nA = false, nB = false, o;
        flux_hllc_both(L, R, eos, nA, nB, fa, gb, o);
        if (side == 0) {
            FA = fa;
            GB = gb;
            nanA = nA;
            nanB = nB;
            odd = o & live;
            if (__builtin_expect(!__any(odd), 1)) return;
            L = mirrored(B);
            R = mirrored(A);
        } else if (odd) {
            GB = mirrored(fa);
            nanB = nA;
        }
    }
}

// HLL and Rusanov evaluated once.  From B's side the bounds are A's negated and
// exchanged, so each sum holds the same products, as x - y for y - x: its
// rounded value is A's, negated, and GB = FA.  Not so where a wave speed is
// NaN (`odd` above); there B's side is evaluated.
template <int FLUX>
__device__ __forceinline__ void flux_even_pair(const Z& A, const Z& B, const Eos& eos, bool live, bool& nanA,
                                               bool& nanB, Q& FA, Q& GB) {
    const double cA = eos_c(eos, A.r, A.p), cB = eos_c(eos, B.r, B.p);
    const bool odd =
        live & (__builtin_isunordered(A.u - cA, B.u - cB) | __builtin_isunordered(A.u + cA, B.u + cB));
    FA = num_flux<FLUX>(A, B, eos, nanA);
    GB = FA;
    nanB = nanA;
    if (__builtin_expect(__any(odd), 0)) {
        bool n = false;
        const Q g = mirrored(num_flux<FLUX>(mirrored(B), mirrored(A), eos, n));
        if (odd) {
            GB = g;
            nanB = n;
        }
    }
}

template <int FLUX>
__device__ __forceinline__ void flux_pair(const Z& A, const Z& B, const Eos& eos, bool live, bool& nanA, bool& nanB,
                                          Q& FA, Q& GB) {
    static_assert(FLUX >= 1 && FLUX <= 3, "Rusanov, HLL, HLLC");
    nanA = nanB = false;
    if constexpr (FLUX == 3) flux_hllc_pair(A, B, eos, live, nanA, nanB, FA, GB);
    else flux_even_pair<FLUX>(A, B, eos, live, nanA, nanB, FA, GB);
}

// The same with the isolation mode's HLL flux on `robust` lanes.
template <int FLUX>
__device__ __forceinline__ void flux_pair_robust(const Z& A, const Z& B, bool robust, const Eos& eos, bool live,
                                                 bool& nanA, bool& nanB, Q& FA, Q& GB) {
    bool nA = false, nB = false;
    flux_pair<FLUX>(A, B, eos, live, nA, nB, FA, GB);
    if constexpr (FLUX != 2) {
        if (__builtin_expect(__any(robust), 0)) {
            bool mA = false, mB = false;
            Q fa, gb;
            flux_pair<2>(A, B, eos, live, mA, mB, fa, gb);
            if (robust) {
                FA = fa;
                GB = gb;
                nA = mA;
                nB = mB;
            }
        }
    }
    nanA |= nA;
    nanB |= nB;
}

}  // namespace zfv
