// A face's flux from both of its cells (zfv_pair.hpp) on the host: flux_pair's GB
// against the second evaluation it stands for, value for value, and how often a
// wavefront is asked for that second evaluation.
#include <cstdint>
#include <cstdio>
#include <initializer_list>
#include <limits>

static int asked = 0;   // lanes that asked a wavefront to evaluate again
static bool __any(bool b) {
    asked += b;
    return b;
}
#include "hip/hip_runtime.h"
#include "zfv_pair.hpp"

using namespace zfv;

static uint64_t seed = 1;
static double uniform() {
    seed = seed * 6364136223846793005ULL + 1442695040888963407ULL;
    return (double)(seed >> 11) / 9007199254740992.0;
}
static bool same(double a, double b) { return a == b || (a != a && b != b); }
static bool same(const Q& a, const Q& b) {
    return same(a.r, b.r) && same(a.mx, b.mx) && same(a.my, b.my) && same(a.E, b.E);
}

static int failures = 0;

template <int FLUX>
static void check(const Z& A, const Z& B, const Eos& eos, bool live) {
    bool nA = false, nB = false, mA = false, mB = false;
    Q FA, GB;
    flux_pair<FLUX>(A, B, eos, live, nA, nB, FA, GB);
    const Q fA = num_flux<FLUX>(A, B, eos, mA);
    const Q gB = mirrored(num_flux<FLUX>(mirrored(B), mirrored(A), eos, mB));
    if (!same(FA, fA) || nA != mA || !same(GB, gB) || nB != mB) {
        if (failures++ < 5)
            printf("flux %d: A %g %g %g %g %g B %g %g %g %g %g\n", FLUX, A.r, A.u, A.v, A.p, A.e, B.r, B.u, B.v, B.p,
                   B.e);
    }
}

template <int FLUX>
static void run() {
    const Eos eos{1.4, 0.0, 0.0};
    const double odd[] = {0.0, -0.0, 1e-310, 1e300, -1.0, std::numeric_limits<double>::infinity(),
                          -std::numeric_limits<double>::infinity(), std::numeric_limits<double>::quiet_NaN()};
    auto state = [&](double speed) {
        Z z{0.1 + uniform(), speed * (uniform() - 0.5), uniform() - 0.5, 0.1 + uniform(), 0.0};
        z.e = z.p / (0.4 * z.r);
        return z;
    };
    for (int k = 0; k < 200000; ++k) {
        const double speed = k % 3 == 0 ? 0.5 : (k % 3 == 1 ? 4.0 : 20.0);
        const Z A = state(speed), B = state(speed);
        asked = 0;
        check<FLUX>(A, B, eos, true);
        if (asked) {
            ++failures;
            printf("flux %d: a state asked for a second evaluation\n", FLUX);
        }
    }
    for (int k = 0; k < 20000; ++k) {   // no states: the second evaluation where a wave speed is NaN
        Z z[2] = {state(1.0), state(1.0)};
        double* const f[5] = {&z[k & 1].r, &z[k & 1].u, &z[k & 1].v, &z[k & 1].p, &z[k & 1].e};
        *f[(k >> 1) % 5] = odd[(k / 10) % 8];
        if (k % 7 == 0) z[1 - (k & 1)].r = odd[(k / 80) % 8];
        check<FLUX>(z[0], z[1], eos, true);
    }
    // a lane without a face does not ask, one with a face does
    for (const bool live : {false, true}) {
        bool nA, nB;
        Q FA, GB;
        asked = 0;
        flux_pair<FLUX>(state(1.0), Z{0.0, 0.0, 0.0, 0.0, 0.0}, eos, live, nA, nB, FA, GB);
        if ((asked != 0) != live) {
            ++failures;
            printf("flux %d: zeros in a lane %s a face: asked %d\n", FLUX, live ? "with" : "without", asked);
        }
    }
}

int main() {
    run<1>();
    run<2>();
    run<3>();
    printf("failures: %d\n", failures);
    return failures != 0;
}
