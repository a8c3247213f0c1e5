/*
 * The correctly rounded sin, cos and acos of voxelyze_amd/csrc/vx_math.h against binary128
 * (libquadmath) rounded once, on the host: over the ranges the step meets, next to multiples of
 * pi/2, and at acos's ends.  Also the short series' distance from the exact value, which has to
 * stay inside the interval its rounding test assumes.  Prints "0 failures" and exits 0.
 */
#include <cmath>
#include <cstdio>
#include <random>

#include <quadmath.h>

#include "../../voxelyze_amd/csrc/vx_math.h"

using namespace vx;

static long bad = 0;
static double worst = 0;
static std::mt19937_64 rng(11);
static double U(double a, double b) { return std::uniform_real_distribution<double>(a, b)(rng); }

static void angle(double x) {
    const double s = (double)sinq(x), c = (double)cosq(x);
    double s1, c1;
    cr_sincos(x, &s1, &c1);
    if (s1 != s || c1 != c || cr_sin(x) != s) {
        if (bad++ < 10) printf("sin/cos of %a\n", x);
    }
    const double kq = rint(x * (1.0 / VX_PIO2_HI));
    const dd r = dd_reduce(x, kq);
    if (std::fabs(r.hi) < 0x1p-24) return;
    for (int cosine = 0; cosine < 2; cosine++) {
        const dd v = dd_short_series(r, cosine);
        const bool asCos = (((int)kq & 1) != 0) != (cosine != 0);
        const __float128 e = fabsq(asCos ? cosq(x) : sinq(x)), g = fabsq((__float128)v.hi + v.lo);
        worst = std::fmax(worst, (double)fabsq((g - e) / e));
    }
}
static void cosine(double w) {
    if (w <= -1.0 || w >= 1.0) return;
    if (cr_acos(w) != (double)acosq(w) && bad++ < 10) printf("acos of %a\n", w);
}

int main() {
    for (int i = 0; i < 200000; i++) {
        angle(U(-2.0, 2.0));
        angle(std::exp(U(-20.0, 0.0)));
        angle(U(-1e6, 1e6));
        angle(std::floor(U(0.0, 5000.0)) * M_PI_2 * (1 + U(-1e-9, 1e-9)));
        cosine(U(-1.0, 1.0));
        cosine(1.0 - std::exp(U(-30.0, 0.0)));
        cosine(-1.0 + std::exp(U(-30.0, 0.0)));
        cosine(std::cos(U(0.0, 0.3)));
    }
    for (int k = -8; k <= 8; k++)
        for (int d = -3; d <= 3; d++) angle(k * M_PI_2 + d * 2e-16);
    if (worst > 0.5 * VX_ZIV) bad++;
    printf("short series within 2^%.1f, rounding test at 2^%.0f\n%ld failures\n", std::log2(worst), std::log2(VX_ZIV), bad);
    return bad ? 1 : 0;
}
