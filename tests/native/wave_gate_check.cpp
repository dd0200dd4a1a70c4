// Checks the condition under which the wave kernel forms the dissipation's
// quotients from reciprocals (no_subnormal of xbg_math.h): for <n> random cells
// (seed) that pass it, no quotient is subnormal and each equals the IEEE one.
// Cells lie over and beyond the condition's limits, bins near its smallest.
// Prints the cells that passed and the faults; exits non-zero on a fault.
#include <cmath>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <random>

#include "../../xbeach_gpu_amd/csrc/xbg_math.h"

static uint32_t bf(float f) { uint32_t u; std::memcpy(&u, &f, 4); return u; }
static bool same(float x, float y) { return (x != x && y != y) || bf(x) == bf(y); }

int main(int argc, char** argv) {
    if (argc < 3) return 2;
    const long n = std::atol(argv[1]);
    std::mt19937_64 g(std::strtoull(argv[2], nullptr, 10));
    auto uni = [&](double a, double b) { return a + (b - a) * (double)(g() >> 11) / 9007199254740992.0; };
    auto lg = [&](double a, double b) { return (float)std::exp(uni(std::log(a), std::log(b))); };
    long passed = 0, capped = 0, bad = 0;
    for (long i = 0; i < n; i++) {
        const float c = g() % 4 ? lg(0.05, 40.0) : lg(0.9e-10, 1.1e10);
        const float E = g() % 3 ? lg(1e-7, 1e8) : 1e-7f;
        const float D = g() % 8 ? (float)(E * lg(0.9 * 9.3e-10, 1e3)) : 0.0f;
        const float gb = g() % 8 ? (float)(c * lg(0.9e-5, 1e2)) : 0.0f;
        const float idiv = g() % 3 ? lg(1.0, 1.1e6) : 1.0f;
        const float lim = 8.1e-28f * (g() % 2 ? idiv : 1.0f);
        float e[4], r[4];
        uint32_t m = 0xffffffffu;
        for (int k = 0; k < 4; k++) {
            e[k] = g() % 8 ? lim * lg(0.999, g() % 2 ? 4.0 : 1e30) : 0.0f;
            r[k] = g() % 8 ? lim * lg(0.999, g() % 2 ? 4.0 : 1e30) : 0.0f;
            m = xm::nonzero_min(xm::nonzero_min(m, e[k]), r[k]);
        }
        if (!xm::no_subnormal(c, D, E, gb, idiv, m)) continue;
        passed++;
        if (idiv > 64.0f) capped++;
        const double rE = 1.0 / (double)E, c0 = c, rc = 1.0 / c0, hc = 0.5 * rc;
        for (int k = 0; k < 4; k++) {
            const float p = (idiv != 1.0f ? e[k] / idiv : e[k]) * D, q = p / E;
            const float t = (float)uni(-3.2, 3.2), cx = c * xm::cosf(t), cy = c * xm::sinf(t), s2 = cx * cx + cy * cy;
            const float num = gb * r[k], u = num / std::sqrt(s2);
            if (std::fpclassify(q) == FP_SUBNORMAL || !same(xm::div_by(p, rE), q)) bad++;
            if (std::fpclassify(u) == FP_SUBNORMAL || !same(xm::div_near(num, xm::sqrt_near(s2, c0, hc), rc), u)) bad++;
        }
    }
    std::printf("passed %ld of %ld cells, %ld capped by more than 64, faults %ld\n", passed, n, capped, bad);
    return bad || passed * 100 < n || capped * 1000 < n ? 1 : 0;
}
