// Checks the correctly rounded operations of xbg_math.h that the wave kernel
// uses for its per-bin square root and divisions against the IEEE operations.
//   near <n> <seed>   n random c: sqrt_near for every float s within 40 ulp of
//                     c*c and for the squares the kernel forms, div_near for
//                     random and edge numerators over those square roots
//   by <n> <seed>     n random divisors, div_by for random and edge numerators
// Subnormal quotients are left out, as the kernel forms them by a division;
// that no quotient which should be subnormal comes out otherwise is checked.
// Prints "mismatches N" and exits non-zero on a mismatch.
#include <cmath>
#include <cstdint>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <random>

#include "../../xbeach_gpu_amd/csrc/xbg_math.h"

static float fb(uint32_t u) { float f; std::memcpy(&f, &u, 4); return f; }
static uint32_t bf(float f) { uint32_t u; std::memcpy(&u, &f, 4); return u; }
static bool same(float x, float y) { return (x != x && y != y) || bf(x) == bf(y); }
static bool sub(float x) { return std::fpclassify(x) == FP_SUBNORMAL; }
// the kernel's division: the fast form, the operation where it is subnormal
static bool ok(float fast, float exact) { return sub(fast) || same(fast, exact); }

int main(int argc, char** argv) {
    if (argc < 4) return 2;
    const long n = std::atol(argv[2]);
    std::mt19937_64 g(std::strtoull(argv[3], nullptr, 10));
    auto uni = [&](double a, double b) { return a + (b - a) * (double)(g() >> 11) / 9007199254740992.0; };
    auto edge = [&](int k) {
        const float e[] = {0.0f, -0.0f, fb(1), fb(0x007fffff), fb(0x00800000), fb(0x7f7fffff), INFINITY, NAN, 1.0f, 1e-30f};
        return e[k % 10];
    };
    long bad = 0;
    if (!std::strcmp(argv[1], "near")) {
        for (long i = 0; i < n; i++) {
            const float c = (float)(i % 3 ? std::exp(uni(std::log(0.05), std::log(40.0)))
                                          : std::exp(uni(std::log(1.01e-10), std::log(0.99e10))));
            const double c0 = c, rc = 1.0 / c0, hc = 0.5 * rc;
            auto check = [&](float s) {
                const float q = std::sqrt(s), qn = xm::sqrt_near(s, c0, hc);
                if (!same(q, qn)) bad++;
                for (int k = 0; k < 4; k++) {
                    const float a = k == 0 ? edge((int)(g() % 10)) : fb((uint32_t)(g() >> 32));
                    if (!ok(xm::div_near(a, q, rc), a / q)) bad++;
                }
            };
            const float s0 = c * c;
            for (int u = -40; u <= 40; u++) check(fb(bf(s0) + u));
            for (int k = 0; k < 8; k++) {
                const float t = (float)uni(-3.2, 3.2), cx = c * xm::cosf(t), cy = c * xm::sinf(t);
                check(cx * cx + cy * cy);
            }
        }
    } else {
        for (long i = 0; i < n; i++) {
            const float b = (float)(i % 2 ? std::exp(uni(std::log(1e-7), std::log(1e38))) : std::exp(uni(std::log(1e-3), std::log(1e5))));
            const double rb = 1.0 / (double)b;
            for (int k = 0; k < 200; k++) {
                // random bits, edges, and numerators whose quotient is near a midpoint or subnormal
                const float a = k < 100 ? fb((uint32_t)(g() >> 32))
                                : k < 110 ? edge(k)
                                : k < 160 ? b * fb((bf(1.0f) & 0xff800000u) | (uint32_t)(g() & 0x7fffff))
                                          : (float)((double)b * (double)fb((uint32_t)(g() % 0x01000000)));
                if (!ok(xm::div_by(a, rb), a / b)) bad++;
            }
        }
    }
    std::printf("mismatches %ld\n", bad);
    return bad ? 1 : 0;
}
