// Prints a hash over the bits of the elementary functions of xbg_math.h at many
// arguments: the same for any way in which their multiply-adds are compiled.
#include <cmath>
#include <cstdint>
#include <cstdio>
#include <cstring>

#include "../../xbeach_gpu_amd/csrc/xbg_math.h"

int main() {
    uint64_t h = 1469598103934665603ull, s = 88172645463325252ull;
    auto add = [&](double v) {
        uint64_t b;
        if (v != v) v = NAN;
        std::memcpy(&b, &v, 8);
        h = (h ^ (b & 0x7fffffffffffffffull ? b : 0)) * 1099511628211ull;
    };
    for (int i = 0; i < 400000; i++) {
        s ^= s << 13;
        s ^= s >> 7;
        s ^= s << 17;
        const double u = (double)(s >> 11) / 9007199254740992.0, x = (u - 0.5) * (i % 2 ? 80.0 : 4.0);
        add(xm::exp(x));
        add(xm::sinh(x));
        add(xm::tanh(x));
        add(xm::sin(x));
        add(xm::cos(x));
        add(xm::log(std::fabs(x) + 1e-30));
        add(xm::pow(std::fabs(x) + 1e-6, 1.2));
        const float c = (float)(0.1 + 30.0 * u), q = c * (1.0f + 1e-7f);
        add(xm::sqrt_near(c * c, c, 0.5 / c));
        add(xm::div_near((float)x, q, 1.0 / c));
    }
    std::printf("%016llx\n", (unsigned long long)h);
}
