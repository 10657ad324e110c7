// rare_range (rare_bound.h): the sums of random candidates, in 64 bits, lie in the range that their codes give.
#include <cstdio>
#include <random>

#include "../../thundergbm_amd/csrc/rare_bound.h"

using namespace tgbm;

int main() {
    std::mt19937_64 rng(1);
    auto uniform = [&](double a, double b) { return std::uniform_real_distribution<double>(a, b)(rng); };
    long outside = 0, trials = 0;
    for (int t = 0; t < 60000; ++t) {
        const int kind = t % 5, n = (int)std::exp(uniform(0, std::log(4096.0)));
        const float gq = (float)std::rint(std::exp2(uniform(0, 50))), hq = (float)std::rint(std::exp2(uniform(0, 50)));
        const float inv = (float)std::exp2(-std::floor(uniform(0, 40)));
        const RareBound u{gq * inv / kRareSteps, hq * inv / kRareSteps, 0, 0};
        RareCell whole{0, 0}, part{0, 0};
        double g_min = 0, g_max = 0, h_min = 0, h_max = 0;
        const int in_part = kind == 0 ? 0 : (int)uniform(0, n);
        const double step = std::floor(uniform(0, 1023)) / kRareSteps;
        for (int i = 0; i < n; ++i) {
            // just above a step, so that every code is off by nearly one; of one sign, of two, or spread
            double x = kind <= 1 ? std::min(1.0, step + 1e-6) : kind == 2 ? step : uniform(0, 1);
            if (kind >= 3 && uniform(0, 1) < 0.5) x = -x;
            if (kind == 1 && t % 2) x = -x;
            const float g = (float)std::rint(x * gq), h = (float)std::rint((kind <= 2 ? 1 - step : uniform(0, 1)) * hq);
            const unsigned w = rare_word(5, g, h, gq, hq);
            const RareCell c{rare_addend(w), w >> 22};
            const bool p = i < in_part;
            (p ? part : whole) = (p ? part : whole) + c;
            const double sg = (double)g * inv, sh = (double)h * inv;
            g_min += p ? std::min(0.0, sg) : sg;
            g_max += p ? std::max(0.0, sg) : sg;
            h_min += p ? 0 : sh;
            h_max += sh;
        }
        const RareRange r = rare_range(whole, part, u);
        ++trials;
        if (!(r.g_min <= g_min && g_max <= r.g_max && r.h_min <= h_min && h_max <= r.h_max)) {
            if (++outside <= 5)
                std::printf("kind %d, %d values: g [%.9g, %.9g] in [%.9g, %.9g], h [%.9g, %.9g] in [%.9g, %.9g]\n", kind, n, g_min,
                            g_max, r.g_min, r.g_max, h_min, h_max, r.h_min, r.h_max);
        }
    }
    std::printf("%ld of %ld outside\n", outside, trials);
    return outside != 0;
}
