// Host-side check of steps.h's mean_rounding: for running sums and densities
// from zero over the subnormal numbers to 4096, the correction is finite and at
// most an ulp of the largest number in it (a mean of rounding errors, each at
// most half an ulp).  Prints "ok <n>" or the first miss.
#include <stdio.h>

#include "../../deepdrr_amd/csrc/steps.h"

static uint64_t rng = 0x9E3779B97F4A7C15ull;
static float uniform() {
    rng ^= rng << 13;
    rng ^= rng >> 7;
    rng ^= rng << 17;
    return (float)((rng >> 20) & 0xffffff) / 16777216.0f;
}

static bool check(float cur, float lo, float hi) {
    const float m = drr::mean_rounding(cur, lo, hi);
    const float top = fmaxf(fabsf(cur) + fabsf(lo), fabsf(cur) + fabsf(hi));
    const float ulp = nextafterf(top, INFINITY) - top;
    if (isfinite(m) && fabsf(m) <= ulp) return true;
    printf("miss cur %.9g lo %.9g hi %.9g: %.9g\n", cur, lo, hi, m);
    return false;
}

int main() {
    // tails of smooth densities: subnormal, just normal, and beside a large sum
    const float tails[][3] = {{0.0f, 1e-40f, 3e-40f}, {1.0f, 1e-40f, 3e-40f}, {0.0f, 1e-35f, 1.0001e-35f},
                              {1e-40f, 0.0f, 1e-45f}, {700.0f, 3e-39f, 1e-45f}, {0.0f, -1e-40f, 2e-40f}};
    for (const auto &t : tails)
        if (!check(t[0], t[1], t[2])) return 1;
    long long n = 0;
    for (int k = 0; k < 4000000; k++) {
        auto number = [&]() {
            if (uniform() < 0.02f) return 0.0f;
            const float x = ldexpf(1.0f + uniform(), (int)(uniform() * 161.0f) - 149);  // 2^-149 .. 2^12
            return uniform() < 0.1f ? -x : x;
        };
        const float cur = fabsf(number()), lo = number();
        // the other end: near, a little off, or anywhere
        const float r = uniform();
        const float hi = r < 0.4f ? lo * (1.0f + ldexpf(uniform(), -(int)(uniform() * 22.0f))) : r < 0.5f ? lo : number();
        if (!check(cur, lo, hi)) return 1;
        n++;
    }
    printf("ok %lld\n", n);
    return 0;
}
