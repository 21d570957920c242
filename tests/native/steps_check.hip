// Host-side check of steps.h: skip_steps, air_steps and stretch against the
// plain FP32 loops they stand for, over steps, starting points and limits from
// the start of the sequence to where it no longer moves.  Prints "ok <n>" or
// the first miss.
#include <stdio.h>

#include "../../deepdrr_amd/csrc/steps.h"

static uint64_t rng = 0x9E3779B97F4A7C15ull;
static float uniform() {
    rng ^= rng << 13;
    rng ^= rng >> 7;
    rng ^= rng << 17;
    return (float)((rng >> 20) & 0xffffff) / 16777216.0f;
}

int main() {
    long long n = 0;
    const float steps[] = {0.1f, 0.25f, 0.125f, 1.0f / 3.0f, 1.3f, 0.0078125f, 0.05f, 7.0f, 0.1f * 3.0f, 0.75f};
    for (float step : steps) {
        for (int trial = 0; trial < 400; trial++) {
            // start points over the binades, some on coarse grids (ties)
            float a0 = ldexpf(1.0f + uniform(), (int)(uniform() * 22.0f) - 2);
            if (trial % 3 == 0) a0 = floorf(a0 * 8.0f) / 8.0f;
            if (trial % 41 == 0) a0 = 0.0f;
            if (trial % 50 == 1) a0 = ldexpf(1.0f + uniform(), 23);
            const int N = 1 + (int)(uniform() * 40000.0f);
            const float lim = a0 + step * (float)N * (1.6f * uniform() - 0.1f);
            float a = a0;
            int t = 0;
            while (t < N && a < lim) {
                a += step;
                ++t;
            }
            float b = a0;
            int u = 0;
            drr::skip_steps(N, lim, step, b, u);
            if (a != b || t != u) {
                printf("skip_steps: step %g from %.9g to %.9g, N %d: %.9g %d, not %.9g %d\n", step, a0, lim, N, b, u, a, t);
                return 1;
            }
            // the stretch: every sample it spans, at a0 + k inc, as the loop reaches it
            if (a0 > 0.0f && lim >= a0) {
                float inc;
                const int m = drr::stretch(a0, step, lim, N, inc);
                if (m < 1 || m > N) {
                    printf("stretch: step %g from %.9g: %d samples of %d\n", step, a0, m, N);
                    return 1;
                }
                float x = a0;
                for (int k = 0; k < m; k++) {
                    if (x != __builtin_fmaf((float)k, inc, a0) || (k > 0 && !(x <= lim))) {
                        printf("stretch: step %g from %.9g to %.9g: sample %d of %d at %.9g\n", step, a0, lim, k, m, x);
                        return 1;
                    }
                    x += step;
                }
                if (x != __builtin_fmaf((float)(m - 1), inc, a0) + step) {
                    printf("stretch: step %g from %.9g: ends at %.9g\n", step, a0, x);
                    return 1;
                }
            }
            float p = (float)((double)(a0 / step) * DRR_AIR_DENSITY), q = p;
            for (int k = 0; k < t; k++) p = drr::add_air(p);
            drr::air_steps(t, q);
            if (p != q) {
                printf("air_steps: %d from %.9g: %.9g, not %.9g\n", t, (float)((double)(a0 / step) * DRR_AIR_DENSITY), q, p);
                return 1;
            }
            ++n;
        }
    }
    printf("ok %lld\n", n);
    return 0;
}
