// steps.h -- the march's FP32 sequences `x += d` taken many steps at a time with
// the results of the single additions, and the mean of what such additions
// round off.  Host code runs them too, to check them against the plain loops.
#pragma once

#include <hip/hip_runtime.h>
#include <math.h>
#include <stdint.h>

#define DRR_AIR_DENSITY 0.1129  // double, as project_kernel.cu:6

namespace drr {

__host__ __device__ __forceinline__ float add_air(float a) {
    // area_density[AIR] += AIR_DENSITY evaluates in double (project_kernel.cu:526)
    return (float)((double)a + DRR_AIR_DENSITY);
}

// Stretches of a sequence x_{k+1} = fl(x_k + d) that are an exact arithmetic
// progression: while the results stay in x's binade every addition rounds d to
// the same multiple of that binade's ulp, and the only thing that can make two
// increments differ, a tie going to the even neighbour, shows in the first two
// of them (after one step every x is even and the increments repeat).  So with
// x1 = fl(x + d) and x2 = fl(x1 + d), equal increments x1 - x = x2 - x1 = inc
// mean x_k = x + k inc, exactly, as long as x_k is below the binade's top.
__host__ __device__ __forceinline__ float binade_top(float x) {  // x > 0, normal
    return __builtin_bit_cast(float, (__builtin_bit_cast(uint32_t, x) & 0x7f800000u) + 0x00800000u);
}

// Steps certainly before `lim` on the progression from x, at most `most` (0 if
// inc <= 0): the quotient's rounding and one step of slack stay below the 2
// taken off.
__host__ __device__ __forceinline__ int steps_below(float x, float inc, float lim, int most) {
    if (!(inc > 0.0f)) return 0;
    const int k = (int)fminf(fmaxf((lim - x) / inc - 2.0f, 0.0f), 4194304.0f);
    return k < most ? k : most;
}

// `while (t < N && alpha < lim) { alpha += step; ++t; }` with the results of
// the same FP32 additions: jumps of many steps inside a binade of alpha
// (above), single steps around its end.  From a source about 700 mm away that
// is some 10 binades instead of 7000 additions a ray (1-17 % of a ray's work
// at 512 and 128 voxels).
__host__ __device__ __forceinline__ void skip_steps(int N, float lim, float step, float &alpha, int &t) {
    while (t < N && alpha < lim) {
        const float a1 = alpha + step, inc = a1 - alpha, a2 = a1 + step;
        if (inc == 0.0f) {  // alpha no longer moves
            t = N;
            break;
        }
        const int k = a2 - a1 == inc ? steps_below(alpha, inc, fminf(lim, binade_top(alpha)), N - t) : 0;
        if (k > 0) {
            alpha = __builtin_fmaf((float)k, inc, alpha);
            t += k;
        } else {
            alpha = a1;
            ++t;
        }
    }
}

// n times acc = add_air(acc), by the same argument (the double addition's
// rounding, too, is the same all over a binade of acc).
__host__ __device__ __forceinline__ void air_steps(int n, float &acc) {
    while (n > 0) {
        const float c1 = add_air(acc), inc = c1 - acc, c2 = add_air(c1);
        const int k = (acc > 0.0f && c2 - c1 == inc) ? steps_below(acc, inc, binade_top(acc), n) : 0;
        if (k > 0) {
            acc = __builtin_fmaf((float)k, inc, acc);
            n -= k;
        } else {
            acc = c1;
            --n;
        }
    }
}

// Samples of a stretch that starts at alpha (<= mx) and is an exact progression
// with increment inc = fl(alpha + step) - alpha: those up to mx and inside
// alpha's binade, at most `most`; 1 where the two first increments differ.
__host__ __device__ __forceinline__ int stretch(float alpha, float step, float mx, int most, float &inc) {
    const float a1 = alpha + step, a2 = a1 + step;
    inc = a1 - alpha;
    if (inc == 0.0f) return most;  // alpha does not move
    if (a2 - a1 != inc) return 1;
    // the last k with alpha + k inc <= lim: the quotient's floor is off by at
    // most one below 2^22
    const float lim = fminf(mx, __builtin_bit_cast(float, __builtin_bit_cast(uint32_t, binade_top(alpha)) - 1u));
    float k = floorf(fminf((lim - alpha) / inc, 4194304.0f));
    if (__builtin_fmaf(k, inc, alpha) > lim)
        k -= 1.0f;
    else if (__builtin_fmaf(k + 1.0f, inc, alpha) <= lim)
        k += 1.0f;
    const int n = (int)k + 1;
    return n < most ? n : most;
}

// What rounding to cur's precision adds to the mean of samples that are added to
// cur one by one, where the samples run from lo to hi.  The rounding error of a
// term x is a sawtooth in x, whose integral is its square, so over a ramp the
// mean of the errors is (el^2 - eh^2) / (2 (hi - lo)) with those at the ends.
__host__ __device__ __forceinline__ float mean_rounding(float cur, float lo, float hi) {
    const float el = ((cur + lo) - cur) - lo, eh = ((cur + hi) - cur) - hi, d = hi - lo;
    const float s = 0.5f * (el + eh);
    // el - eh is d where the ends round to the same value.  A difference too
    // small for its own rounding to leave anything of it, or for its reciprocal
    // to be a number (smooth densities have subnormal tails), counts as none.
#ifdef __HIP_DEVICE_COMPILE__
    const float id = __builtin_amdgcn_rcpf(d);
#else
    const float id = 1.0f / d;
#endif
    return fabsf(d) > __builtin_fmaf(9.5367432e-7f, fabsf(hi), 1e-30f) ? s * ((el - eh) * id) : s;
}

}  // namespace drr
