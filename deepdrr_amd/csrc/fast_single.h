// fast_single.h -- the fast march with every sample added singly (single_sums of
// the context), for images whose photons are then counted with noise.
//
// A Poisson count drawn for a given seed is a step function of its mean: where
// the photon probability moves by a rounding, one count in some thousand comes
// out one photon off, and the image with noise moves by a hundred times what
// the image without it does.  So views that feed the noise are marched with
// the sums in the order in which they were always added, sample by sample,
// and a seed's noise stays what it was: with fast_march.h's sums that of eight
// views of 500 x 400 differs by 1.4e-4 of the image.
//
// The samples t in [t, tlim), all of weight 1, have the same FP32 alpha sequence
// as sample_v1 and, in cells whose labels agree, the same sequential FP32
// additions into the area densities, but each sample's density is formed far
// more cheaply than by the exact filter.  Along the ray the trilinear density
// of a cell is a cubic in the distance u = alpha - a0 from the sample where the
// ray entered the cell; on entering a cell its four coefficients are formed
// from the 8 corner densities, the entry fractions and the ray direction, with
// the distance to the exit face, and each sample then costs three multiply-adds
// and the loop's bookkeeping.  The entry sample uses the exact march's position
// and floor; the samples after it are placed by the exact alpha sequence (u is
// exact) on the exact line instead of at their rounded FP32 positions, and a
// sample within rounding of a face may take either cell (the density is
// continuous there).  A cell with two labels splits the density by the second
// label's fraction, also a cubic (single_run); a cell with more takes the exact
// filter's formulas.  The sums stay within about 1e-7 relative of the exact
// march's; nothing depends on the launch or on other lanes.
//
// VALU issue bounds it.  The sums live in LDS, one word per lane and label
// (in registers the entry block took a compare and a select per material, and
// their lane masks spilled 95 scalar registers through the loop), and a
// sample's distance from the cell's first is k inc, with no alpha to follow:
// 8 views of 500 x 400 through 256 x 256 x 300 march in 3.88 ms, 4.60 before.  The
// next cell's record is loaded before this one's samples, for the small
// launches, which wait for it (fast_march.h): 4 views of 356 x 225 through
// 150 x 172 x 79 take 0.85 ms, 0.95 without.
#pragma once

#include "fast_march.h"

namespace drr {

// Waves per SIMD of the kernels that march so: at an earlier stage 8 views of 500 x 400
// took 4.06 ms at 5 and 4.09 at 6 (with spills), 2 views of 299 x 102 0.87 and 0.91, 4 views of
// 356 x 225 0.85 and 0.94.
constexpr int SINGLE_WAVES = 5;

// How a kernel marches a single-volume view.
enum : int { MARCH_V1_EXACT, MARCH_V1_FAST, MARCH_V1_SINGLE };
inline int march_v1_mode(const drr_ctx *ctx, int march) {
    if (march != DRR_MARCH_FAST) return MARCH_V1_EXACT;
    return ctx->single_sums ? MARCH_V1_SINGLE : MARCH_V1_FAST;
}
inline int march_v1_mode(const drr_ctx *ctx) { return march_v1_mode(ctx, ctx->scene.march); }

// Of a two-label cell (tw): the second label's share of the density at the sample
// at al, at its FP32 position (that of the exact filter), by nested lerps of the
// densities and of the label's indicators (first corners v, differences e along
// x); rho becomes the first label's.  Otherwise 0, and rho stays.
__device__ __forceinline__ float second_share(const Cell &c, float al, float sx, float sy, float sz, float rix,
                                              float riy, float riz, float v00, float v10, float v01, float v11,
                                              float e00, float e10, float e01, float e11, float &rho, bool tw) {
    const float fx = __builtin_fmaf(al, rix, sx) - (c.bx + 1.0f);
    const float fy = __builtin_fmaf(al, riy, sy) - (c.by + 1.0f);
    const float fz = __builtin_fmaf(al, riz, sz) - (c.bz + 1.0f);
    const float a00 = __builtin_fmaf(fx, c.d0.y - c.d0.x, c.d0.x);
    const float a10 = __builtin_fmaf(fx, c.d0.w - c.d0.z, c.d0.z);
    const float a01 = __builtin_fmaf(fx, c.d1.y - c.d1.x, c.d1.x);
    const float a11 = __builtin_fmaf(fx, c.d1.w - c.d1.z, c.d1.z);
    const float b0 = __builtin_fmaf(fy, a10 - a00, a00), b1 = __builtin_fmaf(fy, a11 - a01, a01);
    const float x = __builtin_fmaf(fz, b1 - b0, b0);
    const float i00 = __builtin_fmaf(fx, e00, v00), i10 = __builtin_fmaf(fx, e10, v10);
    const float i01 = __builtin_fmaf(fx, e01, v01), i11 = __builtin_fmaf(fx, e11, v11);
    const float j0 = __builtin_fmaf(fy, i10 - i00, i00), j1 = __builtin_fmaf(fy, i11 - i01, i01);
    const float xq = x * __builtin_fmaf(fz, j1 - j0, j0);
    rho = tw ? x - xq : rho;
    return tw ? xq : 0.0f;
}

// The samples t in [t, tlim), all of weight 1; on return alpha and t are those
// after them.  a: the sums, every one of them in LDS (a.cur is not used), and in
// a.cm the material whose sum the last cell's samples went to first.
template <int M>
__device__ __forceinline__ void single_run(const VolDev &vol, LdsAccum &a, bool &uni, float sx, float sy, float sz,
                                           float rix, float riy, float riz, float step, float &alpha, int &t,
                                           int tlim, float amax) {
    // Cell by cell: every lane still marching enters the cell of its current
    // sample together (one execution of the long cell-entry block for the whole
    // wave), then runs that cell's samples.  A cell's sample count n is fixed on entry:
    // the samples at u = 0, step, 2 step, ... (for a far source, at the FP32
    // increment) before the exit distance (at least the entry sample, at
    // most the samples left before tlim); a sample within the FP32 alpha
    // sequence's drift of the face may so fall to either cell, where the
    // density is continuous.
    //
    // Materials: a cell whose labels agree adds each sample's density to the sum
    // of its material.  A cell with exactly two labels
    // (nearly every cell on a material boundary) forms each sample's density
    // and the fraction f_q of its second label q at the sample's FP32 position,
    // as the exact filter does (across a boundary the density changes by up to
    // several g/cm^3 per voxel, so that position's rounding shows at 1e-5 in
    // the sums, unlike in a cell of one material), each by nested lerps:
    // rho (1 - f_q) goes to the sum of the first material and rho f_q to that of
    // q; the first is the one that the ray's last samples went to, if the cell
    // has it.  A cell with three or more labels takes the exact filter's
    // formulas.
    if (t >= tlim) return;
    // exit distances in steps (reciprocals to 1 ulp are plenty there), kept in
    // registers (an empty asm stops the compiler from forming them again on
    // every cell entry)
    const float istep = 1.0f / step;
    float jx = rix == 0.0f ? 0.0f : __builtin_amdgcn_rcpf(rix) * istep;
    float jy = riy == 0.0f ? 0.0f : __builtin_amdgcn_rcpf(riy) * istep;
    float jz = riz == 0.0f ? 0.0f : __builtin_amdgcn_rcpf(riz) * istep;
    float hx = rix == 0.0f ? INFINITY : (rix < 0.0f ? 0.0f : jx);
    float hy = riy == 0.0f ? INFINITY : (riy < 0.0f ? 0.0f : jy);
    float hz = riz == 0.0f ? INFINITY : (riz < 0.0f ? 0.0f : jz);
    // Each FP32 `alpha += step` moves alpha by step rounded to alpha's ulp, off
    // step by up to half an ulp.  Below 2^14 steps (about 1.6 m at 0.1 mm) that
    // is under 2^-11 of a step and the samples a cell's count assumes stay
    // within rounding of its face.  Beyond (a far source: at 4 km alpha moves a
    // quarter step more, or not at all) the exit distances are scaled by step
    // over the larger of the increments at the ray's current alpha and at its
    // largest, those of the two binades a far ray spans, so a cell's count ends
    // at its exit face (a ray that also crosses lower binades, starting near its
    // source, has their increments within 3/4 of an ulp of amax of these); where
    // alpha stops moving, every entry takes one sample.
    if (amax > 16384.0f * step) {
        const float s_lo = (alpha + step) - alpha, s_hi = (amax + step) - amax;
        const float fac = (s_lo > 0.0f && s_hi > 0.0f) ? step / fmaxf(s_lo, s_hi) : 0.0f;
        jx *= fac;
        jy *= fac;
        jz *= fac;
        hx = fac > 0.0f ? hx * fac : 0.0f;
        hy = fac > 0.0f ? hy * fac : 0.0f;
        hz = fac > 0.0f ? hz * fac : 0.0f;
    }
    asm volatile("" : "+v"(jx), "+v"(jy), "+v"(jz), "+v"(hx), "+v"(hy), "+v"(hz));
    // alpha moves by inc from sample to sample while it stays below top (steps.h)
    float inc = 0.0f, top = -INFINITY;
    float px = sample_pos(sx, alpha, rix), py = sample_pos(sy, alpha, riy), pz = sample_pos(sz, alpha, riz);
    Cell next;
    next.load(vol, floorf(px), floorf(py), floorf(pz));
    while (t < tlim) {
        const float a0 = alpha;  // u = alpha - a0
        if (!(a0 < top)) {
            const float a1 = a0 + step, a2 = a1 + step;
            inc = a1 - a0;
            top = a2 - a1 == inc ? binade_top(a0) : a0;
        }
        const Cell c = next;
        const float bx = c.bx, by = c.by, bz = c.bz;
        uni = c.uni;
        const float fx = px - bx, fy = py - by, fz = pz - bz;
        // density = ((c3 u + c2) u + c1) u + c0
        const Cubic fc = cell_cubic(c.d0.x, c.d0.y - c.d0.x, c.d0.z, c.d0.w - c.d0.z, c.d1.x, c.d1.y - c.d1.x,
                                    c.d1.z, c.d1.w - c.d1.z, fx, fy, fz, rix, riy, riz);
        // per axis, the exit face is reached after fma(-f, j, h) steps with
        // j = 1 / (r step) and h = j going up, 0 going down (j = 0, h = +inf
        // where r = 0)
        const float nex =
            fminf(__builtin_fmaf(-fx, jx, hx), fminf(__builtin_fmaf(-fy, jy, hy), __builtin_fmaf(-fz, jz, hz)));
        // the samples before the exit face, clamped to [1, tlim - t] after
        // the conversion (which saturates infinities and takes NaN to 0), so
        // every entry takes at least one sample
        int n = min(max((int)ceilf(nex), 1), tlim - t);
        t += n;
        bool tw = false, ex = false;  // two labels; three or more
        int m1 = (int)c.l1, m2 = 0;   // the first and second material
        // two labels: the indicators of the second as lerps along x
        float v00, v10, v01, v11, e00, e10, e01, e11;
        if (!c.uni) {
            const uint32_t l0 = c.l0;
            const uint32_t la = l0 & 0xfu;
            const uint32_t xa = l0 ^ (la * 0x11111111u);  // nonzero nibbles: corners not la
            const uint32_t lb = (l0 >> (__builtin_ctz(xa) & ~3u)) & 0xfu;
            const uint32_t xb = l0 ^ (lb * 0x11111111u);
            const uint32_t na = nz_nibbles(xa), nb = nz_nibbles(xb);
            tw = (na & nb) == 0u;
            ex = !tw;
            const bool sw = (int)lb == a.cm;
            m1 = (int)(sw ? lb : la);
            m2 = (int)(sw ? la : lb);
            const uint32_t iq = sw ? na : nb;  // bit set: corner not the second
            v00 = (iq & 0x8u) ? 0.f : 1.f;
            v10 = (iq & 0x800u) ? 0.f : 1.f;
            v01 = (iq & 0x80000u) ? 0.f : 1.f;
            v11 = (iq & 0x8000000u) ? 0.f : 1.f;
            e00 = ((iq & 0x80u) ? 0.f : 1.f) - v00;
            e10 = ((iq & 0x8000u) ? 0.f : 1.f) - v10;
            e01 = ((iq & 0x800000u) ? 0.f : 1.f) - v01;
            e11 = ((iq & 0x80000000u) ? 0.f : 1.f) - v11;
            a.cm = ex ? -1 : m1;
        } else {
            a.cm = m1;
        }
        float *pa = a.sums + LDS_LANES * m1, *pb = a.sums + LDS_LANES * m2;
        float cur = *pa, sq = *pb;
        alpha = __builtin_fmaf((float)n, inc, a0);
        px = sample_pos(sx, alpha, rix), py = sample_pos(sy, alpha, riy), pz = sample_pos(sz, alpha, riz);
        next.load(vol, floorf(px), floorf(py), floorf(pz));
        const bool even = alpha <= top;  // alpha - a0 is k inc at the cell's k-th sample, exactly
        const int ne = even & !ex ? n : 0;
        float u = 0.0f, al = a0;
        if (tw) {
            for (int k = 0; k < ne; ++k) {
                float rho;
                sq += second_share(c, al, sx, sy, sz, rix, riy, riz, v00, v10, v01, v11, e00, e10, e01, e11, rho, true);
                cur += rho;
                al += inc;
            }
        } else {
            for (int k = 0; k < ne; ++k) {
                cur += __builtin_fmaf(__builtin_fmaf(__builtin_fmaf(fc.c3, u, fc.c2), u, fc.c1), u, fc.c0);
                u += inc;
            }
        }
        if (!even) {  // across a binade's top, step by step
            alpha = a0;
            for (int k = 0; k < n; ++k) {
                const float u = alpha - a0;
                float rho = __builtin_fmaf(__builtin_fmaf(__builtin_fmaf(fc.c3, u, fc.c2), u, fc.c1), u, fc.c0);
                const float xq = second_share(c, alpha, sx, sy, sz, rix, riy, riz, v00, v10, v01, v11, e00, e10, e01, e11, rho, tw);
                sq += xq;
                cur += rho;
                alpha += step;
            }
            px = sample_pos(sx, alpha, rix), py = sample_pos(sy, alpha, riy), pz = sample_pos(sz, alpha, riz);
            next.load(vol, floorf(px), floorf(py), floorf(pz));
        }
        if (tw) *pb = sq;
        if (ex) {
            float al = a0;
            for (int k = 0; k < n; ++k) {
                float w[8];
                weights8(__builtin_fmaf(al, rix, sx) - (bx + 1.0f), __builtin_fmaf(al, riy, sy) - (by + 1.0f),
                         __builtin_fmaf(al, riz, sz) - (bz + 1.0f), w);
                add_mixed(a.sums, c.l0, w, trilerp(c.d0, c.d1, w));
                al += step;
            }
        } else {
            *pa = cur;
        }
    }
}

// Single-volume march (project_kernel.cu:334-584 with NUM_VOLUMES == 1).
// On return ad[] holds the final area densities in g/cm^2.
template <int M, bool ATTEN>
__device__ __forceinline__ void march_fast_single(const Geo1 &g, const VolDev &vol, int udx, int vdx,
                                                  float step, int air, float *sums, float (&ad)[M]) {
    RayV1 r;
    march_setup_v1(g, udx, vdx, step, r);
    clear_sums<M>(sums, vol.n_labels);
    float acc = 0.0f;  // air accumulator while no volume is sampled
    if (ATTEN) acc = (float)((double)acc + (double)(r.minA / step) * DRR_AIR_DENSITY);

    const int N = r.N;
    float alpha = r.minA;
    int t = 0;
    if (r.trace) {
        const float sx = g.s[0], sy = g.s[1], sz = g.s[2];
        const float rix = r.ri[0], riy = r.ri[1], riz = r.ri[2];
        // Phase 1: steps well before the volume: only the alpha sequence.
        const float rdom = fmaxf(fabsf(rix), fmaxf(fabsf(riy), fabsf(riz)));
        const float lim = r.mnv - (1.0f / rdom + 2.0f * step);
        skip_steps(N, lim, step, alpha, t);
        if (ATTEN) air_steps(t, acc);
        // Phase 2: the cells of the last voxel before the volume, from the last of
        // which the first cell inside takes its first material (single_run).
        Cell c;
        while (t < N && alpha < r.mnv) {
            const float px = sample_pos(sx, alpha, rix);
            const float py = sample_pos(sy, alpha, riy);
            const float pz = sample_pos(sz, alpha, riz);
            const float bx = floorf(px), by = floorf(py), bz = floorf(pz);
            if (!c.have || bx != c.bx || by != c.by || bz != c.bz) c.load(vol, bx, by, bz);
            if (ATTEN) acc = add_air(acc);
            alpha += step;
            ++t;
        }
        if (ATTEN) sums[LDS_LANES * air] = acc;
        // Phase 3: inside [minAlpha_vol, maxAlpha_vol]: sample and accumulate.
        // While the ray is in a cell whose 8 labels agree (material m0), only
        // ad[m0] changes; it is kept in `cur` and written back on leaving, so
        // every FP32 addition is the one the reference performs.  The end
        // samples t == 0 and t == N-1 carry weight 0.5 (project_kernel.cu:
        // 541), the others 1.
        LdsAccum acc3{sums};
        if (c.have && c.uni) acc3.open((int)c.l1);
        // The loop runs while t < tlim with no test on alpha: tlim is at most
        // the last weight-1 sample (N - 2) and at most the samples whose alpha
        // is certainly <= maxAlpha_vol.  Each FP32 `alpha += step` adds at
        // most step + 2^-24 (|mxv| + step) while alpha <= mxv, so with
        // inc = step + 2^-23 (|mxv| + step) the next K = floor((mxv - alpha)
        // / inc) - 2 samples stay inside (the -2 covers the FP32 quotient and
        // difference).  Past tlim the loop re-enters one sample at a time with
        // the full test; the last sample (t == N-1) re-enters with weight 0.5.
        float wt = (0 == t) ? 0.5f : 1.0f;
        const float inc = step + 1.1920929e-7f * (fabsf(r.mxv) + step);
        const float kf = (r.mxv - alpha) / inc - 2.0f;
        // (clamped in float to a range the conversion holds, then to N - 1 in
        // integers, where (float)(N - 1 - t) could round up)
        int tlim = min(t + (int)__builtin_amdgcn_fmed3f(kf, 0.0f, 16777216.0f), N - 1);
        for (;;) {
            // a sample of weight 0.5 (the first, the last) takes the exact filter
            if (wt != 1.0f && t < tlim) {
                sample_lds(vol, c, acc3, sample_pos(sx, alpha, rix), sample_pos(sy, alpha, riy),
                           sample_pos(sz, alpha, riz), wt);
                wt = 1.0f;
                alpha += step;
                ++t;
            }
            if (t < tlim) {
                const int m = acc3.cm;
                acc3.open(-1);  // every sum to LDS
                acc3.cm = m;
                bool uni = true;
                single_run<M>(vol, acc3, uni, sx, sy, sz, rix, riy, riz, step, alpha, t, tlim, r.mxv);
                // the next sample enters its cell anew; a running sum goes on only in
                // a material whose samples were one label's
                const int cm = uni ? acc3.cm : -1;
                acc3.cm = -1;
                acc3.open(cm);
                c = Cell{};
            }
            // a fresh comparison after the loop (an empty asm hides alpha's
            // in-loop history), so the loop does not carry one
            asm volatile("" : "+v"(alpha));
            if (!(alpha <= r.mxv) || t >= N) break;
            if (t == N - 1) wt = 0.5f;
            tlim = t + 1;
        }
        acc3.open(-1);
        if (ATTEN) acc = sums[LDS_LANES * air];
    }
    // Phase 4: the rest of the steps sample nothing.
    if (ATTEN) {
        air_steps(N - t, acc);
        acc = (float)((double)acc + (double)((r.L - r.maxA) / step) * DRR_AIR_DENSITY);
        sums[LDS_LANES * air] = acc;
    }
#pragma unroll
    for (int m = 0; m < M; m++) ad[m] = sums[LDS_LANES * m] * step;
#pragma unroll
    for (int m = 0; m < M; m++) ad[m] /= 10.0f;
}

// LDS of a launch that marches so.
inline size_t march_bytes(int march, int n_materials, int n_labels) {
    return march == MARCH_V1_EXACT ? 0 : sums_bytes(n_materials, n_labels);
}

// The single-volume march of a thread of a block of at most LDS_LANES.
template <int M, bool ATTEN, int MARCH>
__device__ __forceinline__ void march_single_volume(const Geo1 &g, const VolDev &vol, int udx, int vdx, float step,
                                                    int air, float (&ad)[M]) {
    if constexpr (MARCH != MARCH_V1_EXACT) {
        if constexpr (MARCH == MARCH_V1_FAST)
            march_fast<M, ATTEN>(g, vol, udx, vdx, step, air, thread_sums(), ad);
        else
            march_fast_single<M, ATTEN>(g, vol, udx, vdx, step, air, thread_sums(), ad);
    } else {
        march_v1<M, ATTEN>(g, vol, udx, vdx, step, air, ad);
    }
}

}  // namespace drr
