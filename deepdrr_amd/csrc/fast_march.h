// fast_march.h -- the fast single-volume march (DRR_MARCH_FAST), shared by the
// plain and batched kernels.
//
// The samples are those of the exact march (march.h): the same FP32 sequence
// `alpha += step`, weight 1 except for the ends of the ray; what differs is how
// their densities are formed and added, so values differ from the exact
// march's by rounding.  The ray is taken cell by cell.
//
// * Along the ray the trilinear density of a cell is a cubic in the distance u
//   from the middle of the cell's samples, formed from the 8 corner densities,
//   the fractions there and the ray direction.  The samples sit at u = k inc
//   about that middle (inc: alpha's exact increment, march.h), so the odd
//   powers cancel and their sum is n c0 + c2 sum(u^2): a cell costs about 90
//   vector instructions whatever its number of samples.
// * The reference adds the samples one by one in FP32, and in a long sum those
//   roundings are as large as the 1e-5 the fast march promises to stay within
//   of them (4e-5 on the clinical view where every cell is summed at once).
//   So a material whose running sum has passed FAST_CLOSED_SUM is added sample
//   by sample again.  Below that a cell's mean takes what the roundings add to
//   it where they do not cancel, in a density that hardly changes from sample to
//   sample (mean_rounding; without it a smooth body's image came to 2.6e-5 of
//   the exact march's, with it to 7.4e-6).  A cell of constant density is summed
//   at once at any size of the sum, unless that takes the sum to its next
//   binade: within one its samples all round the same way.
// * A cell with two labels (nearly every cell on a material boundary) splits
//   the density by the second label's fraction f, also a cubic: the sum of
//   density x f has the even moments up to u^6, about the mean of the samples'
//   FP32 positions, where the exact filter places them (across a metal
//   boundary the density changes by several g/cm^3 per voxel, and the
//   positions' rounding shows in the images).  Where a sum is long, each
//   sample's density and fraction are formed by nested lerps at its position.
// * A cell with three or more labels takes the exact filter's formulas.
//
// Every lane enters its next cell together with the others (one execution of
// the entry block for the wave), and each kind of cell runs its block and its
// loop over the samples for its own lanes.  (With the loops after all blocks, wave
// votes as their tests and 0/1 factors as the lanes' choices, for the scalar
// instructions that lanes' own branches take, a sample cost 7 vector
// instructions in place of 5, one of two labels 39 in place of 30 for every lane
// of the wave: 16 clinical views 85.5 ms, 73.3 after it (launches apart; back to
// back 80 to 84); 48 mixed 17.6, 16.5.)  The materials' sums live in LDS, one word per lane and
// label: an entry reads and writes the words its labels name, which in
// registers takes a compare and a select per material and holds the
// materials' registers and lane masks through the loop.  The record of the
// cell after is loaded before the present one is summed: the wait for it was
// most of a small launch, where no other wave fills it (one view of 256^2
// through 128^3: 323 us without, 274 with; 16 views of 1536^2 through the
// clinical CT: 97.2 ms, 86.4), and does nothing where VALU issue is the bound
// (48 views of 765 x 768: 17.9 ms either way).  Nothing depends on
// the launch or on other lanes, so results are the same from run to run and
// from kernel to kernel.
#pragma once

#include "march.h"

namespace drr {

// Running sum (density x step, mm g/cm^3) up to which cells are summed at once:
// images of clinical views are then within 7.8e-6 of the exact march's (6.4e-6
// with every sample added singly, 1.2e-5 at 128, 1.6e-5 at 204.8), at 16.5 ms
// for 48 mixed views (when singly took 24.2, this took 17.5).
constexpr float FAST_CLOSED_SUM = 102.4f;
// The same in units of the sums (density), whose ulp is what the additions round
// to: at steps below 0.1 mm this is the smaller.  With the physical sum alone,
// images at steps of 0.05, 0.01 and 0.004 mm were 6.4e-6, 3.0e-5 and 7.6e-5 from the exact
// march's on the clinical CT (3.8e-6, 4.5e-6, 5.1e-6 with this), 2.2e-5, 4.5e-5 and 3.0e-4
// on rays along a boundary of two labels (4.0e-6, 1.4e-6, 1.2e-6).
constexpr float FAST_CLOSED_UNITS = 1024.0f;
// Samples of a cell that are summed at once, so that the sum is not far past the
// bound where a cell has many (voxels of 20 mm at a step of 0.1: 9.4e-6 without,
// 6.7e-6 with; of up to 6 mm it changes nothing).
constexpr int FAST_CLOSED_SAMPLES = 64;
// Waves per SIMD of the kernels that march fast: 89 registers hold the entry
// block and the record on its way (with 9 more, 6 waves spilled 16: 7.4 ms
// against 5.7 on the clinical view; 4 waves: 5.7).
constexpr int FAST_WAVES = 5;

// A trilinear interpolant along the ray p(u) = p_m + u r as a cubic in u:
// value(u) = ((c3 u + c2) u + c1) u + c0, from the lerps along x of the corner
// pairs (0yz, 1yz) (first corners vYZ, differences xYZ) and the fractions f of
// p_m against the cell.
struct Cubic {
    float c0, c1, c2, c3;
};
__device__ __forceinline__ Cubic cell_cubic(float v00, float x00, float v10, float x10, float v01, float x01,
                                            float v11, float x11, float fx, float fy, float fz, float rx, float ry,
                                            float rz) {
    // x: e_yz(u) = A_yz + B_yz u
    const float A00 = __builtin_fmaf(fx, x00, v00), A10 = __builtin_fmaf(fx, x10, v10);
    const float A01 = __builtin_fmaf(fx, x01, v01), A11 = __builtin_fmaf(fx, x11, v11);
    const float B00 = rx * x00, B10 = rx * x10, B01 = rx * x01, B11 = rx * x11;
    // y: g_z(u) = G_z0 + G_z1 u + G_z2 u^2
    const float P0 = A10 - A00, Q0 = B10 - B00, P1 = A11 - A01, Q1 = B11 - B01;
    const float G00 = __builtin_fmaf(fy, P0, A00), G01 = __builtin_fmaf(fy, Q0, __builtin_fmaf(ry, P0, B00));
    const float G02 = ry * Q0;
    const float G10 = __builtin_fmaf(fy, P1, A01), G11 = __builtin_fmaf(fy, Q1, __builtin_fmaf(ry, P1, B01));
    const float G12 = ry * Q1;
    // z: the cubic
    const float D0 = G10 - G00, D1 = G11 - G01, D2 = G12 - G02;
    Cubic k;
    k.c0 = __builtin_fmaf(fz, D0, G00);
    k.c1 = __builtin_fmaf(fz, D1, __builtin_fmaf(rz, D0, G01));
    k.c2 = __builtin_fmaf(fz, D2, __builtin_fmaf(rz, D1, G02));
    k.c3 = rz * D2;
    return k;
}

// Bit 3 of nibble d is set where nibble d of x is nonzero (exact per nibble:
// the low three bits plus 7 carry into bit 3 and never into the next nibble).
__device__ __forceinline__ uint32_t nz_nibbles(uint32_t x) {
    return (((x & 0x77777777u) + 0x77777777u) | x) & 0x88888888u;
}

// One sample of weight wt by the exact filter's formulas, added to the sums.
template <int M>
__device__ __forceinline__ void fast_sample(const Cell &c, float *acc, float fx, float fy, float fz, float wt) {
    float w[8];
    weights8(fx, fy, fz, w);
    const float x = wt * trilerp(c.d0, c.d1, w);
#pragma unroll 1
    for (int m = 0; m < M; m++) {
        const uint32_t xm = c.l0 ^ (0x11111111u * (uint32_t)m);
        if (((xm - 0x11111111u) & ~xm & 0x88888888u) == 0u) continue;  // no corner has it
        float sm = 0.0f;
#pragma unroll
        for (int d = 0; d < 8; d++) sm += (corner_label(c.l0, c.l1, d) == (uint32_t)m) ? w[d] : 0.0f;
        acc[LDS_LANES * m] = __builtin_fmaf(x, sm, acc[LDS_LANES * m]);
    }
}

// The samples t in [t, tlim) of a stretch over which alpha moves by inc, all of
// weight 1.  acut: FAST_CLOSED_SUM in units of the sums.
template <int M>
__device__ __forceinline__ void fast_run(const VolDev &vol, float *acc, float sx, float sy, float sz, float rix,
                                         float riy, float riz, float step, float inc, float acut, float alpha, int t,
                                         int tlim) {
    // exit distances in steps (reciprocals to 1 ulp are plenty there): per axis
    // the exit face is reached after fma(-f, j, h) steps with j = 1 / (r inc)
    // and h = j going up, 0 going down (j = 0, h = +inf where r = 0).  They stay
    // in registers (an empty asm stops the compiler from forming them again on
    // every entry).  Where alpha does not move every entry takes one sample.
    const float iinc = inc > 0.0f ? 1.0f / inc : 0.0f;
    float jx = rix == 0.0f ? 0.0f : __builtin_amdgcn_rcpf(rix) * iinc;
    float jy = riy == 0.0f ? 0.0f : __builtin_amdgcn_rcpf(riy) * iinc;
    float jz = riz == 0.0f ? 0.0f : __builtin_amdgcn_rcpf(riz) * iinc;
    const float hno = inc > 0.0f ? INFINITY : 0.0f;
    float hx = rix == 0.0f ? hno : (rix < 0.0f ? 0.0f : jx);
    float hy = riy == 0.0f ? hno : (riy < 0.0f ? 0.0f : jy);
    float hz = riz == 0.0f ? hno : (riz < 0.0f ? 0.0f : jz);
    asm volatile("" : "+v"(jx), "+v"(jy), "+v"(jz), "+v"(hx), "+v"(hy), "+v"(hz));
    const float inc2_12 = inc * inc * (1.0f / 12.0f);
    if (t >= tlim) return;
    float px = sample_pos(sx, alpha, rix), py = sample_pos(sy, alpha, riy), pz = sample_pos(sz, alpha, riz);
    Cell next;
    next.load(vol, floorf(px), floorf(py), floorf(pz));
    while (t < tlim) {
        const float alpha0 = alpha;
        const Cell c = next;
        const float bx = c.bx, by = c.by, bz = c.bz;
        const float fx = px - bx, fy = py - by, fz = pz - bz;
        const float nex =
            fminf(__builtin_fmaf(-fx, jx, hx), fminf(__builtin_fmaf(-fy, jy, hy), __builtin_fmaf(-fz, jz, hz)));
        // the samples before the exit face, clamped to [1, tlim - t] after the
        // conversion (which saturates infinities and takes NaN to 0), so every
        // entry takes at least one sample; one within rounding of the face may
        // fall to either cell (the density is continuous)
        int n = min(min(max((int)ceilf(nex), 1), FAST_CLOSED_SAMPLES), tlim - t);
        t += n;
        const float nf = (float)n;
        const float um = inc * __builtin_fmaf(0.5f, nf, -0.5f);  // from the entry sample to the middle
        alpha = __builtin_fmaf(nf, inc, alpha);
        px = sample_pos(sx, alpha, rix), py = sample_pos(sy, alpha, riy), pz = sample_pos(sz, alpha, riz);
        next.load(vol, floorf(px), floorf(py), floorf(pz));
        const float mx = __builtin_fmaf(rix, um, fx), my = __builtin_fmaf(riy, um, fy), mz = __builtin_fmaf(riz, um, fz);
        // sum of u^2 over the samples
        const float S2 = inc2_12 * (nf * __builtin_fmaf(nf, nf, -1.0f));
        const uint32_t l0 = c.l0, la = l0 & 0xfu;
        float *pa = acc + LDS_LANES * la;
        if (c.uni) {
            float cur = *pa;
            const Cubic fc = cell_cubic(c.d0.x, c.d0.y - c.d0.x, c.d0.z, c.d0.w - c.d0.z, c.d1.x, c.d1.y - c.d1.x,
                                        c.d1.z, c.d1.w - c.d1.z, mx, my, mz, rix, riy, riz);
            const float h = 0.5f * inc * nf, h2 = h * h;  // the samples' extent is [-h, h]
            const float ev = __builtin_fmaf(fc.c2, h2, fc.c0), od = h * __builtin_fmaf(fc.c3, h2, fc.c1);
            const bool flat = (fc.c1 == 0.0f) & (fc.c2 == 0.0f);
            bool closed = flat | (cur < acut);
            if (closed) {  // beyond the bound only within cur's binade
                const float to = cur + __builtin_fmaf(fc.c2, S2, nf * (fc.c0 + mean_rounding(cur, ev - od, ev + od)));
                closed = (cur < acut) | ((__float_as_uint(to) ^ __float_as_uint(cur)) < 0x00800000u);
                cur = closed ? to : cur;
            }
            if (!closed) {
                float u = -um;
                for (int k = 0; k < n; ++k) {
                    cur += __builtin_fmaf(__builtin_fmaf(__builtin_fmaf(fc.c3, u, fc.c2), u, fc.c1), u, fc.c0);
                    u += inc;
                }
            }
            *pa = cur;
            continue;
        }
        const uint32_t xa = l0 ^ (la * 0x11111111u);  // nonzero nibbles: corners not la
        const uint32_t lb = (l0 >> (__builtin_ctz(xa) & ~3u)) & 0xfu;
        const uint32_t xb = l0 ^ (lb * 0x11111111u);
        const uint32_t na = nz_nibbles(xa), nb = nz_nibbles(xb);  // nb bit set: corner not lb
        float al = alpha0;
        if ((na & nb) != 0u) {  // three or more labels
            for (int k = 0; k < n; ++k) {
                fast_sample<M>(c, acc, __builtin_fmaf(al, rix, sx) - (bx + 1.0f),
                               __builtin_fmaf(al, riy, sy) - (by + 1.0f), __builtin_fmaf(al, riz, sz) - (bz + 1.0f),
                               1.0f);
                al += step;
            }
            continue;
        }
        float *pb = acc + LDS_LANES * lb;
        float cur = *pa, sq = *pb;
        // the second label's indicators of the corners as lerps along x: 0 or 1,
        // 0 or +-1
        const float v00 = (nb & 0x8u) ? 0.f : 1.f, x00 = ((nb & 0x80u) ? 0.f : 1.f) - v00;
        const float v10 = (nb & 0x800u) ? 0.f : 1.f, x10 = ((nb & 0x8000u) ? 0.f : 1.f) - v10;
        const float v01 = (nb & 0x80000u) ? 0.f : 1.f, x01 = ((nb & 0x800000u) ? 0.f : 1.f) - v01;
        const float v11 = (nb & 0x8000000u) ? 0.f : 1.f, x11 = ((nb & 0x80000000u) ? 0.f : 1.f) - v11;
        if (fmaxf(cur, sq) < acut) {
            // The middle's fractions as the mean of the samples' FP32
            // positions: the exact filter's positions round with the same
            // sign over many samples, which along a boundary adds up (with
            // the entry's alone, oblique clinical views came to 2e-5 of the
            // exact march's, with three samples' to 1.2e-5).
            float qx = 0.0f, qy = 0.0f, qz = 0.0f;
            for (int k = 0; k < n; ++k) {
                qx += __builtin_fmaf(al, rix, sx) - (bx + 1.0f);
                qy += __builtin_fmaf(al, riy, sy) - (by + 1.0f);
                qz += __builtin_fmaf(al, riz, sz) - (bz + 1.0f);
                al += inc;
            }
            const float rn = __builtin_amdgcn_rcpf(nf);
            qx *= rn;
            qy *= rn;
            qz *= rn;
            const Cubic g = cell_cubic(v00, x00, v10, x10, v01, x01, v11, x11, qx, qy, qz, rix, riy, riz);
            const Cubic fc = cell_cubic(c.d0.x, c.d0.y - c.d0.x, c.d0.z, c.d0.w - c.d0.z, c.d1.x, c.d1.y - c.d1.x,
                                        c.d1.z, c.d1.w - c.d1.z, qx, qy, qz, rix, riy, riz);
            const float S4 = S2 * (inc2_12 * 0.6f) * __builtin_fmaf(3.0f * nf, nf, -7.0f);
            const float S6 = S2 * (inc2_12 * inc2_12 * (9.0f / 7.0f)) *
                             __builtin_fmaf(nf * nf, __builtin_fmaf(3.0f * nf, nf, -18.0f), 31.0f);
            const float p2 = __builtin_fmaf(fc.c0, g.c2, __builtin_fmaf(fc.c1, g.c1, fc.c2 * g.c0));
            const float p4 = __builtin_fmaf(fc.c1, g.c3, __builtin_fmaf(fc.c2, g.c2, fc.c3 * g.c1));
            const float sum_q = __builtin_fmaf(
                nf, fc.c0 * g.c0, __builtin_fmaf(S2, p2, __builtin_fmaf(S4, p4, S6 * (fc.c3 * g.c3))));
            sq += sum_q;
            cur += __builtin_fmaf(fc.c2, S2, nf * fc.c0) - sum_q;
        } else {
            // density and second fraction at each sample's FP32 position, by
            // nested lerps
            for (int k = 0; k < n; ++k) {
                const float gx = __builtin_fmaf(al, rix, sx) - (bx + 1.0f);
                const float gy = __builtin_fmaf(al, riy, sy) - (by + 1.0f);
                const float gz = __builtin_fmaf(al, riz, sz) - (bz + 1.0f);
                const float a00 = __builtin_fmaf(gx, c.d0.y - c.d0.x, c.d0.x);
                const float a10 = __builtin_fmaf(gx, c.d0.w - c.d0.z, c.d0.z);
                const float a01 = __builtin_fmaf(gx, c.d1.y - c.d1.x, c.d1.x);
                const float a11 = __builtin_fmaf(gx, c.d1.w - c.d1.z, c.d1.z);
                const float b0 = __builtin_fmaf(gy, a10 - a00, a00), b1 = __builtin_fmaf(gy, a11 - a01, a01);
                const float x = __builtin_fmaf(gz, b1 - b0, b0);
                const float i00 = __builtin_fmaf(gx, x00, v00), i10 = __builtin_fmaf(gx, x10, v10);
                const float i01 = __builtin_fmaf(gx, x01, v01), i11 = __builtin_fmaf(gx, x11, v11);
                const float j0 = __builtin_fmaf(gy, i10 - i00, i00), j1 = __builtin_fmaf(gy, i11 - i01, i01);
                const float xq = x * __builtin_fmaf(gz, j1 - j0, j0);
                sq += xq;
                cur += x - xq;
                al += step;
            }
        }
        *pb = sq;
        *pa = cur;
    }
}

// The single-volume march (project_kernel.cu:334-584 with NUM_VOLUMES == 1).
// acc: this thread's sums in LDS, material m at acc[LDS_LANES * m].  On return
// ad[] holds the final area densities in g/cm^2.
template <int M, bool ATTEN>
__device__ __forceinline__ void march_fast(const Geo1 &g, const VolDev &vol, int udx, int vdx, float step, int air,
                                           float *acc, float (&ad)[M]) {
    RayV1 r;
    march_setup_v1(g, udx, vdx, step, r);
    clear_sums<M>(acc, vol.n_labels);
    float air_sum = 0.0f;
    if (ATTEN) air_sum = (float)((double)air_sum + (double)(r.minA / step) * DRR_AIR_DENSITY);
    const int N = r.N;
    float alpha = r.minA;
    int t = 0;
    if (r.trace) {
        const float sx = g.s[0], sy = g.s[1], sz = g.s[2];
        const float rix = r.ri[0], riy = r.ri[1], riz = r.ri[2];
        skip_steps(N, r.mnv, step, alpha, t);
        if (ATTEN) {
            air_steps(t, air_sum);
            acc[LDS_LANES * air] = air_sum;
        }
        // Stretches over which alpha is an exact arithmetic progression (march.h),
        // ending at the volume's exit or the binade's top; anything else one
        // sample at a time.
        const float acut = fminf(FAST_CLOSED_SUM / step, FAST_CLOSED_UNITS);
        while (alpha <= r.mxv && t < N) {
            if (t == 0 || t == N - 1) {  // weight 0.5
                const float px = sample_pos(sx, alpha, rix), py = sample_pos(sy, alpha, riy),
                            pz = sample_pos(sz, alpha, riz);
                Cell c;
                c.load(vol, floorf(px), floorf(py), floorf(pz));
                fast_sample<M>(c, acc, px - c.bx, py - c.by, pz - c.bz, 0.5f);
                alpha += step;
                ++t;
                continue;
            }
            const float a0 = alpha;
            float inc;
            const int m = stretch(a0, step, r.mxv, N - 1 - t, inc);
            fast_run<M>(vol, acc, sx, sy, sz, rix, riy, riz, step, inc, acut, alpha, t, t + m);
            t += m;
            // the addition after the last sample may leave the binade
            alpha = __builtin_fmaf((float)(m - 1), inc, a0) + step;
        }
        if (ATTEN) air_sum = acc[LDS_LANES * air];
    }
    if (ATTEN) {
        air_steps(N - t, air_sum);
        air_sum = (float)((double)air_sum + (double)((r.L - r.maxA) / step) * DRR_AIR_DENSITY);
        acc[LDS_LANES * air] = air_sum;
    }
#pragma unroll
    for (int m = 0; m < M; m++) ad[m] = acc[LDS_LANES * m] * step;
#pragma unroll
    for (int m = 0; m < M; m++) ad[m] /= 10.0f;
}

}  // namespace drr
