// march.h -- per-ray DRR march on CDNA4, shared by the plain, batched and
// adjoint kernels.
//
// Semantics are those of deepdrr's projectKernel
// (deepdrr/projector/project_kernel.cu:195-646): same FP32 operation order,
// IEEE division and sqrt, and no implicit contraction (-ffp-contract=off);
// three multiply-adds per sample are fused explicitly, where nvcc's default
// --fmad=true fuses the reference's expressions: the sample position
// (402-404), the area-density accumulation (543-547) and, in this engine's
// exact-weight trilinear filter, its running sum.  Differences are in *how*
// the work is done, never in the values:
//   * the 8 label corners and 8 density corners of a trilinear cell are read
//     once per cell change from the cell-expanded layout (drr_internal.h) and
//     kept in registers while the ray stays in the cell; the reference keeps
//     the labels (project_kernel.cu:394-431) and re-reads density texels at
//     every step (542);
//   * for a single volume the steps before the volume are skipped, with the
//     alpha the same sequential FP32 `alpha += step` (552) reaches
//     (skip_steps); the label cache needs no step before the first sample (the
//     labels a fetch returns depend on the cell alone, see Cell);
//   * a cell whose 8 labels agree sums the weights once instead of per
//     material; a fused multiply-add with a zero fraction leaves an
//     accumulator unchanged, so the result is bit-identical to the
//     per-material sums (451-455, 543-547).
// The fast march (fast_march.h, DRR_MARCH_FAST) is the one place where values
// differ from the reference's, by rounding only.
#pragma once

#include "drr_internal.h"
#include "steps.h"

namespace drr {

__device__ __forceinline__ void ray_dir(const float *W, int udx, int vdx, float &rx, float &ry,
                                        float &rz, float &L) {
    // (float)udx + 0.5 (a double literal) is exact for udx < 2^23.
    const float u = (float)udx + 0.5f;
    const float v = (float)vdx + 0.5f;
    rx = u * W[0] + v * W[1] + W[2];
    ry = u * W[3] + v * W[4] + W[5];
    rz = u * W[6] + v * W[7] + W[8];
    L = sqrtf(rx * rx + ry * ry + rz * rz);
    const float inv = 1.0f / L;
    rx *= inv;
    ry *= inv;
    rz *= inv;
}

// Slab clip of one volume (project_kernel.cu:274-315).  Returns do_trace.
__device__ __forceinline__ bool slab(const float *A, const float *s, const float *lo,
                                     const float *hi, float mrl, float rx, float ry, float rz,
                                     float ri[3], float &mn, float &mx) {
    ri[0] = A[0] * rx + A[1] * ry + A[2] * rz + A[3] * 0.0f;
    ri[1] = A[4] * rx + A[5] * ry + A[6] * rz + A[7] * 0.0f;
    ri[2] = A[8] * rx + A[9] * ry + A[10] * rz + A[11] * 0.0f;
    mn = 0.0f;
    mx = mrl > 0 ? mrl : INFINITY;
#pragma unroll
    for (int a = 0; a < 3; a++) {
        if (0.0f != ri[a]) {
            const float reci = 1.0f / ri[a];
            const float a0 = (lo[a] - s[a]) * reci;
            const float a1 = (hi[a] - s[a]) * reci;
            mn = fmaxf(mn, fminf(a0, a1));
            mx = fminf(mx, fmaxf(a0, a1));
        } else if (lo[a] > s[a] || s[a] > hi[a]) {
            return false;
        }
    }
    return true;
}

// Sample position along one axis: the reference's s + alpha * r - 1.0f, with
// the multiply-add fused as nvcc fuses it by default (--fmad=true); the
// oracle uses the same fmaf.
__device__ __forceinline__ float sample_pos(float s, float alpha, float r) {
    return __builtin_fmaf(alpha, r, s) - 1.0f;
}

// Volume arrays live in device global memory.  Pointers that reach a kernel
// through a table in memory (the batch's volume list) are generic to the
// compiler, which then emits flat loads (slower, and they also wait on the
// LDS counter); reading through an address-space-1 pointer gives global loads.
typedef const __attribute__((address_space(1))) float gfloat;
typedef const __attribute__((address_space(1))) uint32_t guint;

__device__ __forceinline__ int clamp_cell(float b, int n) {
    // cell index in [-1, n-1]; clamp in float (one v_med3_f32) so that huge
    // values stay defined before the conversion
    const float c = __builtin_amdgcn_fmed3f(b, -1.0f, (float)(n - 1));
    return (int)c;
}

__device__ __forceinline__ void weights8(float fx, float fy, float fz, float w[8]) {
    const float gx = 1.0f - fx, gy = 1.0f - fy, gz = 1.0f - fz;
    w[0] = gx * gy * gz;
    w[1] = fx * gy * gz;
    w[2] = gx * fy * gz;
    w[3] = fx * fy * gz;
    w[4] = gx * gy * fz;
    w[5] = fx * gy * fz;
    w[6] = gx * fy * fz;
    w[7] = fx * fy * fz;
}

__device__ __forceinline__ uint32_t corner_label(uint32_t l0, uint32_t, int d) {
    return (l0 >> (4 * d)) & 0xfu;
}

// Density at the sample: corner densities weighted by the same exact FP32
// weights, summed in corner order starting from the first product, each
// further term fused into the running sum.
__device__ __forceinline__ float trilerp(const float4 &d0, const float4 &d1, const float w[8]) {
    float rho = w[0] * d0.x;
    rho = __builtin_fmaf(w[1], d0.y, rho);
    rho = __builtin_fmaf(w[2], d0.z, rho);
    rho = __builtin_fmaf(w[3], d0.w, rho);
    rho = __builtin_fmaf(w[4], d1.x, rho);
    rho = __builtin_fmaf(w[5], d1.y, rho);
    rho = __builtin_fmaf(w[6], d1.z, rho);
    rho = __builtin_fmaf(w[7], d1.w, rho);
    return rho;
}

template <int M>
__device__ __forceinline__ float get_m(const float (&a)[M], int idx) {
    float r = 0.0f;
#pragma unroll
    for (int m = 0; m < M; m++) r = (m == idx) ? a[m] : r;
    return r;
}

template <int M>
__device__ __forceinline__ void set_m(float (&a)[M], int idx, float val) {
#pragma unroll
    for (int m = 0; m < M; m++) a[m] = (m == idx) ? val : a[m];
}

// Labels of the 8 corners of the sample at p with base b = floor(p): the
// reference point-samples L[clamp(floor(p + d))] (project_kernel.cu:421-425).
// Every p the march forms is fl(q - 1) for an FP32 q (sample_pos), and for
// such p with |p| < 2^22 the sum p + 1 is exact: for q >= 0.5, q - 1 is exact
// (Sterbenz, and 1 is a multiple of ulp(q) below 2^24), so fl(p + 1) = q; for
// p <= -0.5, |p| - 1 is a multiple of ulp(p).  Hence floor(p + d) = b + d.
// For |p| >= 2^22 the sample is over 2^22 - 16384 voxels outside the volume,
// where b + 1, b + 2 (and b) all clamp to the same edge voxel.  So the labels
// are always L[clamp(b + d)], which is exactly the cell record of
// clamp(b, -1, n-1): l0 = corner labels as nibbles, l1 = common label or ~0.
//
// Cached trilinear cell of the ray: base, 8 labels, 8 densities and whether
// the labels agree (l1 = their common label).  Before the first load the base
// is far from any sample (the fractions p - b test as outside [0, 1)).
struct Cell {
    float bx = -1.0e30f, by = -1.0e30f, bz = -1.0e30f;
    bool have = false;
    bool uni = false;
    uint32_t l0 = 0, l1 = 0;  // corner labels (nibbles); common label or ~0
    float4 d0 = make_float4(0.f, 0.f, 0.f, 0.f), d1 = make_float4(0.f, 0.f, 0.f, 0.f);

    // Cell of base (x, y, z): clamped to [-1, n-1] per axis, its index formed
    // in FP32 (VolDev: exact integers), records read from the biased bases.
    __device__ __forceinline__ void load(const VolDev &vol, float x, float y, float z) {
        const float cx = __builtin_amdgcn_fmed3f(x, -1.0f, vol.cmax[0]);
        const float cy = __builtin_amdgcn_fmed3f(y, -1.0f, vol.cmax[1]);
        const float cz = __builtin_amdgcn_fmed3f(z, -1.0f, vol.cmax[2]);
        const uint32_t ib = cell_index_biased(vol, cx, cy, cz);  // index + 0x4B000000
        gfloat *rp = (gfloat *)(vol.cells_b + (uint64_t)ib * (4u * DRR_CELL_WORDS));
        d0 = make_float4(rp[0], rp[1], rp[2], rp[3]);
        d1 = make_float4(rp[4], rp[5], rp[6], rp[7]);
        l0 = ((guint *)rp)[8];
        l1 = ((guint *)rp)[9];
        uni = l1 != 0xffffffffu;
        bx = x;
        by = y;
        bz = z;
        have = true;
    }
};

// Running area density of the current uniform material: ad[cm] lives in
// `cur` across consecutive uniform cells of one material and is written back
// only when the material changes (cm < 0: none).
struct Accum {
    float cur = 0.0f;
    int cm = -1;
};

// One in-volume sample of the single-volume march at position p
// (project_kernel.cu:394-547) with weight wt (0.5 at the ends of the ray, else 1).
template <int M>
__device__ __forceinline__ void sample_v1(const VolDev &vol, Cell &c, float (&ad)[M], Accum &a, float px,
                                          float py, float pz, float wt) {
    // floor(p) is the cached base exactly when every fraction p - b lies in
    // [0, 1): p - b is exact there, and rounding is monotonic.  As unsigned
    // bits, [0, 1) is [0, 0x3f800000); -0, negatives and NaN fall outside.
    float fx = px - c.bx, fy = py - c.by, fz = pz - c.bz;
    const uint32_t fmax = max(max(__float_as_uint(fx), __float_as_uint(fy)), __float_as_uint(fz));
    if (fmax >= 0x3f800000u) {
        const float bx = floorf(px), by = floorf(py), bz = floorf(pz);
        c.load(vol, bx, by, bz);
        fx = px - bx;
        fy = py - by;
        fz = pz - bz;
        const int ncm = (int)c.l1;  // the common material, -1 if the labels differ
        if (ncm != a.cm) {
            if (a.cm >= 0) set_m<M>(ad, a.cm, a.cur);
            a.cm = ncm;
            a.cur = get_m<M>(ad, ncm);
        }
    }
    float w[8];
    weights8(fx, fy, fz, w);
    const float rho = trilerp(c.d0, c.d1, w);
    const float x = wt * rho;
    const float ssum = ((((((w[0] + w[1]) + w[2]) + w[3]) + w[4]) + w[5]) + w[6]) + w[7];
    // uniform cell: seg[m0] = ssum, all other fractions 0
    a.cur = c.uni ? __builtin_fmaf(x, ssum, a.cur) : a.cur;
    if (!c.uni) {
        // Labels differ: per material present among the 8 corners (a zero
        // nibble of l0 ^ m * 0x11111111, by the borrow test), its fraction in
        // corner order; an absent material's fraction is 0 and leaves ad[m]
        // unchanged (fma(x, 0, a) = a for a >= 0), so it is skipped.
#pragma unroll
        for (int m = 0; m < M; m++) {
            const uint32_t xm = c.l0 ^ (0x11111111u * (uint32_t)m);
            if (((xm - 0x11111111u) & ~xm & 0x88888888u) != 0u) {
                float sm = 0.0f;
#pragma unroll
                for (int d = 0; d < 8; d++) sm += (corner_label(c.l0, c.l1, d) == (uint32_t)m) ? w[d] : 0.0f;
                ad[m] = __builtin_fmaf(x, sm, ad[m]);
            }
        }
    }
}

// Occupancy target of the march kernels: up to 5 materials the march fits in
// 64 VGPRs (8 waves per SIMD) without spills in its sample loops; more
// materials get more registers.
template <int M>
struct MarchOcc {
    static constexpr int waves = M <= 5 ? 8 : 5;
};

// Per-ray state of the single-volume march, filled by march_setup_v1.
struct RayV1 {
    float rx, ry, rz, L;
    float ri[3];
    float mnv, mxv;
    float minA, maxA;
    int N;
    bool trace;
};

__device__ __forceinline__ void march_setup_v1(const Geo1 &g, int udx, int vdx, float step, RayV1 &r) {
    ray_dir(g.W, udx, vdx, r.rx, r.ry, r.rz, r.L);
    r.minA = r.L;
    r.maxA = 0.0f;
    r.trace = false;
    r.ri[0] = r.ri[1] = r.ri[2] = 0.0f;
    r.mnv = 0.0f;
    r.mxv = 0.0f;
    if (g.en) {
        r.trace = slab(g.A, g.s, g.lo, g.hi, g.mrl, r.rx, r.ry, r.rz, r.ri, r.mnv, r.mxv);
        if (r.trace) {
            r.minA = fminf(r.minA, r.mnv);
            r.maxA = fmaxf(r.maxA, r.mxv);
        }
    }
    r.N = (int)ceilf((r.maxA - r.minA) / step);
}

// Single-volume march (project_kernel.cu:334-584 with NUM_VOLUMES == 1).
// On return ad[] holds the final area densities in g/cm^2.
template <int M, bool ATTEN>
__device__ __forceinline__ void march_v1(const Geo1 &g, const VolDev &vol, int udx, int vdx,
                                         float step, int air, float (&ad)[M]) {
    RayV1 r;
    march_setup_v1(g, udx, vdx, step, r);
#pragma unroll
    for (int m = 0; m < M; m++) ad[m] = 0.0f;
    float acc = 0.0f;  // air accumulator while no volume is sampled
    if (ATTEN) acc = (float)((double)acc + (double)(r.minA / step) * DRR_AIR_DENSITY);

    const int N = r.N;
    float alpha = r.minA;
    int t = 0;
    if (r.trace) {
        const float sx = g.s[0], sy = g.s[1], sz = g.s[2];
        const float rix = r.ri[0], riy = r.ri[1], riz = r.ri[2];
        // Steps before the volume: only the alpha sequence.  The labels a sample
        // is split by depend on its cell alone (Cell), so the label
        // cache needs no steps before the first sample.
        skip_steps(N, r.mnv, step, alpha, t);
        if (ATTEN) air_steps(t, acc);  // one per step so far
        Cell c;
        if (ATTEN) set_m<M>(ad, air, acc);
        // Inside [minAlpha_vol, maxAlpha_vol]: sample and accumulate.
        // While the ray is in a cell whose 8 labels agree (material m0), only
        // ad[m0] changes; it is kept in `cur` and written back on leaving, so
        // every FP32 addition is the one the reference performs.  The end
        // samples t == 0 and t == N-1 carry weight 0.5 (project_kernel.cu:
        // 541), the others 1.
        Accum acc3;
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
            while (t < tlim) {
                sample_v1<M>(vol, c, ad, acc3, sample_pos(sx, alpha, rix), sample_pos(sy, alpha, riy),
                             sample_pos(sz, alpha, riz), wt);
                wt = 1.0f;
                alpha += step;
                ++t;
            }
            // a fresh comparison after the loop (an empty asm hides alpha's
            // in-loop history), so the loop does not carry one
            asm volatile("" : "+v"(alpha));
            if (!(alpha <= r.mxv) || t >= N) break;
            if (t == N - 1) wt = 0.5f;
            tlim = t + 1;
        }
        if (acc3.cm >= 0) set_m<M>(ad, acc3.cm, acc3.cur);
        if (ATTEN) acc = get_m<M>(ad, air);
    }
    // The rest of the steps sample nothing.
    if (ATTEN) {
        air_steps(N - t, acc);
        acc = (float)((double)acc + (double)((r.L - r.maxA) / step) * DRR_AIR_DENSITY);
        set_m<M>(ad, air, acc);
    }
#pragma unroll
    for (int m = 0; m < M; m++) ad[m] *= step;
#pragma unroll
    for (int m = 0; m < M; m++) ad[m] /= 10.0f;
}

// The materials' sums in LDS, one word per thread and material (m at
// sums[LDS_LANES m] from the thread's first; consecutive lanes in consecutive
// banks): an access by a label known only at run time is one LDS access, where
// registers take a compare and a select per material and hold M registers and
// their masks through the march.  There is a word for every label of the volumes
// (sums_bytes): a scene may come to have fewer materials than the volumes were
// made with, whose labels then go to no material, but have their words.
constexpr int LDS_LANES = 256;  // threads per block of the kernels that use them

inline int max_labels(const ViewDev &vd, int n_volumes) {
    int n = 0;
    for (int i = 0; i < n_volumes; i++) n = vd.vol[i].n_labels > n ? vd.vol[i].n_labels : n;
    return n;
}

inline size_t sums_bytes(int n_materials, int n_labels) {
    return sizeof(float) * LDS_LANES * (n_materials > n_labels ? n_materials : n_labels);
}

template <int M>
__device__ __forceinline__ void clear_sums(float *sums, int n_labels) {
#pragma unroll
    for (int m = 0; m < M; m++) sums[LDS_LANES * m] = 0.0f;
    for (int m = M; m < n_labels; m++) sums[LDS_LANES * m] = 0.0f;
}

// This thread's words, of the LDS that the launch asked for with sums_bytes.
__device__ __forceinline__ float *thread_sums() {
    extern __shared__ float lane_sums[];
    return lane_sums + threadIdx.x;
}

// Running sum of the current one-label material of such sums.
struct LdsAccum {
    float *sums;
    float cur = 0.0f;
    int cm = -1;
    __device__ __forceinline__ void open(int m) {  // m < 0: none
        if (m != cm) {
            if (cm >= 0) sums[LDS_LANES * cm] = cur;
            cm = m;
            if (m >= 0) cur = sums[LDS_LANES * m];
        }
    }
};

// Adds x times each label's fraction of the weights w (summed in corner order)
// to its material's sum, for a cell whose labels differ: label by label of
// those the corners have (an absent one's fraction is 0 and leaves its sum alone).
__device__ __forceinline__ void add_mixed(float *sums, uint32_t l0, const float (&w)[8], float x) {
    uint32_t left = 0x11111111u;  // corners whose label is still to be added
    do {
        const uint32_t m = (l0 >> __builtin_ctz(left)) & 0xfu;
        const uint32_t d0 = l0 ^ (m * 0x11111111u);  // nibble 0: the corner has label m
        const uint32_t other = (((d0 & 0x77777777u) + 0x77777777u) | d0) >> 3;  // bit 4d set: another label
        float sm = 0.0f;
#pragma unroll
        for (int d = 0; d < 8; d++) sm += ((other >> (4 * d)) & 1u) ? 0.0f : w[d];
        sums[LDS_LANES * m] = __builtin_fmaf(x, sm, sums[LDS_LANES * m]);
        left &= other;
    } while (left != 0u);
}

// sample_v1 with the sums in LDS.
__device__ __forceinline__ void sample_lds(const VolDev &vol, Cell &c, LdsAccum &a, float px, float py, float pz,
                                           float wt) {
    float fx = px - c.bx, fy = py - c.by, fz = pz - c.bz;
    if (max(max(__float_as_uint(fx), __float_as_uint(fy)), __float_as_uint(fz)) >= 0x3f800000u) {
        const float bx = floorf(px), by = floorf(py), bz = floorf(pz);
        c.load(vol, bx, by, bz);
        fx = px - bx;
        fy = py - by;
        fz = pz - bz;
        a.open((int)c.l1);
    }
    float w[8];
    weights8(fx, fy, fz, w);
    const float x = wt * trilerp(c.d0, c.d1, w);
    const float ssum = ((((((w[0] + w[1]) + w[2]) + w[3]) + w[4]) + w[5]) + w[6]) + w[7];
    a.cur = c.uni ? __builtin_fmaf(x, ssum, a.cur) : a.cur;
    if (!c.uni) add_mixed(a.sums, c.l0, w, x);
}

// Mesh terms of a ray for march_multi: `inside(alpha)` says whether a
// subtractive mesh hides the sample at alpha (called with increasing alpha,
// project_kernel.cu:498-521), `until()` the largest alpha up to which that
// answer holds, and `add(ad)` adds the additive mesh area densities after the
// step scaling (569-579).  NoMesh is the scene without meshes.
struct NoMesh {
    __device__ __forceinline__ bool inside(float) { return false; }
    __device__ __forceinline__ float until() const { return INFINITY; }
    template <int M>
    __device__ __forceinline__ void add(float (&)[M]) {}
};

// Waves per SIMD of the kernels that run march_multi: 80 registers, a few
// spilled outside the sample loops (4 waves without spills: 4.27 ms against
// 3.98 on a 768^2 view of three volumes; 8: 3.73 there, 2.74 against 2.70 with
// a mesh, and twice the spills).
constexpr int MULTI_WAVES = 6;

// Steps a lane takes in march_multi before it looks again at what the other
// lanes of its wave wait for: lanes that leave a stretch early (an implant's
// edge runs through the wave) idle until the others come to its end (128 steps:
// +7 %, no limit: +75 %).
constexpr int MULTI_STRETCH = 48;

// The alphas at which the bases floor(p) of volumes i and j can agree, as
// [lo, hi] (lo > hi: none): |p_i - p_j| is linear in alpha and must be below
// one voxel on every axis, here below g, which leaves room for the rounding
// of FP32 positions and for two steps between the compared samples.
__device__ __forceinline__ void same_base(const float *si, const float *ri, const float *sj, const float *rj,
                                          float step, float amax, float &lo, float &hi) {
    lo = -INFINITY;
    hi = INFINITY;
#pragma unroll
    for (int a = 0; a < 3; a++) {
        const float D = si[a] - sj[a], E = ri[a] - rj[a], r = fabsf(ri[a]) + fabsf(rj[a]);
        const float g = 1.25f + 2.0f * step * r + 1e-6f * (fabsf(si[a]) + fabsf(sj[a]) + amax * r);
        if (E == 0.0f) {
            if (!(fabsf(D) < g)) hi = -INFINITY;
        } else {
            const float iE = 1.0f / E, a0 = (-g - D) * iE, a1 = (g - D) * iE;
            lo = fmaxf(lo, fminf(a0, a1));
            hi = fminf(hi, fmaxf(a0, a1));
        }
    }
}

// General march for 1..V volumes with priorities and the label cache shared
// across volumes (project_kernel.cu:394-553), bit for bit, in less work:
//   * steps before the first volume and after the last only advance alpha (and
//     the outside air), in jumps (steps.h);
//   * where one volume has the sole say (the usual case: alone, or on top by
//     its priority) its samples are taken by march_v1's loop up to the next
//     event on the ray: a volume's entry or exit, a mesh's, the stretch below;
//     a volume is looked at only where it counts;
//   * the shared label cache hands a volume another volume's labels only where
//     the two volumes' bases floor(p) agree.  The stretch of the ray where any
//     two can (same_base) follows the cache volume by volume, as the reference
//     does at every step; elsewhere each sample's labels are its own cell's.
//     Outside that stretch consecutive bases differ, so every lookup replaces
//     the cache and its state at the stretch's start does not matter.  A ray
//     that starts inside it starts at least one voxel of the first volume
//     early: hits and misses depend on the bases alone, and were there no
//     miss in that window, all bases would stay that of its start, but the
//     first volume's changes.
template <int V, int M, typename Mesh = NoMesh>
__device__ __forceinline__ void march_multi(const ViewDev &vd, int udx, int vdx, float step,
                                            int atten, int air, float *sums, float (&ad)[M], Mesh mesh = Mesh()) {
    float rx, ry, rz, L;
    ray_dir(vd.W, udx, vdx, rx, ry, rz, L);
    float minA = L, maxA = 0.0f;
    int n_labels = 0;
#pragma unroll
    for (int i = 0; i < V; i++) n_labels = max(n_labels, vd.vol[i].n_labels);
    clear_sums<M>(sums, n_labels);
    constexpr int VA = V > 0 ? V : 1;  // array extent (V = 0: meshes only)
    float ri[VA][3], mnv[VA], mxv[VA];
    float first = INFINITY, last = -INFINITY;  // the ray's part inside any volume
    float rfirst = 0.0f;                       // largest speed (voxels per mm) in the first volume
    bool have_first = false;
#pragma unroll
    for (int i = 0; i < V; i++) {
        ri[i][0] = ri[i][1] = ri[i][2] = 0.0f;
        mnv[i] = INFINITY;  // never inside
        mxv[i] = -INFINITY;
        if (!vd.en[i]) continue;
        float mn, mx;
        if (slab(vd.A[i], vd.s[i], vd.lo[i], vd.hi[i], vd.max_ray_length, rx, ry, rz, ri[i], mn, mx)) {
            mnv[i] = mn;
            mxv[i] = mx;
            minA = fminf(minA, mn);
            maxA = fmaxf(maxA, mx);
            if (mn <= mx) {
                first = fminf(first, mn);
                last = fmaxf(last, mx);
            }
        }
        if (!have_first) rfirst = fmaxf(fabsf(ri[i][0]), fmaxf(fabsf(ri[i][1]), fabsf(ri[i][2])));
        have_first = true;
    }
    const int N = (int)ceilf((maxA - minA) / step);
    LdsAccum acc{sums};
    acc.open(air);
    if (atten) acc.cur = (float)(0.0 + (double)(minA / step) * DRR_AIR_DENSITY);
    // steps outside every volume, up to lim: only the air
    float alpha = minA;
    int t = 0;
    auto advance = [&](float lim) __attribute__((always_inline)) {
        if (!atten) {
            skip_steps(N, lim, step, alpha, t);
            return;
        }
        acc.open(air);
        while (t < N && alpha < lim) {
            const bool hidden = mesh.inside(alpha);
            const float e = mesh.until();
            const float up = e < INFINITY ? __uint_as_float(__float_as_uint(e) + 1u) : INFINITY;  // alpha < up: alpha <= e
            const int t0 = t;
            skip_steps(N, fminf(lim, up), step, alpha, t);
            if (!hidden) air_steps(t - t0, acc.cur);
        }
    };

    if (V > 0) {
        float c0 = INFINITY, c1 = -INFINITY;  // where the label cache is followed
#pragma unroll
        for (int i = 0; i < V; i++)
#pragma unroll
            for (int j = i + 1; j < V; j++)
                if (vd.en[i] && vd.en[j]) {
                    float lo, hi;
                    same_base(vd.s[i], ri[i], vd.s[j], ri[j], step, last, lo, hi);
                    if (lo <= hi) {
                        c0 = fminf(c0, lo - 4.0f * step);
                        c1 = fmaxf(c1, hi + 4.0f * step);
                    }
                }
        const float early = 1.0f / rfirst + 2.0f * step;
        advance(c0 < first && c1 >= first - early ? first - early : first);

        Cell c;       // the open cell of volume cv
        int cv = -1;
        float pbx = 0.0f, pby = 0.0f, pbz = 0.0f;  // the shared cache: base and labels
        uint32_t s0 = 0, s1 = 0;
        bool have = false;
        while (t < N && alpha <= last) {
            // what holds at alpha, and up to which alpha (e) it holds
            const bool follow = (alpha >= c0) & (alpha <= c1);
            const bool hidden = mesh.inside(alpha);
            float e = mesh.until();
            if (V > 1) e = fminf(e, alpha < c0 ? c0 : (follow ? c1 : INFINITY));
            int cp = V, n_at = 0, users = 0;
            bool use[VA];
#pragma unroll
            for (int i = 0; i < V; i++) {
                const bool in = (alpha >= mnv[i]) & (alpha <= mxv[i]);
                e = fminf(e, alpha < mnv[i] ? mnv[i] : (in ? mxv[i] : INFINITY));
                const bool lower = in & (vd.prio[i] < cp), same = in & (vd.prio[i] == cp);
                n_at = lower ? 1 : n_at + (same ? 1 : 0);
                cp = lower ? vd.prio[i] : cp;
            }
#pragma unroll
            for (int i = 0; i < V; i++) {
                // the volumes of the chosen priority count where the ray meets
                // them at all (mnv finite), inside or not
                use[i] = vd.en[i] == 1 && (n_at > 0) & (vd.prio[i] == cp) & (mnv[i] < INFINITY);
                users += use[i] ? 1 : 0;
            }
            // steps certainly before e (as march_v1 bounds its loop), short of
            // the half-weight ends
            const float inc = step + 1.1920929e-7f * (fminf(fabsf(e), 1.0e30f) + step);
            const int k = (int)__builtin_amdgcn_fmed3f((e - alpha) / inc - 2.0f, 0.0f, 16777216.0f);
            const int tl = t > 0 ? min(t + min(k, MULTI_STRETCH), N - 1) : 0;
            if (!follow && t < tl) {
                if (hidden | (n_at == 0)) {
                    const int t0 = t;
                    skip_steps(tl, INFINITY, step, alpha, t);
                    if (!hidden && atten) {
                        acc.open(air);
                        air_steps(t - t0, acc.cur);
                    }
                    continue;
                }
                if (users == 1) {  // one volume, weight 1
#pragma unroll
                    for (int i = 0; i < V; i++) {
                        if (!use[i]) continue;
                        if (V > 1 && cv != i) c = Cell();
                        cv = i;
                        if (c.have) acc.open((int)c.l1);
                        while (t < tl) {
                            sample_lds(vd.vol[i], c, acc, sample_pos(vd.s[i][0], alpha, ri[i][0]),
                                       sample_pos(vd.s[i][1], alpha, ri[i][1]),
                                       sample_pos(vd.s[i][2], alpha, ri[i][2]), 1.0f);
                            alpha += step;
                            ++t;
                        }
                    }
                    continue;
                }
            }
            // one step, whatever holds
            float weight = n_at > 0 ? 1.0f / (float)n_at : 0.0f;
            weight *= (0 == t || N - 1 == t) ? 0.5f : 1.0f;
            cv = -1;
#pragma unroll
            for (int i = 0; i < V; i++) {
                if (!vd.en[i] || !(use[i] | follow)) continue;
                const float px = sample_pos(vd.s[i][0], alpha, ri[i][0]);
                const float py = sample_pos(vd.s[i][1], alpha, ri[i][1]);
                const float pz = sample_pos(vd.s[i][2], alpha, ri[i][2]);
                c.load(vd.vol[i], floorf(px), floorf(py), floorf(pz));
                uint32_t l0 = c.l0, l1 = c.l1;
                if (V > 1 && follow) {
                    if (!have || c.bx != pbx || c.by != pby || c.bz != pbz) {
                        s0 = l0;
                        s1 = l1;
                        pbx = c.bx;
                        pby = c.by;
                        pbz = c.bz;
                        have = true;
                    }
                    l0 = s0;
                    l1 = s1;
                }
                if (hidden | !use[i]) continue;
                float w[8];
                weights8(px - c.bx, py - c.by, pz - c.bz, w);
                const float x = weight * trilerp(c.d0, c.d1, w);
                acc.open((int)l1);
                if (l1 != 0xffffffffu) {  // one label: the other fractions are 0
                    const float ssum = ((((((w[0] + w[1]) + w[2]) + w[3]) + w[4]) + w[5]) + w[6]) + w[7];
                    acc.cur = __builtin_fmaf(x, ssum, acc.cur);
                } else {
                    add_mixed(sums, l0, w, x);
                }
            }
            if (!hidden & (n_at == 0) & (atten != 0)) {
                acc.open(air);
                acc.cur = add_air(acc.cur);
            }
            alpha += step;
            ++t;
        }
    }
    if (atten) {
        advance(INFINITY);
        acc.open(air);
        acc.cur = (float)((double)acc.cur + (double)((L - maxA) / step) * DRR_AIR_DENSITY);
    }
    acc.open(-1);
#pragma unroll
    for (int m = 0; m < M; m++) ad[m] = sums[LDS_LANES * m] * step;
    mesh.add(ad);
#pragma unroll
    for (int m = 0; m < M; m++) ad[m] /= 10.0f;
}

// Spectral Beer-Lambert sum (project_kernel.cu:637-646).
template <int M>
__device__ __forceinline__ void spectral(const SpectrumDev &sp, const float (&ad)[M], float &intensity,
                                         float &photon_prob) {
    float I = 0.0f, P = 0.0f;
    for (int b = 0; b < sp.n_bins; b++) {
        float e = 0.0f;
#pragma unroll
        for (int m = 0; m < M; m++) e += ad[m] * sp.mu[b * M + m];
        const float p = expf(-1.f * e) * sp.pdf[b];
        P += p;
        I += sp.energies[b] * p;
    }
    intensity = I;
    photon_prob = P;
}

// Solid angle of pixel (udx, vdx) (project_kernel.cu:14-133).
__device__ __forceinline__ float solid_angle(const float *W, int udx, int vdx) {
    float cx[4], cy[4], cz[4], cm[4];
    const float cu_off[4] = {0.f, 1.f, 1.f, 0.f};
    const float cv_off[4] = {0.f, 0.f, 1.f, 1.f};
#pragma unroll
    for (int c = 0; c < 4; c++) {
        const float cu = udx + cu_off[c];
        const float cv = vdx + cv_off[c];
        cx[c] = cu * W[0] + cv * W[1] + W[2];
        cy[c] = cu * W[3] + cv * W[4] + W[5];
        cz[c] = cu * W[6] + cv * W[7] + W[8];
        cm[c] = sqrtf((cx[c] * cx[c]) + (cy[c] * cy[c]) + (cz[c] * cz[c]));
    }
    const float x02 = (cy[0] * cz[2]) - (cz[0] * cy[2]);
    const float y02 = (cz[0] * cx[2]) - (cx[0] * cz[2]);
    const float z02 = (cx[0] * cy[2]) - (cy[0] * cx[2]);
    const float d01 = (cx[0] * cx[1]) + (cy[0] * cy[1]) + (cz[0] * cz[1]);
    const float d02 = (cx[0] * cx[2]) + (cy[0] * cy[2]) + (cz[0] * cz[2]);
    const float d03 = (cx[0] * cx[3]) + (cy[0] * cy[3]) + (cz[0] * cz[3]);
    const float d12 = (cx[1] * cx[2]) + (cy[1] * cy[2]) + (cz[1] * cz[2]);
    const float d23 = (cx[2] * cx[3]) + (cy[2] * cy[3]) + (cz[2] * cz[3]);
    const float n012 = fabsf((cx[1] * x02) + (cy[1] * y02) + (cz[1] * z02));
    const float n023 = fabsf((cx[3] * x02) + (cy[3] * y02) + (cz[3] * z02));
    const float den012 = (cm[0] * cm[1] * cm[2]) + (d01 * cm[2]) + (d02 * cm[1]) + (d12 * cm[0]);
    const float den023 = (cm[0] * cm[2] * cm[3]) + (d02 * cm[3]) + (d03 * cm[2]) + (d23 * cm[0]);
    float s012 = 2.f * atan2f(n012, den012);
    if (s012 < 0.0f) s012 += 3.141592654f;
    float s023 = 2.f * atan2f(n023, den023);
    if (s023 < 0.0f) s023 += 3.141592654f;
    return s012 + s023;
}

// Tile -> pixel mapping: a 64-lane wave covers an 8x8 pixel tile (a ray
// packet whose samples fall in neighbouring cells at each depth).
__device__ __forceinline__ void lane_pixel(int tile_x, int tile_y, int lane, int &udx, int &vdx) {
    udx = tile_x * 8 + (lane & 7);
    vdx = tile_y * 8 + (lane >> 3);
}

}  // namespace drr
