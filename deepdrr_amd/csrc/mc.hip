// mc.hip -- Monte-Carlo X-ray transport with Woodcock (delta) tracking.
//
// deepdrr removed its scatter simulation (projector.py:527-531 raises for
// scatter_num > 0) and keeps only MC-GPU's data files and a RITA sampler
// (mcgpu_*.py, rita.py).  This kernel implements the MC-GPU method (Badal &
// Badano 2009): photons from a point source, energies from the spectrum,
// Woodcock tracking through the voxel phantom against a majorant attenuation
// coefficient, photoelectric absorption, Compton scattering (Klein-Nishina,
// Kahn's rejection sampling) and Rayleigh scattering (Thomson angular
// distribution), and scoring of the energy reaching each detector pixel split
// into primary / single Compton / single Rayleigh / multiple scatter.
// Cross sections are power laws mu_x = rho * a_x[m] * (E / 60 keV)^(-k_x).
// Random numbers: RANECU (L'Ecuyer 1988, as in PENELOPE and MC-GPU), one
// stream per history seeded from (seed, history index) by SplitMix64.
//
// Local majorants: one global majorant (the densest voxel's attenuation, here
// a titanium rod) made a photon in soft tissue take ~155 flights, most of them
// virtual.  The volume is cut into 16x16x16-voxel bricks, and each brick stores
// the component-wise maxima of density x (photoelectric, Compton, Rayleigh)
// coefficient over its voxels (k_mc_bricks, per call); its majorant at energy
// E is maj_pe f_pe(E) + maj_c f_c(E) + maj_r f_r(E), which bounds every
// voxel's attenuation in FP32 too (products and sums round monotonically).  A
// flight draws its optical depth once and walks the bricks along the
// direction (Amanatides-Woo), spending depth at each brick's own majorant;
// where it runs out is the tentative collision, accepted as real with
// probability mu(voxel) / mu(brick).  This is delta tracking with a piecewise
// constant majorant, unbiased like the global one (Badal & Badano 2009 use a
// global majorant; the local form is standard in Woodcock trackers).
//
// GPU mapping: every lane owns one history at a time and is in one of a few
// states (a brick of its flight, a tentative collision, an interaction, ...);
// each pass of the wave's loop runs the states' blocks one after the other for
// the lanes that wait there.  What bounds it is VALU issue times the lanes that
// are active in it: run flight by flight the blocks had 5.3 of 64 lanes active
// on average.  So the short and frequent blocks (a brick step, the verdict on
// a collision, the start of a flight) run on their own, the brick loop until a
// share of its lanes has left it, and the long and rare ones (a trial of a
// sampler, a turn, scoring, a new history) only once enough lanes wait for
// any of them.  A lane's own sequence of operations and random numbers stays
// what it is, so the flights, brick steps and scores do.  Measured on a 512^3
// phantom with 1.6e7 histories: 7.55 ms flight by flight, 4.98 ms so (15 of 64
// lanes active).
#include <hip/hip_runtime.h>

#include "drr_internal.h"

namespace {

struct Ranecu {
    int s1, s2;
};

__device__ __forceinline__ uint64_t splitmix64(uint64_t &x) {
    uint64_t z = (x += 0x9E3779B97F4A7C15ull);
    z = (z ^ (z >> 30)) * 0xBF58476D1CE4E5B9ull;
    z = (z ^ (z >> 27)) * 0x94D049BB133111EBull;
    return z ^ (z >> 31);
}

__device__ __forceinline__ Ranecu seed_history(uint64_t seed, uint64_t h) {
    uint64_t x = seed ^ (h * 0xD1B54A32D192ED03ull);
    Ranecu r;
    r.s1 = (int)(splitmix64(x) % 2147483562ull) + 1;
    r.s2 = (int)(splitmix64(x) % 2147483398ull) + 1;
    return r;
}

// RANECU: two multiplicative congruential generators (Schrage's method),
// combined.  Every product has factors below 2^24 (s / 53668 < 40014 and so
// on), so the full-rate 24-bit multiplies give them.
__device__ __forceinline__ float ranecu(Ranecu &r) {
    const uint32_t i1 = (uint32_t)r.s1 / 53668u;
    r.s1 = (int)(__umul24(40014u, (uint32_t)r.s1 - __umul24(i1, 53668u)) - __umul24(i1, 12211u));
    if (r.s1 < 0) r.s1 += 2147483563;
    const uint32_t i2 = (uint32_t)r.s2 / 52774u;
    r.s2 = (int)(__umul24(40692u, (uint32_t)r.s2 - __umul24(i2, 52774u)) - __umul24(i2, 3791u));
    if (r.s2 < 0) r.s2 += 2147483399;
    int z = r.s1 - r.s2;
    if (z < 1) z += 2147483562;
    return fminf((float)z * 4.656612873077393e-10f, 0.99999994f);
}

// Rotate unit direction (u, v, w) by polar cos(theta) and azimuth phi in
// [0, 2 pi) (the hardware sine and cosine: a few ulp, ample for sampling).
__device__ __forceinline__ void rotate(float &u, float &v, float &w, float ct, float phi) {
    const float st = sqrtf(fmaxf(0.0f, 1.0f - ct * ct));
    const float cp = __cosf(phi), sp = __sinf(phi);
    if (fabsf(w) > 0.99999f) {
        u = st * cp;
        v = st * sp;
        w = (w > 0.0f ? 1.0f : -1.0f) * ct;
    } else {
        const float it = rsqrtf(1.0f - w * w), t = (1.0f - w * w) * it;
        const float sit = st * it;
        const float nu = u * ct + sit * (u * w * cp - v * sp);
        const float nv = v * ct + sit * (v * w * cp + u * sp);
        const float nw = w * ct - t * st * cp;
        u = nu;
        v = nv;
        w = nw;
    }
    const float n = rsqrtf(u * u + v * v + w * w);
    u *= n;
    v *= n;
    w *= n;
}

// One trial of Klein-Nishina by Kahn's method: whether it is accepted; eta is
// the ratio of the energies.
__device__ __forceinline__ bool compton_trial(Ranecu &rng, float E, float &eta) {
    const float k = E * (1.0f / 510.99895f), ik = 1.0f / k;
    const float b1 = (1.0f + 2.0f * k) / (9.0f + 2.0f * k);
    const float r1 = ranecu(rng), r2 = ranecu(rng), r3 = ranecu(rng);
    const bool low = r1 <= b1;
    const float q = 1.0f + 2.0f * k * r2;
    eta = low ? q : (1.0f + 2.0f * k) / q;
    const float ie = 1.0f / eta, ct = 1.0f - (eta - 1.0f) * ik;
    return r3 <= (low ? 4.0f * (ie - 1.0f / (eta * eta)) : 0.5f * (ct * ct + ie));
}

// cos(theta) of an accepted trial, and the scattered energy.
__device__ __forceinline__ float compton_angle(float eta, float &E) {
    const float k = E * (1.0f / 510.99895f), ik = 1.0f / k;
    const float ct = 1.0f - (eta - 1.0f) * ik;
    E = E / eta;
    return fminf(1.0f, fmaxf(-1.0f, ct));
}

constexpr int MAX_TRIALS = 1000;  // of a rejection sampler, then the last is taken

struct Photon {
    float x[3], d[3];
    float E;
    int nc, nr;
};

constexpr float TWO_PI = 6.283185307179586f;

// (E / 60 keV)^(-k) of the three processes from one log2 and three exp2.
__device__ __forceinline__ void cross_sections(const drr_mc_params_t &p, float E, float &fpe, float &fc, float &fr) {
    const float l = __log2f(E * (1.0f / 60.0f));
    fpe = exp2f(-p.k_pe * l);
    fc = exp2f(-p.k_compton * l);
    fr = exp2f(-p.k_rayleigh * l);
}
constexpr float E_MIN = 5.0f;  // keV: lower energies are absorbed locally
constexpr int BRICK = 16;      // voxels per brick edge (a power of two)

struct Bricks {
    const float4 *maj;  // [nbz][nby][nbx]: (max rho a_pe, max rho a_c, max rho a_r, 0)
    int nb[3];
};

}  // namespace

// One wave per brick: lane l reads voxels l, l + 64, ... of the brick in x-fastest
// order (rows of BRICK contiguous records), then the wave reduces.
__global__ __launch_bounds__(256) void k_mc_bricks(const uint2 *__restrict__ vox, int nx, int ny, int nz,
                                                   drr_mc_params_t p, Bricks b, int64_t n_bricks) {
    const int64_t bi = (int64_t)blockIdx.x * 4 + (threadIdx.x >> 6);
    const int lane = threadIdx.x & 63;
    if (bi >= n_bricks) return;  // whole waves leave together
    const int bx = (int)(bi % b.nb[0]), by = (int)((bi / b.nb[0]) % b.nb[1]), bz = (int)(bi / ((int64_t)b.nb[0] * b.nb[1]));
    float mpe = 0.0f, mc = 0.0f, mr = 0.0f;
    for (int v = lane; v < BRICK * BRICK * BRICK; v += 64) {
        const int i = bx * BRICK + v % BRICK, j = by * BRICK + (v / BRICK) % BRICK, k = bz * BRICK + v / (BRICK * BRICK);
        if (i < nx && j < ny && k < nz) {
            const uint2 rv = vox[((int64_t)k * ny + j) * nx + i];
            const float rho = __uint_as_float(rv.x);
            const int m = (int)rv.y;
            mpe = fmaxf(mpe, rho * p.a_pe[m]);
            mc = fmaxf(mc, rho * p.a_compton[m]);
            mr = fmaxf(mr, rho * p.a_rayleigh[m]);
        }
    }
    for (int o = 32; o > 0; o >>= 1) {
        mpe = fmaxf(mpe, __shfl_xor(mpe, o));
        mc = fmaxf(mc, __shfl_xor(mc, o));
        mr = fmaxf(mr, __shfl_xor(mr, o));
    }
    if (lane == 0) const_cast<float4 *>(b.maj)[bi] = make_float4(mpe, mc, mr, 0.0f);
}

// The schedule; us of a scatter call on the 512^3 phantom with 1.6e7 histories.
// Waves per SIMD: 6 5550, 7 4980, 8 5150 (spills)
constexpr int MC_WAVES = 7;
// lanes waiting for the long blocks before they run: 24 5210, 32 4980, 40 5060
constexpr int MC_WAIT = 32;
// sixteenths of the brick loop's lanes still in it when it ends: 3 5070, 4 4980;
// at an earlier stage 2 and 6 were 1 % and 2 % slower than 4, 8 7 %
constexpr int MC_STOP = 4;

// What a lane's photon waits for (from REAL on: the long blocks).
enum : int {
    WALK,  // the next brick of its flight
    HIT,   // the verdict on a tentative collision
    FLY,   // a new flight
    REAL,  // an interaction
    COMP,  // a trial of the Compton sampler
    RAYL,  // a trial of the Rayleigh sampler
    OUT,   // the detector: it has left the box (or was never in it)
    DEAD,  // a new history
    DONE,  // nothing: the lane's histories are spent
};

__global__ __launch_bounds__(256, MC_WAVES) void k_mc(const uint2 *__restrict__ vox, int nx, int ny, int nz, drr_mc_params_t p,
                                            Bricks bk, int64_t first, int64_t count, uint64_t seed, float *img,
                                            float *img2, unsigned long long *nsteps, unsigned long long *nbsteps) {
    __shared__ float s_e[DRR_MAX_BINS], s_cdf[DRR_MAX_BINS];
    __shared__ float s_a[3][DRR_MAX_MATERIALS];
    for (int i = threadIdx.x; i < p.n_bins; i += blockDim.x) {
        s_e[i] = p.energies_keV[i];
        s_cdf[i] = p.cdf[i];
    }
    for (int i = threadIdx.x; i < p.n_materials; i += blockDim.x) {
        s_a[0][i] = p.a_pe[i];
        s_a[1][i] = p.a_compton[i];
        s_a[2][i] = p.a_rayleigh[i];
    }
    __syncthreads();
    const int64_t stride = (int64_t)gridDim.x * blockDim.x;
    int64_t h = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    const int W = p.det_width, H = p.det_height;
    const int64_t npix = (int64_t)W * H;
    // pixel coordinates along u and v are (hit - origin) . u / |u|^2
    const float iuu = 1.0f / (p.detector_u[0] * p.detector_u[0] + p.detector_u[1] * p.detector_u[1] + p.detector_u[2] * p.detector_u[2]);
    const float ivv = 1.0f / (p.detector_v[0] * p.detector_v[0] + p.detector_v[1] * p.detector_v[1] + p.detector_v[2] * p.detector_v[2]);
    const float *A = p.ijk_from_world;
    const int n3[3] = {nx, ny, nz};
    unsigned long long steps = 0, bsteps = 0;
    uint32_t steps_h = 0, bsteps_h = 0;  // of the current history
    Photon ph{};
    Ranecu rng{1, 1};
    float fpe = 0.f, fc = 0.f, fr = 0.f;
    float t_exit = 0.f;
    // the direction: bricks per step along each axis (signed, in the brick
    // table) and the distance between brick faces (inf across the direction)
    int sl[3] = {0, 0, 0};
    float td[3] = {0.f, 0.f, 0.f};
    // the flight: brick, bricks left before the box's side and distance to the
    // next face along each axis, the distance flown, the optical depth left,
    // the brick's majorant
    int lin = 0, left_b[3] = {0, 0, 0};
    float tn[3] = {0.f, 0.f, 0.f};
    float t = 0.f, tau = 0.f, mub = 0.f;
    float mt = 0.f, mpe = 0.f, mc = 0.f;  // of an interaction's voxel
    int tries = 0;
    int state = h < count ? DEAD : DONE;
    for (;;) {
        const int n_wait = __popcll(__ballot(state >= REAL)), n_done = __popcll(__ballot(state == DONE));
        if (n_done == 64) break;
        // The long blocks run once MC_WAIT lanes wait for them, or no photon flies.
        if (n_wait - n_done >= MC_WAIT || n_wait == 64) {
            bool turn = false;  // the photon has a new direction
            float ct = 1.0f;
            if (state == REAL) {
                const float u = ranecu(rng) * mt;
                // below mpe: photoelectric absorption
                state = u < mpe ? DEAD : (u < mpe + mc ? COMP : RAYL);
                tries = 0;
            }
            // one trial of each sampler: a lane whose trial fails waits for the
            // next round, where others join it
            if (state == COMP) {
                float eta;
                if (compton_trial(rng, ph.E, eta) || ++tries == MAX_TRIALS) {
                    ct = compton_angle(eta, ph.E);
                    ph.nc++;
                    turn = true;
                }
            }
            if (state == RAYL) {  // Thomson's (1 + cos^2) / 2 by rejection
                ct = 2.0f * ranecu(rng) - 1.0f;
                if (ranecu(rng) <= 0.5f * (1.0f + ct * ct) || ++tries == MAX_TRIALS) {
                    ph.nr++;
                    turn = true;
                }
            }
            if (turn && (ph.E < E_MIN || ph.nc + ph.nr > p.max_interactions)) {
                turn = false;
                state = DEAD;
            }
            if (state == OUT) {
                // out of the box (t_exit 0: never in it), straight to the detector plane
                state = DEAD;
                for (int a = 0; a < 3; a++) ph.x[a] += t_exit * ph.d[a];
                const float dn = ph.d[0] * p.detector_normal[0] + ph.d[1] * p.detector_normal[1] + ph.d[2] * p.detector_normal[2];
                const float tp = ((p.detector_origin[0] - ph.x[0]) * p.detector_normal[0] +
                                  (p.detector_origin[1] - ph.x[1]) * p.detector_normal[1] +
                                  (p.detector_origin[2] - ph.x[2]) * p.detector_normal[2]) / dn;
                if (!(dn <= 0.0f) && !(tp < 0.0f)) {
                    float r[3];
                    for (int a = 0; a < 3; a++) r[a] = ph.x[a] + tp * ph.d[a] - p.detector_origin[a];
                    const float fu = (r[0] * p.detector_u[0] + r[1] * p.detector_u[1] + r[2] * p.detector_u[2]) * iuu;
                    const float fv = (r[0] * p.detector_v[0] + r[1] * p.detector_v[1] + r[2] * p.detector_v[2]) * ivv;
                    if (fu >= 0.0f && fv >= 0.0f && fu < (float)W && fv < (float)H) {
                        const int iu = min((int)fu, W - 1), iv = min((int)fv, H - 1);
                        const int cls = (ph.nc + ph.nr == 0) ? 0 : (ph.nc == 1 && ph.nr == 0) ? 1 : (ph.nr == 1 && ph.nc == 0) ? 2 : 3;
                        const int64_t o = cls * npix + (int64_t)iv * W + iu;
                        unsafeAtomicAdd(img + o, ph.E);
                        if (img2) unsafeAtomicAdd(img2 + o, ph.E * ph.E);
                    }
                }
            }
            bool born = false;
            if (state == DEAD) {
                steps += steps_h;
                bsteps += bsteps_h;
                steps_h = bsteps_h = 0;
                state = DONE;
                if (h < count) {
                    born = true;
                    turn = true;
                    rng = seed_history(seed, (uint64_t)(first + h));
                    h += stride;
                    // energy from the spectrum
                    const float u = ranecu(rng);
                    int lo = 0, hi = p.n_bins - 1;
                    while (lo < hi) {
                        const int mid = (lo + hi) >> 1;
                        if (s_cdf[mid] >= u) hi = mid; else lo = mid + 1;
                    }
                    ph.E = s_e[lo];
                    // direction uniform in the cone about the axis
                    ph.d[0] = p.cone_axis[0];
                    ph.d[1] = p.cone_axis[1];
                    ph.d[2] = p.cone_axis[2];
                    ct = 1.0f - ranecu(rng) * (1.0f - p.cone_cos);
                    ph.x[0] = p.source_world[0];
                    ph.x[1] = p.source_world[1];
                    ph.x[2] = p.source_world[2];
                    ph.nc = ph.nr = 0;
                }
            }
            if (turn) {
                rotate(ph.d[0], ph.d[1], ph.d[2], ct, TWO_PI * ranecu(rng));
                // the volume box [-0.5, n-0.5] in IJK: entry (of a new photon) and exit
                float tmin = 0.0f, tmax = INFINITY;
                bool hit = true;
                int row = 1;
#pragma unroll
                for (int a = 0; a < 3; a++) {
                    const float q0 = A[4 * a] * ph.x[0] + A[4 * a + 1] * ph.x[1] + A[4 * a + 2] * ph.x[2] + A[4 * a + 3];
                    const float dq = A[4 * a] * ph.d[0] + A[4 * a + 1] * ph.d[1] + A[4 * a + 2] * ph.d[2];
                    const float idq = 1.0f / dq;  // one division per axis
                    const float hi = (float)n3[a] - 0.5f;
                    if (dq != 0.0f) {
                        const float t0 = (-0.5f - q0) * idq, t1 = (hi - q0) * idq;
                        tmin = fmaxf(tmin, fminf(t0, t1));
                        tmax = fminf(tmax, fmaxf(t0, t1));
                    } else if (q0 < -0.5f || q0 > hi) {
                        hit = false;
                    }
                    td[a] = dq != 0.0f ? (float)BRICK * fabsf(idq) : INFINITY;
                    sl[a] = dq > 0.0f ? row : -row;
                    row *= bk.nb[a];
                }
                state = FLY;
                t_exit = fmaxf(tmax, 0.0f);
                if (born) {
                    const bool in = hit && tmin < tmax;
                    state = in ? FLY : OUT;
                    t_exit = in ? tmax - tmin : 0.0f;
                    if (in)
                        for (int a = 0; a < 3; a++) ph.x[a] += tmin * ph.d[a];
                }
                cross_sections(p, ph.E, fpe, fc, fr);
            }
        }
        if ((state == HIT) | (state == FLY)) {
            if (state == HIT) {
                t += tau / mub;
                for (int a = 0; a < 3; a++) ph.x[a] += t * ph.d[a];
                t_exit -= t;
            }
            float qp[3];
            for (int a = 0; a < 3; a++)
                qp[a] = A[4 * a] * ph.x[0] + A[4 * a + 1] * ph.x[1] + A[4 * a + 2] * ph.x[2] + A[4 * a + 3] + 0.5f;
            if (state == HIT) {
                int ix[3];
                for (int a = 0; a < 3; a++) ix[a] = min(max((int)floorf(qp[a]), 0), n3[a] - 1);
                const int64_t vi = ((int64_t)ix[2] * ny + ix[1]) * nx + ix[0];
                const uint2 rv = vox[vi];  // (density bits, label)
                const float rho = __uint_as_float(rv.x);
                const int m = (int)rv.y;
                mpe = rho * s_a[0][m] * fpe;
                mc = rho * s_a[1][m] * fc;
                const float mr = rho * s_a[2][m] * fr;
                mt = mpe + mc + mr;
                state = ranecu(rng) * mub < mt ? REAL : FLY;
            }
            if (state == FLY) {
                // one flight: optical depth tau spent brick by brick at each
                // brick's majorant, up to a tentative collision or the box exit
                ++steps_h;
                tau = -__logf(ranecu(rng));
                lin = 0;
#pragma unroll
                for (int a = 0; a < 3; a++) {
                    const int bi = min(max((int)floorf(qp[a] * (1.0f / BRICK)), 0), bk.nb[a] - 1);
                    const bool up = sl[a] > 0, across = td[a] == INFINITY;
                    const float idq = copysignf(td[a] * (1.0f / BRICK), up ? 1.0f : -1.0f);  // 1 / dq: BRICK is a power of 2
                    tn[a] = across ? INFINITY : fmaxf(((float)(BRICK * (up ? bi + 1 : bi)) - qp[a]) * idq, 0.0f);
                    left_b[a] = up ? bk.nb[a] - 1 - bi : bi;
                    lin += abs(sl[a]) * bi;
                }
                t = 0.0f;
                state = WALK;
            }
        }
        // brick by brick, until more lanes wait for what comes after
        const int stop = (__popcll(__ballot(state == WALK)) * MC_STOP) >> 4;
        int left;
        do {
            if (state == WALK) {
                ++bsteps_h;
                const float4 mj = bk.maj[(uint32_t)lin];
                mub = (mj.x * fpe + mj.y * fc) + mj.z * fr;
                // the axis whose face comes first
                const bool a0 = (tn[0] <= tn[1]) & (tn[0] <= tn[2]), a1 = !a0 & (tn[1] <= tn[2]), a2 = !(a0 | a1);
                const float tnext = fminf(a0 ? tn[0] : (a1 ? tn[1] : tn[2]), t_exit);
                const float depth = mub * (tnext - t);
                if ((mub > 0.0f) & (tau < depth)) {
                    state = HIT;
                } else {
                    tau -= mub > 0.0f ? depth : 0.0f;
                    t = tnext;
                    tn[0] += a0 ? td[0] : 0.0f;
                    tn[1] += a1 ? td[1] : 0.0f;
                    tn[2] += a2 ? td[2] : 0.0f;
                    lin += a0 ? sl[0] : (a1 ? sl[1] : sl[2]);
                    left_b[0] -= a0 ? 1 : 0;
                    left_b[1] -= a1 ? 1 : 0;
                    left_b[2] -= a2 ? 1 : 0;
                    if ((tnext >= t_exit) | ((left_b[0] | left_b[1] | left_b[2]) < 0)) state = OUT;
                }
            }
            left = __popcll(__ballot(state == WALK));
        } while (left > stop);
    }
    if (nsteps) {
        for (int o = 32; o > 0; o >>= 1) steps += __shfl_xor(steps, o);
        if ((threadIdx.x & 63) == 0) atomicAdd(nsteps, steps);
    }
    if (nbsteps) {
        for (int o = 32; o > 0; o >>= 1) bsteps += __shfl_xor(bsteps, o);
        if ((threadIdx.x & 63) == 0) atomicAdd(nbsteps, bsteps);
    }
}

extern "C" int drr_mc_scatter(drr_ctx *ctx, const drr_volume *vol, const drr_mc_params_t *params,
                              int64_t first_history, int64_t n_histories, uint64_t seed, float *image,
                              float *image2, int64_t *n_steps, int64_t *n_brick_steps, void *stream) {
    if (!ctx || !vol || !params || !image) return drr_set_error(DRR_ERR_INVALID, "drr_mc_scatter: NULL argument");
    if (vol->ctx != ctx) return drr_set_error(DRR_ERR_INVALID, "drr_mc_scatter: volume of another context");
    const drr_mc_params_t &p = *params;
    if (p.n_materials < 1 || p.n_materials > DRR_MAX_MATERIALS || p.n_bins < 1 || p.n_bins > DRR_MAX_BINS)
        return drr_set_error(DRR_ERR_INVALID, "drr_mc_scatter: n_materials in [1,16] and n_bins in [1,256]");
    if (p.det_width < 1 || p.det_height < 1 || first_history < 0 || n_histories < 0)
        return drr_set_error(DRR_ERR_INVALID, "drr_mc_scatter: bad detector size or history range");
    if (!(p.cone_cos > -1.0f && p.cone_cos < 1.0f))
        return drr_set_error(DRR_ERR_INVALID, "drr_mc_scatter: cone_cos must be in (-1, 1)");
    if (!(p.cdf[p.n_bins - 1] >= 0.999f))
        return drr_set_error(DRR_ERR_INVALID, "drr_mc_scatter: cdf must end at 1");
    if (p.max_interactions < 1) return drr_set_error(DRR_ERR_INVALID, "drr_mc_scatter: max_interactions >= 1");
    if (ctx->have_scene && p.n_materials < ctx->scene.n_materials)
        return drr_set_error(DRR_ERR_INVALID, "drr_mc_scatter: tables must cover every label of the scene");
    if (n_histories == 0) return DRR_OK;
    int prev = -1;
    (void)hipGetDevice(&prev);
    if (prev != ctx->device) DRR_HIP_CHECK(hipSetDevice(ctx->device));
    drr_volume *v = const_cast<drr_volume *>(vol);
    int rc = drr_volume_ensure_linear(v);
    if (rc) return rc;
    const drr_mc_params_t &pp = p;
    int cus = 0;
    DRR_HIP_CHECK(hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, ctx->device));
    // Every lane takes histories h, h + stride, ...: a grid larger than what is
    // resident at once would leave its later blocks a full share of work to
    // start only when the first ones finish, so the grid is capped there.
    int per_cu = 0;
    DRR_HIP_CHECK(hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, k_mc, 256, 0));
    int64_t blocks = (n_histories + 255) / 256;
    const int64_t cap = (int64_t)cus * (per_cu > 0 ? per_cu : 1);
    if (blocks > cap) blocks = cap;
    hipStream_t st = (hipStream_t)stream;
    // the brick majorants of these cross sections, in stream-ordered memory
    Bricks bk{};
    bk.nb[0] = (v->nx + BRICK - 1) / BRICK;
    bk.nb[1] = (v->ny + BRICK - 1) / BRICK;
    bk.nb[2] = (v->nz + BRICK - 1) / BRICK;
    const int64_t n_bricks = (int64_t)bk.nb[0] * bk.nb[1] * bk.nb[2];
    float4 *maj = nullptr;
    hipError_t e = hipMallocAsync((void **)&maj, sizeof(float4) * n_bricks, st);
    if (e == hipErrorOutOfMemory && DevPool::drop_all()) {
        (void)hipGetLastError();
        e = hipMallocAsync((void **)&maj, sizeof(float4) * n_bricks, st);
    }
    if (e != hipSuccess) {
        if (prev >= 0 && prev != ctx->device) (void)hipSetDevice(prev);
        return drr_hip_error(e, "hipMallocAsync(brick majorants)");
    }
    bk.maj = maj;
    (void)hipEventRecord(ctx->ev0, st);
    k_mc_bricks<<<(unsigned)((n_bricks + 3) / 4), 256, 0, st>>>(v->lin_vox, v->nx, v->ny, v->nz, pp, bk, n_bricks);
    k_mc<<<(unsigned)blocks, 256, 0, st>>>(v->lin_vox, v->nx, v->ny, v->nz, pp, bk, first_history,
                                         n_histories, seed, image, image2,
                                         reinterpret_cast<unsigned long long *>(n_steps),
                                         reinterpret_cast<unsigned long long *>(n_brick_steps));
    e = hipGetLastError();
    (void)hipEventRecord(ctx->ev1, st);
    ctx->timed = true;
    (void)hipFreeAsync(maj, st);
    if (prev >= 0 && prev != ctx->device) (void)hipSetDevice(prev);
    if (e != hipSuccess) return drr_hip_error(e, "drr_mc_scatter launch");
    return DRR_OK;
}
