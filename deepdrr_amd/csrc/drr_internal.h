// drr_internal.h -- shared definitions of the HIP library (not installed).
//
// Volume layout in HBM ("cell-expanded"): for a volume of nx*ny*nz voxels the
// library stores one 40-byte record per trilinear cell (i, j, k), i in
// [-1, nx-1] (same for j, k), i.e. (nx+1)(ny+1)(nz+1) cells, i fastest:
//   words 0-7   : 8 float32 corner densities, corner d = dx + 2 dy + 4 dz
//                 holding D[clamp(i+dx)][clamp(j+dy)][clamp(k+dz)]   (32 B)
//   word 8      : the 8 corner labels as 4-bit fields, corner d at bits
//                 4d..4d+3 (labels are < DRR_MAX_MATERIALS = 16)
//   word 9      : their common label if all 8 agree, else ~0          (8 B)
// A ray sample with base = floor(p) reads cell clamp(base, -1, n-1): three
// loads from one address (16 + 16 + 8 bytes) replace the 16 scattered texel
// fetches of the reference's texture path (project_kernel.cu:421-425, 542).
// Clamping the cell index reproduces clamp-to-edge addressing exactly.
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

#include <memory>
#include <mutex>
#include <string>

#include "../../include/deepdrr_amd.h"

// Small device buffers (job tables, keys, flags) of a context's calls, kept from
// call to call: hipMalloc and hipFree cost about 20 us each and hipFree waits for
// the whole device, where a call over a few small views takes a millisecond.  A
// buffer is put back only after the GPU work that uses it has ended, so any
// thread or stream may take it next.  At most 32 buffers and 64 MB of up to 16 MB
// each are kept, and one of up to 2 GB: a volume's cells, which a fit makes anew
// for every density (freeing 87 MB takes 0.3 ms); it serves that size alone and
// is freed when another is asked for.  All are freed with the context, those that
// outlive it by their owner, and every context's when an allocation of the library
// (drr_device_malloc) finds no memory.
class DevPool {
  public:
    DevPool() {
        std::lock_guard<std::mutex> lk(all_mu_);
        next_ = all_;
        all_ = this;
    }
    ~DevPool() {
        {
            std::lock_guard<std::mutex> lk(all_mu_);
            DevPool **at = &all_;
            while (*at != this) at = &(*at)->next_;
            *at = next_;
        }
        (void)drop();
    }
    DevPool(const DevPool &) = delete;
    DevPool &operator=(const DevPool &) = delete;

    // Contents undefined; `size` is what has to be given back with the buffer.
    hipError_t take(size_t bytes, void **p, size_t *size);

    void put(void *p, size_t size) {
        {
            std::lock_guard<std::mutex> lk(mu_);
            if (size > BIG) {
                if (size <= ((size_t)2 << 30) && !big_.p) {
                    big_ = Buf{size, p};
                    return;
                }
            } else if (n_ < MOST && held_ + size <= ((size_t)64 << 20)) {
                free_[n_++] = Buf{size, p};
                held_ += size;
                return;
            }
        }
        (void)hipFree(p);
    }

    // Free what every context keeps; whether there was anything.
    static bool drop_all() {
        std::lock_guard<std::mutex> lk(all_mu_);
        bool any = false;
        for (DevPool *q = all_; q; q = q->next_) any |= q->drop();
        return any;
    }

  private:
    struct Buf {
        size_t size;
        void *p;
    };
    static constexpr size_t BIG = (size_t)16 << 20;
    static constexpr int MOST = 32;
    bool drop() {
        Buf all[MOST + 1];
        int n;
        {
            std::lock_guard<std::mutex> lk(mu_);
            n = n_;
            for (int i = 0; i < n; i++) all[i] = free_[i];
            if (big_.p) all[n++] = big_;
            n_ = 0;
            held_ = 0;
            big_ = Buf{0, nullptr};
        }
        for (int i = 0; i < n; i++) (void)hipFree(all[i].p);
        return n > 0;
    }
    std::mutex mu_;
    Buf free_[MOST];
    Buf big_{0, nullptr};
    int n_ = 0;
    size_t held_ = 0;  // bytes in free_
    DevPool *next_ = nullptr;
    static inline std::mutex all_mu_;
    static inline DevPool *all_ = nullptr;
};

// hipMalloc that has the contexts give back what they keep before it fails.
inline hipError_t drr_device_malloc(void **p, size_t bytes) {
    hipError_t e = hipMalloc(p, bytes);
    if (e == hipErrorOutOfMemory && DevPool::drop_all()) {
        (void)hipGetLastError();
        e = hipMalloc(p, bytes);
    }
    return e;
}
template <typename T>
inline hipError_t drr_device_malloc(T **p, size_t bytes) {
    return drr_device_malloc(reinterpret_cast<void **>(p), bytes);
}

inline hipError_t DevPool::take(size_t bytes, void **p, size_t *size) {
    const size_t unit = bytes > ((size_t)1 << 20) ? (size_t)1 << 20 : 4096;
    const size_t n = (bytes + unit - 1) / unit * unit;
    void *stale = nullptr;
    {
        std::lock_guard<std::mutex> lk(mu_);
        if (n > BIG) {
            const Buf b = big_;
            big_ = Buf{0, nullptr};
            if (b.p && b.size == n) {
                *size = n;
                *p = b.p;
                return hipSuccess;
            }
            stale = b.p;
        } else {
            int best = n_;  // the smallest that fits and is not over twice as large
            for (int i = 0; i < n_; i++)
                if (free_[i].size >= n && free_[i].size <= 2 * n && (best == n_ || free_[i].size < free_[best].size))
                    best = i;
            if (best < n_) {
                *size = free_[best].size;
                *p = free_[best].p;
                held_ -= *size;
                free_[best] = free_[--n_];
                return hipSuccess;
            }
        }
    }
    if (stale) (void)hipFree(stale);
    *size = n;
    return drr_device_malloc(p, n);
}

// A buffer of a pool, given back when its owner drops it.
class PoolBuf {
  public:
    PoolBuf() = default;
    PoolBuf(const PoolBuf &) = delete;
    PoolBuf &operator=(const PoolBuf &) = delete;
    ~PoolBuf() { reset(); }
    hipError_t take(const std::shared_ptr<DevPool> &pool, size_t bytes) {
        reset();
        const hipError_t e = pool->take(bytes, &p_, &size_);
        if (e == hipSuccess)
            pool_ = pool;
        else
            p_ = nullptr;
        return e;
    }
    void reset() {
        if (p_) pool_->put(p_, size_);
        p_ = nullptr;
        pool_.reset();
    }
    // Where the wait for the buffer's work failed: nobody gets it, and hipFree waits.
    void discard() {
        if (p_) (void)hipFree(p_);
        p_ = nullptr;
        pool_.reset();
    }
    template <typename T>
    T *as(size_t byte_offset = 0) const {
        return reinterpret_cast<T *>(static_cast<char *>(p_) + byte_offset);
    }

  private:
    std::shared_ptr<DevPool> pool_;
    void *p_ = nullptr;
    size_t size_ = 0;
};

struct drr_volume_s {
    drr_ctx *ctx = nullptr;
    int device = 0;  // HIP device of the allocation (outlives the context)
    int nx = 0, ny = 0, nz = 0;
    int64_t n_cells = 0;
    int n_labels = 0;  // every label is below it: the scene's materials when the volume was made
    PoolBuf cell_buf;
    uint32_t *cells = nullptr;  // DRR_CELL_WORDS 32-bit words per cell
    // voxel-order records [nz][ny][nx] of (density bits, label), made on first
    // use by the Monte-Carlo path: a nearest-voxel lookup is one 8-byte load
    // (one memory sector, where separate density and label arrays take two)
    uint2 *lin_vox = nullptr;
    float max_density = 0.0f;
};

struct drr_ctx_s {
    int device = 0;
    int n_cus = 0;  // compute units
    std::shared_ptr<DevPool> pool = std::make_shared<DevPool>();
    // The stream that plans are captured on (nothing runs on it), one for all:
    // making a stream takes up to a millisecond.
    std::mutex cap_mu;
    hipStream_t cap = nullptr;
    drr_scene_t scene{0.1f, 0, 0, 0, DRR_MARCH_EXACT};
    bool have_scene = false;
    bool single_sums = false;  // the fast march adds every sample singly (drr_ctx_set_single_sums)
    int n_bins = 0;
    float *d_energies = nullptr;  // [B]
    float *d_pdf = nullptr;       // [B]
    float *d_mu = nullptr;        // [B * M]
    hipEvent_t ev0 = nullptr, ev1 = nullptr;
    bool timed = false;
};

// ---- error plumbing (defined in runtime.hip) ------------------------------
int drr_set_error(int code, const std::string &msg);
int drr_hip_error(hipError_t e, const char *what);

#define DRR_HIP_CHECK(expr)                                   \
    do {                                                      \
        hipError_t _e = (expr);                               \
        if (_e != hipSuccess) return drr_hip_error(_e, #expr); \
    } while (0)

// ---- kernel parameter blocks ------------------------------------------------

#define DRR_CELL_WORDS 10  // words of one cell record: 8 densities, 2 label words

// One volume as the march sees it.
struct VolDev {
    int nx, ny, nz;
    // Cell index in FP32 arithmetic for clamped cell coordinates (cx, cy, cz)
    // (march.h, Cell::load): with e1 = cz * a1 + (cy * b1 + c1) and
    // e2 = cy * b2 + (cx + c2) (parameters from vol_index_params),
    //   (uint32)e1 * s1 + bits(e2) = index + 0x4B000000,
    // every intermediate an exact integer below 2^24.
    float a1, b1, c1, b2, c2;
    uint32_t s1;
    float cmax[3];  // nx - 1, ny - 1, nz - 1: the largest cell coordinate
    uint64_t cells_b;  // address of the record of index -0x4B000000
    int n_labels;      // every label of the cells is below it
};
static_assert(sizeof(VolDev) == 64, "the fixed scratch of drr_project_jobs_noalloc holds as many volumes as ever");

// Parameters of the FP32 cell index.  Form A ((nx+1)(ny+1) <= 2^23):
// e1 = cz + 1, e2 = (cy+1)(nx+1) + (cx+1) + 2^23, s1 = (nx+1)(ny+1).  Form B
// ((nz+1)(ny+1) <= 2^23): e1 = (cz+1)(ny+1) + (cy+1), e2 = cx + 1 + 2^23,
// s1 = nx+1.  Dimensions <= 16384 and fewer than 2^31 cells leave no volume
// outside both forms ((nx+1)(ny+1) > 2^23 forces nz+1 < 256).  bits(e2) of
// an integer e2 in [2^23, 2^24) is 0x4B000000 + (e2 - 2^23); the bias is
// taken off the base addresses instead of each index.
inline VolDev vol_index_params(const uint32_t *cells, int nx, int ny, int nz) {
    VolDev d{};
    d.nx = nx;
    d.ny = ny;
    d.nz = nz;
    d.cmax[0] = (float)(nx - 1);
    d.cmax[1] = (float)(ny - 1);
    d.cmax[2] = (float)(nz - 1);
    const double nx1 = nx + 1.0, ny1 = ny + 1.0, nz1 = nz + 1.0;
    const double two23 = 8388608.0;
    if (nx1 * ny1 <= two23) {
        d.a1 = 1.0f;
        d.b1 = 0.0f;
        d.c1 = 1.0f;
        d.b2 = (float)nx1;
        d.c2 = (float)(nx1 + 1.0 + two23);
        d.s1 = (uint32_t)(nx1 * ny1);
    } else {  // then nz + 1 < 256, so (nz+1)(ny+1) < 2^23
        d.a1 = (float)ny1;
        d.b1 = 1.0f;
        d.c1 = (float)(ny1 + 1.0);
        d.b2 = 0.0f;
        d.c2 = (float)(1.0 + two23);
        d.s1 = (uint32_t)nx1;
        (void)nz1;
    }
    d.cells_b = (uint64_t)(uintptr_t)cells - (uint64_t)0x4B000000u * (4u * DRR_CELL_WORDS);
    return d;
}

// Everything the per-ray march needs for one view of up to V volumes.
struct ViewDev {
    float W[9];
    float max_ray_length;
    int width, height;
    float A[DRR_MAX_VOLUMES][12];
    float s[DRR_MAX_VOLUMES][3];
    float lo[DRR_MAX_VOLUMES][3];
    float hi[DRR_MAX_VOLUMES][3];
    int prio[DRR_MAX_VOLUMES];
    int en[DRR_MAX_VOLUMES];
    VolDev vol[DRR_MAX_VOLUMES];
};

// One view of a single volume: the uniforms of the single-volume march.
struct Geo1 {
    float W[9];
    float mrl;
    int width, height;
    float A[12];
    float s[3];
    float lo[3];
    float hi[3];
    int en;
};

inline void view_to_geo1(const drr_view_t &v, Geo1 &g) {
    for (int i = 0; i < 9; i++) g.W[i] = v.world_from_index[i];
    g.mrl = v.max_ray_length;
    g.width = v.width;
    g.height = v.height;
    for (int i = 0; i < 12; i++) g.A[i] = v.vol[0].ijk_from_world[i];
    for (int i = 0; i < 3; i++) {
        g.s[i] = v.vol[0].source_ijk[i];
        g.lo[i] = v.vol[0].bounds_lo[i];
        g.hi[i] = v.vol[0].bounds_hi[i];
    }
    g.en = v.vol[0].enabled;
}

struct SpectrumDev {
    const float *energies;
    const float *pdf;
    const float *mu;
    int n_bins;
};

// Index + 0x4B000000 of the cell at clamped coordinates (cx, cy, cz), each an
// integer in [-1, n-1] held in FP32 (the march's Cell::load; host code runs it
// too, to check it against integer arithmetic).
__host__ __device__ __forceinline__ uint32_t cell_index_biased(const VolDev &v, float cx, float cy, float cz) {
    const float e1 = __builtin_fmaf(cz, v.a1, __builtin_fmaf(cy, v.b1, v.c1));
    const float e2 = __builtin_fmaf(cy, v.b2, cx + v.c2);
    uint32_t bits;
    __builtin_memcpy(&bits, &e2, 4);
#ifdef __HIP_DEVICE_COMPILE__
    return __umul24((uint32_t)e1, v.s1) + bits;  // both below 2^24: a full-rate multiply-add
#else
    return (uint32_t)e1 * v.s1 + bits;
#endif
}

inline VolDev vol_to_dev(const drr_volume *v) {
    VolDev d = vol_index_params(v->cells, v->nx, v->ny, v->nz);
    d.n_labels = v->n_labels;
    return d;
}

inline void view_to_dev(const drr_view_t &v, const drr_volume *const *vols, ViewDev &d) {
    for (int i = 0; i < 9; i++) d.W[i] = v.world_from_index[i];
    d.max_ray_length = v.max_ray_length;
    d.width = v.width;
    d.height = v.height;
    for (int k = 0; k < DRR_MAX_VOLUMES; k++) {
        const drr_view_volume_t &vv = v.vol[k];
        for (int i = 0; i < 12; i++) d.A[k][i] = vv.ijk_from_world[i];
        for (int i = 0; i < 3; i++) {
            d.s[k][i] = vv.source_ijk[i];
            d.lo[k][i] = vv.bounds_lo[i];
            d.hi[k][i] = vv.bounds_hi[i];
        }
        d.prio[k] = vv.priority;
        d.en[k] = vv.enabled;
        if (k < v.n_volumes && vols && vols[k]) {
            d.vol[k] = vol_to_dev(vols[k]);
        } else {
            d.vol[k] = vol_index_params(nullptr, 1, 1, 1);
        }
    }
}

// Validation shared by the entry points.
int drr_check_view(const drr_ctx *ctx, const drr_volume *const *vols, const drr_view_t *view);
// Every float of the view's geometry is finite (else DRR_ERR_INVALID).
int drr_check_view_finite(const drr_view_t *view);

// Make vol->lin_vox and vol->max_density if absent (runtime.hip).
int drr_volume_ensure_linear(drr_volume *vol);

// Launchers implemented in forward.hip (used by batch/adjoint code).
// bad (may be NULL) becomes nonzero if a label is not below n_labels.
int drr_launch_expand(const float *density, const uint8_t *labels, int n_labels, uint32_t *bad, int nx, int ny, int nz,
                      uint32_t *cells, hipStream_t st);
