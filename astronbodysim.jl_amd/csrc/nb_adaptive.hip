// nb_adaptive.hip -- adaptive (block, power-of-two) timesteps on the GPU.
//
// Follows the reference's CPU semantics (src/base/Timestep.jl), which its GPU
// kernels restate (src/directsumgpu/timestep.jl:1-47,103-154,178-192):
//   get_timestep      dt = sqrt(2 eta h / |a|), capped by MaxStep; errors when
//                     dt < MinStep or the integer step is <= 0; the integer
//                     step is the largest TimeBase / 2^k not above dt/TimeInterval
//                     (src/base/Timestep.jl:1-23)
//   init_timesteps    Ti_endstep = get_timestep, Ti_begstep = 0  (:29-39)
//   half kick         Vel += Acc * forward * 0.5 * (Ti_end - Ti_beg) * TimeInterval (:105-114)
//   advance           active particles (Ti_endstep == system time): new step,
//                     kick from the middle of the old step to the middle of the
//                     new one, Ti_beg = Ti_end, Ti_end += step  (:47-82)
//   min end step      minimum over Ti_endstep and TimeBase  (:135-144)
//   drift             every particle by (t_int - last_t_int) * TimeInterval (:169-179)
// The force is evaluated for the active particles only; inactive particles
// keep their accelerations (the reference CPU path does; its GPU path zeroes
// them, src/directsumgpu/gravity.jl:43).
#include <hip/hip_runtime.h>
#include <algorithm>
#include <cstring>
#include <math.h>

#include "nb_block.h"
#include "nb_ctx.h"

namespace nb {

static int launch_ok(const char *what) {
    hipError_t e = hipGetLastError();
    if (e != hipSuccess) {
        set_error("launch of %s failed: %s", what, hipGetErrorString(e));
        return NB_ERR_HIP;
    }
    return NB_OK;
}

static inline unsigned gridn(int64_t n) { return (unsigned)((n + 255) / 256); }

struct AdaptParams {
    double time_interval;
    int64_t time_base;
    double err_tol;
    double min_step;
    double max_step;
};

// Error flags: 1 = dt < MinStep, 2 = integer step <= 0.
__device__ __forceinline__ int64_t get_timestep_dev(double ax, double ay, double az, double h,
                                                    const AdaptParams &p, unsigned &flag) {
    const double ac = sqrt(ax * ax + ay * ay + az * az);
    double dt = sqrt(2.0 * p.err_tol * h / ac);
    if (dt > p.max_step) dt = p.max_step;
    if (dt < p.min_step) flag |= 1u;
    const double ti_step = dt / p.time_interval;
    if (!(ti_step > 0.0)) flag |= 2u;
    int64_t ti_min = p.time_base;
    while ((double)ti_min > ti_step && ti_min > 0) ti_min >>= 1;
    return ti_min;
}

template <typename T>
__global__ void k_init_timesteps(const double *__restrict__ ax, const double *__restrict__ ay,
                                 const double *__restrict__ az, const double *__restrict__ h,
                                 int64_t n, AdaptParams p, int64_t *__restrict__ te,
                                 int64_t *__restrict__ tb, unsigned *flag) {
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    unsigned f = 0;
    te[i] = get_timestep_dev(ax[i], ay[i], az[i], h[i], p, f);
    tb[i] = 0;
    if (f) atomicOr(flag, f);
}

template <typename T>
__global__ void k_adaptive_half_kick(T *__restrict__ vx, T *__restrict__ vy, T *__restrict__ vz,
                                     const double *__restrict__ ax, const double *__restrict__ ay,
                                     const double *__restrict__ az, const int64_t *__restrict__ te,
                                     const int64_t *__restrict__ tb, int64_t n, double forward,
                                     double interval) {
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    const double c = forward * 0.5 * (double)(te[i] - tb[i]) * interval;
    vx[i] += (T)(ax[i] * c);
    vy[i] += (T)(ay[i] * c);
    vz[i] += (T)(az[i] * c);
}

template <typename T>
__global__ void k_adaptive_drift(T *__restrict__ x, T *__restrict__ y, T *__restrict__ z,
                                 const T *__restrict__ vx, const T *__restrict__ vy,
                                 const T *__restrict__ vz, int64_t n, double dt) {
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    const T d = (T)dt;
    x[i] += vx[i] * d;
    y[i] += vy[i] * d;
    z[i] += vz[i] * d;
}

// Minimum end step and the number of particles at it: (m, k) pairs combine as
// (min, sum of the counts of the operands at that minimum).  Start value
// (time_base, 0), so an empty range leaves (time_base, 0).
constexpr int MINRED_BLOCKS = 256;

struct MinCount {
    int64_t m, k;
};
__device__ __forceinline__ void add_step(MinCount &r, int64_t v) {
    if (v < r.m) {
        r.m = v;
        r.k = 1;
    } else if (v == r.m) {
        ++r.k;
    }
}

// A block's (min, count, error flags), written to its slot of the pinned host
// array that the host combines after its one wait per block step.
__device__ __forceinline__ void store_min_count(MinCount r, unsigned flags, int64_t *__restrict__ out) {
    __shared__ int64_t sm[4], sk[4];
    __shared__ unsigned sf[4];
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) {
        const int64_t m2 = __shfl_xor(r.m, off, 64), k2 = __shfl_xor(r.k, off, 64);
        const int64_t mm = m2 < r.m ? m2 : r.m;
        r.k = (r.m == mm ? r.k : 0) + (m2 == mm ? k2 : 0);
        r.m = mm;
        flags |= (unsigned)__shfl_xor((int)flags, off, 64);
    }
    const int w = threadIdx.x >> 6;
    if ((threadIdx.x & 63) == 0) { sm[w] = r.m; sk[w] = r.k; sf[w] = flags; }
    __syncthreads();
    if (threadIdx.x != 0) return;
    int64_t mm = sm[0], kk = 0;
    unsigned f = 0;
#pragma unroll
    for (int q = 1; q < 4; ++q) mm = sm[q] < mm ? sm[q] : mm;
#pragma unroll
    for (int q = 0; q < 4; ++q) {
        kk += sm[q] == mm ? sk[q] : 0;
        f |= sf[q];
    }
    out[3 * blockIdx.x] = mm;
    out[3 * blockIdx.x + 1] = kk;
    out[3 * blockIdx.x + 2] = (int64_t)f;
}

__global__ __launch_bounds__(256) void k_min_count(const int64_t *__restrict__ te, int64_t n, int64_t base,
                                                   int64_t *__restrict__ out) {
    MinCount r{base, 0};
    for (int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x; i < n; i += (int64_t)gridDim.x * 256)
        add_step(r, te[i]);
    store_min_count(r, 0, out);
}

// The active particles' kick and new steps, and the minimum and count of the
// timeline that results, in one pass.
template <typename T>
__global__ __launch_bounds__(256) void k_adaptive_advance(
    T *__restrict__ vx, T *__restrict__ vy, T *__restrict__ vz, const double *__restrict__ ax,
    const double *__restrict__ ay, const double *__restrict__ az, const double *__restrict__ h,
    int64_t *__restrict__ te, int64_t *__restrict__ tb, int64_t n, int64_t t_int, AdaptParams p,
    int64_t *__restrict__ out) {
    MinCount r{p.time_base, 0};
    unsigned flags = 0;
    for (int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x; i < n; i += (int64_t)gridDim.x * 256) {
        int64_t end = te[i];
        if (end == t_int) {
            int64_t ti_step = get_timestep_dev(ax[i], ay[i], az[i], h[i], p, flags);
            if (t_int == p.time_base) ti_step = 0;
            if (p.time_base - t_int < ti_step) ti_step = p.time_base - t_int;
            const double tstart = (double)(tb[i] + end) / 2.0;
            const double tend = (double)end + 0.5 * (double)ti_step;
            const double dt = (tend - tstart) * p.time_interval;
            vx[i] += (T)(ax[i] * dt);
            vy[i] += (T)(ay[i] * dt);
            vz[i] += (T)(az[i] * dt);
            tb[i] = end;
            end += ti_step;
            te[i] = end;
        }
        add_step(r, end);
    }
    store_min_count(r, flags, out);
}

// Active particles of each 256 (Morton-ordered) ones: the ballots of their
// waves and their count.
__global__ __launch_bounds__(256) void k_active_masks(const int64_t *__restrict__ te, int64_t n, int64_t t_int,
                                                      uint64_t *__restrict__ mask, int *__restrict__ count) {
    __shared__ int c[4];
    const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
    const uint64_t b = __builtin_amdgcn_ballot_w64(i < n && te[i] == t_int);
    const int w = threadIdx.x >> 6;
    if ((threadIdx.x & 63) == 0) {
        mask[(int64_t)blockIdx.x * 4 + w] = b;
        c[w] = __popcll(b);
    }
    __syncthreads();
    if (threadIdx.x == 0) count[blockIdx.x] = c[0] + c[1] + c[2] + c[3];
}

// The counts of the blocks before each, by one workgroup: every thread adds up a
// run of them, then writes its run's prefix.  It pays from SCAN_FROM blocks on: a
// compaction of no active particles took 72 us at 2^22 without it and 65 with it,
// 39 and 43 at 2^21, 1.87 and 0.36 ms at 2^25.
constexpr unsigned SCAN_FROM = 1 << 14;
constexpr int SCAN_THREADS = 1024;
__global__ __launch_bounds__(SCAN_THREADS) void k_scan_counts(const int *__restrict__ count, int nblk,
                                                              int64_t *__restrict__ before) {
    __shared__ int64_t part[SCAN_THREADS];
    const int per = (nblk + SCAN_THREADS - 1) / SCAN_THREADS;
    const int64_t b0 = (int64_t)per * threadIdx.x;
    const int64_t b1 = b0 + per < nblk ? b0 + per : nblk;
    int64_t sum = 0;
    for (int64_t b = b0; b < b1; ++b) sum += count[b];
    part[threadIdx.x] = sum;
    __syncthreads();
    for (int off = 1; off < SCAN_THREADS; off <<= 1) {
        const int64_t v = (int)threadIdx.x >= off ? part[threadIdx.x - off] : 0;
        __syncthreads();
        part[threadIdx.x] += v;
        __syncthreads();
    }
    int64_t k = part[threadIdx.x] - sum;
    for (int64_t b = b0; b < b1; ++b) {
        before[b] = k;
        k += count[b];
    }
}

// The active particles in order, gathered as targets.  Every block adds up the
// counts of the blocks before it (a few KB in L2), so the ordered compaction
// takes this launch and k_active_masks: with a device-wide select in between a
// block step had four more launches.  That work grows with the square of the
// blocks: from SCAN_FROM of them on k_scan_counts has added them up (before_all).
template <typename T>
__global__ __launch_bounds__(256) void k_gather_active(
    const T *__restrict__ x, const T *__restrict__ y, const T *__restrict__ z, const double *__restrict__ h,
    int64_t n, const uint64_t *__restrict__ mask, const int *__restrict__ count,
    const int64_t *__restrict__ before_all, int64_t *__restrict__ idx,
    int64_t *__restrict__ total, T *__restrict__ gx, T *__restrict__ gy, T *__restrict__ gz,
    double *__restrict__ gh) {
    __shared__ int64_t part[4];
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
    int64_t k;
    if (before_all) {   // (uniform over the launch)
        k = before_all[blockIdx.x];
    } else {
        int64_t before = 0;
        for (int b = threadIdx.x; b < (int)blockIdx.x; b += 256) before += count[b];
        before = wave_sum(before);
        if (lane == 0) part[w] = before;
        __syncthreads();
        k = part[0] + part[1] + part[2] + part[3];
    }
    const uint64_t *m = mask + (int64_t)blockIdx.x * 4;
    uint64_t mine = 0;
#pragma unroll
    for (int q = 0; q < 4; ++q) {
        if (q < w) k += __popcll(m[q]);
        if (q == w) mine = m[q];
    }
    if (blockIdx.x == gridDim.x - 1 && threadIdx.x == 255) *total = k + __popcll(mine);
    if (!((mine >> lane) & 1)) return;
    k += __popcll(mine & ((1ull << lane) - 1));
    const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
    idx[k] = i;
    gx[k] = x[i];
    gy[k] = y[i];
    gz[k] = z[i];
    gh[k] = h[i];
}

__global__ void k_scatter_acc(const double *__restrict__ gax, const double *__restrict__ gay,
                              const double *__restrict__ gaz, const int64_t *__restrict__ idx,
                              int64_t na, double *__restrict__ ax,
                              double *__restrict__ ay, double *__restrict__ az) {
    const int64_t k = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (k >= na) return;
    const int64_t i = idx[k];
    ax[i] = gax[k];
    ay[i] = gay[k];
    az[i] = gaz[k];
}

__global__ void k_steps_in(const int64_t *__restrict__ e, const int64_t *__restrict__ b,
                           const int64_t *__restrict__ perm, int64_t n, int64_t *__restrict__ te,
                           int64_t *__restrict__ tb) {
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    const int64_t u = perm ? perm[i] : i;
    te[i] = e[u];
    tb[i] = b[u];
}

}  // namespace nb

using namespace nb;

namespace {

AdaptParams params_of(const nb_ctx *c) {
    AdaptParams p;
    p.time_interval = c->ad.time_interval;
    p.time_base = c->ad.time_base;
    p.err_tol = c->ad.err_tol;
    p.min_step = c->ad.min_step;
    p.max_step = c->ad.max_step;
    return p;
}

int check_adaptive(nb_ctx *c) {
    clear_error();
    if (!c) {
        set_error("null context");
        return NB_ERR_INVALID;
    }
    NB_HIP(hipSetDevice(c->dev));
    if (!c->uploaded) {
        set_error("no particle data uploaded");
        return NB_ERR_STATE;
    }
    if (!c->ad.red) {
        set_error("adaptive timesteps not initialised (call nb_adaptive_init)");
        return NB_ERR_STATE;
    }
    return NB_OK;
}

int flag_error(nb_ctx *c, unsigned f) {
    if (f) {
        NB_HIP(hipMemsetAsync(c->flag, 0, sizeof(unsigned), c->stream));
        NB_HIP(hipStreamSynchronize(c->stream));
        set_error(f & 1 ? "Timestep < MinStep" : "Wrong integer timestep");
        return NB_ERR_TIMESTEP;
    }
    return NB_OK;
}

int read_flag(nb_ctx *c) {
    unsigned f = 0;
    NB_HIP(hipMemcpyAsync(&f, c->flag, sizeof f, hipMemcpyDeviceToHost, c->stream));
    NB_HIP(hipStreamSynchronize(c->stream));
    return flag_error(c, f);
}

int min_blocks(const nb_ctx *c) {
    return (int)std::min<int64_t>(MINRED_BLOCKS, std::max<int64_t>(1, (c->n + 255) / 256));
}

// (minimum end step, particles at it, error flags) from the blocks' slots, once
// the kernel that wrote them has run.
int read_steps(nb_ctx *c, int64_t (&r)[3]) {
    NB_HIP(hipStreamSynchronize(c->stream));
    r[0] = c->ad.time_base;
    r[1] = r[2] = 0;
    for (int b = 0; b < min_blocks(c); ++b) {
        const int64_t *p = c->ad.red + 3 * b;
        if (p[0] < r[0]) {
            r[0] = p[0];
            r[1] = p[1];
        } else if (p[0] == r[0]) {
            r[1] += p[1];
        }
        r[2] |= p[2];
    }
    return NB_OK;
}

}  // namespace

extern "C" {

int nb_adaptive_init(nb_ctx *c, double time_interval, int64_t time_base, double err_tol,
                     double min_step, double max_step) {
    clear_error();
    if (!c) {
        set_error("null context");
        return NB_ERR_INVALID;
    }
    NB_HIP(hipSetDevice(c->dev));
    if (!c->uploaded) {
        set_error("no particle data uploaded");
        return NB_ERR_STATE;
    }
    if (!(time_interval > 0.0) || time_base <= 0 || !(err_tol > 0.0) || !(min_step >= 0.0) ||
        !(max_step > 0.0)) {
        set_error("invalid adaptive timestep parameters");
        return NB_ERR_INVALID;
    }
    c->ad.next_valid = false;
    c->ad.time_interval = time_interval;
    c->ad.time_base = time_base;
    c->ad.err_tol = err_tol;
    c->ad.min_step = min_step;
    c->ad.max_step = max_step;
    const size_t n = (size_t)std::max<int64_t>(c->n, 1);
    if (!c->ad.red) {   // (the last of the allocations: a call that failed among them starts over)
        dfree(c->ti_end); dfree(c->ti_beg);
        dfree(c->ad.mask); dfree(c->ad.count); dfree(c->ad.before); dfree(c->ad.idx); dfree(c->ad.cnt); dfree(c->ad.buf);
        NB_TRY(dalloc(&c->ti_end, sizeof(int64_t) * n));
        NB_TRY(dalloc(&c->ti_beg, sizeof(int64_t) * n));
        const size_t nblk = (n + 255) / 256;
        NB_TRY(dalloc(&c->ad.mask, sizeof(uint64_t) * 4 * nblk));
        NB_TRY(dalloc(&c->ad.count, sizeof(int) * nblk));
        if (nblk >= SCAN_FROM) NB_TRY(dalloc(&c->ad.before, sizeof(int64_t) * nblk));
        NB_TRY(dalloc(&c->ad.idx, sizeof(int64_t) * n));
        NB_TRY(dalloc(&c->ad.cnt, sizeof(int64_t) * 2));
        NB_TRY(dalloc(&c->ad.buf, sizeof(double) * 7 * n));
        NB_HIP(hipHostMalloc((void **)&c->ad.red, sizeof(int64_t) * 3 * MINRED_BLOCKS, hipHostMallocDefault));
    }
    NB_HIP(hipMemsetAsync(c->flag, 0, sizeof(unsigned), c->stream));
    if (c->n > 0) {
        k_init_timesteps<double><<<gridn(c->n), 256, 0, c->stream>>>(
            c->ax, c->ay, c->az, c->h, c->n, params_of(c), c->ti_end, c->ti_beg, c->flag);
        NB_TRY(launch_ok("k_init_timesteps"));
    }
    return read_flag(c);
}

int nb_adaptive_half_kick(nb_ctx *c, int32_t forward) {
    NB_TRY(check_adaptive(c));
    if (forward != 1 && forward != -1) {
        set_error("forward must be +1 or -1");
        return NB_ERR_INVALID;
    }
    if (c->n == 0) return NB_OK;
    if (c->is_double)
        k_adaptive_half_kick<double><<<gridn(c->n), 256, 0, c->stream>>>(
            (double *)c->vx, (double *)c->vy, (double *)c->vz, c->ax, c->ay, c->az, c->ti_end,
            c->ti_beg, c->n, (double)forward, c->ad.time_interval);
    else
        k_adaptive_half_kick<float><<<gridn(c->n), 256, 0, c->stream>>>(
            (float *)c->vx, (float *)c->vy, (float *)c->vz, c->ax, c->ay, c->az, c->ti_end,
            c->ti_beg, c->n, (double)forward, c->ad.time_interval);
    return launch_ok("k_adaptive_half_kick");
}

int nb_adaptive_min_endstep(nb_ctx *c, int64_t *min_endstep) {
    NB_TRY(check_adaptive(c));
    if (!min_endstep) {
        set_error("null output");
        return NB_ERR_INVALID;
    }
    // after a kick the reduction has already been read back with its flag
    if (!c->ad.next_valid) {
        int64_t r[3];
        k_min_count<<<min_blocks(c), 256, 0, c->stream>>>(c->ti_end, c->n, c->ad.time_base, c->ad.red);
        NB_TRY(launch_ok("k_min_count"));
        NB_TRY(read_steps(c, r));
        c->ad.next_min = r[0];
        c->ad.next_count = r[1];
        c->ad.next_valid = true;
    }
    *min_endstep = c->ad.next_min;
    return NB_OK;
}

int nb_adaptive_drift(nb_ctx *c, int64_t from_int, int64_t to_int) {
    NB_TRY(check_adaptive(c));
    const double dt = (double)(to_int - from_int) * c->ad.time_interval;
    if (c->n == 0) return NB_OK;
    if (c->is_double)
        k_adaptive_drift<double><<<gridn(c->n), 256, 0, c->stream>>>(
            (double *)c->x, (double *)c->y, (double *)c->z, (const double *)c->vx,
            (const double *)c->vy, (const double *)c->vz, c->n, dt);
    else
        k_adaptive_drift<float><<<gridn(c->n), 256, 0, c->stream>>>(
            (float *)c->x, (float *)c->y, (float *)c->z, (const float *)c->vx,
            (const float *)c->vy, (const float *)c->vz, c->n, dt);
    return launch_ok("k_adaptive_drift");
}

int nb_adaptive_compute_force(nb_ctx *c, int64_t t_int, int64_t *nactive) {
    NB_TRY(check_adaptive(c));
    if (c->n == 0) {
        if (nactive) *nactive = 0;
        return NB_OK;
    }
    hipStream_t s = c->stream;
    const int64_t n = c->n;
    // The count is known without a wait when t_int is the minimum end step
    // reduced since Ti_endstep last changed (the usual block step); the
    // kernels below read the device count, which equals it.
    int64_t na = -1;
    if (c->ad.next_valid && t_int == c->ad.next_min) na = c->ad.next_count;
    if (na == n) {   // everyone active: the plain path
        if (nactive) *nactive = na;
        return ctx_run_force(c, false, true);
    }
    // ordered compaction of the active particles (deterministic)
    const unsigned nblk_n = gridn(n);
    const int64_t *before = nblk_n >= SCAN_FROM ? c->ad.before : nullptr;
    k_active_masks<<<nblk_n, 256, 0, s>>>(c->ti_end, n, t_int, c->ad.mask, c->ad.count);
    NB_TRY(launch_ok("k_active_masks"));
    if (before) {
        k_scan_counts<<<1, SCAN_THREADS, 0, s>>>(c->ad.count, (int)nblk_n, c->ad.before);
        NB_TRY(launch_ok("k_scan_counts"));
    }
    double *gh = c->ad.buf;
    double *gax = gh + n, *gay = gax + n, *gaz = gay + n;
    void *gx = gaz + n;
    void *gy = (char *)gx + (c->is_double ? 8 : 4) * (size_t)n;
    void *gz = (char *)gy + (c->is_double ? 8 : 4) * (size_t)n;
    if (c->is_double)
        k_gather_active<double><<<nblk_n, 256, 0, s>>>(
            (const double *)c->x, (const double *)c->y, (const double *)c->z, c->h, n, c->ad.mask, c->ad.count,
            before, c->ad.idx, c->ad.cnt, (double *)gx, (double *)gy, (double *)gz, gh);
    else
        k_gather_active<float><<<nblk_n, 256, 0, s>>>(
            (const float *)c->x, (const float *)c->y, (const float *)c->z, c->h, n, c->ad.mask, c->ad.count,
            before, c->ad.idx, c->ad.cnt, (float *)gx, (float *)gy, (float *)gz, gh);
    NB_TRY(launch_ok("k_gather_active"));
    if (na < 0) {
        NB_HIP(hipMemcpyAsync(&na, c->ad.cnt, sizeof na, hipMemcpyDeviceToHost, s));
        NB_HIP(hipStreamSynchronize(s));
    }
    if (nactive) *nactive = na;
    if (na == 0) return NB_OK;
    if (na == n) return ctx_run_force(c, false, true);
    NB_TRY(launch_tile_boxes(c->x, c->y, c->z, c->is_double, n, c->h, 0.0, c->tile_box, c->sub_box, s));
    // Few active targets still fill the GPU: the sources are split into segments
    // (partials reduced in a fixed order).  Below 2^14 targets the matrix-core
    // path gives way to the wavefront kernel, whose segments go down to one
    // quarter: 20 targets among 60000 took 52 us in 59 blocks, 8.7 us here.
    // Above, about 16384 blocks even out the last round (4180 blocks on the 1024
    // that fit: five rounds for four), with the target geometry stored once; the
    // wavefront kernel takes them too once its waves walk whole segments (49500 /
    // 64900 targets 0.94 / 1.47 ms in 2048 blocks, 0.83 / 1.34 in 12500 and more).
    const int64_t nblk = (na + BS - 1) / BS, rounds = std::min<int64_t>((16384 + nblk - 1) / nblk, 64);
    int far = c->is_double || c->tun.far_path == FAR_MFMA_BF16 ? c->tun.far_path : FAR_VALU;
    if (far == FAR_MFMA_BF16 && na < (1 << 14)) far = FAR_VALU;
    const Geometry g = c->mode != NB_MODE_FP64 && wave_path(far, 1, false, true)
                           ? wave_launch_geometry(na, n, na < WAVE_SPLIT_BELOW ? 1 : rounds, 256)
                           : geometry(na, n, 1, rounds);
    const int nseg = g.nseg;
    // (the buffer holds part_cap segments of n targets)
    NB_TRY(ctx_ensure_part(c, (int)std::max<int64_t>((na * nseg + n - 1) / n, 2)));
    const bool central = c->mode == NB_MODE_SPLIT_CENTRAL && c->ncentral > 0;
    // the segments' sums go straight to the particles when nothing follows
    const bool direct = nseg > 1 && !central && c->bg.empty() && !(c->mond_acc0 > 0.0);
    auto common = [&](auto &a) {
        a.th = gh; a.nt = na; a.ns = n;
        a.tile_box = c->tile_box; a.sub_box = c->sub_box;
        a.nseg = nseg; a.seg_len = g.seg_len; a.nblk_i = g.nblk_i; a.wave_split = g.wave_split; a.G = c->G;
        a.ax = gax; a.ay = gay; a.az = gaz; a.pot = nullptr; a.part = c->part;
        if (nblk * nseg >= 2048) {
            a.tgeo = c->tgeo;
            a.tbg = c->tbg;
            a.nflag = c->nflag_cap >= (size_t)(nblk * nseg * NW) ? c->nflag : nullptr;
        }
    };
    if (far_path_weighted(far) && c->mode != NB_MODE_FP64) NB_TRY(ctx_ensure_source_weights(c));
    if (c->is_double) {
        ForceArgs<double> a{};
        common(a);
        a.tx = (const double *)gx; a.ty = (const double *)gy; a.tz = (const double *)gz;
        a.sx = (const double *)c->x; a.sy = (const double *)c->y; a.sz = (const double *)c->z;
        a.sm = (const double *)c->m;
        a.use_origin = 1;
        a.skip_src = central ? c->central : nullptr;
        if (c->mode == NB_MODE_FP64) {
            NB_TRY(launch_force_f64(a, false, s));
        } else {
            if (far_path_weighted(far)) a.sw = c->wsrc;
            NB_TRY(launch_force_split(a, 1, false, s, far));
        }
        if (nseg > 1 && !direct)
            NB_TRY(launch_finalize(c->part, nseg, na, c->G, gax, gay, gaz, nullptr, false, s));
        if (central) {
            // FP64 central terms for the active targets
            ForceArgs<double> b = a;
            b.sx = c->cx; b.sy = c->cy; b.sz = c->cz; b.sm = c->cm; b.ns = c->ncentral;
            b.skip_src = nullptr; b.tile_box = nullptr; b.sub_box = nullptr; b.accumulate = 1;
            b.nseg = 1; b.part = nullptr;
            b.seg_len = ((c->ncentral + BS - 1) / BS) * BS;
            NB_TRY(ctx_gather_central(c));
            NB_TRY(launch_force_f64(b, false, s));
        }
    } else {
        ForceArgs<float> a{};
        common(a);
        a.tx = (const float *)gx; a.ty = (const float *)gy; a.tz = (const float *)gz;
        a.sx = (const float *)c->x; a.sy = (const float *)c->y; a.sz = (const float *)c->z;
        a.sm = (const float *)c->m;
        a.use_origin = 0;
        if (far == FAR_MFMA_BF16) a.sw = c->wsrc;
        NB_TRY(launch_force_f32(a, 1, false, s, true, far));
        if (nseg > 1 && !direct)
            NB_TRY(launch_finalize(c->part, nseg, na, c->G, gax, gay, gaz, nullptr, false, s));
    }
    if (direct)
        return launch_finalize(c->part, nseg, na, c->G, c->ax, c->ay, c->az, nullptr, false, s, true, c->ad.idx);
    // post-processing of the active targets, in the order of
    // src/base/PostProcessing/Force.jl:33-46: background fields, then MOND
    for (const BgField &f : c->bg)
        NB_TRY(background(gx, gy, gz, na, c->is_double, f, gax, gay, gaz, nullptr, s));
    if (c->mond_acc0 > 0.0) NB_TRY(mond(gax, gay, gaz, na, c->mond_acc0, c->mond_index, s));
    k_scatter_acc<<<gridn(na), 256, 0, s>>>(gax, gay, gaz, c->ad.idx, na, c->ax, c->ay, c->az);
    NB_TRY(launch_ok("k_scatter_acc"));
    return NB_OK;
}

int nb_adaptive_kick(nb_ctx *c, int64_t t_int) {
    NB_TRY(check_adaptive(c));
    if (c->n == 0) return NB_OK;
    c->ad.next_valid = false;
    if (c->is_double)
        k_adaptive_advance<double><<<min_blocks(c), 256, 0, c->stream>>>(
            (double *)c->vx, (double *)c->vy, (double *)c->vz, c->ax, c->ay, c->az, c->h, c->ti_end,
            c->ti_beg, c->n, t_int, params_of(c), c->ad.red);
    else
        k_adaptive_advance<float><<<min_blocks(c), 256, 0, c->stream>>>(
            (float *)c->vx, (float *)c->vy, (float *)c->vz, c->ax, c->ay, c->az, c->h, c->ti_end,
            c->ti_beg, c->n, t_int, params_of(c), c->ad.red);
    NB_TRY(launch_ok("k_adaptive_advance"));
    // the new timeline's next sync point comes back with the error flags
    int64_t r[3];
    NB_TRY(read_steps(c, r));
    NB_TRY(flag_error(c, (unsigned)r[2]));
    c->ad.next_min = r[0];
    c->ad.next_count = r[1];
    c->ad.next_valid = true;
    return NB_OK;
}

int nb_adaptive_set_steps(nb_ctx *c, const int64_t *endstep, const int64_t *begstep) {
    NB_TRY(check_adaptive(c));
    c->ad.next_valid = false;
    const int64_t n = c->n;
    if (n == 0) return NB_OK;
    if (!endstep || !begstep) {
        set_error("endstep and begstep are required");
        return NB_ERR_INVALID;
    }
    for (int64_t i = 0; i < n; ++i) {
        if (begstep[i] < 0 || endstep[i] < begstep[i] || endstep[i] > c->ad.time_base) {
            set_error("step %lld: begstep %lld / endstep %lld outside 0 <= beg <= end <= TimeBase",
                      (long long)i, (long long)begstep[i], (long long)endstep[i]);
            return NB_ERR_INVALID;
        }
    }
    // staging: the gathered-target buffer holds 7n doubles, 2n int64 fit
    int64_t *se = (int64_t *)c->ad.buf, *sb = se + n;
    NB_HIP(hipMemcpyAsync(se, endstep, sizeof(int64_t) * n, hipMemcpyHostToDevice, c->stream));
    NB_HIP(hipMemcpyAsync(sb, begstep, sizeof(int64_t) * n, hipMemcpyHostToDevice, c->stream));
    k_steps_in<<<gridn(n), 256, 0, c->stream>>>(se, sb, c->perm, n, c->ti_end, c->ti_beg);
    NB_TRY(launch_ok("k_steps_in"));
    NB_HIP(hipStreamSynchronize(c->stream));
    return NB_OK;
}

int nb_adaptive_get_steps(nb_ctx *c, int64_t *endstep, int64_t *begstep) {
    NB_TRY(check_adaptive(c));
    const int64_t n = c->n;
    if (n == 0) return NB_OK;
    std::vector<int64_t> e((size_t)n), b((size_t)n), perm;
    NB_HIP(hipMemcpyAsync(e.data(), c->ti_end, sizeof(int64_t) * n, hipMemcpyDeviceToHost, c->stream));
    NB_HIP(hipMemcpyAsync(b.data(), c->ti_beg, sizeof(int64_t) * n, hipMemcpyDeviceToHost, c->stream));
    if (c->perm) {
        perm.resize((size_t)n);
        NB_HIP(hipMemcpyAsync(perm.data(), c->perm, sizeof(int64_t) * n, hipMemcpyDeviceToHost,
                              c->stream));
    }
    NB_HIP(hipStreamSynchronize(c->stream));
    for (int64_t i = 0; i < n; ++i) {
        const int64_t u = c->perm ? perm[(size_t)i] : i;
        if (endstep) endstep[u] = e[(size_t)i];
        if (begstep) begstep[u] = b[(size_t)i];
    }
    return NB_OK;
}

}  // extern "C"
