// nb_sort.hip -- Morton (Z-order) reordering of the internal particle order.
//
// Spatially sorted particles make each target block and each source tile
// compact: the per-block FP32 origin then resolves close pairs to the block's
// extent, and most (block, tile) pairs are separated by more than the
// softening length, so they take the unchecked Newtonian path.  The caller's
// order is kept in `perm` (internal -> caller index); downloads scatter back.
// No reference counterpart: the reference evaluates particles in input order.
#include <hip/hip_runtime.h>
#include <cstring>
#include <rocprim/device/device_radix_sort.hpp>

#include "nb_block.h"
#include "nb_ctx.h"

namespace nb {

static int check_launch(const char *what) {
    hipError_t e = hipGetLastError();
    if (e != hipSuccess) {
        set_error("launch of %s failed: %s", what, hipGetErrorString(e));
        return NB_ERR_HIP;
    }
    return NB_OK;
}

// Global box from the per-tile boxes (one block, fixed order).
__global__ __launch_bounds__(256) void k_global_box(const double *__restrict__ tb, int64_t ntiles,
                                                    double *__restrict__ box) {
    __shared__ double red[6][256];
    double v[6] = {1e300, 1e300, 1e300, -1e300, -1e300, -1e300};
    for (int64_t t = threadIdx.x; t < ntiles; t += 256) {
#pragma unroll
        for (int d = 0; d < 3; ++d) {
            v[d] = fmin(v[d], tb[t * 8 + d]);
            v[3 + d] = fmax(v[3 + d], tb[t * 8 + 3 + d]);
        }
    }
#pragma unroll
    for (int q = 0; q < 6; ++q) red[q][threadIdx.x] = v[q];
    __syncthreads();
    for (int off = 128; off > 0; off >>= 1) {
        if ((int)threadIdx.x < off) {
#pragma unroll
            for (int q = 0; q < 3; ++q) red[q][threadIdx.x] = fmin(red[q][threadIdx.x], red[q][threadIdx.x + off]);
#pragma unroll
            for (int q = 3; q < 6; ++q) red[q][threadIdx.x] = fmax(red[q][threadIdx.x], red[q][threadIdx.x + off]);
        }
        __syncthreads();
    }
    if (threadIdx.x < 6) box[threadIdx.x] = red[threadIdx.x][0];
}

__device__ __forceinline__ uint64_t spread21(uint64_t v) {
    v &= 0x1fffff;
    v = (v | (v << 32)) & 0x1f00000000ffffULL;
    v = (v | (v << 16)) & 0x1f0000ff0000ffULL;
    v = (v | (v << 8)) & 0x100f00f00f00f00fULL;
    v = (v | (v << 4)) & 0x10c30c30c30c30c3ULL;
    v = (v | (v << 2)) & 0x1249249249249249ULL;
    return v;
}

// Morton key of a position in the box (lo xyz, hi xyz).
__device__ __forceinline__ uint64_t morton_key(const double (&p)[3], const double *box) {
    const double scale = 2097151.0;  // 2^21 - 1
    uint64_t c[3];
#pragma unroll
    for (int d = 0; d < 3; ++d) {
        const double lo = box[d], ext = box[3 + d] - box[d];
        double u = ext > 0.0 ? (p[d] - lo) / ext : 0.0;
        u = fmin(fmax(u, 0.0), 1.0);
        c[d] = (uint64_t)(u * scale);
    }
    return spread21(c[0]) | (spread21(c[1]) << 1) | (spread21(c[2]) << 2);
}

template <typename T>
__global__ void k_morton(const T *__restrict__ x, const T *__restrict__ y, const T *__restrict__ z,
                         int64_t n, const double *__restrict__ box, uint64_t *__restrict__ key,
                         int64_t *__restrict__ idx) {
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    const double p[3] = {(double)x[i], (double)y[i], (double)z[i]};
    key[i] = morton_key(p, box);
    idx[i] = i;
}

// The particle arrays that follow a re-sort, gathered by one permutation in
// one pass (elements of 1, 4 or 8 bytes) into their own areas of the spare
// buffer, then copied back in a second pass: two launches for all of them.
// The last one is the permutation to the caller's order (perm_old, or, when
// null, the identity).
constexpr int MAX_SORTED_ARRAYS = 17;
struct GatherSet {
    void *arr[MAX_SORTED_ARRAYS];
    int64_t off[MAX_SORTED_ARRAYS];   // byte offset of the array's area in the spare buffer
    int size[MAX_SORTED_ARRAYS];      // bytes per element
    int count;
    const int64_t *perm_old;
};

// Element k of array a to element i of its area in the spare buffer.
__device__ __forceinline__ void gather_one(const GatherSet &g, int a, int64_t k, int64_t i, char *__restrict__ spare) {
    char *dst = spare + g.off[a];
    if (a == g.count - 1) ((int64_t *)dst)[i] = g.perm_old ? g.perm_old[k] : k;
    else if (g.size[a] == 8) ((uint64_t *)dst)[i] = ((const uint64_t *)g.arr[a])[k];
    else if (g.size[a] == 4) ((uint32_t *)dst)[i] = ((const uint32_t *)g.arr[a])[k];
    else ((uint8_t *)dst)[i] = ((const uint8_t *)g.arr[a])[k];
}

// (blockIdx.y: the array.  A loop over the arrays in each thread waited for one
// array's loads after the other: the copy back of 1000 particles took 6.5 us.)
__global__ void k_gather_set(GatherSet g, const int64_t *__restrict__ idx, int64_t n,
                             char *__restrict__ spare) {
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) gather_one(g, blockIdx.y, idx[i], i, spare);
}

// The whole order of a small system in one launch, up to the copy back: every
// workgroup finds the box and all keys for itself (positions come from the L2),
// its 64 particles' places are the numbers of smaller keys (of equal ones, those
// before it: the order of a stable sort), counted by its 16 waves, and each
// wave moves some of the arrays there.  Small systems are bound by launches:
// with the box, key, sort, gather, permutation and copy kernels launched one by
// one a re-sort was eight to ten of them, about 36 us; a step with one re-sort in
// sixteen took 12.3 us at 300 particles, 13.3 at 1000, 24.0 at 4096 and 43.0 at
// 8000 with them, 10.5, 11.6, 21.8 and 41.0 with this one (13 us at 1000, 22 at 4096) and the copy
// back.
// Every workgroup reads all positions, so the gain falls with n (and the keys
// have to fit the LDS): RANK_UPTO.
constexpr int RANK_WAVES = 16;
constexpr int64_t RANK_UPTO = 8192;   // keys in LDS
template <typename T>
__global__ __launch_bounds__(64 * RANK_WAVES) void k_rank_gather(GatherSet g, const T *__restrict__ x,
                                                                 const T *__restrict__ y, const T *__restrict__ z,
                                                                 int n, char *__restrict__ spare) {
    __shared__ uint64_t key[RANK_UPTO];
    __shared__ double red[RANK_WAVES][6];
    __shared__ int below[RANK_WAVES][64];
    constexpr int TH = 64 * RANK_WAVES, PER = RANK_UPTO / TH;
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
    // the positions: all loads in flight at once (past the end: the last one's)
    T p[PER][3];
#pragma unroll
    for (int u = 0; u < PER; ++u) {
        if (u * TH >= n) break;
        const int i = u * TH + threadIdx.x < n ? u * TH + threadIdx.x : n - 1;
        p[u][0] = x[i];
        p[u][1] = y[i];
        p[u][2] = z[i];
    }
    double v[6] = {1e300, 1e300, 1e300, -1e300, -1e300, -1e300};
#pragma unroll
    for (int u = 0; u < PER; ++u) {
        if (u * TH >= n) break;
#pragma unroll
        for (int d = 0; d < 3; ++d) {
            v[d] = fmin(v[d], (double)p[u][d]);
            v[3 + d] = fmax(v[3 + d], (double)p[u][d]);
        }
    }
#pragma unroll
    for (int d = 0; d < 3; ++d) {
        v[d] = wave_min(v[d]);
        v[3 + d] = wave_max(v[3 + d]);
    }
    if (lane == 0) {
#pragma unroll
        for (int d = 0; d < 6; ++d) red[w][d] = v[d];
    }
    __syncthreads();
#pragma unroll
    for (int d = 0; d < 3; ++d) {   // (one wave's result per lane, repeated)
        v[d] = wave_min(red[lane % RANK_WAVES][d]);
        v[3 + d] = wave_max(red[lane % RANK_WAVES][3 + d]);
    }
#pragma unroll
    for (int u = 0; u < PER; ++u) {
        if (u * TH >= n) break;
        const double q[3] = {(double)p[u][0], (double)p[u][1], (double)p[u][2]};
        if (u * TH + (int)threadIdx.x < n) key[u * TH + threadIdx.x] = morton_key(q, v);
    }
    __syncthreads();
    const int i0 = blockIdx.x * 64, i = i0 + lane;
    const uint64_t mine = i < n ? key[i] : 0;
    const int per = (n + RANK_WAVES - 1) / RANK_WAVES;
    const int j0 = per * w < n ? per * w : n, j1 = j0 + per < n ? j0 + per : n;
    int count = 0;
    // before these 64, among them, and after them (one broadcast LDS read per key
    // and wave; ballots over 64 keys at a time took twice as long)
    const int a1 = j1 < i0 ? j1 : i0;
#pragma unroll 16
    for (int j = j0; j < a1; ++j) count += key[j] <= mine;
    const int b0 = j0 > i0 ? j0 : i0, b1 = j1 < i0 + 64 ? j1 : i0 + 64;
#pragma unroll 4
    for (int j = b0; j < b1; ++j) count += key[j] < mine || (key[j] == mine && j < i);
#pragma unroll 16
    for (int j = j0 > i0 + 64 ? j0 : i0 + 64; j < j1; ++j) count += key[j] < mine;
    below[w][lane] = count;
    __syncthreads();
    int place = 0;
#pragma unroll
    for (int u = 0; u < RANK_WAVES; ++u) place += below[u][lane];
    if (i >= n) return;
    for (int a = w; a < g.count; a += RANK_WAVES) gather_one(g, a, i, place, spare);
}

__global__ void k_copy_back_set(GatherSet g, int64_t n, const char *__restrict__ spare) {
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    const int a = blockIdx.y;
    const char *src = spare + g.off[a];
    if (g.size[a] == 8) ((uint64_t *)g.arr[a])[i] = ((const uint64_t *)src)[i];
    else if (g.size[a] == 4) ((uint32_t *)g.arr[a])[i] = ((const uint32_t *)src)[i];
    else ((uint8_t *)g.arr[a])[i] = ((const uint8_t *)src)[i];
}

// Bytes of spare buffer for the largest set, of 8-byte elements.
static size_t spare_bytes(int64_t n) { return (size_t)MAX_SORTED_ARRAYS * 8 * (size_t)n; }

static void add_array(GatherSet &g, void *arr, int size, int64_t n) {
    const int64_t off = g.count ? g.off[g.count - 1] + ((g.size[g.count - 1] * n + 7) / 8) * 8 : 0;
    g.arr[g.count] = arr;
    g.off[g.count] = off;
    g.size[g.count] = size;
    ++g.count;
}

// The order of the Morton keys, in the second half of S.idx.
static int sort_keys(nb_ctx *c) {
    const int64_t n = c->n;
    hipStream_t s = c->stream;
    SortState &S = c->sort;
    if (!S.tmp) {
        dfree(S.keys); dfree(S.idx); dfree(S.box);
        NB_TRY(dalloc(&S.keys, sizeof(uint64_t) * 2 * (size_t)n));
        NB_TRY(dalloc(&S.idx, sizeof(int64_t) * 2 * (size_t)n));
        NB_TRY(dalloc(&S.box, sizeof(double) * 8));
        size_t bytes = 0;
        NB_HIP(rocprim::radix_sort_pairs(nullptr, bytes, S.keys, S.keys + n, S.idx, S.idx + n,
                                         (size_t)n, 0, 63, s));
        NB_TRY(dalloc(&S.tmp, bytes));
        S.tmp_bytes = bytes;
    }
    const int64_t ntiles = (n + BS - 1) / BS;
    NB_TRY(launch_tile_boxes(c->x, c->y, c->z, c->is_double, n, nullptr, 0.0, c->tile_box, nullptr, s));
    k_global_box<<<1, 256, 0, s>>>(c->tile_box, ntiles, S.box);
    NB_TRY(check_launch("k_global_box"));
    const unsigned g = (unsigned)((n + 255) / 256);
    if (c->is_double)
        k_morton<double><<<g, 256, 0, s>>>((const double *)c->x, (const double *)c->y,
                                           (const double *)c->z, n, S.box, S.keys, S.idx);
    else
        k_morton<float><<<g, 256, 0, s>>>((const float *)c->x, (const float *)c->y,
                                          (const float *)c->z, n, S.box, S.keys, S.idx);
    NB_TRY(check_launch("k_morton"));
    size_t bytes = S.tmp_bytes;
    NB_HIP(rocprim::radix_sort_pairs(S.tmp, bytes, S.keys, S.keys + n, S.idx, S.idx + n, (size_t)n,
                                     0, 63, s));
    return NB_OK;
}

int morton_reorder(nb_ctx *c) {
    const int64_t n = c->n;
    if (n < 2) return NB_OK;
    hipStream_t s = c->stream;
    SortState &S = c->sort;
    const unsigned g = (unsigned)((n + 255) / 256);
    const bool small = n <= RANK_UPTO;
    if (!S.spare) NB_TRY(dalloc(&S.spare, spare_bytes(n)));
    GatherSet set{};
    const int es = c->is_double ? 8 : 4;
    for (void *a : {c->x, c->y, c->z, c->vx, c->vy, c->vz, c->m}) add_array(set, a, es, n);
    for (void *a : {(void *)c->h, (void *)c->ax, (void *)c->ay, (void *)c->az, (void *)c->pot}) add_array(set, a, 8, n);
    if (c->coll) add_array(set, c->coll, 1, n);
    if (c->central) add_array(set, c->central, 1, n);
    if (c->ad.red) {
        add_array(set, c->ti_end, 8, n);
        add_array(set, c->ti_beg, 8, n);
    }
    // internal position i takes old position idx[i]; perm_new[i] = perm_old[idx[i]]
    int64_t *perm = c->perm;
    if (!perm) NB_TRY(dalloc(&perm, sizeof(int64_t) * (size_t)n));
    set.perm_old = c->perm;
    add_array(set, perm, 8, n);
    auto gather = [&]() -> int {
        if (small) {
            const unsigned gr = (unsigned)((n + 63) / 64);
            if (c->is_double)
                k_rank_gather<double><<<gr, 64 * RANK_WAVES, 0, s>>>(set, (const double *)c->x, (const double *)c->y,
                                                                     (const double *)c->z, (int)n, (char *)S.spare);
            else
                k_rank_gather<float><<<gr, 64 * RANK_WAVES, 0, s>>>(set, (const float *)c->x, (const float *)c->y,
                                                                    (const float *)c->z, (int)n, (char *)S.spare);
            return check_launch("k_rank_gather");
        }
        NB_TRY(sort_keys(c));
        k_gather_set<<<dim3(g, set.count), 256, 0, s>>>(set, S.idx + n, n, (char *)S.spare);
        return check_launch("k_gather_set");
    };
    auto move = [&]() -> int {
        NB_TRY(gather());
        k_copy_back_set<<<dim3(g, set.count), 256, 0, s>>>(set, n, (const char *)S.spare);
        return check_launch("k_copy_back_set");
    };
    const int rc = move();
    if (rc != NB_OK) {
        if (!c->perm) dfree(perm);
        return rc;
    }
    c->perm = perm;
    NB_TRY(ctx_rebuild_central(c));
    S.valid = true;
    c->wsrc_valid = false;   // the source weights follow the masses' order
    return NB_OK;
}

void sort_free(nb_ctx *c) {
    SortState &S = c->sort;
    dfree(S.tmp);
    dfree(S.keys);
    dfree(S.idx);
    dfree(S.box);
    dfree(S.spare);
    S.tmp_bytes = 0;
    S.valid = false;
}

}  // namespace nb
