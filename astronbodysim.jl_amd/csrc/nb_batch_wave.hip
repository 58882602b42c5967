// nb_batch_wave.hip -- the ensemble's all-pairs kernel of far path 0 with one
// target per lane.
#include <hip/hip_runtime.h>
#include <stdint.h>

#include "nb_batch.h"
#include "nb_wave.h"

namespace nb {

// Far path 0 with one target per lane (wave_force): one workgroup per quarter
// (64 targets) of an item.  The system's source tiles are cut into PARTS parts, of
// which each of the W waves takes one, or two one after the other.  A part's FP64
// sums are its own, and the parts' are added pair by pair in order, so a system's
// bits depend on the system alone, not on W, which follows from the size of the
// whole ensemble.  A wave without a tile leaves at once: with one to four waves
// of eight at work on systems of one to four tiles, the others held the places of
// the next workgroups until the barrier (700 systems of 256 bodies 113 us a force).
// The origins, classes and FP32 sums of a tile are force_block's, so the results
// are too (but for the order of the FP64 sums).  Bound by FP32 VALU issue on large
// ensembles (2.85e12 pairs/s on the 512 clusters below); the block-wide
// persistent kernel that it replaced held a workgroup at its barriers for the
// slowest of four waves, and a small ensemble gave it few waves with long
// source loops: an item of 16384 sources took about 0.9 ms alone.
//
// The items come in order of cost, so the last workgroups are the shortest, and
// ITEM_RUN consecutive ones (quarters of one system, or of a few) run on the
// same XCD, whose L2 then holds their sources.  Runs of 8, 16 and 32 are alike
// (within 0.7 % on 512 clusters); 256 leave the XCDs unequal work (5 % slower).
//
// A force call with its tile boxes against that kernel (clusters of 256 to 16384
// bodies, log-uniform): 512 clusters 5.47 -> 5.13 ms, 200 2.30 -> 1.96, 64
// 1.16 -> 0.80, 32 1.05 -> 0.52, 8 0.48 -> 0.10; 700 systems of 256 bodies
// 56 -> 42 us, 6000 of 100 239 -> 147, 399 of 1 to 399 57 -> 37.
constexpr unsigned ITEM_RUN = 16, XCDS = 8;
constexpr int PARTS = 8;   // (of one tile at least: a system of few tiles has empty ones)
template <bool ACC, bool POT>
constexpr int NVALUES = (ACC ? 3 : 0) + (POT ? 1 : 0);

// The sums of quarter b of the items, by a whole workgroup.  LEAVE: its waves
// without a part end here; else every wave returns, by way of the same barriers.
template <bool ACC, bool POT, int W, bool LEAVE>
__device__ __forceinline__ void item_quarter(const BatchArgs &a, unsigned b, WaveStage<double> (&st)[W],
                                             double (&red)[W][NVALUES<ACC, POT>][64]) {
    constexpr int NV = NVALUES<ACC, POT>;
    constexpr int V0 = ACC ? 0 : 3;
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
    const int64_t item = a.items[b / NQ];
    const int s = (int)(item >> 32);
    const int64_t o0 = a.off[s], o1 = a.off[s + 1];
    const int64_t qt = (item & 0xffffffffll) * NQ + b % NQ;   // the targets' quarter of the system
    const int64_t i0 = o0 + qt * SB;
    if (i0 >= o1) return;   // (the whole workgroup)
    const int64_t i = i0 + lane;
    const int64_t ic = i < o1 ? i : o1 - 1;
    const int64_t tb = a.tile_base[s], nt = (o1 - o0 + BS - 1) / BS;
    const auto part = [&](int g) { return o0 + nt * g / PARTS * BS; };   // its first source
    constexpr int MINE = PARTS / W;
    static_assert(MINE == 1 || MINE == 2, "a wave takes one part or two");
    const int g0 = wave * MINE;
    const int64_t j0 = part(g0), jm = part(g0 + 1), j1 = g0 + MINE < PARTS ? part(g0 + MINE) : o1;
    unsigned busy = 0;   // the waves with a part
#pragma unroll
    for (int w = 0; w < W; ++w) busy |= (unsigned)(nt * w / W < nt * (w + 1) / W) << w;
    double v[4];   // ax, ay, az, pot
    if (LEAVE && j0 >= j1) return;   // (never the last wave, which adds up; a barrier waits for the waves that remain)
    if (j0 < j1) {
        wave_force<double, ACC, POT, true>(st[wave], a.x[ic], a.y[ic], a.z[ic], a.h[ic], nullptr, a.x, a.y, a.z, a.m,
                                           a.skip_src, a.sub_box + (tb * NQ + (j0 - o0) / SB) * 8, a.tile_box, j0,
                                           j1, v[0], v[1], v[2], v[3], a.tgeo + (tb + qt / NQ) * TG_STRIDE,
                                           (int)(qt % NQ), MINE == 2 ? (int)((jm - j0) / SB) - 1 : -1, red[wave]);
        if (MINE == 2 && jm > j0) {   // the pair's sum
#pragma unroll
            for (int q = 0; q < NV; ++q) v[V0 + q] = red[wave][q][lane] + v[V0 + q];
        }
#pragma unroll
        for (int q = 0; q < NV; ++q) red[wave][q][lane] = v[V0 + q];
    }
    __syncthreads();
    if (wave < W - 1) return;
#pragma unroll
    for (int q = 0; q < NV; ++q) v[V0 + q] = 0.0;
#pragma unroll
    for (int g = 0; g < PARTS; g += 2) {
        const int w = g / MINE;
#pragma unroll
        for (int q = 0; q < NV; ++q) {
            double p = busy >> w & 1 ? red[w][q][lane] : 0.0;
            if (MINE == 1) p += busy >> (w + 1) & 1 ? red[w + 1][q][lane] : 0.0;
            v[V0 + q] += p;
        }
    }
    if (i >= o1) return;
    const double G = a.Gs[s];
    if (ACC) {
        a.ax[i] = G * v[0];
        a.ay[i] = G * v[1];
        a.az[i] = G * v[2];
    }
    if (POT) a.pot[i] = -G * v[3];
}

// PERSISTENT: nb_batch_tuning.blocks workgroups go through the quarters, of eight
// waves each (64 clusters of 200 to 3000 bodies on 8 / 64 / 512 workgroups:
// 3.72 / 0.50 / 0.115 ms a force, by four waves 4.88 / 0.66 / 0.137).
template <bool ACC, bool POT, int W, bool PERSISTENT>
__global__ __launch_bounds__(64 * W) __attribute__((amdgpu_waves_per_eu(ACC &&POT ? 5 : 6)))
void k_batch_wave(BatchArgs a) {
    __shared__ WaveStage<double> st[W];
    __shared__ double red[W][NVALUES<ACC, POT>][64];
    if constexpr (PERSISTENT) {
        const unsigned total = (unsigned)(a.nitems * NQ);
        for (unsigned b = blockIdx.x; b < total; b += gridDim.x) {
            item_quarter<ACC, POT, W, false>(a, b, st, red);
            __syncthreads();   // red is read before the next quarter's sums
        }
    } else {
        unsigned b = blockIdx.x;
        if (b < gridDim.x / (ITEM_RUN * XCDS) * (ITEM_RUN * XCDS)) {
            const unsigned slot = b / XCDS;
            b = (slot / ITEM_RUN * XCDS + b % XCDS) * ITEM_RUN + slot % ITEM_RUN;
        }
        item_quarter<ACC, POT, W, true>(a, b, st, red);
    }
}

template <int W, bool PERSISTENT>
static void launch(const BatchArgs &a, bool pot, bool acc, unsigned nb, hipStream_t s) {
    const unsigned bs = 64 * W;
    if (pot && acc) k_batch_wave<true, true, W, PERSISTENT><<<nb, bs, 0, s>>>(a);
    else if (pot) k_batch_wave<false, true, W, PERSISTENT><<<nb, bs, 0, s>>>(a);
    else k_batch_wave<true, false, W, PERSISTENT><<<nb, bs, 0, s>>>(a);
}

// Four waves per 64 targets, or eight while the launch has fewer workgroups
// than this: eight / four waves took 48 / 62 us a force at 52 workgroups, 273 /
// 302 at 776 and 459 / 479 at 2100, but 713 / 710 at 3600 and 5.66 / 5.57 ms at
// 33000; sixteen were slower from 776 on (all timed in a form that split the
// sources by quarters instead of tiles).  Four also where no system has more than four tiles
// (1 to 399 bodies in 399 systems: 38 us by four waves, 41 by eight).
constexpr int64_t EIGHT_WAVES_BELOW = 3072;

int launch_batch_wave(const BatchArgs &a, int64_t max_n, int blocks, bool pot, bool acc, hipStream_t s) {
    if (a.nitems <= 0) return NB_OK;
    if (a.nitems * NQ > INT32_MAX) {
        set_error("ensemble force grid too large (%lld items)", (long long)a.nitems);
        return NB_ERR_INVALID;
    }
    const unsigned nb = (unsigned)(a.nitems * NQ);
    if (blocks > 0 && (unsigned)blocks < nb) launch<2 * NW, true>(a, pot, acc, (unsigned)blocks, s);
    else if (nb < EIGHT_WAVES_BELOW && max_n > NW * BS) launch<2 * NW, false>(a, pot, acc, nb, s);
    else launch<NW, false>(a, pot, acc, nb, s);
    hipError_t e = hipGetLastError();
    if (e != hipSuccess) {
        set_error("launch of k_batch_wave failed: %s", hipGetErrorString(e));
        return NB_ERR_HIP;
    }
    return NB_OK;
}

}  // namespace nb
