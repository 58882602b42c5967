// nb_force.hip -- all-pairs gravity kernels for one system (gfx950).
//
// Replaces compute_force_gpu_kernel  src/directsumgpu/gravity.jl:22-34 (one
// thread per target, sources re-read from global memory) with an LDS-tiled
// kernel: each block owns BS*TPT targets held in registers and streams the
// sources through a double-buffered LDS stage of BS particles; every lane
// reads the same source (LDS broadcast).  Pair arithmetic is FP32 (v_rsq_f32);
// each tile's FP32 partial sums are folded into FP64 accumulators.  The block
// routine itself, with its per-wave tile classes (softening-checked, hi/lo
// Newtonian, far) and the optional matrix-core far tiles, is force_block in
// nb_block.h.
#include <hip/hip_runtime.h>
#include <float.h>
#include <stdint.h>

#include "nb_block.h"
#include "nb_internal.h"
#include "nb_pair.h"
#include "nb_wave.h"

namespace nb {

// FP32-pair kernel.  T = double (SPLIT: FP64 state, per-block origin, hi/lo
// coordinates on near tiles) or float (FP32 state: absolute coordinates, or,
// with the bf16 far tiles, the SPLIT layout of the FP32 positions).  MF
// selects the matrix-core far tiles (TPT 1, forces or potentials alone).
// ACC = false writes the potential only.
// PASS: every tile (PASS_ALL), or the far half of a split bf16 launch
// (PASS_FAR): the far tiles' sums, with the waves that left near tiles out
// flagged in a.nflag (which holds zeros between launches) for k_force_near.
template <typename T, int TPT, bool POT, int MF = 0, bool ACC = true, int PASS = PASS_ALL>
__global__ __launch_bounds__(BS) __attribute__((amdgpu_waves_per_eu(MF == 4 ? 4 : 3))) void k_force_f32(ForceArgs<T> a) {
    __shared__ BlockShared<T, MF> sh;
    const int tid = threadIdx.x;
    const int logical = xcd_remap(blockIdx.x, gridDim.x);
    const int seg = logical / a.nblk_i;
    const int ib = logical - seg * a.nblk_i;
    const int64_t i0 = (int64_t)ib * (BS * TPT);
    const int64_t j0 = (int64_t)seg * a.seg_len;
    const int64_t j1 = (j0 + a.seg_len < a.ns) ? j0 + a.seg_len : a.ns;
    double Ax[TPT], Ay[TPT], Az[TPT], Aq[TPT];
    bool valid[TPT];
    const bool had_near = force_block<T, TPT, POT, MF, ACC, PASS>(sh, a.tx, a.ty, a.tz, a.th, a.th_const, i0, a.nt, a.sx, a.sy, a.sz,
                             a.sm, a.sw, j0, j1, a.tile_box + (j0 / BS) * 8,
                             a.sub_box ? a.sub_box + (j0 / BS) * (NQ * 8) : nullptr,
                             a.tgeo ? a.tgeo + (int64_t)ib * TG_STRIDE : nullptr,
                             a.tbg ? a.tbg + (int64_t)ib * BS * 16 : nullptr, a.skip_src,
                             a.use_origin != 0, Ax, Ay, Az, Aq, valid);
    // (one plain byte store per wave that left near tiles out)
    if (PASS == PASS_FAR && had_near && (tid & 63) == 0) a.nflag[(int64_t)logical * NW + (tid >> 6)] = 1;
#pragma unroll
    for (int k = 0; k < TPT; ++k) {
        if (!valid[k]) continue;
        const int64_t i = target_of<TPT>(i0, k, tid);
        if (a.nseg == 1) {
            if (ACC) {
                a.ax[i] = a.G * Ax[k];
                a.ay[i] = a.G * Ay[k];
                a.az[i] = a.G * Az[k];
            }
            if (POT) a.pot[i] = -a.G * Aq[k];
        } else {
            double *p = a.part + (int64_t)seg * 4 * a.nt;
            if (ACC) {
                p[i] = Ax[k];
                p[a.nt + i] = Ay[k];
                p[2 * a.nt + i] = Az[k];
            }
            if (POT) p[3 * a.nt + i] = Aq[k];
        }
    }
}

// Segments g, g + NW, ... of target i's partial sums (part: [nseg][4][n], from
// the first of the NV values on), in order.
// SHARED: other workgroups of this launch wrote them.
template <bool SHARED, int NV>
__device__ __forceinline__ void group_sums(const double *part, int64_t n, int nseg, int64_t i, int grp,
                                           double (&s)[NV]) {
    const double *p = part + i;
    constexpr int U = 4;   // segments in flight; past the end: the last one's, not added
    for (int g = grp; g < nseg; g += U * NW) {
        double t[U][NV];
#pragma unroll
        for (int u = 0; u < U; ++u) {
            const int gu = g + u * NW < nseg ? g + u * NW : nseg - 1;
#pragma unroll
            for (int q = 0; q < NV; ++q) {
                const double *e = p + ((int64_t)gu * 4 + q) * n;
                t[u][q] = SHARED ? __hip_atomic_load(e, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) : *e;
            }
        }
#pragma unroll
        for (int u = 0; u < U; ++u)
            if (g + u * NW < nseg) {
#pragma unroll
                for (int q = 0; q < NV; ++q) s[q] += t[u][q];
            }
    }
}

// The waves' values, added in order in wave 0.
template <int NV>
__device__ __forceinline__ void add_waves(double (&s)[NV], double (&red)[NW - 1][NV][64]) {
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    if (wave > 0) {
#pragma unroll
        for (int q = 0; q < NV; ++q) red[wave - 1][q][lane] = s[q];
    }
    __syncthreads();
    if (wave > 0) return;
#pragma unroll
    for (int w = 0; w < NW - 1; ++w)
#pragma unroll
        for (int q = 0; q < NV; ++q) s[q] += red[w][q][lane];
}

// The sums over all segments of target i (v: it exists), s being segment seg's
// in wave 0: true in wave 0 of the workgroup that is the last of its 64 targets'
// to arrive, whose s they then are (added as k_finalize adds them).
// The segments' sums cross XCDs: they are written and read as agent-scope
// atomics, which pass the XCDs' L2s by, and a workgroup counts itself in
// (arrived) once its own are written; the last one leaves the count at zero.
// (Plain stores between agent-scope fences write back and invalidate an L2 per
// workgroup: k_force_step on 4096 particles took 175 us.)
// The atomics are relaxed, so the language's memory model does not order the sums
// before the count: that rests on gfx950, where an agent-scope store is
// acknowledged (vmcnt) once it is past the L2, and an agent-scope load reads past
// it.  The wait below is the acknowledgement of every store of the wave.
template <int NV>
__device__ __forceinline__ bool last_arrival(double (&s)[NV], double *part, int64_t n, int nseg, int seg, int64_t i,
                                             bool v, unsigned *arrived, double (&red)[NW - 1][NV][64], int &last) {
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
    if (wave == 0) {
        if (v) {
            double *p = part + (int64_t)seg * 4 * n + i;
#pragma unroll
            for (int q = 0; q < NV; ++q) __hip_atomic_store(p + q * n, s[q], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        }
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");   // this wave's sums are written
        if (lane == 0) {
            last = __hip_atomic_fetch_add(arrived, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) ==
                   (unsigned)nseg - 1;
            if (last) *arrived = 0;
        }
    }
    __syncthreads();
    if (!last) return false;
#pragma unroll
    for (int q = 0; q < NV; ++q) s[q] = 0.0;
    if (v) group_sums<true>(part, n, nseg, i, wave, s);
    add_waves(s, red);
    return wave == 0;
}

// Far path 0 with one target per lane (wave_force).
// split = 0: wave w of workgroup ib owns the targets 64 (NW ib + w).. and walks
// the whole segment; the waves share the scalar cache's lines of its sources,
// nothing else.
// split = 1 (few targets): the waves share the targets 64 ib.. and take a part
// of the segment each, down to 16 sources, and their sums meet in LDS in a
// fixed order: the same waves on a quarter of the segments, so a quarter of the
// partial sums to write and to add up.
// FIN (split, several segments): the last workgroup of its 64 targets to arrive
// adds the segments' sums (last_arrival), which spares the launch of k_finalize.
// Held to 6 waves per SIMD (two values spilled outside the pair loops;
// 5 without): 60000 particles in FP32 986 -> 929 us a force, 30011 in split
// precision 312 -> 308 us.  Against the block-wide kernel that it replaced (one
// force call with its boxes and segment sums, split precision, Plummer): 1000
// particles 32 -> 12.5 us, 4096 35 -> 22, 16384 130 -> 106, 30011 333 -> 301;
// FP32 60000 1030 -> 929.
template <typename T, bool ACC, bool POT, bool FIN>
__global__ __launch_bounds__(BS) __attribute__((amdgpu_waves_per_eu(ACC &&POT && sizeof(T) == 8 ? 5 : 6)))
void k_force_wave(ForceArgs<T> a, int split) {
    constexpr int NV = (ACC ? 3 : 0) + (POT ? 1 : 0);
    __shared__ WaveStage<T> st[NW];
    __shared__ double red[NW - 1][NV][64];
    __shared__ int last;
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
    const int logical = xcd_remap(blockIdx.x, gridDim.x);
    const int seg = logical / a.nblk_i;
    const int ib = logical - seg * a.nblk_i;
    const int64_t i0 = split ? (int64_t)ib * 64 : (int64_t)ib * BS + wave * 64;
    if (i0 >= a.nt) return;   // (split: never)
    const int64_t i = i0 + lane;
    const int64_t ic = i < a.nt ? i : a.nt - 1;
    int64_t j0 = (int64_t)seg * a.seg_len;
    int64_t j1 = (j0 + a.seg_len < a.ns) ? j0 + a.seg_len : a.ns;
    if (split) {   // (segments of 1, 2 or a multiple of 4 quarters: no part starts inside a quarter and leaves it)
        const int64_t part = a.seg_len / NW;
        j0 = j0 + part * wave < j1 ? j0 + part * wave : j1;
        j1 = j0 + part < j1 ? j0 + part : j1;
    }
    constexpr int V0 = ACC ? 0 : 3;
    double v[4];   // ax, ay, az, pot
    wave_force<T, ACC, POT>(st[wave], a.tx[ic], a.ty[ic], a.tz[ic], a.th ? a.th[ic] : a.th_const,
                            a.tbox ? a.tbox + (i0 / 64) * 8 : nullptr, a.sx, a.sy, a.sz, a.sm, a.skip_src,
                            a.sub_box ? a.sub_box + (j0 / SB) * 8 : nullptr,
                            a.sub_box ? nullptr : a.tile_box + (j0 / BS) * 8, j0, j1, v[0], v[1], v[2], v[3]);
    double s[NV];
#pragma unroll
    for (int q = 0; q < NV; ++q) s[q] = v[V0 + q];
    if (split) {
        add_waves(s, red);
        if constexpr (FIN) {
            if (!last_arrival(s, a.part + V0 * a.nt, a.nt, a.nseg, seg, i, i < a.nt, a.arrived + ib, red, last)) return;
        } else {
            if (wave > 0) return;
        }
    }
    if (i >= a.nt) return;
    if (FIN || a.nseg == 1) {
        if (ACC) {
            a.ax[i] = a.G * s[0];
            a.ay[i] = a.G * s[1];
            a.az[i] = a.G * s[2];
        }
        if (POT) a.pot[i] = -a.G * s[NV - 1];
    } else {
        double *p = a.part + (int64_t)seg * 4 * a.nt;
#pragma unroll
        for (int q = 0; q < NV; ++q) p[(V0 + q) * a.nt + i] = s[q];
    }
}

template <typename T>
static void launch_wave(ForceArgs<T> a, bool pot, bool acc, hipStream_t s) {
    const int split = a.wave_split;
    if (split) a.nblk_i = (int)((a.nt + 63) / 64);
    const unsigned nb = (unsigned)((int64_t)a.nblk_i * a.nseg);
    const bool fin = split && a.nseg > 1 && a.arrived;
#define NB_W(A_, P_)                                                       \
    do {                                                                   \
        if (fin) k_force_wave<T, A_, P_, true><<<nb, BS, 0, s>>>(a, split); \
        else k_force_wave<T, A_, P_, false><<<nb, BS, 0, s>>>(a, split);    \
    } while (0)
    if (pot && acc) NB_W(true, true);
    else if (pot) NB_W(false, true);
    else NB_W(true, false);
#undef NB_W
}

// Near pass of a split bf16 launch (forces only): one wavefront per
// workgroup, one workgroup per (force block, wave) of the far pass.  The
// waves the far pass flagged add their near quarters (near_wave) to the same
// outputs and clear their flags; the rest return at once.  Each wave runs on
// its own, so a wave with many near tiles holds no other wave's resources.
template <typename T>
__global__ __launch_bounds__(64) void k_force_near(ForceArgs<T> a) {
    __shared__ NearShared<T, FAR_MFMA_BF16> sh;
    const int lw = xcd_remap(blockIdx.x, gridDim.x);
    if (!a.nflag[lw]) return;   // wave-uniform
    if (threadIdx.x == 0) a.nflag[lw] = 0;
    const int logical = lw / NW, wave = lw - logical * NW;
    const int seg = logical / a.nblk_i;
    const int ib = logical - seg * a.nblk_i;
    const int64_t i0 = (int64_t)ib * BS;
    const int64_t j0 = (int64_t)seg * a.seg_len;
    const int64_t j1 = (j0 + a.seg_len < a.ns) ? j0 + a.seg_len : a.ns;
    double Ax, Ay, Az;
    bool valid;
    near_wave<T, FAR_MFMA_BF16>(sh, wave, a.tx, a.ty, a.tz, a.th, a.th_const, i0, a.nt, a.sx, a.sy, a.sz, a.sm,
                                j0, j1, a.tile_box + (j0 / BS) * 8,
                                a.sub_box ? a.sub_box + (j0 / BS) * (NQ * 8) : nullptr,
                                a.tgeo + (int64_t)ib * TG_STRIDE, a.skip_src, Ax, Ay, Az, valid);
    if (!valid) return;
    const int64_t i = i0 + wave * 64 + (threadIdx.x & 63);
    if (a.nseg == 1) {
        a.ax[i] += a.G * Ax;
        a.ay[i] += a.G * Ay;
        a.az[i] += a.G * Az;
    } else {
        double *p = a.part + (int64_t)seg * 4 * a.nt;
        p[i] += Ax;
        p[a.nt + i] += Ay;
        p[2 * a.nt + i] += Az;
    }
}

// The bf16 matrix-core force launch (forces only, 1 target per lane): one
// kernel, or the far and near passes when the caller provides the flags
// and the target blocks' stored geometry (several source segments).
// The split pays where near tiles are few (FP64 state: the collision at 2^20
// has 1.8 % of its pairs in them, and its far loop alone runs about 10 %
// faster); with FP32 state (the FP32 Plummer sphere at 2^16: 18 %) the near
// pass cost more than it saved, so that launch stays in one kernel.
template <typename T>
static void launch_bf16_forces(const ForceArgs<T> &a, int64_t nb, hipStream_t s) {
    if constexpr (sizeof(T) == 8) {
        if (a.nflag && a.tgeo) {
            k_force_f32<T, 1, false, FAR_MFMA_BF16, true, PASS_FAR><<<(unsigned)nb, BS, 0, s>>>(a);
            k_force_near<T><<<(unsigned)(nb * NW), 64, 0, s>>>(a);
            return;
        }
    }
    k_force_f32<T, 1, false, FAR_MFMA_BF16><<<(unsigned)nb, BS, 0, s>>>(a);
}

// The origin and wave geometry of each target block (force_block's first
// steps), stored once per force call for launches whose target blocks meet
// several source segments.  hilo: the force kernel's near tiles have a
// close class (FP64 state).
template <typename T, int TPT, bool ROWS>
__global__ __launch_bounds__(BS) void k_target_geom(ForceArgs<T> a, bool hilo) {
    __shared__ double red[11][NW];
    const int tid = threadIdx.x;
    const int64_t i0 = (int64_t)blockIdx.x * (BS * TPT);
    double px[TPT], py[TPT], pz[TPT], ph[TPT];
    bool valid[TPT];
#pragma unroll
    for (int k = 0; k < TPT; ++k) {
        const int64_t i = target_of<TPT>(i0, k, tid);
        valid[k] = i < a.nt;
        px[k] = valid[k] ? (double)a.tx[i] : 0.0;
        py[k] = valid[k] ? (double)a.ty[i] : 0.0;
        pz[k] = valid[k] ? (double)a.tz[i] : 0.0;
        ph[k] = valid[k] ? (a.th ? a.th[i] : a.th_const) : 0.0;
    }
    BlockStats st;
    block_stats<TPT>(px, py, pz, ph, valid, a.use_origin != 0, red, st);
    const double ox = uniform_f64(st.ox), oy = uniform_f64(st.oy), oz = uniform_f64(st.oz);
    const WaveGeom wg = wave_geometry<TPT>(px, py, pz, ph, valid, ox, oy, oz, hilo);
    store_target_geom(a.tgeo + (int64_t)blockIdx.x * TG_STRIDE, ox, oy, oz, wg, tid >> 6, tid & 63);
    if constexpr (ROWS) {   // the lanes' bf16 B operands (TPT 1)
        nb_bf8 Bg[4];
        target_b_operands(px[0] - ox, py[0] - oy, pz[0] - oz, tid & 63, Bg);
        nb_u4v *b = reinterpret_cast<nb_u4v *>(a.tbg + ((int64_t)blockIdx.x * BS + tid) * 16);
#pragma unroll
        for (int g = 0; g < 4; ++g) b[g] = __builtin_bit_cast(nb_u4v, Bg[g]);
    }
}

// FP64-pair kernel (correctness mode, and the FP64 central-body terms).
// Bound by FP64 VALU issue: 16 FP64 operations, a v_rsq_f64 and a 32-bit range
// test per pair (newton_f64), where the former kernel spent about 60 on sqrt
// and divide.  A workgroup's four waves share 64 targets and take a quarter
// of the segment's sources each (their sums meet in LDS in a fixed order), so
// a small system still gives every SIMD waves: 2048 particles are 32 groups of
// targets and, in 32 segments, 1024 workgroups.  The source index is wave-uniform, so the
// sources come through scalar loads and sit in SGPRs: no LDS staging and no
// barrier in the loop.  Measured: 10007 particles 199 -> 92 us a launch, 2048
// (forces and potentials) 56 -> 14 us.  Where 64-target workgroups would be too many for one
// launch (split = 0) each wave has 64 targets of its own and the whole segment.
constexpr int F64_GROUP = 4;   // sources per softening test

template <bool POT>
__device__ __forceinline__ void sources_f64(const double *__restrict__ sx, const double *__restrict__ sy,
                                            const double *__restrict__ sz, const double *__restrict__ sm,
                                            int64_t j0, int64_t j1, double xi, double yi, double zi, double h,
                                            double &Ax, double &Ay, double &Az, double &Aq) {
    const double hinv = 1.0 / h, hinv3 = hinv * hinv * hinv;
    unsigned first, count;
    fast_f64_window(h, first, count);
    int64_t j = j0;
    for (; j + F64_GROUP <= j1; j += F64_GROUP) {
        double dx[F64_GROUP], dy[F64_GROUP], dz[F64_GROUP], fac[F64_GROUP], q[F64_GROUP];
        bool fast[F64_GROUP], all = true;
#pragma unroll
        for (int g = 0; g < F64_GROUP; ++g) {
            dx[g] = sx[j + g] - xi;
            dy[g] = sy[j + g] - yi;
            dz[g] = sz[j + g] - zi;
            const double r2 = r2_pair(dx[g], dy[g], dz[g]);
            fast[g] = fast_f64(r2, first, count);
            all = all && fast[g];
            newton_f64<POT>(r2, sm[j + g], fac[g], q[g]);
        }
        if (__builtin_expect(!all, 0)) {
#pragma unroll
            for (int g = 0; g < F64_GROUP; ++g)
                if (!fast[g]) terms_f64(dx[g], dy[g], dz[g], sm[j + g], h, hinv, hinv3, fac[g], q[g]);
        }
#pragma unroll
        for (int g = 0; g < F64_GROUP; ++g) {
            Ax = __builtin_fma(dx[g], fac[g], Ax);
            Ay = __builtin_fma(dy[g], fac[g], Ay);
            Az = __builtin_fma(dz[g], fac[g], Az);
            if (POT) Aq += q[g];
        }
    }
    for (; j < j1; ++j) pair_f64<POT>(sx[j], sy[j], sz[j], sm[j], xi, yi, zi, h, hinv, hinv3, Ax, Ay, Az, Aq);
}

// FIN (split, several segments): as in k_force_wave.
template <bool POT, bool FIN>
__global__ __launch_bounds__(BS) void k_force_f64(ForceArgs<double> a, int split) {
    constexpr int NV = POT ? 4 : 3;
    __shared__ double red[NW - 1][NV][64];
    __shared__ int last;
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
    const int logical = xcd_remap(blockIdx.x, gridDim.x);
    const int seg = logical / a.nblk_i;
    const int ib = logical - seg * a.nblk_i;
    const int64_t i = split ? (int64_t)ib * 64 + lane : (int64_t)ib * BS + threadIdx.x;
    const bool valid = i < a.nt;
    const double xi = valid ? a.tx[i] : 0.0, yi = valid ? a.ty[i] : 0.0, zi = valid ? a.tz[i] : 0.0;
    const double h = valid ? (a.th ? a.th[i] : a.th_const) : 1.0;
    double Ax = 0.0, Ay = 0.0, Az = 0.0, Aq = 0.0;
    int64_t j0 = (int64_t)seg * a.seg_len;
    int64_t j1 = (j0 + a.seg_len < a.ns) ? j0 + a.seg_len : a.ns;
    if (split) {
        const int64_t part = (j1 - j0 + NW - 1) / NW;
        j0 = j0 + part * wave < j1 ? j0 + part * wave : j1;
        j1 = j0 + part < j1 ? j0 + part : j1;
    }
    sources_f64<POT>(a.sx, a.sy, a.sz, a.sm, j0, j1, xi, yi, zi, h, Ax, Ay, Az, Aq);
    if (split) {   // (uniform over the launch)
        double v[NV] = {Ax, Ay, Az};
        if (POT) v[NV - 1] = Aq;
        add_waves(v, red);
        if constexpr (FIN) {
            if (!last_arrival(v, a.part, a.nt, a.nseg, seg, i, valid, a.arrived + ib, red, last)) return;
        } else {
            if (wave > 0) return;
        }
        Ax = v[0];
        Ay = v[1];
        Az = v[2];
        if (POT) Aq = v[NV - 1];
    }
    if (!valid) return;
    if (FIN || a.nseg == 1) {
        if (!FIN && a.accumulate) {
            a.ax[i] += Ax * a.G;
            a.ay[i] += Ay * a.G;
            a.az[i] += Az * a.G;
            if (POT) a.pot[i] -= Aq * a.G;
        } else {
            a.ax[i] = Ax * a.G;
            a.ay[i] = Ay * a.G;
            a.az[i] = Az * a.G;
            if (POT) a.pot[i] = -Aq * a.G;
        }
    } else {
        double *p = a.part + (int64_t)seg * 4 * a.nt;
        p[i] = Ax;
        p[a.nt + i] = Ay;
        p[2 * a.nt + i] = Az;
        if (POT) p[3 * a.nt + i] = Aq;
    }
}

// One target's per-segment partial sums, added by the W waves of a workgroup
// (64 targets): wave w takes the segments w, w + W, ..., and lane l of wave 0
// adds the waves' sums in order of w for target i, so results repeat.  Bound
// by the latency of the loads where n is small: one thread per target walked
// all the segments serially on n / 256 workgroups.  Four waves up to 64
// segments; the hundreds that a few probe points take get sixteen (782
// segments x 1009 points: 27 -> 20 us).
constexpr int FIN_WAVES = 4, FIN_WAVES_MANY = 16, FIN_MANY = 64;

template <bool ACC, bool POT>
struct PartSums {
    static constexpr int NV = (ACC ? 3 : 0) + (POT ? 1 : 0);
    double v[NV];
};
template <bool ACC, bool POT, int W>
__device__ __forceinline__ bool sum_partials(const double *__restrict__ part, int nseg, int64_t n, int64_t i,
                                             double (&red)[W - 1][PartSums<ACC, POT>::NV][64],
                                             PartSums<ACC, POT> &r) {
    constexpr int NV = PartSums<ACC, POT>::NV;
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
#pragma unroll
    for (int q = 0; q < NV; ++q) r.v[q] = 0.0;
    if (i < n) {
        const double *p = part + (ACC ? 0 : 3) * n + i;
        // (eight segments in flight; past the end: the last one's, not added)
        constexpr int U = 8;
        for (int s = w; s < nseg; s += U * W) {
            double t[U][NV];
#pragma unroll
            for (int u = 0; u < U; ++u) {
                const int su = s + u * W < nseg ? s + u * W : nseg - 1;
#pragma unroll
                for (int q = 0; q < NV; ++q) t[u][q] = p[((int64_t)su * 4 + q) * n];
            }
#pragma unroll
            for (int u = 0; u < U; ++u)
                if (s + u * W < nseg) {
#pragma unroll
                    for (int q = 0; q < NV; ++q) r.v[q] += t[u][q];
                }
        }
    }
    if (w > 0) {
#pragma unroll
        for (int q = 0; q < NV; ++q) red[w - 1][q][lane] = r.v[q];
    }
    __syncthreads();
    if (w > 0 || i >= n) return false;
#pragma unroll
    for (int u = 0; u < W - 1; ++u)
#pragma unroll
        for (int q = 0; q < NV; ++q) r.v[q] += red[u][q][lane];
    return true;
}

// Sum the per-segment partials in a fixed order and apply G (64 targets per
// workgroup).  Measured with four waves: 59 segments x 30011 potentials
// 27 -> 5.4 us, 63 segments x 16001 forces 21 -> 6.7 us.
template <bool ACC, bool POT, int W>
__global__ __launch_bounds__(64 * W) void k_finalize(const double *__restrict__ part, int nseg, int64_t n, double G,
                                                     double *__restrict__ ax, double *__restrict__ ay,
                                                     double *__restrict__ az, double *__restrict__ pot,
                                                     const int64_t *__restrict__ idx) {
    __shared__ double red[W - 1][PartSums<ACC, POT>::NV][64];
    const int64_t k = (int64_t)blockIdx.x * 64 + (threadIdx.x & 63);
    PartSums<ACC, POT> r;
    if (!sum_partials<ACC, POT, W>(part, nseg, n, k, red, r)) return;
    const int64_t i = idx ? idx[k] : k;
    if constexpr (ACC) {
        ax[i] = G * r.v[0];
        ay[i] = G * r.v[1];
        az[i] = G * r.v[2];
    }
    if constexpr (POT) pot[i] = -G * r.v[PartSums<ACC, POT>::NV - 1];
}

// Bounding box of each BS-source tile (lo xyz, hi xyz) and, when sub is not
// null, of each of its NQ quarters (the sources of one wave; an empty quarter
// gets lo = DBL_MAX, hi = -DBL_MAX) with the quarter's largest h in slot 6.
// One block per tile; thread t holds the position of source BS * blockIdx.x + t
// (v: the source exists).
__device__ __forceinline__ void tile_box_block(double px, double py, double pz, double ph, bool v,
                                               double *__restrict__ box, double *__restrict__ sub,
                                               double (&red)[6][NW]) {
    double lo[3] = {DBL_MAX, DBL_MAX, DBL_MAX}, hi[3] = {-DBL_MAX, -DBL_MAX, -DBL_MAX};
    if (v) {
        lo[0] = hi[0] = px;
        lo[1] = hi[1] = py;
        lo[2] = hi[2] = pz;
    }
#pragma unroll
    for (int d = 0; d < 3; ++d) {
        lo[d] = wave_min(lo[d]);
        hi[d] = wave_max(hi[d]);
    }
    const double hm = sub ? wave_max(v ? ph : 0.0) : 0.0;
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
    if (lane == 0) {
#pragma unroll
        for (int d = 0; d < 3; ++d) { red[d][w] = lo[d]; red[3 + d][w] = hi[d]; }
    }
    if (sub && lane == 0) {
        double *o = sub + ((int64_t)blockIdx.x * NQ + w) * 8;
#pragma unroll
        for (int d = 0; d < 3; ++d) { o[d] = lo[d]; o[3 + d] = hi[d]; }
        o[6] = hm;
    }
    if (!box) return;   // (uniform over the launch)
    __syncthreads();
    if (threadIdx.x < 6) {
        const int q = threadIdx.x;
        double r = red[q][0];
        for (int ww = 1; ww < NW; ++ww) r = q < 3 ? fmin(r, red[q][ww]) : fmax(r, red[q][ww]);
        box[(int64_t)blockIdx.x * 8 + q] = r;
    }
}

template <typename T>
__global__ __launch_bounds__(BS) void k_tile_boxes(const T *__restrict__ x, const T *__restrict__ y,
                                                   const T *__restrict__ z, int64_t n,
                                                   const double *__restrict__ h, double h_const,
                                                   double *__restrict__ box, double *__restrict__ sub) {
    __shared__ double red[6][NW];
    const int64_t j = (int64_t)blockIdx.x * BS + threadIdx.x;
    const bool v = j < n;
    tile_box_block(v ? (double)x[j] : 0.0, v ? (double)y[j] : 0.0, v ? (double)z[j] : 0.0,
                   v && h ? h[j] : h_const, v, box, sub, red);
}

// Kick of particle j from the FP64 sums of its force (without G): the central
// bodies' FP64 terms, Acc = G sum, Vel += Acc dt.
template <typename T>
__device__ __forceinline__ void kick_particle(const StepArgs &a, int64_t j, const double (&s)[3], T px, T py, T pz,
                                              double ph, T &ux, T &uy, T &uz) {
    double fx = a.G * s[0], fy = a.G * s[1], fz = a.G * s[2];
    if (a.ncentral > 0) {
        const double hinv = 1.0 / ph, hinv3 = hinv * hinv * hinv;
        double bx = 0.0, by = 0.0, bz = 0.0, bq = 0.0;
        const double *c = a.c_in;
        const int64_t k = a.ncentral;
        for (int64_t u = 0; u < k; ++u)
            pair_f64<false>(c[u], c[k + u], c[2 * k + u], c[3 * k + u], (double)px, (double)py, (double)pz, ph, hinv,
                            hinv3, bx, by, bz, bq);
        fx += bx * a.G;
        fy += by * a.G;
        fz += bz * a.G;
    }
    a.ax[j] = fx;
    a.ay[j] = fy;
    a.az[j] = fz;
    const T c = (T)a.dt;
    ux += (T)fx * c;
    uy += (T)fy * c;
    uz += (T)fz * c;
    ((T *)a.vx)[j] = ux;
    ((T *)a.vy)[j] = uy;
    ((T *)a.vz)[j] = uz;
}

// Drift of particle j (v: it exists): Pos += Vel (t_new - t_old), stored to
// xn.., particle 0 publishing t_new; a central body's new position goes to c_out.
template <typename T>
__device__ __forceinline__ void drift_particle(const StepArgs &a, int64_t j, bool v, T ux, T uy, T uz, T &px, T &py,
                                               T &pz) {
    const double t_old = a.time[a.rd];
    const double t_new = t_old + a.dt;
    if (j == 0) a.time[a.wr] = t_new;
    if (!v) return;
    const T d = (T)(t_new - t_old);
    px += ux * d;
    py += uy * d;
    pz += uz * d;
    ((T *)a.xn)[j] = px;
    ((T *)a.yn)[j] = py;
    ((T *)a.zn)[j] = pz;
    if (a.ncentral > 0 && a.central[j]) {
        for (int64_t u = 0; u < a.ncentral; ++u)
            if (a.cidx[u] == j) {
                a.c_out[u] = (double)px;
                a.c_out[a.ncentral + u] = (double)py;
                a.c_out[2 * a.ncentral + u] = (double)pz;
                a.c_out[3 * a.ncentral + u] = (double)((const T *)a.m)[j];
            }
    }
}

// The per-particle part of a KDK step, between one force launch and the next
// (one workgroup per 256 particles): the sums of the force's segments, the
// central bodies' FP64 terms and the kick (a.kick), then the next step's drift
// (a.drift) with the tile boxes of the drifted positions and, with GEO, the
// block's target geometry as k_target_geom<T, 1, ROWS> stores it.
// Bound by launch and load latency up to 10^5 particles, hence one launch for
// all of it: 64 steps of 1000 particles 1047 us with a launch each for the
// sums and kick and for the drift and boxes, 968 us in one; a disc of 16001
// with a central star (six launches a step) 1007 and 937 us per 8 steps.
// The segments' sums are split over four groups of 256 threads and meet in
// LDS in a fixed order; the first group does the rest.
//   kick:  Acc = G sum (+ central terms), Vel += Acc dt
//   drift: Pos += Vel (t_new - t_old), block 0 publishing t_new = time[rd] + dt
//          to time[wr] (rd != wr)
// The central bodies' terms read their positions from c_in, and the drift
// leaves the new ones in c_out: other workgroups still read the old ones.
constexpr int STEP_GROUPS = NW;   // (the groups of group_sums)
template <typename T, bool GEO, bool ROWS>
__global__ __launch_bounds__(BS * STEP_GROUPS) void k_step(StepArgs a) {
    __shared__ double sums[STEP_GROUPS - 1][3][BS];
    __shared__ double red[6][NW];
    __shared__ double gred[GEO ? 11 : 1][NW];
    const int tid = threadIdx.x & (BS - 1), grp = threadIdx.x / BS;
    const int64_t j = (int64_t)blockIdx.x * BS + tid;
    const bool v = j < a.n;
    const T *x = (T *)a.x, *y = (T *)a.y, *z = (T *)a.z, *vx = (T *)a.vx, *vy = (T *)a.vy, *vz = (T *)a.vz;
    T px = 0, py = 0, pz = 0, ux = 0, uy = 0, uz = 0;
    double ph = 0.0;
    if (grp == 0 && v) {
        px = x[j]; py = y[j]; pz = z[j];
        ux = vx[j]; uy = vy[j]; uz = vz[j];
        ph = a.h[j];
    }
    if (a.kick) {
        double s[3] = {0.0, 0.0, 0.0};
        if (v) group_sums<false, 3>(a.part, a.n, a.nseg, j, grp, s);
        if (grp > 0) {
#pragma unroll
            for (int q = 0; q < 3; ++q) sums[grp - 1][q][tid] = s[q];
        }
        __syncthreads();
        if (grp == 0 && v) {
#pragma unroll
            for (int g = 0; g < STEP_GROUPS - 1; ++g)
#pragma unroll
                for (int q = 0; q < 3; ++q) s[q] += sums[g][q][tid];
            kick_particle<T>(a, j, s, px, py, pz, ph, ux, uy, uz);
        }
    }
    if (!a.drift || grp > 0) return;   // (a barrier waits for the waves that remain)
    drift_particle<T>(a, j, v, ux, uy, uz, px, py, pz);
    tile_box_block((double)px, (double)py, (double)pz, ph, v, a.box, a.sub, red);
    if constexpr (GEO) {
        double gx[1] = {(double)px}, gy[1] = {(double)py}, gz[1] = {(double)pz};
        double gh[1] = {ph};
        bool gv[1] = {v};
        BlockStats st;
        block_stats<1>(gx, gy, gz, gh, gv, a.use_origin != 0, gred, st);
        const double ox = uniform_f64(st.ox), oy = uniform_f64(st.oy), oz = uniform_f64(st.oz);
        const WaveGeom wg = wave_geometry<1>(gx, gy, gz, gh, gv, ox, oy, oz, sizeof(T) == 8);
        store_target_geom(a.tgeo + (int64_t)blockIdx.x * TG_STRIDE, ox, oy, oz, wg, tid >> 6, tid & 63);
        if constexpr (ROWS) {
            nb_bf8 Bg[4];
            target_b_operands(gx[0] - ox, gy[0] - oy, gz[0] - oz, tid & 63, Bg);
            nb_u4v *b = reinterpret_cast<nb_u4v *>(a.tbg + ((int64_t)blockIdx.x * BS + tid) * 16);
#pragma unroll
            for (int g = 0; g < 4; ++g) b[g] = __builtin_bit_cast(nb_u4v, Bg[g]);
        }
    }
}

// A whole step of a small system in one launch: k_force_wave's forces on targets
// that share waves, then, in the workgroup that is the last of its 64 targets'
// segments to arrive, k_step's sums, kick and drift of those targets.
// Positions are double-buffered: other workgroups still read the old ones.
// Small systems are bound by the chain of memory latencies from the targets'
// load to the new boxes.
// A step in split precision, two launches -> one: 300 particles 13.8 -> 12.3 us,
// 1000 14.4 -> 13.3, 2000 18.5 -> 15.5, 4096 26.5 -> 23.9, 8000 44.8 -> 43.0,
// 30000 308 -> 304; FP32: 1000 13.3 -> 12.8, 4096 22.7 -> 19.4, 16001 87.1 ->
// 86.5 (with shorter re-sorts and DPP reductions since then: 9.3, 10.9, 12.4,
// 20.3 and 39.9 us at 300 to 8000).
template <typename T>
__global__ __launch_bounds__(BS) __attribute__((amdgpu_waves_per_eu(5))) void k_force_step(ForceArgs<T> a,
                                                                                           StepArgs st) {
    __shared__ WaveStage<T> stage[NW];
    __shared__ double red[NW - 1][3][64];
    __shared__ int last;
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
    const int logical = xcd_remap(blockIdx.x, gridDim.x);
    const int seg = logical / a.nblk_i;
    const int ib = logical - seg * a.nblk_i;
    const int64_t i0 = (int64_t)ib * 64, i = i0 + lane, ic = i < a.nt ? i : a.nt - 1;
    int64_t j0 = (int64_t)seg * a.seg_len;
    int64_t j1 = (j0 + a.seg_len < a.ns) ? j0 + a.seg_len : a.ns;
    const int64_t part = a.seg_len / NW;
    j0 = j0 + part * wave < j1 ? j0 + part * wave : j1;
    j1 = j0 + part < j1 ? j0 + part : j1;
    const T xt = a.tx[ic], yt = a.ty[ic], zt = a.tz[ic];
    const double ph = a.th[ic];
    double s[3], q;
    wave_force<T, true, false, false, true>(stage[wave], xt, yt, zt, ph, a.tbox + (i0 / 64) * 8, a.sx, a.sy, a.sz, a.sm,
                               a.skip_src, a.sub_box + (j0 / SB) * 8, a.tile_box, j0, j1, s[0], s[1], s[2], q);
    add_waves(s, red);
    const bool v = i < a.nt;
    T ux = 0, uy = 0, uz = 0;
    if (wave == 0 && v) {   // (requested before the wait for the sums' stores)
        ux = ((const T *)st.vx)[i];
        uy = ((const T *)st.vy)[i];
        uz = ((const T *)st.vz)[i];
    }
    if (a.nseg == 1 ? wave > 0 : !last_arrival(s, a.part, a.nt, a.nseg, seg, i, v, st.arrived + ib, red, last)) return;
    T px = xt, py = yt, pz = zt;
    if (v) kick_particle<T>(st, i, s, px, py, pz, ph, ux, uy, uz);
    if (!st.drift) return;
    drift_particle<T>(st, i, v, ux, uy, uz, px, py, pz);
    const double p[3] = {(double)px, (double)py, (double)pz};
    double *o = st.sub + (i0 / 64) * 8;
#pragma unroll
    for (int d = 0; d < 3; ++d) {   // the new box of these 64 (lanes without a particle: none)
        const double lo = wave_min(v ? p[d] : DBL_MAX), hi = wave_max(v ? p[d] : -DBL_MAX);
        if (lane == 0) { o[d] = lo; o[3 + d] = hi; }
    }
    const double hm = wave_max(v ? ph : 0.0);
    if (lane == 0) o[6] = hm;
}

// ---------------------------------------------------------------------------
// Launchers
// ---------------------------------------------------------------------------
static int check_launch(const char *what) {
    hipError_t e = hipGetLastError();
    if (e != hipSuccess) {
        set_error("launch of %s failed: %s", what, hipGetErrorString(e));
        return NB_ERR_HIP;
    }
    return NB_OK;
}

int launch_tile_boxes(const void *x, const void *y, const void *z, int is_double, int64_t n,
                      const double *h, double h_const, double *box, double *sub_box, hipStream_t s) {
    if (n <= 0) return NB_OK;
    const int64_t ntiles = (n + BS - 1) / BS;
    if (is_double)
        k_tile_boxes<double><<<(unsigned)ntiles, BS, 0, s>>>((const double *)x, (const double *)y,
                                                            (const double *)z, n, h, h_const, box, sub_box);
    else
        k_tile_boxes<float><<<(unsigned)ntiles, BS, 0, s>>>((const float *)x, (const float *)y,
                                                           (const float *)z, n, h, h_const, box, sub_box);
    return check_launch("k_tile_boxes");
}

// With several source segments, store each target block's geometry first
// (a.tgeo); otherwise the force kernel derives it (tgeo = nullptr).
// rows: the force kernel takes bf16 matrix-core far tiles (TPT 1), whose
// B operands are stored as well (a.tbg).
template <typename T>
static int prepare_target_geom(ForceArgs<T> &a, int tpt, hipStream_t s, bool rows = false) {
    if (!a.tgeo || a.nseg <= 1 || a.nblk_i <= 0) {
        a.tgeo = nullptr;
        a.tbg = nullptr;
        return NB_OK;
    }
    // already written by the step's drift (one target per lane), with the B
    // operands when this launch takes them
    if (tpt == 1 && a.tgeo_ready && (a.tgeo_ready == 2 || !rows || !a.tbg)) {
        if (!rows || !a.tbg) a.tbg = nullptr;
        return NB_OK;
    }
    const bool hilo = sizeof(T) == 8;
    if (!rows || tpt != 1 || !a.tbg) a.tbg = nullptr;
    if (tpt == 1 && a.tbg) k_target_geom<T, 1, true><<<(unsigned)a.nblk_i, BS, 0, s>>>(a, hilo);
    else if (tpt == 1) k_target_geom<T, 1, false><<<(unsigned)a.nblk_i, BS, 0, s>>>(a, hilo);
    else if (tpt == 2) k_target_geom<T, 2, false><<<(unsigned)a.nblk_i, BS, 0, s>>>(a, hilo);
    else if (tpt == 4) k_target_geom<T, 4, false><<<(unsigned)a.nblk_i, BS, 0, s>>>(a, hilo);
    else {
        a.tgeo = nullptr;
        a.tbg = nullptr;
        return NB_OK;
    }
    return check_launch("k_target_geom");
}

template <typename T, int MF>
static int launch_f32_impl(ForceArgs<T> a, int tpt, bool pot, hipStream_t s, bool acc) {
    const int64_t nb = (int64_t)a.nblk_i * a.nseg;
    if (nb <= 0) return NB_OK;
    if (nb > INT32_MAX) {
        set_error("force grid too large (%lld blocks)", (long long)nb);
        return NB_ERR_INVALID;
    }
    if (wave_path(MF, tpt, pot, acc)) {
        launch_wave<T>(a, pot, acc, s);
        return check_launch("k_force_wave");
    }
    NB_TRY(prepare_target_geom(a, tpt, s));
    dim3 g((unsigned)nb), b(BS);
#define NB_L(TPT_, POT_) k_force_f32<T, TPT_, POT_, (POT_ ? 0 : MF)><<<g, b, 0, s>>>(a)
#define NB_LP(TPT_) k_force_f32<T, TPT_, true, 0, false><<<g, b, 0, s>>>(a)
    if (tpt == 1) {
        if constexpr (MF != FAR_VALU) NB_L(1, false);   // (the others take k_force_wave)
    } else if (tpt == 2) { if (pot && !acc) NB_LP(2); else if (pot) NB_L(2, true); else NB_L(2, false); }
    else if (tpt == 4) { if (pot && !acc) NB_LP(4); else if (pot) NB_L(4, true); else NB_L(4, false); }
    else {
        set_error("unsupported targets_per_thread %d", tpt);
        return NB_ERR_INVALID;
    }
#undef NB_L
#undef NB_LP
    return check_launch("k_force_f32");
}

int launch_force_f32(const ForceArgs<float> &a, int tpt, bool pot, hipStream_t s, bool acc,
                     int far_path) {
    if (!acc && !pot) acc = true;
    if (far_path == FAR_MFMA_BF16 && tpt == 1 && (!pot || !acc)) {
        // FP32 state through the per-block FP64 origin: hi/lo near tiles, bf16
        // matrix-core squared distances on the far tiles (forces or potential alone)
        const int64_t nb = (int64_t)a.nblk_i * a.nseg;
        if (nb <= 0) return NB_OK;
        if (nb > INT32_MAX) {
            set_error("force grid too large (%lld blocks)", (long long)nb);
            return NB_ERR_INVALID;
        }
        ForceArgs<float> b = a;
        b.use_origin = 1;
        NB_TRY(prepare_target_geom(b, 1, s, true));
        if (pot) k_force_f32<float, 1, true, FAR_MFMA_BF16, false><<<(unsigned)nb, BS, 0, s>>>(b);
        else launch_bf16_forces(b, nb, s);
        return check_launch("k_force_f32<float, bf16 mfma>");
    }
    return launch_f32_impl<float, FAR_VALU>(a, tpt, pot, s, acc);
}
int launch_force_split(const ForceArgs<double> &a_in, int tpt, bool pot, hipStream_t s, int far_path,
                       bool acc) {
    if (!acc && !pot) acc = true;
    ForceArgs<double> a = a_in;
    if (far_path == FAR_MFMA_BF16 && tpt == 1 && pot && !acc) {
        const int64_t nb = (int64_t)a.nblk_i * a.nseg;
        if (nb <= 0) return NB_OK;
        NB_TRY(prepare_target_geom(a, tpt, s, true));
        k_force_f32<double, 1, true, FAR_MFMA_BF16, false><<<(unsigned)nb, BS, 0, s>>>(a);
        return check_launch("k_force_f32<bf16 mfma, potential>");
    }
    if ((far_path == FAR_MFMA_SUM || far_path == FAR_MFMA_R2) && tpt == 1 && !pot) {
        const int64_t nb = (int64_t)a.nblk_i * a.nseg;
        if (nb <= 0) return NB_OK;
        NB_TRY(prepare_target_geom(a, tpt, s));
        if (far_path == FAR_MFMA_R2) k_force_f32<double, 1, false, FAR_MFMA_R2><<<(unsigned)nb, BS, 0, s>>>(a);
        else k_force_f32<double, 1, false, FAR_MFMA_SUM><<<(unsigned)nb, BS, 0, s>>>(a);
        return check_launch("k_force_f32<mfma>");
    }
    if (far_path == FAR_MFMA_BF16 && tpt == 1 && !pot) {
        const int64_t nb = (int64_t)a.nblk_i * a.nseg;
        if (nb <= 0) return NB_OK;
        NB_TRY(prepare_target_geom(a, tpt, s, true));
        launch_bf16_forces(a, nb, s);
        return check_launch("k_force_f32<bf16 mfma>");
    }
    if (far_path == FAR_WEIGHTED) return launch_f32_impl<double, FAR_WEIGHTED>(a, tpt, pot, s, acc);
    return launch_f32_impl<double, FAR_VALU>(a, tpt, pot, s, acc);
}

template <typename T>
__global__ void k_source_weights(const T *__restrict__ m, int64_t n, float *__restrict__ w) {
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    const double mi = (double)m[i];
    w[i] = mi > 0.0 ? (float)(1.0 / cbrt(mi * mi)) : 0.0f;
}

int launch_source_weights(const void *m, bool is_double, int64_t n, float *w, hipStream_t s) {
    if (n <= 0) return NB_OK;
    const unsigned g = (unsigned)((n + 255) / 256);
    if (is_double) k_source_weights<double><<<g, 256, 0, s>>>((const double *)m, n, w);
    else k_source_weights<float><<<g, 256, 0, s>>>((const float *)m, n, w);
    return check_launch("k_source_weights");
}

int launch_force_f64(const ForceArgs<double> &a_in, bool pot, hipStream_t s) {
    ForceArgs<double> a = a_in;
    if (a.nt <= 0 || a.nseg <= 0) return NB_OK;
    const int split = f64_split(a.nt, a.nseg);
    a.nblk_i = (int)(split ? (a.nt + 63) / 64 : (a.nt + BS - 1) / BS);
    const unsigned nb = (unsigned)((int64_t)a.nblk_i * a.nseg);
    const bool fin = split && a.nseg > 1 && a.arrived;
    if (pot && fin) k_force_f64<true, true><<<nb, BS, 0, s>>>(a, split);
    else if (pot) k_force_f64<true, false><<<nb, BS, 0, s>>>(a, split);
    else if (fin) k_force_f64<false, true><<<nb, BS, 0, s>>>(a, split);
    else k_force_f64<false, false><<<nb, BS, 0, s>>>(a, split);
    return check_launch("k_force_f64");
}

int launch_step(const StepArgs &a, bool is_double, hipStream_t s) {
    if (a.n <= 0) return NB_OK;
    const unsigned nt = (unsigned)((a.n + BS - 1) / BS), bs = BS * STEP_GROUPS;
    const bool g = a.drift && a.tgeo, r = g && a.tbg;
#define NB_ST(T_)                                                       \
    do {                                                                \
        if (r) k_step<T_, true, true><<<nt, bs, 0, s>>>(a);             \
        else if (g) k_step<T_, true, false><<<nt, bs, 0, s>>>(a);       \
        else k_step<T_, false, false><<<nt, bs, 0, s>>>(a);             \
    } while (0)
    if (is_double) NB_ST(double);
    else NB_ST(float);
#undef NB_ST
    return check_launch("k_step");
}

template <typename T>
static int force_step(ForceArgs<T> f, const StepArgs &st, hipStream_t s) {
    if (f.nt <= 0) return NB_OK;
    f.nblk_i = (int)((f.nt + 63) / 64);
    k_force_step<T><<<(unsigned)((int64_t)f.nblk_i * f.nseg), BS, 0, s>>>(f, st);
    return check_launch("k_force_step");
}
int launch_force_step(const ForceArgs<float> &f, const StepArgs &st, hipStream_t s) { return force_step(f, st, s); }
int launch_force_step(const ForceArgs<double> &f, const StepArgs &st, hipStream_t s) { return force_step(f, st, s); }

int launch_finalize(const double *part, int nseg, int64_t n, double G, double *ax, double *ay,
                    double *az, double *pot, bool with_pot, hipStream_t s, bool with_acc, const int64_t *idx) {
    if (n <= 0) return NB_OK;
    const unsigned nb = (unsigned)((n + 63) / 64);
#define NB_FIN(A_, P_)                                                                                          \
    do {                                                                                                        \
        if (nseg > FIN_MANY)                                                                                    \
            k_finalize<A_, P_, FIN_WAVES_MANY><<<nb, 64 * FIN_WAVES_MANY, 0, s>>>(part, nseg, n, G, ax, ay, az, pot, idx); \
        else                                                                                                    \
            k_finalize<A_, P_, FIN_WAVES><<<nb, 64 * FIN_WAVES, 0, s>>>(part, nseg, n, G, ax, ay, az, pot, idx);     \
    } while (0)
    if (with_pot && with_acc) NB_FIN(true, true);
    else if (with_pot) NB_FIN(false, true);
    else if (with_acc) NB_FIN(true, false);
#undef NB_FIN
    return check_launch("k_finalize");
}

}  // namespace nb
