// nb_wave.h -- the wavefront-level all-pairs routine of far path 0 with one
// target per lane, shared by the one-system kernel (nb_force.hip) and the
// ragged ensemble kernel (nb_batch_wave.hip).
#pragma once
#include <hip/hip_runtime.h>
#include <float.h>
#include <stdint.h>

#include "nb_block.h"
#include "nb_internal.h"
#include "nb_pair.h"

namespace nb {

// A wavefront owns 64 consecutive targets and walks its source range on its
// own, one quarter (SB = 64 sources) at a time: no workgroup barrier, so a wave
// with many near quarters holds no other wave up, and a small system still
// gives every SIMD waves (64 sources each, instead of 256 per block).
//
// Bound: FP32 VALU issue where the grid fills the chip, the latency of one
// quarter where it does not.  The LDS broadcast port is the other limit of a
// block-wide tile loop (a 32-byte FP64 record is two ds_read_b128 per source
// and wave, 64 CU-cycles for four SIMDs against about 62 VALU cycles), so the
// near quarters take the source positions through scalar loads (the source
// index is wave-uniform): FP64 separations are formed from the positions
// themselves, FP32 masses come four at a time from LDS.  Only the mid quarters
// of an FP64 state read staged records (hi coordinates relative to the wave's
// origin, one ds_read_b128 per source).
//
// The classes are those of force_block's far path 0 (nb_block.h), by quarter,
// from the wave's own box and with the box's centre as the FP64 origin: soft
// (a pair may lie inside some target's h), close (FP64 state: gap <= R/2, R
// the wave's half extent), else mid (FP32 state: every unsoftened quarter takes
// the FP32 positions).  A block-wide origin had R about 1.6 times as large, so
// fewer quarters are close here.
template <typename T>
struct WaveStage {
    static constexpr bool D = sizeof(T) == 8;
    float4 hi[D ? SB : 1];   // source relative to the wave's origin, and its mass
    float m[SB];             // masses (0: excluded or past the end)
    double geo[8];           // the wave's box and squared class distances, read once per 64 quarters
};

template <typename T>
using scalar_ptr = const __attribute__((address_space(4))) T *;
template <typename T>
__device__ __forceinline__ scalar_ptr<T> as_scalar(const T *p) {
    return (scalar_ptr<T>)(uintptr_t)p;
}

struct SoftF32 {
    float h2c, h2, hinv, hinv3;
};

// Four consecutive values at a wave-uniform address, in scalar registers.
template <typename T>
struct Four {
    typedef T vec __attribute__((ext_vector_type(4), aligned(sizeof(T))));
};
template <typename T>
__device__ __forceinline__ typename Four<T>::vec load_four(scalar_ptr<T> p) {
    return *reinterpret_cast<const __attribute__((address_space(4))) typename Four<T>::vec *>(p);
}

// cnt sources at (sx, sy, sz) (wave-uniform addresses), masses in LDS, four at
// a time: the next four are requested as soon as the separations of these have
// left the scalar registers, so that their latency runs beside the rest (scalar
// and LDS loads share a counter, hence the masses too), and one test per
// group finds a pair inside some target's h.
// LATE: the masses are requested after their last use in the group: requested
// earlier, they were copied to other registers on every trip of k_batch_wave's
// unchecked loop (2.5 % of 512 clusters).
template <typename T, bool CHECKED, bool ACC, bool POT, bool LATE>
__device__ __forceinline__ void near_sources(scalar_ptr<T> sx, scalar_ptr<T> sy, scalar_ptr<T> sz,
                                             const float *__restrict__ sm, int cnt, T xt, T yt, T zt,
                                             const SoftF32 &t, float &ax, float &ay, float &az, float &aq) {
    constexpr int GR = 4;
    using V = typename Four<T>::vec;
    const int full = cnt & ~(GR - 1);
    if (full > 0) {
        V x = load_four<T>(sx), y = load_four<T>(sy), z = load_four<T>(sz);
        float4 m4 = *reinterpret_cast<const float4 *>(sm);
#pragma unroll 1
        for (int j = 0; j < full; j += GR) {
            const float m[GR] = {m4.x, m4.y, m4.z, m4.w};
            float dx[GR], dy[GR], dz[GR], r2[GR], fac[GR], q[GR];
#pragma unroll
            for (int g = 0; g < GR; ++g) {
                dx[g] = (float)(x[g] - xt);
                dy[g] = (float)(y[g] - yt);
                dz[g] = (float)(z[g] - zt);
            }
            const int jn = j + GR < full ? j + GR : 0;
            x = load_four<T>(sx + jn);
            y = load_four<T>(sy + jn);
            z = load_four<T>(sz + jn);
            if (!LATE) m4 = *reinterpret_cast<const float4 *>(sm + jn);
#pragma unroll
            for (int g = 0; g < GR; ++g) {
                r2[g] = __builtin_fmaf(dx[g], dx[g], __builtin_fmaf(dy[g], dy[g], dz[g] * dz[g]));
                const float ri = __builtin_amdgcn_rsqf(r2[g]);
                q[g] = m[g] * ri;
                fac[g] = q[g] * (ri * ri);
            }
            if (LATE) m4 = *reinterpret_cast<const float4 *>(sm + jn);
            if (CHECKED) {
                const float rmin = fminf(fminf(r2[0], r2[1]), fminf(r2[2], r2[3]));
                if (__builtin_expect(rmin < t.h2c, 0)) {
#pragma unroll
                    for (int g = 0; g < GR; ++g)
                        if (r2[g] < t.h2c) spline_f32(r2[g], m[g], t.h2, t.hinv, t.hinv3, fac[g], q[g]);
                }
            }
#pragma unroll
            for (int g = 0; g < GR; ++g) {
                if (ACC) {
                    ax = __builtin_fmaf(fac[g], dx[g], ax);
                    ay = __builtin_fmaf(fac[g], dy[g], ay);
                    az = __builtin_fmaf(fac[g], dz[g], az);
                }
                if (POT) aq += q[g];
            }
            // (keeps the requests above in this iteration)
            asm volatile("" : "+s"(x), "+s"(y), "+s"(z));
        }
    }
#pragma unroll 1
    for (int j = full; j < cnt; ++j) {
        const float dx = (float)(sx[j] - xt), dy = (float)(sy[j] - yt), dz = (float)(sz[j] - zt);
        const float r2 = __builtin_fmaf(dx, dx, __builtin_fmaf(dy, dy, dz * dz));
        const float ri = __builtin_amdgcn_rsqf(r2);
        float q = sm[j] * ri;
        float fac = q * (ri * ri);
        if (CHECKED && r2 < t.h2c) spline_f32(r2, sm[j], t.h2, t.hinv, t.hinv3, fac, q);
        if (ACC) {
            ax = __builtin_fmaf(fac, dx, ax);
            ay = __builtin_fmaf(fac, dy, ay);
            az = __builtin_fmaf(fac, dz, az);
        }
        if (POT) aq += q;
    }
}

// The sums of one wave: targets (xt, yt, zt, h), one per lane (lanes without a
// target of their own repeat one), against the sources [j0, j1).
// tbox, when not null: the box and largest h of the wave's targets (lo xyz,
// hi xyz, h); else reduced here.  sub_box: the boxes of the quarters from j0
// on, or, when null, tile_box: the boxes of the BS-source tiles from j0 on.
// TILES: the origin, box and classes are those of the targets' block (tgeo, its
// stored record, and the wave's place gw in it) and the FP32 sums run over a
// whole tile (j0 starts one), as in force_block, whose sums these then are.  After
// quarter qm, the last of a tile, the sums so far go to mid and start again.
// EARLY (with sub_box): the first quarter's sources and the boxes of the first 64 quarters (one
// per lane) are requested before anything waits for the targets, in 15 more
// registers (4096 particles 24.5 -> 23.9 us a step of k_force_step; at six
// waves per SIMD they spill, and 30011 particles take 3 % longer).
// Returns FP64 sums without G.
template <typename T, bool ACC, bool POT, bool TILES = false, bool EARLY = false>
__device__ __forceinline__ void wave_force(WaveStage<T> &st, T xt, T yt, T zt, double h,
                                           const double *__restrict__ tbox, const T *__restrict__ sx,
                                           const T *__restrict__ sy, const T *__restrict__ sz,
                                           const T *__restrict__ sm, const uint8_t *__restrict__ skip_src,
                                           const double *__restrict__ sub_box,
                                           const double *__restrict__ tile_box, int64_t j0, int64_t j1,
                                           double &Ax, double &Ay, double &Az, double &Aq,
                                           const double *__restrict__ tgeo = nullptr, int gw = 0, int qm = -1,
                                           double (*mid)[64] = nullptr) {
    constexpr bool D = WaveStage<T>::D;
    const int lane = threadIdx.x & 63;
    // the next quarter's sources are loaded while the current one is computed
    // (index clamped into the range, validity decided at staging)
    T rx, ry, rz, rm;
    unsigned rskip = 0;
    auto fetch = [&](int64_t j) {
        const int64_t jc = j < j1 ? j : j1 - 1;
        if (D) { rx = sx[jc]; ry = sy[jc]; rz = sz[jc]; }
        rm = sm[jc];
        if (skip_src) rskip = skip_src[jc];
    };
    double bx[6];
    if constexpr (EARLY) {
        if (j0 < j1) fetch(j0 + lane);
        if (j0 + lane * SB < j1) {
#pragma unroll
            for (int d = 0; d < 6; ++d) bx[d] = sub_box[lane * 8 + d];
        }
    }
    double o[3];
    if constexpr (TILES) {
        if (lane < 8) st.geo[lane] = tgeo[3 + 9 * gw + lane];
#pragma unroll
        for (int d = 0; d < 3; ++d) o[d] = uniform_f64(tgeo[d]);
    } else {
        double lo[3], hi[3], hmax, rb = 0.0;
        if (tbox) {
#pragma unroll
            for (int d = 0; d < 3; ++d) { lo[d] = tbox[d]; hi[d] = tbox[3 + d]; }
            hmax = tbox[6];
        } else {
            const double p[3] = {(double)xt, (double)yt, (double)zt};
#pragma unroll
            for (int d = 0; d < 3; ++d) { lo[d] = wave_min(p[d]); hi[d] = wave_max(p[d]); }
            hmax = wave_max(h);
        }
#pragma unroll
        for (int d = 0; d < 3; ++d) {
            // FP32 state: no origin (the margin then covers the coordinates' own size)
            o[d] = D ? uniform_f64(0.5 * lo[d] + 0.5 * hi[d]) : 0.0;
            rb = fmax(rb, fmax(fabs(lo[d] - o[d]), fabs(hi[d] - o[d])));
        }
        const double soft_d = hmax * (1.0 + 1e-6) + 1e-6 * rb + 1e-300;
        const double close_d = D ? fmax(soft_d, 0.5 * rb) : soft_d;
        if (lane == 0) {
#pragma unroll
            for (int d = 0; d < 3; ++d) { st.geo[d] = lo[d]; st.geo[3 + d] = hi[d]; }
            st.geo[6] = soft_d * soft_d;
            st.geo[7] = close_d * close_d;
        }
    }

    const float xi = (float)((double)xt - o[0]), yi = (float)((double)yt - o[1]), zi = (float)((double)zt - o[2]);
    const float hf = (float)h;
    SoftF32 t;
    t.h2 = hf * hf;
    t.h2c = fmaxf(t.h2, FLT_MIN);
    t.hinv = 1.0f / hf;
    t.hinv3 = t.hinv * t.hinv * t.hinv;

    Ax = Ay = Az = Aq = 0.0;
    uint64_t m_soft = 0, m_close = 0;
    if (!EARLY && j0 < j1) fetch(j0 + lane);
    int q = 0;
    float ax = 0.0f, ay = 0.0f, az = 0.0f, aq = 0.0f;
    for (int64_t base = j0; base < j1; base += SB, ++q) {
        {
            const bool rv = base + lane < j1;
            const float m = rv && rskip == 0 ? (float)rm : 0.0f;
            st.m[lane] = m;
            if constexpr (D) {
                st.hi[lane] = rv ? make_float4((float)((double)rx - o[0]), (float)((double)ry - o[1]),
                                               (float)((double)rz - o[2]), m)
                                 : make_float4(PAD_COORD, PAD_COORD, PAD_COORD, 0.0f);
            }
        }
        __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");   // staged before it is read (LDS is in order)
        if (base + SB < j1) fetch(base + SB + lane);
        if ((q & 63) == 0) {   // the classes of the next 64 quarters, one per lane
            const int64_t u = (int64_t)q + lane;
            bool c_soft = false, c_close = false;
            if (j0 + u * SB < j1) {
                WaveGeom wg;
#pragma unroll
                for (int d = 0; d < 3; ++d) { wg.lo[d] = st.geo[d]; wg.hi[d] = st.geo[3 + d]; }
                wg.soft_d2 = st.geo[6];
                wg.close_d2 = st.geo[7];
                const double g2 = EARLY && q == 0
                                      ? tile_gap2(bx, wg)
                                      : tile_gap2(sub_box ? sub_box + u * 8 : tile_box + (u / NQ) * 8, wg);
                c_soft = !(g2 > wg.soft_d2);
                c_close = !(g2 > wg.close_d2);
            }
            m_soft = __builtin_amdgcn_ballot_w64(c_soft);
            m_close = __builtin_amdgcn_ballot_w64(c_close);
        }
        const uint64_t bit = 1ull << (q & 63);
        const int cnt = j1 - base < SB ? (int)(j1 - base) : SB;
        if (m_soft & bit) {
            near_sources<T, true, ACC, POT, false>(as_scalar(sx + base), as_scalar(sy + base), as_scalar(sz + base),
                                                   st.m, cnt, xt, yt, zt, t, ax, ay, az, aq);
        } else if (!D || (m_close & bit)) {
            near_sources<T, false, ACC, POT, TILES>(as_scalar(sx + base), as_scalar(sy + base), as_scalar(sz + base),
                                                    st.m, cnt, xt, yt, zt, t, ax, ay, az, aq);
        } else if constexpr (D) {
#pragma unroll 1
            for (int j = 0; j < cnt; j += 4) {   // (past cnt: padding)
#pragma unroll
                for (int g = 0; g < 4; ++g) {
                    const float4 v = st.hi[j + g];
                    pair_f32<false, POT>(v.x, v.y, v.z, v.w, xi, yi, zi, t.h2c, t.h2, t.hinv, t.hinv3, ax, ay, az,
                                         aq);
                }
            }
        }
        __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");   // read before the next staging
        if (TILES && (q & (NQ - 1)) != NQ - 1 && base + SB < j1) continue;
        if (ACC) { Ax += (double)ax; Ay += (double)ay; Az += (double)az; }
        if (POT) Aq += (double)aq;
        ax = ay = az = aq = 0.0f;
        if (TILES && q == qm) {
            if (ACC) { mid[0][lane] = Ax; mid[1][lane] = Ay; mid[2][lane] = Az; }
            if (POT) mid[ACC ? 3 : 0][lane] = Aq;
            Ax = Ay = Az = Aq = 0.0;
        }
    }
}

}  // namespace nb
