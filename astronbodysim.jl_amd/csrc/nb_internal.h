// nb_internal.h -- host-side internals shared by the C-ABI translation units.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>
#include <algorithm>
#include <string>
#include <vector>

#include "../../include/nbody_mi355x.h"

namespace nb {

// Source tile = one LDS stage = one block of BS threads (NW wavefronts).
constexpr int BS = 256;
constexpr int NW = BS / 64;
// Tile quarters: the SB sources one wave stages.  Their boxes let a wave
// classify a tile quarter by quarter.
constexpr int SB = 64;
constexpr int NQ = BS / SB;
// Doubles per target block of the force kernel's geometry workspace (the
// block origin, then nine per wave).
constexpr int TG_STRIDE = 3 + 9 * (BS / 64) + 1;

void set_error(const char *fmt, ...);
void clear_error();

#define NB_HIP(call)                                                                       \
    do {                                                                                   \
        hipError_t e_ = (call);                                                            \
        if (e_ != hipSuccess) {                                                            \
            ::nb::set_error("%s failed: %s (%s:%d)", #call, hipGetErrorString(e_), __FILE__, \
                            __LINE__);                                                     \
            return NB_ERR_HIP;                                                             \
        }                                                                                  \
    } while (0)

#define NB_TRY(expr)              \
    do {                          \
        int rc_ = (expr);         \
        if (rc_ != NB_OK) return rc_; \
    } while (0)

// Arguments of the FP32-pair all-pairs kernel (modes FP32 / SPLIT).
// Targets and sources may be different arrays (probe points).
template <typename T>
struct ForceArgs {
    const T *tx, *ty, *tz;   // targets (internal order)
    const double *th;        // per-target softening h (nullptr => th_const)
    double th_const;
    int64_t nt;
    const T *sx, *sy, *sz, *sm;  // sources
    int64_t ns;
    const double *tile_box;  // [ntiles][8]: lo xyz, hi xyz, (unused) of each BS-source tile
    const double *sub_box;   // [ntiles][NQ][8]: the same for each tile's quarters (with the quarter's
                             // largest softening length in slot 6), or nullptr
    const double *tbox;      // the same record for every 64 targets (sub_box where targets are the
                             // sources), or nullptr: reduced by the kernel (k_force_wave)
    double *tgeo;            // [nblk_i][TG_STRIDE] workspace for the target blocks' geometry, or nullptr
    int tgeo_ready;          // 1: tgeo holds this call's geometry (written by the step's drift), 2: tbg too
    unsigned *tbg;           // [nblk_i][BS][16] workspace for their bf16 B operands, or nullptr
    uint8_t *nflag;          // [nblk_i * nseg * NW]: waves with near tiles (split passes), or nullptr
    int use_origin;          // 1: per-block FP64 origin (SPLIT), 0: absolute FP32 coordinates
    int nseg;                // source segments (grid = nblk_i * nseg)
    int64_t seg_len;         // sources per segment: a multiple of BS for the block-wide kernels, of SB (a
                             // quarter) for k_force_wave and k_force_f64; below BS, and wherever wave_split
                             // cuts a segment into the waves' parts, these do not start on tiles, so
                             // k_force_wave needs sub_box there
    int nblk_i;              // target blocks
    int wave_split;          // k_force_wave: the waves of a workgroup share 64 targets and split the segment
    double G;
    double *ax, *ay, *az, *pot;  // final outputs (nseg == 1)
    double *part;                // partials [nseg][4][nt] (nseg > 1)
    unsigned *arrived;           // [64-target groups], zeros between launches: where the waves of a workgroup
                                 // share targets, the launch adds the segments' sums itself; or nullptr
    const uint8_t *skip_src;     // sources excluded from the FP32 sum (central bodies) or nullptr
    int accumulate;              // 1: add G*sum to the outputs instead of storing (nseg == 1)
    const float *sw;             // source weights m^(-2/3) (far paths 3 and 4) or nullptr
};

// Far-tile paths (the far_path tuning value; nb_block.h describes each).
constexpr int FAR_VALU = 0;       // 12 VALU + rsq per pair
constexpr int FAR_MFMA_SUM = 1;   // sum on the matrix cores
constexpr int FAR_MFMA_R2 = 2;    // r^2 and sum on the matrix cores (farthest tiles)
constexpr int FAR_WEIGHTED = 3;   // weighted far tiles: 10 VALU + rsq per pair
constexpr int FAR_MFMA_BF16 = 4;  // bf16-split r^2 on the matrix cores, sum on the VALU

// Whether a launch of the FP32-pair kernels takes the wavefront kernel
// (k_force_wave: far path 0, one target per lane; also forces and potentials
// together where the far path has no such kernel), whose source segments may
// be cut at any quarter (SB sources) instead of at tiles.
inline bool wave_path(int far_path, int tpt, bool pot, bool acc) {
    return tpt == 1 && (far_path == FAR_VALU || (pot && (acc || far_path != FAR_MFMA_BF16)));
}

// A launch over target blocks (BS targets per target of a lane) and source
// segments.
struct Geometry {
    int tpt, nseg, nblk_i;
    int64_t seg_len;
    int wave_split = 0;
};

// Segments of whole tiles.
inline Geometry geometry(int64_t nt, int64_t ns, int tpt, int64_t want_seg) {
    Geometry g;
    g.tpt = tpt;
    g.nblk_i = (int)((nt + (int64_t)BS * tpt - 1) / ((int64_t)BS * tpt));
    const int64_t ntiles = std::max<int64_t>((ns + BS - 1) / BS, 1);
    const int64_t nseg = std::min<int64_t>(std::max<int64_t>(want_seg, 1), ntiles);
    const int64_t tiles_per_seg = (ntiles + nseg - 1) / nseg;
    g.seg_len = tiles_per_seg * BS;
    g.nseg = (int)((ntiles + tiles_per_seg - 1) / tiles_per_seg);
    return g;
}

// A k_force_wave launch: the segments are cut at quarters.  Few targets are
// spread over more segments than asked for, up to max_seg (or one per quarter),
// until the chip has about WAVE_FILL workgroups: a wave alone on its SIMD is
// bound by latency.  Below WAVE_SPLIT_BELOW targets the four waves of a
// workgroup share 64 targets and split the segment's sources, by whole quarters
// only where asked (the FP32 sums of a quarter then never depend on the split).
constexpr int WAVE_SEGMENTS = 64;
constexpr int64_t WAVE_FILL = 2048, WAVE_SPLIT_BELOW = 32768;
inline Geometry wave_launch_geometry(int64_t nt, int64_t ns, int64_t want_seg, int64_t max_seg = WAVE_SEGMENTS,
                                     bool whole_quarters = false) {
    Geometry g;
    g.tpt = 1;
    g.nblk_i = (int)((nt + BS - 1) / BS);
    g.wave_split = nt < WAVE_SPLIT_BELOW;
    const int64_t nq = std::max<int64_t>((ns + SB - 1) / SB, 1);
    const int64_t groups = std::max<int64_t>(g.wave_split ? (nt + 63) / 64 : g.nblk_i, 1);
    if (g.wave_split) want_seg = (want_seg + NW - 1) / NW;
    const int64_t fill = std::min<int64_t>((WAVE_FILL + groups - 1) / groups, max_seg);
    const int64_t nseg = std::min<int64_t>(std::max<int64_t>(std::max<int64_t>(want_seg, 1), fill), nq);
    int64_t qs = (nq + nseg - 1) / nseg;
    if (g.wave_split && (qs > 2 || whole_quarters)) qs = (qs + NW - 1) / NW * NW;
    g.seg_len = qs * SB;
    g.nseg = (int)((nq + qs - 1) / qs);
    return g;
}

// A k_force_f64 launch: segments of whole tiles, or, for few targets, of quarters
// until the chip has about WAVE_FILL workgroups (at 1000 particles four tiles
// gave 64 workgroups of four waves with 62 sources each).  A force call with its
// download: 300 to 1000 particles 40.5 -> 34 us, 3000 47.9 -> 43.7; on device
// arrays: 700 21.8 -> 18.8, 3000 28.5 -> 23.3; alike from 5000 on.
inline Geometry f64_launch_geometry(int64_t nt, int64_t ns, int64_t want_seg, int64_t max_seg = WAVE_SEGMENTS) {
    Geometry g = geometry(nt, ns, 1, want_seg);
    const int64_t groups = std::max<int64_t>((nt + 63) / 64, 1), nq = std::max<int64_t>((ns + SB - 1) / SB, 1);
    const int64_t fill = std::min<int64_t>(std::min<int64_t>((WAVE_FILL + groups - 1) / groups, max_seg), nq);
    if (fill > g.nseg) {
        const int64_t qs = (nq + fill - 1) / fill;
        g.seg_len = qs * SB;
        g.nseg = (int)((nq + qs - 1) / qs);
    }
    return g;
}

// Whether the waves of k_force_f64's workgroups share 64 targets: while the
// launch stays under 2^22 workgroups.
inline bool f64_split(int64_t nt, int nseg) { return (nt + 63) / 64 * nseg <= (1 << 22); }

// Passes of the force kernel (force_block): every tile, or the far tiles
// only (the split bf16 matrix-core launch, whose near tiles k_force_near adds).
constexpr int PASS_ALL = 0;
constexpr int PASS_FAR = 1;

// Launchers (nb_force.hip)
// Tile boxes (box) and quarter boxes (sub_box, with the largest of h or h_const
// in slot 6) of n particles; either output may be nullptr.
int launch_tile_boxes(const void *x, const void *y, const void *z, int is_double, int64_t n,
                      const double *h, double h_const, double *box, double *sub_box, hipStream_t s);
// acc = false (with pot) writes the potential alone.
// far_path FAR_MFMA_BF16 (tpt 1, forces or potential alone) runs the FP32
// state relative to a per-block FP64 origin; any other value is far path 0.
int launch_force_f32(const ForceArgs<float> &a, int tpt, bool pot, hipStream_t s, bool acc = true,
                     int far_path = FAR_VALU);
int launch_force_split(const ForceArgs<double> &a, int tpt, bool pot, hipStream_t s,
                       int far_path = 0, bool acc = true);
int launch_force_f64(const ForceArgs<double> &a, bool pot, hipStream_t s);
// w_i = m_i^(-2/3) (0 for massless particles) for the weighted far paths.
int launch_source_weights(const void *m, bool is_double, int64_t n, float *w, hipStream_t s);
inline bool far_path_weighted(int far_path) { return far_path == FAR_WEIGHTED || far_path == FAR_MFMA_BF16; }
// idx, when not null: target k's sums go to element idx[k].
int launch_finalize(const double *part, int nseg, int64_t n, double G, double *ax, double *ay,
                    double *az, double *pot, bool with_pot, hipStream_t s,
                    bool with_acc = true, const int64_t *idx = nullptr);
// The per-particle part of a KDK step (k_step): the kick of the force launch
// before it (from its segments' partial sums) and/or the next step's drift,
// which stores the tile boxes of the drifted positions and what else the force
// call that follows takes from it: with tgeo the target blocks' geometry
// (one target per lane, several segments), with tbg their bf16 B operands.
struct StepArgs {
    int64_t n;
    double dt, G;
    int kick, drift;
    void *x, *y, *z, *vx, *vy, *vz;
    const void *m;
    const double *h;             // target softening lengths
    const double *part;          // kick: [nseg][4][n]
    int nseg;
    double *ax, *ay, *az;
    int64_t ncentral;            // central bodies, with FP64 terms in the kick
    const int64_t *cidx;
    const uint8_t *central;
    const double *c_in;          // their x, y, z, m [4][ncentral] at the force's positions
    double *c_out;               // and where the drift stores the new ones
    double *time;
    int rd, wr;
    void *xn, *yn, *zn;          // where the drift puts the new positions (k_step: may be x, y, z)
    double *box, *sub, *tgeo;    // box may be nullptr
    unsigned *tbg;
    int use_origin;
    unsigned *arrived;           // k_force_step: as in ForceArgs
};
int launch_step(const StepArgs &a, bool is_double, hipStream_t s);
// The forces of far path 0 on targets that share waves (wave_split) and the
// step of their particles in one launch (k_force_step); positions are read from
// f and the drifted ones written to st.xn.. and st.sub, which no workgroup reads.
int launch_force_step(const ForceArgs<float> &f, const StepArgs &st, hipStream_t s);
int launch_force_step(const ForceArgs<double> &f, const StepArgs &st, hipStream_t s);

}  // namespace nb
