// nyl_march.h -- one pass over a multigrid level (k_mg_march): arguments and
// launchers shared by nyl_march.hip and the host code.
#pragma once
#include "nyl_internal.h"

namespace nyl {

// what a pass reads as the solution of its level
enum MarchSrc {
    MS_FIELD = 0,   // src
    MS_ZERO = 1,    // zero (src is not read)
    MS_PROLONG = 2  // src + the prolongation of the coarse level's xc
};

template <typename T, typename TC>
struct MarchArgs {
    Geo g, gc;              // the level, the next coarser one
    const T *src, *b;
    T *dst;                 // the result of the last sweep (src != dst)
    const TC *xc;           // MS_PROLONG: the coarse correction
    TC *bc, *yc;            // restriction: coarse right-hand side, its first sweep from zero
    double omega;
    MGTabs tab;
    double *partials;       // one per block: sum of the input's squared residuals
    float *rout;            // outer residual: r of the input, in the inner precision
    const double *shift;    // outer residual: subtracted from b (null: 0)
    double *xadd;           // MK_UP_ADD: the result is added to xadd instead of stored in dst
    const int *gate;        // the pass does nothing when *gate != 0 (null: always runs)
    int kz;                 // planes per block
};

// One member's share of a batched pass (tiles of 32 x 16 columns): a.kz is
// the member's own, so its block sums do not depend on the batch.
template <typename T, typename TC>
struct MarchItem {
    BHead h;
    int bx, by;
    MarchArgs<T, TC> a;
};
enum MarchKind {
    MK_UP, MK_UP_ADD, MK_DOWN, MK_RESTRICT, MK_PRE, MK_PRE_RESTRICT, MK_ZERO, MK_ZERO_RESTRICT, MK_OUTER
};
// Planes per block of a member's level, and the blocks of a pass over it: the
// member's own, whatever the batch, so that the block sums of its residual
// norms are.  Short marches for small levels (a batch has blocks enough only
// when its members do), longer ones where the blocks exceed NYL_RED_BLOCKS.
// A level of more than NYL_RED_BLOCKS tiles has more blocks than that all the
// same: the partials of a context have room for them (build_layout).
int b_march_kz(const Geo &g);
int64_t b_march_blocks(const Geo &g);
// map: the item of each block (32 bits: a batch may have any number of members)
template <typename T, typename TC>
hipError_t launch_b_march(const MarchItem<T, TC> *items, const uint32_t *map, int64_t nblk,
                          MarchKind kind, const MGTabs &tab, const int *active, hipStream_t s);

// Blocks of a pass over a level, and their march length.  even: the march
// works on plane pairs (restriction or prolongation).
struct MarchGrid {
    int tx, bx, by, bz, kz;
    int blocks() const { return bx * by * bz; }
};
MarchGrid march_grid(const Geo &g, int res, bool even);
// resident blocks per CU of a kind of pass, from its registers: es bytes per
// value, src a MarchSrc, sweeps, restr: with a restriction
constexpr int march_resident(int es, int src, int sweeps, bool restr) {
    if (sweeps == 0) return 6;   // the FP64 outer residual
    if (src == MS_PROLONG) return es == 4 ? 4 : 2;
    if (sweeps == 2 && restr) return src == MS_ZERO ? (es == 4 ? 4 : 3) : (es == 4 ? 3 : 2);
    if (src == MS_ZERO) return es == 4 ? 8 : 6;
    return es == 4 ? (sweeps == 1 ? 4 : 5) : 3;
}

// two sweeps src + P(xc) -> dst
template <typename T, typename TC>
hipError_t launch_march_up(const MarchArgs<T, TC> &a, hipStream_t s);
// one sweep src -> dst, then residual and restriction of dst into bc and yc
template <typename T, typename TC>
hipError_t launch_march_down(const MarchArgs<T, TC> &a, hipStream_t s);
// two sweeps src (null: zero) -> dst, then residual and restriction of dst
// into bc and yc; partials non-null: also the residual norm of src
template <typename T, typename TC>
hipError_t launch_march_pre(const MarchArgs<T, TC> &a, hipStream_t s);
// its blocks (es bytes per value)
MarchGrid march_pre_grid(const Geo &g, int es);
// the residual norm of src alone, block sums over the cells of gr's blocks;
// strips: in the order of k_mg_sweep2t's (tiles of 64 x 8), else of
// launch_march_pre's
template <typename T>
hipError_t launch_march_norm(const MarchArgs<T, T> &a, const MarchGrid &gr, bool strips,
                             hipStream_t s);
// the mixed solve's FP64 residual (b - shift) - A src: its norm, and its
// values in FP32 into rout
hipError_t launch_march_outer(const MarchArgs<double, double> &a, hipStream_t s);

}  // namespace nyl
