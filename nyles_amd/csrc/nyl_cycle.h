// nyl_cycle.h -- the small levels of a V-cycle in one workgroup
// (k_mg_cycle) and the device-side control of a multigrid solve.
#pragma once
#include "nyl_internal.h"

namespace nyl {

#define CYC_T 1024                // threads of the workgroup
#define CYC_R 4                   // most cells of the largest level per thread
#define CYC_MAXLEV 8
#define CYC_ENT 256               // most positions along the axes of the levels together
#define CYC_LDS (154 * 1024)      // bytes of LDS for the levels (160 KB per CU)

// One level of the cycle: its size, the multipliers that divide by nx and
// nx*ny (0: the divisor is 1), the places (bytes) of its three arrays in LDS
// and of its axes' entries in the position table.  a, c hold the solution
// (Jacobi source and destination) with a layer of zeros beyond each wall, b
// the right-hand side.
struct CycleLevel {
    int nx, ny, nz;
    uint32_t mx, mxy;
    uint32_t a, c, b;
    int ex, ey, ez;
    uint32_t size;                // elements of a and c
};

// One position along an axis of a level: the shares of the axis in the places
// (elements of a, c) of the cell and of its two neighbours, and of the coarse
// cells that a prolongation reads; a cell's place is the sum over the axes.
struct alignas(16) CycleEnt {
    uint32_t w[4];   // own | minus << 16, plus | count << 16 | inside << 20,
                     // coarse own | coarse neighbour << 16, 0
};

struct CycleArgs {
    CycleLevel lev[CYC_MAXLEV];   // lev[0] is the largest of the cycle
    int nl, n0;                   // levels; cells of lev[0]
    int nent;
    int px, py, pz;
    int exact;                    // the coarsest level is solved directly
    uint32_t e;                   // LDS place (bytes) of its eigenvector tables
    uint32_t bytes;               // LDS used
    const CycleEnt *ent;          // the position table in memory
    const double *etab;           // the eigenvector tables in memory (coarse_tables)
    double omega;
    MGTabs tab;
};

// Levels l0 .. nlev-1 of a hierarchy as a cycle, es bytes per value of the
// levels above the coarsest (which is FP64); false when they do not fit one
// workgroup (more than CYC_T * CYC_R cells, CYC_ENT positions, or the LDS).
// ent (room for CYC_ENT): the position table.
bool cycle_layout(CycleArgs &a, CycleEnt *ent, const Geo *lev, int l0, int nlev, int es,
                  bool exact, double omega, const MGTabs &tab);

// ---- control of a solve on the device ---------------------------------------
// The stop rule of mgfor's loop (core/mgfor/solvers.f90:17-30) runs where
// its sums are: the host enqueues the V-cycles a solve is expected to need
// and reads the results once, and the pass that writes a V-cycle's result is
// skipped (its gate) from the test that stopped the loop on.
#define CTL_HIST 96
struct MGCtl {
    double normb, shift;          // |b - mean|^2, mean of b (mixed)
    double res;                   // mixed: last outer residual, relative
    double target;                // mixed: squared residual that ends the inner loop, relative
    int stop;                     // the (inner) loop has stopped: V-cycle results are not written
    int outer_stop;               // mixed: the FP64 residual has met the tolerance
    int no_add;                   // mixed: no inner solution to add (outer stop, or inner loop open)
    int rel;                      // mixed: target is relative to the outer residual
    double hist[CTL_HIST];        // the sums of squares of the tests, in order
};

enum CtlKind {
    CTL_NORMB = 0,     // normb = sum; opens the loop
    CTL_SHIFT = 1,     // two sums: mean of b and |b - mean|^2
    CTL_TEST = 2,      // FP64 loop: stop when sum / normb < tol
    CTL_OUTER = 3,     // mixed: FP64 residual of x; sets the inner target
    CTL_INNER = 4,     // mixed: inner residual after V-cycle k
    CTL_NONE = 5       // publish only
};

struct CtlArgs {
    MGCtl *ctl;
    const double *partials;
    int np;            // partial sums (CTL_SHIFT: of each of the two sums)
    int kind;
    int k;             // CTL_INNER: V-cycles of this inner loop so far
    int slot;          // hist entry that receives the sum (-1: none)
    double tol, ncell;
    double inner_red;  // mixed: squared reduction one inner solve is asked for
    int inner_max;     // ... and its most V-cycles when that is the target
    // publication to coherent host memory (dst null: none): normb, shift and
    // hist[0 .. nhist), then the sequence number
    double *dst;
    uint32_t *flag;
    uint32_t seq;
    int nhist;
};
hipError_t launch_ctl(const CtlArgs &c, hipStream_t s);

// the cycle from y (the first sweep of lev[0], replaced by the level's
// correction) and b; a one-level cycle (FP64) writes x instead.  fin
// non-null: a second workgroup runs launch_ctl's work.
template <typename T>
hipError_t launch_mg_cycle(const CycleArgs &a, const T *b, T *y, T *x, const CtlArgs *fin,
                           hipStream_t s);

// one member's cycle in a batch (a.bytes and a.n0 as for the single launch)
template <typename T>
struct CycleItem {
    int member;
    CycleArgs a;
    const T *b;
    T *y, *x;
};
// most: the largest a.n0 of the items
template <typename T>
hipError_t launch_b_cycle(const CycleItem<T> *items, int n, int most, const int *active,
                          hipStream_t s);

}  // namespace nyl
