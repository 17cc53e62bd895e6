// nyl_stencil.hip -- the diagnostic stencils, reductions and ensemble forms of
// the Nyles time step on gfx950 (the stage kernels: nyl_stage.h).
//
// Every FP64 instantiation reproduces the reference's arithmetic operation
// by operation (the library is compiled with -ffp-contract=off), so its
// results are bit-identical to the oracle's.
#include "nyl_stage.h"
#include <initializer_list>

namespace nyl {

// The per-cell diagnostic kernels (div, correct, diag): each thread takes
// NYL_CELL_KZ consecutive planes of its column (when nz is a multiple), in
// the XCD y-slab order of the stage kernel.
#ifndef NYL_CELL_KZ
#define NYL_CELL_KZ 1
#endif
#ifndef NYL_CELL_YSLAB
#define NYL_CELL_YSLAB 0
#endif
static inline int cell_kz(const Geo &g) { return g.nz % NYL_CELL_KZ == 0 ? NYL_CELL_KZ : 1; }
static inline dim3 cell_grid_kz(const Geo &g) {
    return dim3((g.nx + NYL_BX - 1) / NYL_BX, (g.ny + NYL_BY - 1) / NYL_BY, g.nz / cell_kz(g));
}
#if NYL_CELL_YSLAB
#define CELL_BLOCK() xcd_block_yslab()
#else
#define CELL_BLOCK() xcd_block()
#endif

// ---------------------------------------------------------------------------
// The stage kernel as a 2.5-D march (k_stage25).  A block owns a tile of
// S25_TX x S25_TY columns and walks a range of z planes.  Per plane:
//  * the fields that the in-plane (x, y) stencils read -- b, the three
//    vorticity components, u, v, w and ke of plane k, u and v of plane
//    k+1 -- are staged in LDS, each element loaded once, with the halo each
//    stencil reaches (3 cells for the WENO stencils, 1 for the averages);
//  * the x and y tracer face fluxes of the tile are evaluated once each into
//    LDS (the per-cell kernel evaluates every face twice, once for each
//    cell beside it);
//  * the z stencils (the tracer and vortex-force terms 4 and 5) read
//    per-thread register windows of the column (b over k-3..k+3, vor_i and
//    vor_j over k-3..k+2), the z face flux of the tracer and the z-averaged
//    velocities of terms 4 and 5 are carried to the next plane.
// Per cell that is about 9.5 reconstructions instead of 12, and no stencil
// value is gathered from L1/L2.  Every value is the per-cell kernel's
// expression in the same order (stage_cells), so the results are the same
// bits (checked on the CPU against k_stage).  Nothing launches it: its
// registers leave 3 waves per SIMD between the barriers (1.7 ms against 1.0
// for k_stage_flat, FP64 256^3); it stays as an independent form of the
// stage to check k_stage against.
#define S25_TX 64
#define S25_TY 4
#define S25_NT (S25_TX * S25_TY)

constexpr int S25_BW = S25_TX + 6, S25_BH = S25_TY + 6;
constexpr int S25_W1 = S25_TX + 1, S25_H1 = S25_TY + 1;

// Sequencing of the per-cell terms of k_stage25: the LDS column index of
// the next term passes through an empty asm that takes the previous term's
// result, so the next term's loads are not hoisted above it and each term
// holds only its own operands (no instruction is emitted).
#if NYL_STAGE_SEQ
#define S25_SEQ(idx, dep) asm volatile("" : "+v"(idx) : "v"(dep))
#else
#define S25_SEQ(idx, dep) ((void)0)
#endif

template <typename T>
struct S25Lds {
    T b[S25_BH * S25_BW];     // b(k):   x in [-3, TX+3), y in [-3, TY+3)
    T oz[S25_BH * S25_BW];    // vor_k:  same box
    T ox[S25_BH * S25_TX];    // vor_i:  x in [0, TX),    y in [-3, TY+3)
    T oy[S25_TY * S25_BW];    // vor_j:  x in [-3, TX+3), y in [0, TY)
    T u0[S25_H1 * S25_W1];    // u(k):   x in [-1, TX),   y in [0, TY+1)
    T u1[S25_TY * S25_W1];    // u(k+1): x in [-1, TX),   y in [0, TY)
    T v0[S25_H1 * S25_W1];    // v(k):   x in [0, TX+1),  y in [-1, TY)
    T v1[S25_H1 * S25_TX];    // v(k+1): x in [0, TX),    y in [-1, TY)
    T w0[S25_H1 * S25_W1];    // w(k):   x in [0, TX+1),  y in [0, TY+1)
    T ke[S25_H1 * S25_W1];    // ke(k):  x in [0, TX+1),  y in [0, TY+1)
    T fx[S25_TY * S25_W1];    // x-face tracer fluxes, faces -1 .. TX-1 of each row
    T fy[S25_H1 * S25_TX];    // y-face tracer fluxes, faces -1 .. TY-1 of each column
};

// Columns of the LDS boxes for one lane: x = i0 + X0 + lane (lo) and
// x = i0 + X0 + 64 + lane (hi, the lanes past 64 of a wide box), wrapped on
// a periodic axis, -1 off the grid; X0 = -3, -1, 0.  Plane-invariant.
struct S25Cols {
    int lo[3], hi[3];
};
template <int X0>
__device__ constexpr int s25_xi() { return X0 == -3 ? 0 : (X0 == -1 ? 1 : 2); }

// One LDS box: field f of plane offset pl (elements) over x in
// [i0+X0, i0+X0+W), y in [j0+Y0, j0+Y0+H), row-major: wave w fills rows w,
// w+TY, ... (the row's offset is wave-uniform), each lane one or two
// columns.  Periodic positions wrap; positions off a wall axis (or past a
// partial tile) store 0: the closures never read them.
template <typename T, int PY, int X0, int Y0, int W, int H>
__device__ __forceinline__ void s25_box(T *__restrict__ dst, const T *__restrict__ f,
                                        const Geo &g, int j0, int64_t pl, int lane, int wave,
                                        const S25Cols &cc) {
    constexpr uint32_t ES = sizeof(T);
    constexpr int XI = s25_xi<X0>();
    const int lo = cc.lo[XI], hi = cc.hi[XI];
    for (int r = wave; r < H; r += S25_TY) {
        int gj = j0 + Y0 + r;
        if (PY) gj = gj < 0 ? gj + g.ny : (gj >= g.ny ? gj - g.ny : gj);
        const bool rok = gj >= 0 && gj < g.ny;
        const T *__restrict__ row = f + (rok ? pl + (int64_t)gj * g.sy : 0);
        dst[r * W + lane] = (rok && lo >= 0) ? ldb(row, (uint32_t)lo * ES) : T(0);
        if (W > S25_TX && lane < W - S25_TX)
            dst[r * W + S25_TX + lane] = (rok && hi >= 0) ? ldb(row, (uint32_t)hi * ES) : T(0);
    }
}

// A window of n values of the thread's column along z, held in scalars (a
// register array indexed by a selected position would be placed in scratch
// memory); at(d) with a constant d.
template <typename T>
struct S25Win7 {
    T v0, v1, v2, v3, v4, v5, v6;
    __device__ __forceinline__ T at(int d) const {
        switch (d) {
        case 0: return v0; case 1: return v1; case 2: return v2; case 3: return v3;
        case 4: return v4; case 5: return v5; default: return v6;
        }
    }
    __device__ __forceinline__ void shift() { v0 = v1; v1 = v2; v2 = v3; v3 = v4; v4 = v5; v5 = v6; }
};

// vf_flux on staged values: UU(dm) is the averaged contravariant velocity at
// line position md + dm (dm = -1, 0), om(m) the vorticity at line position m
template <typename T, int PER, typename UF, typename OF>
__device__ __forceinline__ T s25_vf(int md, int nd, const UF &UU, const OF &om) {
    T uu_prev;
    if (!PER && md == 0) uu_prev = T(0);   // UU_0 = 0. at the line start
    else uu_prev = UU(-1);
    const T u1d = T(0.5) * (uu_prev + UU(0));
    auto q = [&](int m) -> T {             // q(1) = 0., q(k) = vort(k-1)
        if (!PER && m == 0) return T(0);
        return om(m - 1);
    };
    return face_flux<T, PER>(md, nd, u1d, q);
}

template <typename T, int MODE, int PX, int PY, int PZ>
__global__ __launch_bounds__(S25_NT) void k_stage25(Geo g, StageArgs<T> a, int kz) {
    __shared__ S25Lds<T> L;
    constexpr uint32_t ES = sizeof(T);
    const Blk3 bk = xcd_block();
    const int tid = threadIdx.x;
    const int tx = tid % S25_TX, ty = tid / S25_TX;
    const int i0 = bk.x * S25_TX, j0 = bk.y * S25_TY;
    const int i = i0 + tx, j = j0 + ty;
    const int nz = g.nz;
    const int k0 = bk.z * kz, k1 = k0 + kz < nz ? k0 + kz : nz;
    const bool live = i < g.nx && j < g.ny;
    // the thread's column (threads past a partial tile use column 0, and
    // compute nothing from it)
    const int ic = live ? i : 0, jc = live ? j : 0;
    const int64_t col = (int64_t)jc * g.sy + ic;
    const T cx = T(a.idx2), cy = T(a.idy2), cz = T(a.idz2);
    auto zw = [&](int kk) -> int { return PZ ? (kk < 0 ? kk + nz : (kk >= nz ? kk - nz : kk)) : kk; };
    auto zok = [&](int kk) -> bool { return PZ || (kk >= 0 && kk < nz); };
    // field f at the thread's column (offset dc within the plane), plane kk
    auto colv = [&](const T *__restrict__ f, int kk, int64_t dc) -> T {
        return zok(kk) ? ldb(f, (uint32_t)((int64_t)zw(kk) * g.sz + col + dc) * ES) : T(0);
    };
    // offsets of the x+1 and y+1 neighbours of the column (0 when absent)
    const int64_t dxp = (PX || ic + 1 < g.nx) ? (int64_t)((PX && ic + 1 >= g.nx) ? 1 - g.nx : 1)
                                              : 0;
    const int64_t dyp = (PY || jc + 1 < g.ny) ? ((PY && jc + 1 >= g.ny) ? (1 - g.ny) * g.sy : g.sy)
                                              : 0;
    // register windows along z: b over k-3 .. k+3, vor_i and vor_j over
    // k-3 .. k+2 (the last slot of those unused)
    S25Win7<T> bw, xw, yw;
    bw.v0 = colv(a.b, k0 - 3, 0); bw.v1 = colv(a.b, k0 - 2, 0); bw.v2 = colv(a.b, k0 - 1, 0);
    bw.v3 = colv(a.b, k0, 0); bw.v4 = colv(a.b, k0 + 1, 0); bw.v5 = colv(a.b, k0 + 2, 0);
    xw.v0 = colv(a.ox, k0 - 3, 0); xw.v1 = colv(a.ox, k0 - 2, 0); xw.v2 = colv(a.ox, k0 - 1, 0);
    xw.v3 = colv(a.ox, k0, 0); xw.v4 = colv(a.ox, k0 + 1, 0);
    yw.v0 = colv(a.oy, k0 - 3, 0); yw.v1 = colv(a.oy, k0 - 2, 0); yw.v2 = colv(a.oy, k0 - 1, 0);
    yw.v3 = colv(a.oy, k0, 0); yw.v4 = colv(a.oy, k0 + 1, 0);
    bw.v6 = xw.v5 = xw.v6 = yw.v5 = yw.v6 = T(0);
    // carried from the plane below: the tracer flux through face k-1 and the
    // z-averaged U_k of vortex-force terms 4 (averaged in y) and 5 (in x)
    T fzl = T(0), uu4p = T(0), uu5p = T(0);
    if (PZ || k0 > 0) {
        const T wm = colv(a.w, k0 - 1, 0);
        fzl = face_flux_rel<T, PZ>(zw(k0 - 1), nz, wm * cz,
                                   [&](int d) -> T { return bw.at(d + 2); });
        uu4p = T(0.5) * (wm * cz + colv(a.w, k0 - 1, dyp) * cz);
        uu5p = T(0.5) * (wm * cz + colv(a.w, k0 - 1, dxp) * cz);
    }
    // the lane's box columns
    S25Cols cc;
    {
        const int x0s[3] = {-3, -1, 0};
#pragma unroll
        for (int q = 0; q < 3; q++) {
            int lo = i0 + x0s[q] + tx, hi = lo + S25_TX;
            if (PX) {
                lo = lo < 0 ? lo + g.nx : (lo >= g.nx ? lo - g.nx : lo);
                hi = hi >= g.nx ? hi - g.nx : hi;
            }
            cc.lo[q] = (lo >= 0 && lo < g.nx) ? lo : -1;
            cc.hi[q] = (hi >= 0 && hi < g.nx) ? hi : -1;
        }
    }
    for (int k = k0; k < k1; k++) {
        const int64_t pl = (int64_t)k * g.sz;
        const bool has_kp = zok(k + 1);
        const int64_t plp = (int64_t)zw(k + 1) * g.sz;
        bw.v6 = colv(a.b, k + 3, 0);
        xw.v5 = colv(a.ox, k + 2, 0);
        yw.v5 = colv(a.oy, k + 2, 0);
        const T ke_up = has_kp ? ldb(a.ke, (uint32_t)(plp + col) * ES) : T(0);
        s25_box<T, PY, -3, -3, S25_BW, S25_BH>(L.b, a.b, g, j0, pl, tx, ty, cc);
        s25_box<T, PY, -3, -3, S25_BW, S25_BH>(L.oz, a.oz, g, j0, pl, tx, ty, cc);
        s25_box<T, PY, 0, -3, S25_TX, S25_BH>(L.ox, a.ox, g, j0, pl, tx, ty, cc);
        s25_box<T, PY, -3, 0, S25_BW, S25_TY>(L.oy, a.oy, g, j0, pl, tx, ty, cc);
        s25_box<T, PY, -1, 0, S25_W1, S25_H1>(L.u0, a.u, g, j0, pl, tx, ty, cc);
        s25_box<T, PY, 0, -1, S25_W1, S25_H1>(L.v0, a.v, g, j0, pl, tx, ty, cc);
        s25_box<T, PY, 0, 0, S25_W1, S25_H1>(L.w0, a.w, g, j0, pl, tx, ty, cc);
        s25_box<T, PY, 0, 0, S25_W1, S25_H1>(L.ke, a.ke, g, j0, pl, tx, ty, cc);
        if (has_kp) {
            s25_box<T, PY, -1, 0, S25_W1, S25_TY>(L.u1, a.u, g, j0, plp, tx, ty, cc);
            s25_box<T, PY, 0, -1, S25_TX, S25_H1>(L.v1, a.v, g, j0, plp, tx, ty, cc);
        }
        __syncthreads();
        // tracer face fluxes of the tile: x faces i0-1 .. i0+TX-1 of each
        // row, y faces j0-1 .. j0+TY-1 of each column.  Wave w: the x faces
        // i0-1 .. i0+TX-2 of row w and the y faces of row j0+w-1; then wave 0
        // the y faces of row j0+TY-1 and wave 1 the last x face of each row.
        {
            auto xface = [&](int r, int fr) -> T {
                const int f = i0 + fr;
                if (!((PX || f >= 0) && f < g.nx && j0 + r < g.ny)) return T(0);
                auto q = [&](int m) -> T { return L.b[(r + 3) * S25_BW + (m - i0 + 3)]; };
                return face_flux<T, PX>(f, g.nx, L.u0[r * S25_W1 + fr + 1] * cx, q);
            };
            auto yface = [&](int c, int fr) -> T {
                const int f = j0 + fr;
                if (!((PY || f >= 0) && f < g.ny && i0 + c < g.nx)) return T(0);
                auto q = [&](int m) -> T { return L.b[(m - j0 + 3) * S25_BW + (c + 3)]; };
                return face_flux<T, PY>(f, g.ny, L.v0[(fr + 1) * S25_W1 + c] * cy, q);
            };
            const T fxv = xface(ty, tx - 1);
            L.fx[ty * S25_W1 + tx] = fxv;
            int cq = tx;
            S25_SEQ(cq, fxv);
            const T fyv = yface(cq, ty - 1);
            L.fy[ty * S25_TX + tx] = fyv;
            S25_SEQ(cq, fyv);
            if (ty == 0) L.fy[S25_TY * S25_TX + tx] = yface(cq, S25_TY - 1);
            else if (ty == 1 && tx < S25_TY) L.fx[tx * S25_W1 + S25_TX] = xface(cq, S25_TX - 1);
        }
        __syncthreads();
        if (live) {
            const uint32_t cb = (uint32_t)(pl + col) * ES;
            // tracer b: rhstrac, directions i, j, k (core/tracer.py:63-72)
            T db = T(0);
            {
                const T fl = L.fx[ty * S25_W1 + tx], fr = L.fx[ty * S25_W1 + tx + 1];
                if (!PX && i == 0) db = db - fr;
                else db = (db + fl) - fr;
            }
            {
                const T fl = L.fy[ty * S25_TX + tx], fr = L.fy[(ty + 1) * S25_TX + tx];
                if (!PY && j == 0) db = db - fr;
                else db = (db + fl) - fr;
            }
            const T wc = L.w0[ty * S25_W1 + tx];
            {
                const T fr = face_flux_rel<T, PZ>(k, nz, wc * cz,
                                                  [&](int d) -> T { return bw.at(d + 3); });
                if (!PZ && k == 0) db = db - fr;
                else db = (db + fzl) - fr;
                fzl = fr;
            }
            // vortex force, triplets 'ikj', 'jik', 'kji' (core/vortex_force.py:69-81)
            const bool ex = PX || i < g.nx - 1;
            const bool ey = PY || j < g.ny - 1;
            const bool ez = PZ || k < nz - 1;
            int lx = tx;             // the LDS column, sequenced between the terms
            S25_SEQ(lx, db);
            const T uu4 = T(0.5) * (wc * cz + L.w0[(ty + 1) * S25_W1 + lx] * cz);
            const T uu5 = T(0.5) * (wc * cz + L.w0[ty * S25_W1 + lx + 1] * cz);
            T du = T(0), dv = T(0), dw = T(0);
            // direc(U_i, vor_k, du_j): along x, U_i averaged in y
            if (ey)
                dv = dv - s25_vf<T, PX>(i, g.nx,
                    [&](int dm) -> T {
                        return T(0.5) * (L.u0[ty * S25_W1 + lx + 1 + dm] * cx +
                                         L.u0[(ty + 1) * S25_W1 + lx + 1 + dm] * cx);
                    },
                    [&](int m) -> T { return L.oz[(ty + 3) * S25_BW + (m - i + lx + 3)]; });
            S25_SEQ(lx, dv);
            // flip(U_j, vor_k, du_i): along y, U_j averaged in x
            if (ex)
                du = du + s25_vf<T, PY>(j, g.ny,
                    [&](int dm) -> T {
                        return T(0.5) * (L.v0[(ty + 1 + dm) * S25_W1 + lx] * cy +
                                         L.v0[(ty + 1 + dm) * S25_W1 + lx + 1] * cy);
                    },
                    [&](int m) -> T { return L.oz[(m - j + ty + 3) * S25_BW + (lx + 3)]; });
            S25_SEQ(lx, du);
            // direc(U_j, vor_i, du_k): along y, U_j averaged in z
            if (ez)
                dw = dw - s25_vf<T, PY>(j, g.ny,
                    [&](int dm) -> T {
                        return T(0.5) * (L.v0[(ty + 1 + dm) * S25_W1 + lx] * cy +
                                         L.v1[(ty + 1 + dm) * S25_TX + lx] * cy);
                    },
                    [&](int m) -> T { return L.ox[(m - j + ty + 3) * S25_TX + lx]; });
            S25_SEQ(lx, dw);
            // flip(U_k, vor_i, du_j): along z, U_k averaged in y
            if (ey) {
                const T uu_prev = (!PZ && k == 0) ? T(0) : uu4p;
                const T u1d = T(0.5) * (uu_prev + uu4);
                dv = dv + face_flux_rel<T, PZ>(k, nz, u1d, [&](int d) -> T {
                    if (!PZ && k + d == 0) return T(0);
                    return xw.at(d + 2);
                });
            }
            // direc(U_k, vor_j, du_i): along z, U_k averaged in x
            if (ex) {
                const T uu_prev = (!PZ && k == 0) ? T(0) : uu5p;
                const T u1d = T(0.5) * (uu_prev + uu5);
                du = du - face_flux_rel<T, PZ>(k, nz, u1d, [&](int d) -> T {
                    if (!PZ && k + d == 0) return T(0);
                    return yw.at(d + 2);
                });
            }
            uu4p = uu4;
            uu5p = uu5;
            S25_SEQ(lx, du);
            // flip(U_i, vor_j, du_k): along x, U_i averaged in z
            if (ez)
                dw = dw + s25_vf<T, PX>(i, g.nx,
                    [&](int dm) -> T {
                        return T(0.5) * (L.u0[ty * S25_W1 + lx + 1 + dm] * cx +
                                         L.u1[ty * S25_W1 + lx + 1 + dm] * cx);
                    },
                    [&](int m) -> T { return L.oy[ty * S25_BW + (m - i + lx + 3)]; });

            // bernoulli (core/bernoulli.py:14-23, core/fortran_bernoulli.f90:2-58)
            const T kec = L.ke[ty * S25_W1 + tx];
            if (ex) du = du - (L.ke[ty * S25_W1 + tx + 1] - kec);
            if (ey) dv = dv - (L.ke[(ty + 1) * S25_W1 + tx] - kec);
            if (ez) {
                const T cff = T(0.5 * a.dz);
                dw = dw - (ke_up - kec) + cff * (bw.v4 + bw.v3);
            }
            // viscosity at the last stage (core/model_les.py:140-141)
            if (a.visc) viscosity_cell<T, PX, PY, PZ>(g, a, cb, i, j, k, du, dv, dw);

            const T b0 = bw.v3, u0 = L.u0[ty * S25_W1 + tx + 1];
            const T v0 = L.v0[(ty + 1) * S25_W1 + tx], w0 = wc;
            if (MODE == 0 || MODE == 1 || MODE == 2) {
                stb_stream(a.tb, cb, db); stb_stream(a.tu, cb, du); stb_stream(a.tv, cb, dv); stb_stream(a.tw, cb, dw);
            }
            const T cc = T(a.c);
            if (MODE == 1) {            // s += dt*ds0
                stb(a.bn, cb, b0 + cc * db);
                stb(a.un, cb, u0 + cc * du);
                stb(a.vn, cb, v0 + cc * dv);
                stb(a.wn, cb, w0 + cc * dw);
            } else if (MODE == 2) {     // s += (dt/4.)*(ds1-3*ds0)
                stb(a.bn, cb, b0 + cc * (db - T(3) * ldb(a.d0b, cb)));
                stb(a.un, cb, u0 + cc * (du - T(3) * ldb(a.d0u, cb)));
                stb(a.vn, cb, v0 + cc * (dv - T(3) * ldb(a.d0v, cb)));
                stb(a.wn, cb, w0 + cc * (dw - T(3) * ldb(a.d0w, cb)));
            } else if (MODE == 3) {     // s += (dt/12.)*(8*ds2-ds0-ds1)
                stb(a.bn, cb, b0 + cc * ((T(8) * db - ldb(a.d0b, cb)) - ldb(a.d1b, cb)));
                stb(a.un, cb, u0 + cc * ((T(8) * du - ldb(a.d0u, cb)) - ldb(a.d1u, cb)));
                stb(a.vn, cb, v0 + cc * ((T(8) * dv - ldb(a.d0v, cb)) - ldb(a.d1v, cb)));
                stb(a.wn, cb, w0 + cc * ((T(8) * dw - ldb(a.d0w, cb)) - ldb(a.d1w, cb)));
            } else if (MODE == 4) {     // LFAM3 predictor (core/timescheme.py:144-162)
                const T c2 = T(a.c2), c12 = T(1. / 12.);
                T sb, t1;
                sb = ldb(a.sbb, cb); t1 = sb + c2 * db; stb(a.bn, cb, c12 * (T(5) * t1 + T(8) * b0 - sb)); stb(a.sbb, cb, b0);
                sb = ldb(a.sbu, cb); t1 = sb + c2 * du; stb(a.un, cb, c12 * (T(5) * t1 + T(8) * u0 - sb)); stb(a.sbu, cb, u0);
                sb = ldb(a.sbv, cb); t1 = sb + c2 * dv; stb(a.vn, cb, c12 * (T(5) * t1 + T(8) * v0 - sb)); stb(a.sbv, cb, v0);
                sb = ldb(a.sbw, cb); t1 = sb + c2 * dw; stb(a.wn, cb, c12 * (T(5) * t1 + T(8) * w0 - sb)); stb(a.sbw, cb, w0);
            } else if (MODE == 5) {     // LFAM3 corrector: s = sn + dt*ds
                stb(a.bn, cb, ldb(a.bn, cb) + cc * db);
                stb(a.un, cb, ldb(a.un, cb) + cc * du);
                stb(a.vn, cb, ldb(a.vn, cb) + cc * dv);
                stb(a.wn, cb, ldb(a.wn, cb) + cc * dw);
            } else if (MODE == 6) {     // first LFAM3 step: sn = s; sb = s; s += dt*ds
                stb(a.sbb, cb, b0); stb(a.sbu, cb, u0); stb(a.sbv, cb, v0); stb(a.sbw, cb, w0);
                stb(a.bn, cb, b0 + cc * db);
                stb(a.un, cb, u0 + cc * du);
                stb(a.vn, cb, v0 + cc * dv);
                stb(a.wn, cb, w0 + cc * dw);
            }
        }
        bw.shift();
        xw.shift();
        yw.shift();
        __syncthreads();
    }
}

// The stage combinations of the stage kernel with the tendency read from memory
template <typename T, int MODE>
__global__ __launch_bounds__(256) void k_update(int64_t n, UpdateArgs<T> a) {
    const int64_t q = (int64_t)blockIdx.x * 256 + threadIdx.x;
    if (q >= n) return;
    const T cc = T(a.c);
    if (MODE == 1) {
        a.sn[q] = a.s[q] + cc * a.ds0[q];
    } else if (MODE == 2) {
        a.sn[q] = a.s[q] + cc * (a.ds1[q] - T(3) * a.ds0[q]);
    } else if (MODE == 3) {
        a.sn[q] = a.s[q] + cc * ((T(8) * a.ds2[q] - a.ds0[q]) - a.ds1[q]);
    } else if (MODE == 4) {
        const T c2 = T(a.c2), c12 = T(1. / 12.);
        const T sb = a.sb[q], t1 = sb + c2 * a.ds0[q];
        a.sn[q] = c12 * (T(5) * t1 + T(8) * a.s[q] - sb);
        a.sb[q] = a.s[q];
    } else if (MODE == 5) {
        a.sn[q] = a.sn[q] + cc * a.ds0[q];
    } else if (MODE == 6) {
        a.sb[q] = a.s[q];
        a.sn[q] = a.s[q] + cc * a.ds0[q];
    }
}

template <typename T>
hipError_t launch_update(int64_t n, const UpdateArgs<T> &a, int mode, hipStream_t s) {
    const dim3 grd((unsigned)((n + 255) / 256));
    switch (mode) {
    case 1: NYL_LAUNCH((k_update<T, 1>), grd, dim3(256), 0, s, n, a); break;
    case 2: NYL_LAUNCH((k_update<T, 2>), grd, dim3(256), 0, s, n, a); break;
    case 3: NYL_LAUNCH((k_update<T, 3>), grd, dim3(256), 0, s, n, a); break;
    case 4: NYL_LAUNCH((k_update<T, 4>), grd, dim3(256), 0, s, n, a); break;
    case 5: NYL_LAUNCH((k_update<T, 5>), grd, dim3(256), 0, s, n, a); break;
    case 6: NYL_LAUNCH((k_update<T, 6>), grd, dim3(256), 0, s, n, a); break;
    default: return hipErrorInvalidValue;
    }
    return hipGetLastError();
}

// ---------------------------------------------------------------------------
// Four cells along x per thread: the per-cell kernels here are latency-bound
// at one cell per thread (one 4-byte load per field and cell); the x4 forms
// move the same bytes with 16-byte loads and stores, a quarter of the memory
// instructions.  Each cell's arithmetic is that of div_cell, correct_cell or
// diag_cell, term for term, so the results are the same bits.  They need
// nx % 4 == 0 and 16-byte aligned fields (the workspace is 256-byte aligned).

template <typename T>
struct Q4 {
    T v[4];
};
__device__ __forceinline__ Q4<float> ld4(const float *p) {
    const float4 q = *reinterpret_cast<const float4 *>(p);
    return {{q.x, q.y, q.z, q.w}};
}
__device__ __forceinline__ Q4<double> ld4(const double *p) {
    const double2 a = *reinterpret_cast<const double2 *>(p);
    const double2 b = *reinterpret_cast<const double2 *>(p + 2);
    return {{a.x, a.y, b.x, b.y}};
}
__device__ __forceinline__ void st4(float *p, const Q4<float> &q) {
    *reinterpret_cast<float4 *>(p) = make_float4(q.v[0], q.v[1], q.v[2], q.v[3]);
}
__device__ __forceinline__ void st4(double *p, const Q4<double> &q) {
    *reinterpret_cast<double2 *>(p) = make_double2(q.v[0], q.v[1]);
    *reinterpret_cast<double2 *>(p + 2) = make_double2(q.v[2], q.v[3]);
}
// st4 with the nontemporal hint (the four stores merge into wide ones)
template <typename T>
__device__ __forceinline__ void st4_stream(T *p, const Q4<T> &q) {
#pragma unroll
    for (int m = 0; m < 4; m++) store_stream(p + m, q.v[m]);
}

static inline dim3 cell_grid4(const Geo &g) {
    return dim3((g.nx / 4 + NYL_BX - 1) / NYL_BX, (g.ny + NYL_BY - 1) / NYL_BY, g.nz / cell_kz(g));
}

static inline bool quad_ok(const Geo &g, std::initializer_list<const void *> ptrs) {
    if (g.nx % 4 != 0) return false;
    for (const void *p : ptrs)
        if (p && (reinterpret_cast<uintptr_t>(p) & 15u) != 0) return false;
    return true;
}

// diag_cell for cells i0 .. i0+3; WHAT is the diag_cell selection as a
// compile-time constant.  FP32: every load the selection needs is issued at
// the top of a plane, together (one memory latency per plane; a neighbour
// outside a wall axis is loaded from the own cell instead and never used),
// and the results are stored with the nontemporal hint (the next stage
// kernel reads them): 115 -> 95 us at 256^3.  FP64: the neighbour loads of
// each part just before it and plain stores (the register cost of hoisting
// the FP64 loads lowers occupancy; 206 vs 232 us, and the hint gains nothing).
template <typename T, int WHAT>
__global__ __launch_bounds__(256) void k_diag4(Geo g, DiagArgs<T> a) {
    constexpr bool HOIST = sizeof(T) == 4;
    const Blk3 bk = CELL_BLOCK();
    const int i0 = (bk.x * NYL_BX + threadIdx.x) * 4;
    const int j = bk.y * NYL_BY + threadIdx.y;
    if (i0 >= g.nx || j >= g.ny) return;
    const int kz = g.nz / (int)gridDim.z;
    // x neighbours of the quad's end cells
    const bool hxm = g.px || i0 > 0;                  // cell i0 has an x-1 neighbour
    const int64_t oxm = g.px ? (int64_t)(i0 - wrapi(i0 - 1, g.nx)) : 1;
    const bool ex3 = g.px || i0 + 3 < g.nx - 1;       // cell i0+3 has an x+1 neighbour
    const int64_t oxp3 = g.px ? (int64_t)(wrapi(i0 + 4, g.nx) - (i0 + 3)) : 1;
    const bool ey = g.py || j < g.ny - 1, hym = g.py || j > 0;
    const int64_t oyp = g.py ? (int64_t)(wrapi(j + 1, g.ny) - j) * g.sy : g.sy;
    const int64_t oym = g.py ? (int64_t)(j - wrapi(j - 1, g.ny)) * g.sy : g.sy;
    auto out4 = [&](T *p, const Q4<T> &q) {
        if constexpr (HOIST) st4_stream(p, q);
        else st4(p, q);
    };
    for (int k = bk.z * kz; k < (bk.z + 1) * kz; k++) {
        const int64_t c = (int64_t)k * g.sz + (int64_t)j * g.sy + i0;
        const bool ez = g.pz || k < g.nz - 1, hzm = g.pz || k > 0;
        const int64_t ozp = g.pz ? (int64_t)(wrapi(k + 1, g.nz) - k) * g.sz : g.sz;
        const int64_t ozm = g.pz ? (int64_t)(k - wrapi(k - 1, g.nz)) * g.sz : g.sz;
        const Q4<T> u = ld4(a.u + c), v = ld4(a.v + c), w = ld4(a.w + c);
        T v4 = T(0), w4 = T(0), um0 = T(0);
        Q4<T> uyp{}, wyp{}, vzp{}, uzp{}, vm{}, wm{};
        if (HOIST && (WHAT & 2)) {
            const int64_t cx = c + 3 + (ex3 ? oxp3 : 0);
            const int64_t cy = c + (ey ? oyp : 0), cz = c + (ez ? ozp : 0);
            v4 = a.v[cx];
            w4 = a.w[cx];
            uyp = ld4(a.u + cy); wyp = ld4(a.w + cy);
            vzp = ld4(a.v + cz); uzp = ld4(a.u + cz);
        }
        if (HOIST && (WHAT & 4)) {
            um0 = a.u[c - (hxm ? oxm : 0)];
            vm = ld4(a.v + c - (hym ? oym : 0));
            wm = ld4(a.w + c - (hzm ? ozm : 0));
        }
        if (WHAT & 1) {
            Q4<T> X, Y, Z;
#pragma unroll
            for (int m = 0; m < 4; m++) {
                X.v[m] = u.v[m] * T(a.idx2);
                Y.v[m] = v.v[m] * T(a.idy2);
                Z.v[m] = w.v[m] * T(a.idz2);
            }
            out4(a.Ux + c, X); out4(a.Uy + c, Y); out4(a.Uz + c, Z);
        }
        if (WHAT & 2) {
            if (!HOIST) {
                v4 = ex3 ? a.v[c + 3 + oxp3] : T(0);
                w4 = ex3 ? a.w[c + 3 + oxp3] : T(0);
                if (ey) { uyp = ld4(a.u + c + oyp); wyp = ld4(a.w + c + oyp); }
                if (ez) { vzp = ld4(a.v + c + ozp); uzp = ld4(a.u + c + ozp); }
            }
            Q4<T> OX, OY, OZ;
#pragma unroll
            for (int m = 0; m < 4; m++) {
                const bool ex = m < 3 || ex3;
                const T vxp = m < 3 ? v.v[m + 1] : v4, wxp = m < 3 ? w.v[m + 1] : w4;
                const T uc = u.v[m], vc = v.v[m], wc = w.v[m];
                T oz = T(0);
                if (ex && ey) {
                    oz = vxp - vc - uyp.v[m] + uc;
                    if (a.fpar > 0.0) oz = oz + T(a.fpar);
                }
                T ox = T(0);
                if (ey && ez) ox = wyp.v[m] - wc - vzp.v[m] + vc;
                T oy = T(0);
                if (ez && ex) oy = uzp.v[m] - uc - wxp + wc;
                OX.v[m] = ox; OY.v[m] = oy; OZ.v[m] = oz;
            }
            out4(a.ox + c, OX); out4(a.oy + c, OY); out4(a.oz + c, OZ);
        }
        if (WHAT & 4) {
            if (!HOIST) {
                um0 = hxm ? a.u[c - oxm] : T(0);
                if (hym) vm = ld4(a.v + c - oym);
                if (hzm) wm = ld4(a.w + c - ozm);
            }
            Q4<T> KE;
#pragma unroll
            for (int m = 0; m < 4; m++) {
                const T uc = u.v[m], vc = v.v[m], wc = w.v[m];
                T ke = T(0);
                if (m > 0 || hxm) {
                    const T um = m > 0 ? u.v[m - 1] : um0;
                    const T cff2 = T(0.5 * a.idx2);
                    ke = ke + cff2 * T(0.5) * (uc * uc + um * um);
                }
                if (hym) {
                    const T cff2 = T(0.5 * a.idy2);
                    ke = ke + cff2 * T(0.5) * (vc * vc + vm.v[m] * vm.v[m]);
                }
                if (hzm) {
                    const T cff2 = T(0.5 * a.idz2);
                    ke = ke + cff2 * T(0.5) * (wc * wc + wm.v[m] * wm.v[m]);
                }
                KE.v[m] = ke;
            }
            out4(a.ke + c, KE);
        }
    }
}

template <typename T>
static void launch_diag4(const Geo &g, const DiagArgs<T> &a, int what, hipStream_t s) {
    const dim3 grd = cell_grid4(g), blk(NYL_BX, NYL_BY, 1);
    switch (what & 7) {
    case 1: NYL_LAUNCH((k_diag4<T, 1>), grd, blk, 0, s, g, a); break;
    case 2: NYL_LAUNCH((k_diag4<T, 2>), grd, blk, 0, s, g, a); break;
    case 3: NYL_LAUNCH((k_diag4<T, 3>), grd, blk, 0, s, g, a); break;
    case 4: NYL_LAUNCH((k_diag4<T, 4>), grd, blk, 0, s, g, a); break;
    case 5: NYL_LAUNCH((k_diag4<T, 5>), grd, blk, 0, s, g, a); break;
    case 6: NYL_LAUNCH((k_diag4<T, 6>), grd, blk, 0, s, g, a); break;
    case 7: NYL_LAUNCH((k_diag4<T, 7>), grd, blk, 0, s, g, a); break;
    default: break;
    }
}

// div_cell for cells i0 .. i0+3
template <typename T, typename TO>
__global__ __launch_bounds__(256) void k_div4(Geo g, DivArgs<T, TO> a) {
    const Blk3 bk = CELL_BLOCK();
    const int i0 = (bk.x * NYL_BX + threadIdx.x) * 4;
    const int j = bk.y * NYL_BY + threadIdx.y;
    if (i0 >= g.nx || j >= g.ny) return;
    const int kz = g.nz / (int)gridDim.z;
    const TO cx = TO(a.idx2), cy = TO(a.idy2), cz = TO(a.idz2);
    const bool hxm = g.px || i0 > 0, hym = g.py || j > 0;
    const int64_t oxm = g.px ? (int64_t)(i0 - wrapi(i0 - 1, g.nx)) : 1;
    const int64_t oym = g.py ? (int64_t)(j - wrapi(j - 1, g.ny)) * g.sy : g.sy;
    for (int k = bk.z * kz; k < (bk.z + 1) * kz; k++) {
        const int64_t c = (int64_t)k * g.sz + (int64_t)j * g.sy + i0;
        const bool hzm = g.pz || k > 0;
        const int64_t ozm = g.pz ? (int64_t)(k - wrapi(k - 1, g.nz)) * g.sz : g.sz;
        // every load at once; a neighbour outside a wall axis is read from
        // the own cell and never used
        const Q4<T> u = ld4(a.u + c), v = ld4(a.v + c), w = ld4(a.w + c);
        const T um0 = a.u[c - (hxm ? oxm : 0)];
        const Q4<T> vm = ld4(a.v + c - (hym ? oym : 0)), wm = ld4(a.w + c - (hzm ? ozm : 0));
        Q4<TO> D;
#pragma unroll
        for (int m = 0; m < 4; m++) {
            TO d;
            const TO Uc = TO(u.v[m]) * cx;
            if (m == 0 && !hxm) d = Uc;
            else d = Uc - TO(m > 0 ? u.v[m - 1] : um0) * cx;
            const TO Vc = TO(v.v[m]) * cy;
            if (!hym) d = d + Vc;
            else d = d + (Vc - TO(vm.v[m]) * cy);
            const TO Wc = TO(w.v[m]) * cz;
            if (!hzm) d = d + Wc;
            else d = d + (Wc - TO(wm.v[m]) * cz);
            D.v[m] = d;
        }
        st4(a.out + c, D);
    }
}

// correct_cell for cells i0 .. i0+3 (a cell without the face keeps its value)
template <typename T, typename TX>
__global__ __launch_bounds__(256) void k_correct4(Geo g, CorrectArgs<T, TX> a) {
    const Blk3 bk = CELL_BLOCK();
    const int i0 = (bk.x * NYL_BX + threadIdx.x) * 4;
    const int j = bk.y * NYL_BY + threadIdx.y;
    if (i0 >= g.nx || j >= g.ny) return;
    const int kz = g.nz / (int)gridDim.z;
    const bool ex3 = g.px || i0 + 3 < g.nx - 1;
    const int64_t oxp3 = g.px ? (int64_t)(wrapi(i0 + 4, g.nx) - (i0 + 3)) : 1;
    const bool ey = g.py || j < g.ny - 1;
    const int64_t oyp = g.py ? (int64_t)(wrapi(j + 1, g.ny) - j) * g.sy : g.sy;
    const TX dx2 = TX(a.dx2);
    for (int k = bk.z * kz; k < (bk.z + 1) * kz; k++) {
        const int64_t c = (int64_t)k * g.sz + (int64_t)j * g.sy + i0;
        const bool ez = g.pz || k < g.nz - 1;
        const int64_t ozp = g.pz ? (int64_t)(wrapi(k + 1, g.nz) - k) * g.sz : g.sz;
        const Q4<TX> x = ld4(a.x + c);
        Q4<T> u = ld4(a.u + c), v = ld4(a.v + c), w = ld4(a.w + c);
        const TX x4 = ex3 ? a.x[c + 3 + oxp3] : TX(0);
        Q4<TX> xy{}, xz{};
        if (ey) xy = ld4(a.x + c + oyp);
        if (ez) xz = ld4(a.x + c + ozp);
#pragma unroll
        for (int m = 0; m < 4; m++) {
            const TX pc = x.v[m] * dx2;
            if (m < 3 || ex3) u.v[m] = T(TX(u.v[m]) - ((m < 3 ? x.v[m + 1] : x4) * dx2 - pc));
            if (ey) v.v[m] = T(TX(v.v[m]) - (xy.v[m] * dx2 - pc));
            if (ez) w.v[m] = T(TX(w.v[m]) - (xz.v[m] * dx2 - pc));
        }
        st4(a.u + c, u); st4(a.v + c, v); st4(a.w + c, w);
    }
}

// U_from_u (core/cov_to_contra.py:15-20), vorticity (core/vorticity.py:25-34,
// core/fortran_vorticity.f90:2-28) and kinenergy (core/kinenergy.py:13-24,
// core/fortran_kinenergy.f90:47-55) from the covariant velocity.
template <typename T>
__device__ __forceinline__ void diag_cell(const Geo &g, const DiagArgs<T> &a, int what, int i,
                                          int j, int k) {
    const int64_t c = (int64_t)k * g.sz + (int64_t)j * g.sy + i;
    const T uc = a.u[c], vc = a.v[c], wc = a.w[c];
    if (what & 1) {
        a.Ux[c] = uc * T(a.idx2);
        a.Uy[c] = vc * T(a.idy2);
        a.Uz[c] = wc * T(a.idz2);
    }
    const int64_t oxp = g.px ? (int64_t)(wrapi(i + 1, g.nx) - i) : 1;
    const int64_t oyp = g.py ? (int64_t)(wrapi(j + 1, g.ny) - j) * g.sy : g.sy;
    const int64_t ozp = g.pz ? (int64_t)(wrapi(k + 1, g.nz) - k) * g.sz : g.sz;
    const bool ex = g.px || i < g.nx - 1, ey = g.py || j < g.ny - 1, ez = g.pz || k < g.nz - 1;
    if (what & 2) {
        // vor_k = delta_i u_j - delta_j u_i (flipview('k'): ui=u, uj=v)
        T oz = T(0);
        if (ex && ey) {
            oz = a.v[c + oxp] - vc - a.u[c + oyp] + uc;
            if (a.fpar > 0.0) oz = oz + T(a.fpar);
        }
        // vor_i (flipview('i') = [x][z][y]: ui=v, uj=w)
        T ox = T(0);
        if (ey && ez) ox = a.w[c + oyp] - wc - a.v[c + ozp] + vc;
        // vor_j (flipview('j') = [y][x][z]: ui=w, uj=u)
        T oy = T(0);
        if (ez && ex) oy = a.u[c + ozp] - uc - a.w[c + oxp] + wc;
        a.ox[c] = ox; a.oy[c] = oy; a.oz[c] = oz;
    }
    if (what & 4) {
        // ke = 0; ke(i) += (cff2*0.5)*(u(i)**2+u(i-1)**2) for i >= 2, per direction
        T ke = T(0);
        if (g.px || i > 0) {
            const T um = a.u[c - (g.px ? (int64_t)(i - wrapi(i - 1, g.nx)) : 1)];
            const T cff2 = T(0.5 * a.idx2);
            ke = ke + cff2 * T(0.5) * (uc * uc + um * um);
        }
        if (g.py || j > 0) {
            const T vm = a.v[c - (g.py ? (int64_t)(j - wrapi(j - 1, g.ny)) * g.sy : g.sy)];
            const T cff2 = T(0.5 * a.idy2);
            ke = ke + cff2 * T(0.5) * (vc * vc + vm * vm);
        }
        if (g.pz || k > 0) {
            const T wm = a.w[c - (g.pz ? (int64_t)(k - wrapi(k - 1, g.nz)) * g.sz : g.sz)];
            const T cff2 = T(0.5 * a.idz2);
            ke = ke + cff2 * T(0.5) * (wc * wc + wm * wm);
        }
        a.ke[c] = ke;
    }
}

template <typename T>
__global__ __launch_bounds__(256) void k_diag(Geo g, DiagArgs<T> a, int what) {
    const Blk3 bk = CELL_BLOCK();
    const int i = bk.x * NYL_BX + threadIdx.x;
    const int j = bk.y * NYL_BY + threadIdx.y;
    if (i >= g.nx || j >= g.ny) return;
    const int kz = g.nz / (int)gridDim.z;
    for (int k = bk.z * kz; k < (bk.z + 1) * kz; k++) diag_cell<T>(g, a, what, i, j, k);
}

template <typename T>
hipError_t launch_diag(const Geo &g, const DiagArgs<T> &a, int what, hipStream_t s) {
    if (quad_ok(g, {a.u, a.v, a.w, a.Ux, a.Uy, a.Uz, a.ox, a.oy, a.oz, a.ke}))
        launch_diag4<T>(g, a, what, s);
    else
        NYL_LAUNCH((k_diag<T>), cell_grid_kz(g), dim3(NYL_BX, NYL_BY, 1), 0, s, g, a, what);
    return hipGetLastError();
}

// compute_div (core/projection.py:15-35 over core/fortran_bernoulli.f90:61-97)
// with U = u*idx2 evaluated in place (core/cov_to_contra.py:18-20).
template <typename T, typename TO>
__device__ __forceinline__ void div_cell(const Geo &g, const DivArgs<T, TO> &a, int i, int j,
                                         int k) {
    const int64_t c = (int64_t)k * g.sz + (int64_t)j * g.sy + i;
    // evaluated in the output precision (FP64 right-hand side of the mixed path)
    const TO cx = TO(a.idx2), cy = TO(a.idy2), cz = TO(a.idz2);
    TO d;
    const TO Uc = TO(a.u[c]) * cx;
    if (!g.px && i == 0) d = Uc;
    else d = Uc - TO(a.u[c - (g.px ? (int64_t)(i - wrapi(i - 1, g.nx)) : 1)]) * cx;
    const TO Vc = TO(a.v[c]) * cy;
    if (!g.py && j == 0) d = d + Vc;
    else d = d + (Vc - TO(a.v[c - (g.py ? (int64_t)(j - wrapi(j - 1, g.ny)) * g.sy : g.sy)]) * cy);
    const TO Wc = TO(a.w[c]) * cz;
    if (!g.pz && k == 0) d = d + Wc;
    else d = d + (Wc - TO(a.w[c - (g.pz ? (int64_t)(k - wrapi(k - 1, g.nz)) * g.sz : g.sz)]) * cz);
    a.out[c] = d;
}

template <typename T, typename TO>
__global__ __launch_bounds__(256) void k_div(Geo g, DivArgs<T, TO> a) {
    const Blk3 bk = CELL_BLOCK();
    const int i = bk.x * NYL_BX + threadIdx.x;
    const int j = bk.y * NYL_BY + threadIdx.y;
    if (i >= g.nx || j >= g.ny) return;
    const int kz = g.nz / (int)gridDim.z;
    for (int k = bk.z * kz; k < (bk.z + 1) * kz; k++) div_cell<T, TO>(g, a, i, j, k);
}

template <typename T, typename TO>
hipError_t launch_div(const Geo &g, const T *u, const T *v, const T *w, double idx2,
                      double idy2, double idz2, TO *out, hipStream_t s) {
    DivArgs<T, TO> a;
    a.u = u; a.v = v; a.w = w; a.idx2 = idx2; a.idy2 = idy2; a.idz2 = idz2; a.out = out;
    if (quad_ok(g, {u, v, w, out}))
        NYL_LAUNCH((k_div4<T, TO>), cell_grid4(g), dim3(NYL_BX, NYL_BY, 1), 0, s, g, a);
    else
        NYL_LAUNCH((k_div<T, TO>), cell_grid_kz(g), dim3(NYL_BX, NYL_BY, 1), 0, s, g, a);
    return hipGetLastError();
}

// u -= delta[p] with p = x*dx**2 (core/projection.py:84-87 over
// core/fortran_bernoulli.f90:2-26; p from core/mgfordriver.py:78)
template <typename T, typename TX>
__device__ __forceinline__ void correct_cell(const Geo &g, const CorrectArgs<T, TX> &a, int i,
                                             int j, int k) {
    const int64_t c = (int64_t)k * g.sz + (int64_t)j * g.sy + i;
    const TX *x = a.x;
    const TX pc = x[c] * TX(a.dx2);
    if (g.px || i < g.nx - 1) {
        const int64_t o = g.px ? (int64_t)(wrapi(i + 1, g.nx) - i) : 1;
        a.u[c] = T(TX(a.u[c]) - (x[c + o] * TX(a.dx2) - pc));
    }
    if (g.py || j < g.ny - 1) {
        const int64_t o = g.py ? (int64_t)(wrapi(j + 1, g.ny) - j) * g.sy : g.sy;
        a.v[c] = T(TX(a.v[c]) - (x[c + o] * TX(a.dx2) - pc));
    }
    if (g.pz || k < g.nz - 1) {
        const int64_t o = g.pz ? (int64_t)(wrapi(k + 1, g.nz) - k) * g.sz : g.sz;
        a.w[c] = T(TX(a.w[c]) - (x[c + o] * TX(a.dx2) - pc));
    }
}

template <typename T, typename TX>
__global__ __launch_bounds__(256) void k_correct(Geo g, CorrectArgs<T, TX> a) {
    const Blk3 bk = CELL_BLOCK();
    const int i = bk.x * NYL_BX + threadIdx.x;
    const int j = bk.y * NYL_BY + threadIdx.y;
    if (i >= g.nx || j >= g.ny) return;
    const int kz = g.nz / (int)gridDim.z;
    for (int k = bk.z * kz; k < (bk.z + 1) * kz; k++) correct_cell<T, TX>(g, a, i, j, k);
}

template <typename T, typename TX>
hipError_t launch_correct(const Geo &g, T *u, T *v, T *w, const TX *x, double dx2,
                          hipStream_t s) {
    CorrectArgs<T, TX> a;
    a.u = u; a.v = v; a.w = w; a.x = x; a.dx2 = dx2;
    if (quad_ok(g, {u, v, w, x}))
        NYL_LAUNCH((k_correct4<T, TX>), cell_grid4(g), dim3(NYL_BX, NYL_BY, 1), 0, s, g, a);
    else
        NYL_LAUNCH((k_correct<T, TX>), cell_grid_kz(g), dim3(NYL_BX, NYL_BY, 1), 0, s, g, a);
    return hipGetLastError();
}

template <typename TX, typename T>
__global__ void k_pressure(int64_t n, const TX *__restrict__ x, double dx2, T *__restrict__ p) {
    const int64_t q = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (q < n) p[q] = T(x[q] * TX(dx2));
}

template <typename TX, typename T>
hipError_t launch_pressure(const Geo &g, const TX *x, double dx2, T *p, hipStream_t s) {
    const int64_t n = (int64_t)g.nx * g.ny * g.nz;
    NYL_LAUNCH((k_pressure<TX, T>), dim3((unsigned)((n + 255) / 256)), dim3(256), 0, s,
                       n, x, dx2, p);
    return hipGetLastError();
}

__global__ void k_fill(double *p, int64_t n, double v) {
    const int64_t q = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (q < n) p[q] = v;
}

template <typename T>
__global__ void k_zero(T *p, int64_t n) {
    const int64_t q = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (q < n) p[q] = T(0);
}

template <typename T>
hipError_t launch_zero(T *p, int64_t n, hipStream_t s) {
    if (n <= 0) return hipSuccess;
    NYL_LAUNCH((k_zero<T>), dim3((unsigned)((n + 255) / 256)), dim3(256), 0, s, p, n);
    return hipGetLastError();
}
template hipError_t launch_zero<float>(float *, int64_t, hipStream_t);
template hipError_t launch_zero<double>(double *, int64_t, hipStream_t);

hipError_t launch_fill(double *p, int64_t n, double v, hipStream_t s) {
    if (n <= 0) return hipSuccess;
    NYL_LAUNCH(k_fill, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, s, p, n, v);
    return hipGetLastError();
}

// ---------------------------------------------------------------------------
// Ensemble batches: one launch covers every member (BHead), each block a
// tile of TPB cells of one member (rows of consecutive cells, or a brick:
// StageTile), running the single-member cell functions.  The stage kernel
// is persistent: a fixed grid strides over all tiles; its RK coefficient is
// the host's dt, dt/4., dt/12. of the member's dt (same IEEE operations).

// the autotuner's candidates: rows, then bricks from flat to cubic
const StageTile kStageTiles[NYL_N_TILES] = {
    {128, -1, 0}, {128, 5, 2}, {128, 4, 2}, {128, 3, 2},
    {256, -1, 0}, {256, 6, 2}, {256, 5, 2}, {256, 4, 2}, {256, 3, 3},
    {512, -1, 0}, {512, 6, 3}, {512, 5, 3}, {512, 5, 2}, {512, 4, 3}, {512, 3, 3}};

int64_t stage_tiles(const Geo &g, const StageTile &t) {
    if (t.lx < 0) return ((int64_t)g.nx * g.ny * g.nz + t.tpb - 1) / t.tpb;
    const int tz = t.tpb >> (t.lx + t.ly);
    return (int64_t)((g.nx + (1 << t.lx) - 1) >> t.lx) * ((g.ny + (1 << t.ly) - 1) >> t.ly)
         * ((g.nz + tz - 1) / tz);
}

// cell (i, j, k) of thread th in tile `tile` of a member; false for a thread
// past the member's edge
template <int TPB>
__device__ __forceinline__ bool tile_cell(const Geo &g, int64_t tile, int th, int lx, int ly,
                                          int &i, int &j, int &k) {
    if (lx < 0) return cell_of(g, tile * TPB + th, i, j, k);
    const uint32_t bx = (uint32_t)(g.nx + (1 << lx) - 1) >> lx;
    const uint32_t by = (uint32_t)(g.ny + (1 << ly) - 1) >> ly;
    const uint32_t t = (uint32_t)tile, r = t / bx, c = r / by;
    i = (int)(((t - r * bx) << lx) + (th & ((1 << lx) - 1)));
    j = (int)(((r - c * by) << ly) + ((th >> lx) & ((1 << ly) - 1)));
    k = (int)(c * (uint32_t)(TPB >> (lx + ly)) + (th >> (lx + ly)));
    return i < g.nx && j < g.ny && k < g.nz;
}

template <typename T, int MODE, int PX, int PY, int PZ, int TPB>
__global__ __launch_bounds__(TPB) void k_b_stage(const StageItem<T> *__restrict__ items, int n,
                                                 int64_t nblk, const double *__restrict__ dt,
                                                 int lx, int ly) {
    for (int64_t blk = blockIdx.x; blk < nblk; blk += gridDim.x) {
        const StageItem<T> &it = find_item(items, n, blk);
        int i, j, k;
        if (!tile_cell<TPB>(it.h.g, blk - it.h.start, threadIdx.x, lx, ly, i, j, k)) continue;
        StageArgs<T> a = it.a;
        const double d = dt[it.h.member];
        a.c = MODE == 1 ? d : (MODE == 2 ? d / 4. : d / 12.);
        stage_cells<T, 1, MODE, PX, PY, PZ, false, int32_t, int32_t>(it.h.g, a, i, j, k);
    }
}

int batch_blocks(int64_t ncell) { return (int)((ncell + NYL_BATCH_TPB - 1) / NYL_BATCH_TPB); }

template <typename T, int PX, int PY, int PZ, int TPB>
static void b_stage_p(const StageItem<T> *items, int n, int64_t nblk, int mode, const double *dt,
                      int lx, int ly, hipStream_t s) {
    const unsigned grid = (unsigned)(nblk < 2048 ? nblk : 2048);
    switch (mode) {
    case 1: NYL_LAUNCH((k_b_stage<T, 1, PX, PY, PZ, TPB>), grid, TPB, 0, s, items, n, nblk, dt, lx, ly); break;
    case 2: NYL_LAUNCH((k_b_stage<T, 2, PX, PY, PZ, TPB>), grid, TPB, 0, s, items, n, nblk, dt, lx, ly); break;
    default: NYL_LAUNCH((k_b_stage<T, 3, PX, PY, PZ, TPB>), grid, TPB, 0, s, items, n, nblk, dt, lx, ly); break;
    }
}

template <typename T, int TPB>
static void b_stage_t(const StageItem<T> *items, int n, int64_t nblk, int mode, int perio,
                      const double *dt, int lx, int ly, hipStream_t s) {
    switch (perio) {
    case 0: b_stage_p<T, 0, 0, 0, TPB>(items, n, nblk, mode, dt, lx, ly, s); break;
    case 1: b_stage_p<T, 1, 0, 0, TPB>(items, n, nblk, mode, dt, lx, ly, s); break;
    case 2: b_stage_p<T, 0, 1, 0, TPB>(items, n, nblk, mode, dt, lx, ly, s); break;
    case 3: b_stage_p<T, 1, 1, 0, TPB>(items, n, nblk, mode, dt, lx, ly, s); break;
    case 4: b_stage_p<T, 0, 0, 1, TPB>(items, n, nblk, mode, dt, lx, ly, s); break;
    case 5: b_stage_p<T, 1, 0, 1, TPB>(items, n, nblk, mode, dt, lx, ly, s); break;
    case 6: b_stage_p<T, 0, 1, 1, TPB>(items, n, nblk, mode, dt, lx, ly, s); break;
    default: b_stage_p<T, 1, 1, 1, TPB>(items, n, nblk, mode, dt, lx, ly, s); break;
    }
}

template <typename T>
hipError_t launch_b_stage(const StageItem<T> *items, int n, int64_t nblk, int mode, int perio,
                          const StageTile &tile, const double *dt, hipStream_t s) {
    if (mode < 1 || mode > 3 || nblk <= 0) return hipErrorInvalidValue;
    if (tile.lx >= 0 && (tile.ly < 0 || tile.lx + tile.ly > 9 || (tile.tpb >> (tile.lx + tile.ly)) < 1))
        return hipErrorInvalidValue;
    switch (tile.tpb) {
    case 128: b_stage_t<T, 128>(items, n, nblk, mode, perio, dt, tile.lx, tile.ly, s); break;
    case 256: b_stage_t<T, 256>(items, n, nblk, mode, perio, dt, tile.lx, tile.ly, s); break;
    case 512: b_stage_t<T, 512>(items, n, nblk, mode, perio, dt, tile.lx, tile.ly, s); break;
    default: return hipErrorInvalidValue;
    }
    return hipGetLastError();
}

template <typename T>
__global__ __launch_bounds__(NYL_BATCH_TPB) void k_b_div(const DivItem<T> *__restrict__ items,
                                                         int n) {
    const DivItem<T> &it = find_item(items, n, blockIdx.x);
    int i, j, k;
    if (!cell_of(it.h.g, ((int64_t)blockIdx.x - it.h.start) * NYL_BATCH_TPB + threadIdx.x, i, j, k))
        return;
    div_cell<T, double>(it.h.g, it.a, i, j, k);
}

template <typename T>
hipError_t launch_b_div(const DivItem<T> *items, int n, int64_t nblk, hipStream_t s) {
    NYL_LAUNCH((k_b_div<T>), dim3((unsigned)nblk), NYL_BATCH_TPB, 0, s, items, n);
    return hipGetLastError();
}

template <typename T>
__global__ __launch_bounds__(NYL_BATCH_TPB) void k_b_correct(const CorrItem<T> *__restrict__ items,
                                                             int n) {
    const CorrItem<T> &it = find_item(items, n, blockIdx.x);
    int i, j, k;
    if (!cell_of(it.h.g, ((int64_t)blockIdx.x - it.h.start) * NYL_BATCH_TPB + threadIdx.x, i, j, k))
        return;
    correct_cell<T, double>(it.h.g, it.a, i, j, k);
}

template <typename T>
hipError_t launch_b_correct(const CorrItem<T> *items, int n, int64_t nblk, hipStream_t s) {
    NYL_LAUNCH((k_b_correct<T>), dim3((unsigned)nblk), NYL_BATCH_TPB, 0, s, items, n);
    return hipGetLastError();
}

template <typename T>
__global__ __launch_bounds__(NYL_BATCH_TPB) void k_b_diag(const DiagItem<T> *__restrict__ items,
                                                          int n, int what) {
    const DiagItem<T> &it = find_item(items, n, blockIdx.x);
    int i, j, k;
    if (!cell_of(it.h.g, ((int64_t)blockIdx.x - it.h.start) * NYL_BATCH_TPB + threadIdx.x, i, j, k))
        return;
    diag_cell<T>(it.h.g, it.a, what, i, j, k);
}

template <typename T>
hipError_t launch_b_diag(const DiagItem<T> *items, int n, int64_t nblk, int what, hipStream_t s) {
    NYL_LAUNCH((k_b_diag<T>), dim3((unsigned)nblk), NYL_BATCH_TPB, 0, s, items, n, what);
    return hipGetLastError();
}

#define NYL_B_STENCIL_INST(T)                                                                    \
    template hipError_t launch_b_stage<T>(const StageItem<T> *, int, int64_t, int, int,         \
                                          const StageTile &, const double *, hipStream_t);      \
    template hipError_t launch_b_div<T>(const DivItem<T> *, int, int64_t, hipStream_t);         \
    template hipError_t launch_b_correct<T>(const CorrItem<T> *, int, int64_t, hipStream_t);    \
    template hipError_t launch_b_diag<T>(const DiagItem<T> *, int, int64_t, int, hipStream_t);
NYL_B_STENCIL_INST(double)
NYL_B_STENCIL_INST(float)
#undef NYL_B_STENCIL_INST

template hipError_t launch_update<double>(int64_t, const UpdateArgs<double> &, int, hipStream_t);
template hipError_t launch_update<float>(int64_t, const UpdateArgs<float> &, int, hipStream_t);
template hipError_t launch_diag<double>(const Geo &, const DiagArgs<double> &, int, hipStream_t);
template hipError_t launch_diag<float>(const Geo &, const DiagArgs<float> &, int, hipStream_t);
template hipError_t launch_div<double, double>(const Geo &, const double *, const double *,
                                               const double *, double, double, double, double *,
                                               hipStream_t);
template hipError_t launch_div<float, double>(const Geo &, const float *, const float *,
                                              const float *, double, double, double, double *,
                                              hipStream_t);
template hipError_t launch_correct<double, double>(const Geo &, double *, double *, double *,
                                                   const double *, double, hipStream_t);
template hipError_t launch_correct<float, double>(const Geo &, float *, float *, float *,
                                                  const double *, double, hipStream_t);
template hipError_t launch_pressure<double, double>(const Geo &, const double *, double,
                                                    double *, hipStream_t);

}  // namespace nyl
