// nyl_cycle.hip -- the small levels of a V-cycle in one workgroup, and the
// stop rule of a multigrid solve on the device.
#include "nyl_cycle.h"

namespace nyl {

// ---------------------------------------------------------------------------
// Sum of the partials in launch_final_sum's order (RED_T strided sums, then
// the tree), by the first RED_T threads of a block; the loads of eight
// strides are issued together.  Every thread of the block calls it.
__device__ __forceinline__ double fixed_sum(const double *__restrict__ part, int np, double *sh,
                                            int tid) {
    double acc = 0.0;
    if (tid < RED_T) {
        int q = tid;
        for (; q + 7 * RED_T < np; q += 8 * RED_T) {
            double v[8];
#pragma unroll
            for (int r = 0; r < 8; r++) v[r] = part[q + r * RED_T];
#pragma unroll
            for (int r = 0; r < 8; r++) acc = acc + v[r];
        }
        for (; q < np; q += RED_T) acc = acc + part[q];
        sh[tid] = acc;
    }
    __syncthreads();
    for (int s = RED_T / 2; s > 0; s >>= 1) {
        if (tid < s) sh[tid] = sh[tid] + sh[tid + s];
        __syncthreads();
    }
    const double t = sh[0];
    __syncthreads();
    return t;
}

__device__ __forceinline__ void ctl_body(const CtlArgs &c, double *sh, int tid) {
    double s0 = 0.0, s1 = 0.0;
    if (c.kind != CTL_NONE) s0 = fixed_sum(c.partials, c.np, sh, tid);
    if (c.kind == CTL_SHIFT) s1 = fixed_sum(c.partials + c.np, c.np, sh, tid);
    if (tid != 0) return;
    MGCtl &m = *c.ctl;
    if (c.slot >= 0) m.hist[c.slot] = s0;
    if (c.kind == CTL_NORMB) {
        m.normb = s0;
        m.stop = 0;
    } else if (c.kind == CTL_SHIFT) {
        const double shift = s0 / c.ncell;
        const double nb = s1 - c.ncell * shift * shift;
        m.shift = shift;
        m.normb = nb < 0.0 ? 0.0 : nb;
    } else if (c.kind != CTL_NONE) {
        const double res = m.normb > 0.0 ? s0 / m.normb : 0.0;
        if (c.kind == CTL_TEST) {
            if (res < c.tol) m.stop = 1;
        } else if (c.kind == CTL_OUTER) {
            const bool rel = res * c.inner_red > c.tol;
            m.res = res;
            m.rel = rel;
            m.target = rel ? res * c.inner_red : c.tol;
            m.outer_stop = res < c.tol;
            m.stop = m.outer_stop;
            m.no_add = 1;
        } else if (!m.stop) {
            if (res < m.target || (m.rel && c.k >= c.inner_max)) {
                m.stop = 1;
                m.no_add = 0;
            }
        }
    }
    if (c.dst) {
        c.dst[0] = m.normb;
        c.dst[1] = m.shift;
        for (int q = 0; q < c.nhist; q++) c.dst[2 + q] = m.hist[q];
        __threadfence_system();
        __hip_atomic_store(c.flag, c.seq, __ATOMIC_RELEASE, __HIP_MEMORY_SCOPE_SYSTEM);
    }
}

__global__ __launch_bounds__(RED_T) void k_mg_ctl(CtlArgs c) {
    __shared__ double sh[RED_T];
    ctl_body(c, sh, threadIdx.x);
}

hipError_t launch_ctl(const CtlArgs &c, hipStream_t s) {
    NYL_LAUNCH(k_mg_ctl, dim3(1), dim3(RED_T), 0, s, c);
    return hipGetLastError();
}

// ---------------------------------------------------------------------------
// The levels of a V-cycle that together fit one workgroup's LDS: their down
// legs (second sweep, residual, restriction with the coarse level's first
// sweep), the coarsest level (its second sweep, or the direct solve of a
// level with an odd size) and their up legs (prolongation, two sweeps), one
// barrier per phase.  At these sizes a launch costs more than a level's work
// (3 to 6 us each, two launches and more per level).  Each value has the
// per-cell kernels' expression and order in the level's type, so the result
// is bitwise that of the separate launches.
// One workgroup issues 64 lanes of a SIMD every four clocks, so the work per
// cell is what bounds a large first level: the places of a cell's neighbours
// and of the coarse cells it reads are sums of three table entries (one per
// axis; the zeros beyond a wall are part of the arrays, so nothing is
// selected), evaluated once per leg and kept in registers, those of the
// first level for both of its legs.  In FP64 with four cells per thread (16^3)
// that takes all 128 registers and 15 spills (64 bytes of scratch per lane),
// FP32 115 and none: 26.6 against 13.9 us per V-cycle at 256^3, whose cycle
// starts at 16^3.
__device__ __forceinline__ uint32_t div_by(uint32_t q, uint32_t m) {
    return m ? __umulhi(q, m) : q;
}

// the same value in every lane, as a scalar
__device__ __forceinline__ int uniform(uint32_t v) { return __builtin_amdgcn_readfirstlane((int)v); }

// a level as the phases see it
template <typename T>
struct CycleView {
    int n;
    uint32_t nx, nxy, mx, mxy;
    T *A, *C, *b;
    const CycleEnt *ex, *ey, *ez;
};

// the coefficient tables in a level's type
template <typename T>
struct CycleTab {
    const T *idiag, *pcoef;
};

// the cells of a thread on a level: own place, the neighbours', the shares
// of the coarse places, neighbour count, index.  Lanes past the last cell
// hold cell 0 and store nothing, so the cells of a thread overlap.
template <typename T, int R>
struct CycleCells {
    int own[R], xm[R], xp[R], ym[R], yp[R], zm[R], zp[R], q[R], nw[R], in[R];
    uint32_t cx[R], cy[R], cz[R];
    T id[R];
    bool live[R];
};

template <typename T, int R>
__device__ __forceinline__ void cycle_cells(CycleCells<T, R> &s, const CycleView<T> &v,
                                            const CycleTab<T> &tb, int tid) {
#pragma unroll
    for (int r = 0; r < R; r++) {
        const int t0 = tid + r * CYC_T;
        s.live[r] = t0 < v.n;
        const uint32_t q = s.live[r] ? t0 : 0;
        const uint32_t k = div_by(q, v.mxy), t = q - k * v.nxy;
        const uint32_t j = div_by(t, v.mx), i = t - j * v.nx;
        const CycleEnt x = v.ex[i], y = v.ey[j], z = v.ez[k];
        const int xo = x.w[0] & 0xffff, yo = y.w[0] & 0xffff, zo = z.w[0] & 0xffff;
        s.q[r] = q;
        s.own[r] = xo + yo + zo;
        s.xm[r] = (int)(x.w[0] >> 16) + yo + zo;
        s.xp[r] = (int)(x.w[1] & 0xffff) + yo + zo;
        s.ym[r] = (int)(y.w[0] >> 16) + xo + zo;
        s.yp[r] = (int)(y.w[1] & 0xffff) + xo + zo;
        s.zm[r] = (int)(z.w[0] >> 16) + xo + yo;
        s.zp[r] = (int)(z.w[1] & 0xffff) + xo + yo;
        // neighbour count in the low bits, the prolongation's inside flags above
        const uint32_t f = (x.w[1] >> 16) + (y.w[1] >> 16) + (z.w[1] >> 16);
        s.nw[r] = f & 15;
        s.in[r] = f >> 4;
        s.cx[r] = x.w[2];
        s.cy[r] = y.w[2];
        s.cz[r] = z.w[2];
        s.id[r] = tb.idiag[s.nw[r]];
    }
}

template <typename T, int R>
__device__ __forceinline__ T cycle_sum6(const CycleCells<T, R> &s, const T *a, int r) {
    return a[s.xm[r]] + a[s.xp[r]] + a[s.ym[r]] + a[s.yp[r]] + a[s.zm[r]] + a[s.zp[r]];
}

// one sweep src -> dst, or to memory (out)
template <typename T, int R>
__device__ __forceinline__ void cycle_sweep(const CycleCells<T, R> &s, const T *src, T *dst,
                                            const T *b, T om, T cff1, T *out) {
    T w[R];
#pragma unroll
    for (int r = 0; r < R; r++)
        w[r] = cff1 * src[s.own[r]] + om * (cycle_sum6(s, src, r) - b[s.q[r]]) * s.id[r];
#pragma unroll
    for (int r = 0; r < R; r++)
        if (s.live[r]) {
            if (out) out[s.q[r]] = w[r];
            else dst[s.own[r]] = w[r];
        }
    __syncthreads();
}

// residual of C into A, summed over the eight children of each coarse cell:
// the coarse right-hand side and its first sweep from zero
template <typename T, typename TC, int R>
__device__ __forceinline__ void cycle_restrict(const CycleCells<T, R> &s, const CycleView<T> &v,
                                               const CycleView<TC> &c, const CycleTab<TC> &tc,
                                               double omega, int tid) {
    T w[R];
#pragma unroll
    for (int r = 0; r < R; r++)
        w[r] = v.b[s.q[r]] + T(s.nw[r]) * v.C[s.own[r]] - cycle_sum6(s, v.C, r);
#pragma unroll
    for (int r = 0; r < R; r++)
        if (s.live[r]) v.A[s.own[r]] = w[r];
    __syncthreads();
    if (tid < c.n) {
        const uint32_t k = div_by(tid, c.mxy), t = tid - k * c.nxy;
        const uint32_t j = div_by(t, c.mx), i = t - j * c.nx;
        // the children: position 2i and its plus neighbour, per axis
        const CycleEnt x = v.ex[2 * i], y = v.ey[2 * j], z = v.ez[2 * k];
        const int x0 = x.w[0] & 0xffff, x1 = x.w[1] & 0xffff;
        const int y0 = y.w[0] & 0xffff, y1 = y.w[1] & 0xffff;
        const int z0 = z.w[0] & 0xffff, z1 = z.w[1] & 0xffff;
        const T *f = v.A;
        const TC bv = TC(T(0.5) * (f[x0 + y0 + z0] + f[x1 + y0 + z0] + f[x0 + y1 + z0] +
                                   f[x1 + y1 + z0] + f[x0 + y0 + z1] + f[x1 + y0 + z1] +
                                   f[x0 + y1 + z1] + f[x1 + y1 + z1]));
        const CycleEnt cx = c.ex[i], cy = c.ey[j], cz = c.ez[k];
        const int nw = ((cx.w[1] >> 16) + (cy.w[1] >> 16) + (cz.w[1] >> 16)) & 15;
        const int own = (cx.w[0] & 0xffff) + (cy.w[0] & 0xffff) + (cz.w[0] & 0xffff);
        c.b[tid] = bv;
        c.A[own] = TC(1.0 - omega) * TC(0) + TC(omega) * (TC(0) - bv) * tc.idiag[nw];
    }
    __syncthreads();
}

// A = C + P(X), X the coarse level's correction
template <typename T, typename TC, int R>
__device__ __forceinline__ void cycle_prolong(const CycleCells<T, R> &s, const CycleView<T> &v,
                                              const TC *X, const CycleTab<T> &tb) {
    T w[R];
#pragma unroll
    for (int r = 0; r < R; r++) {
        const int x0 = s.cx[r] & 0xffff, x1 = s.cx[r] >> 16;
        const int y0 = s.cy[r] & 0xffff, y1 = s.cy[r] >> 16;
        const int z0 = s.cz[r] & 0xffff, z1 = s.cz[r] >> 16;
        auto A = [&](int z) -> T {
            return T(9) * T(X[x0 + y0 + z]) + T(3) * T(X[x1 + y0 + z]) +
                   T(3) * T(X[x0 + y1 + z]) + T(X[x1 + y1 + z]);
        };
        const T bmid = A(z0), aside = A(z1);
        w[r] = v.C[s.own[r]] + tb.pcoef[s.in[r]] * (T(3) * bmid + aside);
    }
#pragma unroll
    for (int r = 0; r < R; r++)
        if (s.live[r]) v.A[s.own[r]] = w[r];
    __syncthreads();
}

// the direct solve of the coarsest level, b -> C: the six transforms of
// nyl_coarse.hip in its order (x y z, scaling, z y x); b and A (dense) are
// the scratch
__device__ __forceinline__ void cycle_direct(const CycleArgs &a, const CycleView<double> &v,
                                             int ny, int nz, const double *E0, int tid) {
    const int nx = v.nx, nxy = v.nxy;
    const double *mux = a.etab + CS_MAXX * CS_MAXX + 2 * CS_MAX * CS_MAX;
    const double *muy = mux + CS_MAXX, *muz = muy + CS_MAX;
    for (int s = 0; s < 6; s++) {
        const int ax = s < 3 ? s : 5 - s;
        const double *E = E0 + (ax == 0 ? 0 : (ax == 1 ? nx * nx : nx * nx + ny * ny));
        const int m = ax == 0 ? nx : (ax == 1 ? ny : nz);
        const int st = ax == 0 ? 1 : (ax == 1 ? nx : nxy);
        const double *src = (s & 1) ? v.A : v.b;
        double *dst = (s & 1) ? v.b : v.A;
        const int er = s < 3 ? m : 1, ec = s < 3 ? 1 : m;   // E or its transpose
        for (int q = tid; q < v.n; q += CYC_T) {
            const int k = (int)div_by(q, v.mxy), t = q - k * nxy;
            const int j = (int)div_by(t, v.mx), i = t - j * nx;
            const int p = ax == 0 ? i : (ax == 1 ? j : k);
            const double *line = src + (q - p * st), *row = E + p * er;
            double acc = 0.0;
#pragma unroll 4
            for (int w = 0; w < m; w++) acc = fma(row[w * ec], line[w * st], acc);
            if (s == 2) {
                const double mu = mux[i] + muy[j] + muz[k];
                acc = mu > 0.0 ? -acc / mu : 0.0;
            }
            if (s == 5)
                v.C[(v.ex[i].w[0] & 0xffff) + (v.ey[j].w[0] & 0xffff) + (v.ez[k].w[0] & 0xffff)] =
                    acc;
            else dst[q] = acc;
        }
        __syncthreads();
    }
}

// T: the type of the levels above the coarsest, R: cells of the first level
// per thread
template <typename T, int R>
__device__ __forceinline__ void cycle_body(const CycleArgs &a, const T *__restrict__ gb,
                                           T *__restrict__ gy, T *__restrict__ gx, char *lds,
                                           uint32_t *slev, CycleEnt *ent, double *tb, int tid) {
    const int nl = a.nl, n0 = a.n0;
    // the level and position tables, the coefficients and the fields of the
    // first level in one round of loads; the levels' arrays start at zero
    constexpr int LW = sizeof(CycleLevel) / 4;
    if (tid < CYC_MAXLEV * LW) slev[tid] = reinterpret_cast<const uint32_t *>(a.lev)[tid];
    if (tid < a.nent) ent[tid] = a.ent[tid];
    double *id64 = tb, *pc64 = tb + 8;
    T *idt = reinterpret_cast<T *>(tb + 16), *pct = idt + 8;
    if (tid < 7) { id64[tid] = a.tab.idiag[tid]; idt[tid] = T(a.tab.idiag[tid]); }
    if (tid < 8) { pc64[tid] = a.tab.pcoef[tid]; pct[tid] = T(a.tab.pcoef[tid]); }
    T vb[R], vy[R];
#pragma unroll
    for (int r = 0; r < R; r++) {
        const int q = tid + r * CYC_T;
        vb[r] = q < n0 ? gb[q] : T(0);
        vy[r] = q < n0 ? gy[q] : T(0);
    }
    for (uint32_t q = tid; q < a.bytes / 8; q += CYC_T) reinterpret_cast<double *>(lds)[q] = 0.0;
    __syncthreads();
    auto view = [&](int l, auto t) {
        using TV = decltype(t);
        const uint32_t *w = slev + l * LW;
        CycleView<TV> v;
        v.nx = (uint32_t)uniform(w[0]);
        v.nxy = v.nx * (uint32_t)uniform(w[1]);
        v.n = (int)(v.nxy * (uint32_t)uniform(w[2]));
        v.mx = (uint32_t)uniform(w[3]);
        v.mxy = (uint32_t)uniform(w[4]);
        v.A = reinterpret_cast<TV *>(lds + uniform(w[5]));
        v.C = reinterpret_cast<TV *>(lds + uniform(w[6]));
        v.b = reinterpret_cast<TV *>(lds + uniform(w[7]));
        v.ex = ent + uniform(w[8]);
        v.ey = ent + uniform(w[9]);
        v.ez = ent + uniform(w[10]);
        return v;
    };
    const CycleTab<T> tt = {idt, pct};
    const CycleTab<double> td = {id64, pc64};
    const T om = T(a.omega), cff1 = T(1.0 - a.omega);
    const CycleView<T> v0 = view(0, T());
    CycleCells<T, R> s0;
    cycle_cells(s0, v0, tt, tid);
#pragma unroll
    for (int r = 0; r < R; r++)
        if (s0.live[r]) {
            v0.b[s0.q[r]] = vb[r];
            v0.A[s0.own[r]] = vy[r];
        }
    if (a.exact) {
        const uint32_t *w = slev + (nl - 1) * LW;
        const int nx2 = w[0] * w[0], ny2 = w[1] * w[1], nz2 = w[2] * w[2];
        double *e = reinterpret_cast<double *>(lds + a.e);
        for (int q = tid; q < nx2 + ny2 + nz2; q += CYC_T)
            e[q] = q < nx2 ? a.etab[q]
                           : (q < nx2 + ny2 ? a.etab[CS_MAXX * CS_MAXX + (q - nx2)]
                                            : a.etab[CS_MAXX * CS_MAXX + CS_MAX * CS_MAX +
                                                     (q - nx2 - ny2)]);
    }
    __syncthreads();
    const CycleView<double> vl = view(nl - 1, double());
    // a level's restriction into the next, its prolongation from the next
    auto down = [&](const auto &s, const CycleView<T> &v, int l) {
        cycle_sweep(s, v.A, v.C, v.b, om, cff1, (T *)nullptr);
        if (l + 1 == nl - 1) cycle_restrict(s, v, vl, td, a.omega, tid);
        else cycle_restrict(s, v, view(l + 1, T()), tt, a.omega, tid);
    };
    auto up = [&](const auto &s, const CycleView<T> &v, int l, T *out) {
        if (l + 1 == nl - 1) cycle_prolong(s, v, vl.C, tt);
        else cycle_prolong(s, v, view(l + 1, T()).A, tt);
        for (int h = 0; h < 2; h++)
            cycle_sweep(s, h ? v.C : v.A, h ? v.A : v.C, v.b, om, cff1, h ? out : (T *)nullptr);
    };
    if (nl > 1) down(s0, v0, 0);
    for (int l = 1; l < nl - 1; l++) {
        const CycleView<T> v = view(l, T());
        CycleCells<T, 1> s;
        cycle_cells(s, v, tt, tid);
        down(s, v, l);
    }
    if (a.exact) {
        const uint32_t *w = slev + (nl - 1) * LW;
        cycle_direct(a, vl, uniform(w[1]), uniform(w[2]),
                     reinterpret_cast<const double *>(lds + a.e), tid);
        if (nl == 1) {
#pragma unroll
            for (int r = 0; r < R; r++)
                if (s0.live[r]) gx[s0.q[r]] = v0.C[s0.own[r]];
        }
    } else if (nl == 1) {
        cycle_sweep(s0, v0.A, v0.C, v0.b, om, cff1, gx);
    } else {
        CycleCells<double, 1> s;
        cycle_cells(s, vl, td, tid);
        cycle_sweep(s, vl.A, vl.C, vl.b, a.omega, 1.0 - a.omega, (double *)nullptr);
    }
    for (int l = nl - 2; l >= 1; l--) {
        const CycleView<T> v = view(l, T());
        CycleCells<T, 1> s;
        cycle_cells(s, v, tt, tid);
        up(s, v, l, nullptr);
    }
    if (nl > 1) up(s0, v0, 0, gy);
}

template <typename T, int R>
__global__ __launch_bounds__(CYC_T) void k_mg_cycle(CycleArgs a, const T *gb, T *gy, T *gx,
                                                    CtlArgs fin) {
    __shared__ double lds[CYC_LDS / sizeof(double)];
    __shared__ uint32_t slev[CYC_MAXLEV * sizeof(CycleLevel) / 4];
    __shared__ CycleEnt ent[CYC_ENT];
    __shared__ double tb[32];
    if (blockIdx.x == 1) {
        ctl_body(fin, lds, threadIdx.x);
        return;
    }
    cycle_body<T, R>(a, gb, gy, gx, reinterpret_cast<char *>(lds), slev, ent, tb, threadIdx.x);
}

// the cycles of a batch's members, one workgroup each
template <typename T, int R>
__global__ __launch_bounds__(CYC_T) void k_b_cycle(const CycleItem<T> *__restrict__ items,
                                                   const int *__restrict__ active) {
    __shared__ double lds[CYC_LDS / sizeof(double)];
    __shared__ uint32_t slev[CYC_MAXLEV * sizeof(CycleLevel) / 4];
    __shared__ CycleEnt ent[CYC_ENT];
    __shared__ double tb[32];
    const CycleItem<T> &it = items[blockIdx.x];
    if (!active[it.member]) return;
    cycle_body<T, R>(it.a, it.b, it.y, it.x, reinterpret_cast<char *>(lds), slev, ent, tb,
                     threadIdx.x);
}

template <typename T>
hipError_t launch_b_cycle(const CycleItem<T> *items, int n, int most, const int *active,
                          hipStream_t s) {
    const dim3 grd(n), blk(CYC_T);
    if (most <= CYC_T) NYL_LAUNCH((k_b_cycle<T, 1>), grd, blk, 0, s, items, active);
    else if (most <= 2 * CYC_T) NYL_LAUNCH((k_b_cycle<T, 2>), grd, blk, 0, s, items, active);
    else NYL_LAUNCH((k_b_cycle<T, CYC_R>), grd, blk, 0, s, items, active);
    return hipGetLastError();
}
template hipError_t launch_b_cycle<double>(const CycleItem<double> *, int, int, const int *,
                                           hipStream_t);
template hipError_t launch_b_cycle<float>(const CycleItem<float> *, int, int, const int *,
                                          hipStream_t);

bool cycle_layout(CycleArgs &a, CycleEnt *ent, const Geo *lev, int l0, int nlev, int es,
                  bool exact, double omega, const MGTabs &tab) {
    a = CycleArgs{};
    a.nl = nlev - l0;
    if (l0 < 0 || a.nl < 1 || a.nl > CYC_MAXLEV) return false;
    const int64_t n0 = (int64_t)lev[l0].nx * lev[l0].ny * lev[l0].nz;
    if (n0 > (int64_t)CYC_T * CYC_R) return false;
    a.n0 = (int)n0;
    auto mul = [](uint32_t n) { return n == 1 ? 0u : (uint32_t)((((uint64_t)1 << 32) + n - 1) / n); };
    uint64_t o = 0;
    int ne = 0;
    for (int l = 0; l < a.nl; l++) {
        const Geo &g = lev[l0 + l];
        const int n3[3] = {g.nx, g.ny, g.nz}, p3[3] = {g.px, g.py, g.pz};
        const int64_t n = (int64_t)g.nx * g.ny * g.nz;
        if (l > 0) {   // an exact halving of the level above, one cell per thread
            const Geo &f = lev[l0 + l - 1];
            if (f.nx != 2 * g.nx || f.ny != 2 * g.ny || f.nz != 2 * g.nz || n > CYC_T) return false;
        }
        if (ne + g.nx + g.ny + g.nz > CYC_ENT) return false;
        CycleLevel &v = a.lev[l];
        v.nx = g.nx; v.ny = g.ny; v.nz = g.nz;
        v.mx = mul(g.nx);
        v.mxy = mul((uint32_t)g.nx * g.ny);
        // strides of a, c with a layer beyond each wall, and of the next level
        int64_t st[3], cst[3], size = 1, csize = 1;
        for (int q = 0; q < 3; q++) {
            st[q] = size;
            cst[q] = csize;
            size *= n3[q] + (p3[q] ? 0 : 2);
            csize *= n3[q] / 2 + (p3[q] ? 0 : 2);
        }
        if (size > 0xffff) return false;
        v.size = (uint32_t)size;
        const uint64_t bytes = l == a.nl - 1 ? 8 : es;
        auto take = [&](uint64_t elems) {
            const uint64_t at = o;
            o += (elems * bytes + 7) / 8 * 8;
            return (uint32_t)at;
        };
        v.a = take(size);
        v.c = take(size);
        v.b = take(n);
        int *first[3] = {&v.ex, &v.ey, &v.ez};
        for (int q = 0; q < 3; q++) {
            *first[q] = ne;
            const int m = n3[q], cm = m / 2, w = p3[q] ? 0 : 1;
            auto place = [&](int p, int len, int64_t stride) {   // position p of a line, walls padded
                if (p3[q]) p = ((p % len) + len) % len;
                return (uint32_t)((p + w) * stride);
            };
            for (int p = 0; p < m; p++) {
                const int count = p3[q] ? 2 : (p > 0) + (p < m - 1);
                uint32_t c0 = 0, c1 = 0, inside = 0;
                if (l < a.nl - 1) {
                    const int pc = p >> 1, pn = (p & 1) ? pc + 1 : pc - 1;
                    c0 = place(pc, cm, cst[q]);
                    c1 = place(pn, cm, cst[q]);
                    inside = (p3[q] || (pn >= 0 && pn < cm)) ? 1u << q : 0u;
                }
                CycleEnt &e = ent[ne++];
                e.w[0] = place(p, m, st[q]) | place(p - 1, m, st[q]) << 16;
                e.w[1] = place(p + 1, m, st[q]) | (uint32_t)count << 16 | inside << 20;
                e.w[2] = c0 | c1 << 16;
                e.w[3] = 0;
            }
        }
    }
    const Geo &g = lev[nlev - 1];
    a.px = g.px; a.py = g.py; a.pz = g.pz;
    a.exact = exact;
    a.nent = ne;
    a.bytes = (uint32_t)o;
    a.e = (uint32_t)o;
    if (exact)
        o += 8 * ((uint64_t)g.nx * g.nx + (uint64_t)g.ny * g.ny + (uint64_t)g.nz * g.nz);
    a.omega = omega;
    a.tab = tab;
    return o <= CYC_LDS;
}

template <typename T>
hipError_t launch_mg_cycle(const CycleArgs &a, const T *b, T *y, T *x, const CtlArgs *fin,
                           hipStream_t s) {
    if (a.nl < 1 || (a.nl == 1 && sizeof(T) != 8)) return hipErrorInvalidValue;
    CtlArgs c = {};
    if (fin) c = *fin;
    const dim3 grd(fin ? 2 : 1), blk(CYC_T);
    if (a.n0 <= CYC_T) NYL_LAUNCH((k_mg_cycle<T, 1>), grd, blk, 0, s, a, b, y, x, c);
    else if (a.n0 <= 2 * CYC_T) NYL_LAUNCH((k_mg_cycle<T, 2>), grd, blk, 0, s, a, b, y, x, c);
    else NYL_LAUNCH((k_mg_cycle<T, CYC_R>), grd, blk, 0, s, a, b, y, x, c);
    return hipGetLastError();
}
template hipError_t launch_mg_cycle<double>(const CycleArgs &, const double *, double *, double *,
                                            const CtlArgs *, hipStream_t);
template hipError_t launch_mg_cycle<float>(const CycleArgs &, const float *, float *, float *,
                                           const CtlArgs *, hipStream_t);

}  // namespace nyl
