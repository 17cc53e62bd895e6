// nyl_stage.h -- the explicit right-hand side and stage update (tracer
// advection, vortex force, Bernoulli term, viscosity, time scheme) of the
// Nyles time step on gfx950: device functions, kernels and their launch.
//
// FP64 instantiations reproduce the reference's arithmetic operation by
// operation (the library is compiled with -ffp-contract=off), so their
// results are bit-identical to the oracle's.
#pragma once
#include "nyl_internal.h"

namespace nyl {

#define NYL_BX 64
#define NYL_BY 4

static inline dim3 cell_grid(const Geo &g) {
    return dim3((g.nx + NYL_BX - 1) / NYL_BX, (g.ny + NYL_BY - 1) / NYL_BY, g.nz);
}

// Sequencing of the flux evaluations of the stage kernel.  Its stencil loads
// are invariant (const __restrict__), so the compiler is free to issue the
// loads of all twelve reconstructions before any arithmetic, which needs
// ~180 registers and leaves 2 waves per SIMD.  STAGE_SEQ(idx, dep) passes
// the offset of the next term through an empty asm that also takes the
// previous term's result: the next loads cannot be issued before that result
// exists, each term holds only its own operands and occupancy hides the load
// latency.  No instruction is emitted.
#ifndef NYL_STAGE_SEQ
#define NYL_STAGE_SEQ 1
#endif
#if NYL_STAGE_SEQ
#define STAGE_SEQ(idx, dep) asm volatile("" : "+v"(idx) : "v"(dep))
#else
#define STAGE_SEQ(idx, dep) ((void)0)
#endif

// Stage-kernel loads and stores at a 32-bit byte offset from the field's
// base pointer (the base is uniform, so the load takes it from scalar
// registers and the offset as one 32-bit register: no 64-bit address
// arithmetic per load).  A field is below 4 GiB (checked at context
// creation); offsets wrap modulo 2^32 to the right address.
template <typename T>
__device__ __forceinline__ T ldb(const T *__restrict__ p, uint32_t boff) {
    return *reinterpret_cast<const T *>(reinterpret_cast<const char *>(p) + boff);
}
template <typename T>
__device__ __forceinline__ void stb(T *__restrict__ p, uint32_t boff, T v) {
    *reinterpret_cast<T *>(reinterpret_cast<char *>(p) + boff) = v;
}
template <typename T>
__device__ __forceinline__ void stb_stream(T *__restrict__ p, uint32_t boff, T v) {
    store_stream(reinterpret_cast<T *>(reinterpret_cast<char *>(p) + boff), v);
}

// ---------------------------------------------------------------------------
// The reference's linear upwind branches (linear=.false. in its build:
// core/fortran_upwind.f90:30, core/fortran_vortex_force.f90:28,104), odd
// orders 1, 3, 5.  REAL(4) literals widened; sums left to right as written.

// The order at line position j of the left-biased (qp) or, RIGHT, the
// right-biased (qm) reconstruction; 0: the value is zero.  On a wall line it
// drops near the ends: tracer flavour (core/interpolate_tracer.f90:45-80)
// first order at 0 and n-1, third at 1 and n-2; vortex-force flavour
// (core/interpolate.f90:35-79) qp(-1) = 0, first order at 0 and n-2 (and qm
// at n-1), third at 1 and n-3.
template <bool VF, bool RIGHT>
__device__ __forceinline__ int lin_order(int j, int n, int order, bool per) {
    if (per) return order;
    if (VF && !RIGHT && j < 0) return 0;
    const int last1 = VF ? n - 2 : n - 1;          // first order at 0 and here
    if (j <= 0 || j >= last1) return 1;
    return order == 5 && (j == 1 || j == last1 - 1) ? 3 : order;
}
// The reconstruction of that order from the values at j-2 .. j+2.
template <typename T, bool RIGHT>
__device__ __forceinline__ T lin_value(int ord, T q0, T q1, T q2, T q3, T q4) {
    const T c1 = T(-(1.0f / 6.0f)), c2 = T(5.0f / 6.0f), c3 = T(2.0f / 6.0f);
    const T b1 = T(2.0f / 60.0f), b2 = T(-(13.0f / 60.0f)), b3 = T(47.0f / 60.0f);
    const T b4 = T(27.0f / 60.0f), b5 = T(-(3.0f / 60.0f));
    if (ord == 0) return T(0);
    if (ord == 1) return q2;
    if (ord == 3) {
        if (RIGHT) return c3 * q1 + c2 * q2 + c1 * q3;
        return c1 * q1 + c2 * q2 + c3 * q3;
    }
    if (RIGHT) return b5 * q0 + b4 * q1 + b3 * q2 + b2 * q3 + b1 * q4;
    return b1 * q0 + b2 * q1 + b3 * q2 + b4 * q3 + b5 * q4;
}
// The two upwind contributions at a face from its six values: the left-biased
// reconstruction at line position j times up and the right-biased one at
// j + 1 times um, up/um = 0.5*(U -+ |U|).
template <typename T, bool VF, int PER>
__device__ __forceinline__ void lin_parts(T u, const Stencil6<T> &w, int j, int n, int order, T &a,
                                          T &b) {
    const T au = fabs(u), up = T(0.5) * (u + au), um = T(0.5) * (u - au);
    a = up * lin_value<T, false>(lin_order<VF, false>(j, n, order, PER != 0), w.m2, w.m1, w.z0,
                                 w.p1, w.p2);
    b = um * lin_value<T, true>(lin_order<VF, true>(j + 1, n, order, PER != 0), w.m1, w.z0, w.p1,
                                w.p2, w.p3);
}

// Byte offsets of the cells -3..+3 away along an axis, wrapped on a periodic
// one and held inside the line on a wall axis (the closures read none of the
// values outside).  O: int64_t where the position is the same for the whole
// wavefront -- the load then adds it to the field's base in scalar registers
// -- and int32_t where it differs by lane (32-bit wrapping offsets: a field is
// below 4 GiB).
template <typename O>
struct Line {
    O m3, m2, m1, p1, p2, p3;
};
template <int PER, typename O>
__device__ __forceinline__ Line<O> line_of(int m, int n, O stride) {
    auto off = [&](int d) -> O {
        const int q = m + d;
        return (O)((PER ? wrapi(q, n) : (q < 0 ? 0 : (q >= n ? n - 1 : q))) - m) * stride;
    };
    return Line<O>{off(-3), off(-2), off(-1), off(1), off(2), off(3)};
}
template <typename T, typename O>
__device__ __forceinline__ T ldo(const T *__restrict__ p, uint32_t cb, O off) {
    if constexpr (sizeof(O) == 8)
        return *reinterpret_cast<const T *>(reinterpret_cast<const char *>(p) + off + cb);
    else return ldb(p, cb + (uint32_t)off);
}
// N consecutive cells of a row, loaded and stored as one: one 4- or 8-byte
// element, or 16 bytes (four floats, two doubles; aligned, as N divides nx).
template <typename T, int N>
struct alignas(N * sizeof(T)) Vec {
    T v[N];
};

template <int N, typename T, typename O>
__device__ __forceinline__ Vec<T, N> ldv(const T *__restrict__ p, uint32_t cb, O off) {
    typedef const Vec<T, N> *V;
    const char *b = reinterpret_cast<const char *>(p);
    if constexpr (sizeof(O) == 8) return *reinterpret_cast<V>(b + off + cb);
    else return *reinterpret_cast<V>(b + (uint32_t)(cb + (uint32_t)off));
}
// at the sum of two offsets
template <int N, typename T, typename O, typename E>
__device__ __forceinline__ Vec<T, N> ldv2(const T *__restrict__ p, uint32_t cb, O o, E e) {
    if constexpr (sizeof(O) == sizeof(E)) return ldv<N>(p, cb, o + e);
    else if constexpr (sizeof(O) == 8) return ldv<N>(p, cb + (uint32_t)e, o);
    else return ldv<N>(p, cb + (uint32_t)o, e);
}
template <int N, typename T>
__device__ __forceinline__ Vec<T, N> ldv(const T *__restrict__ p, uint32_t cb) {
    return ldv<N, T, int32_t>(p, cb, 0);
}
template <int N, bool STREAM, typename T>
__device__ __forceinline__ void stv(T *__restrict__ p, uint32_t cb, const Vec<T, N> &x) {
    Vec<T, N> *d = reinterpret_cast<Vec<T, N> *>(reinterpret_cast<char *>(p) + cb);
#if defined(__HIP_DEVICE_COMPILE__)
    if constexpr (STREAM && N > 1) {
        typedef T R __attribute__((ext_vector_type(N)));
        R r;
        __builtin_memcpy(&r, x.v, sizeof(r));
        store_stream(reinterpret_cast<R *>(d), r);
        return;
    }
#endif
    if (STREAM && N == 1) stb_stream(p, cb, x.v[0]);
    else *d = x;
}

// The x axis of N cells: the byte offsets of the elements (N = 1: the cells
// -3..+3 away) or of the 16-byte groups before and after them, wrapped or
// held inside the line as in Line (a group never straddles the line's end).
template <int N>
struct LineX {
    int32_t b2, b1, a1, a2;   // groups -2, -1, +1, +2
    __device__ __forceinline__ int32_t before() const { return b1; }
    __device__ __forceinline__ int32_t after() const { return a1; }
};
template <>
struct LineX<1> : Line<int32_t> {
    __device__ __forceinline__ int32_t before() const { return m1; }
    __device__ __forceinline__ int32_t after() const { return p1; }
};
template <int N, int PER>
__device__ __forceinline__ LineX<N> linex_of(int i, int nx, int es) {
    LineX<N> L;
    if constexpr (N == 1) {
        static_cast<Line<int32_t> &>(L) = line_of<PER, int32_t>(i, nx, es);
    } else {
        auto off = [&](int d) -> int32_t {
            const int q = i + d;
            return ((PER ? wrapi(q, nx) : (q < 0 ? 0 : (q >= nx ? nx - N : q))) - i) * es;
        };
        L = LineX<N>{off(-2 * N), off(-N), off(N), off(2 * N)};
    }
    return L;
}
// The row of f around the N cells: r[4 + d] = the value at i + d, for
// -3 <= d <= N + 2 (HI) or N + 1.
template <int N, bool HI, typename T>
__device__ __forceinline__ void load_row(T (&r)[N + 8], const T *__restrict__ f, uint32_t cb,
                                         const LineX<N> &L) {
    if constexpr (N == 1) {
        r[1] = ldo(f, cb, L.m3); r[2] = ldo(f, cb, L.m2); r[3] = ldo(f, cb, L.m1);
        r[4] = ldb(f, cb);
        r[5] = ldo(f, cb, L.p1); r[6] = ldo(f, cb, L.p2);
        if (HI) r[7] = ldo(f, cb, L.p3);
    } else {
        auto put = [&](int at, int32_t off) {
            const Vec<T, N> a = ldv<N>(f, cb, off);
#pragma unroll
            for (int q = 0; q < N; q++) r[at + q] = a.v[q];
        };
        if (N == 2) put(0, L.b2);
        put(4 - N, L.b1); put(4, 0); put(4 + N, L.a1);
        if (N == 2 && HI) put(4 + 2 * N, L.a2);
    }
}
// N + 1 values of a row from the cell before (LO) or from the first cell on
template <int N, bool LO, typename T, typename O>
__device__ __forceinline__ void load_next(T (&r)[N + 1], const T *__restrict__ f, uint32_t cb,
                                          const LineX<N> &L, O off) {
    const Vec<T, N> c = ldv<N>(f, cb, off);
    const Vec<T, N> s = ldv2<N>(f, cb, LO ? L.before() : L.after(), off);
#pragma unroll
    for (int q = 0; q < N; q++) r[LO ? q + 1 : q] = c.v[q];
    r[LO ? 0 : N] = s.v[LO ? N - 1 : 0];
}

// All six values either upwind direction of a face needs are loaded, and the
// five selected in registers: a wavefront with both directions in it then
// reads whole lines once (selected addresses scatter it over two sets).
//
// The tracer flux at line position m, and its divergence d + flux(m-1) -
// flux(m) with no flux through the ends of a wall line.  WENO
// (core/fortran_upwind.f90:77-81), or, order = 1, 3, 5 (LIN), the linear
// branch (:34-67): fx(i) = up(i)*qp(i) + um(i)*qm(i+1).
template <typename T, int PER, bool LIN>
__device__ __forceinline__ T tracer_flux(int m, int n, T u, const Stencil6<T> &w, int order) {
    if (LIN && order != 0) {
        if (!PER && m == n - 1) return T(0);
        T a, b;
        lin_parts<T, false, PER>(u, w, m, n, order, a, b);
        return a + b;
    }
    return face_of<T, PER>(m, n, u, w);
}
template <typename T, int PER, bool LIN>
__device__ __forceinline__ T tracer_div(T d, T fl, T fr, int m, int order) {
    if (!PER && m == 0) return LIN && order != 0 ? (d + T(0)) - fr : d - fr;
    return (d + fl) - fr;
}
// Along x, N cells: the N + 1 faces are evaluated once.  U_d = ud*cu,
// recomputed from the covariant velocity with the product U_from_u stores
// (core/cov_to_contra.py:15-17).
template <int N, int PER, bool LIN, typename T>
__device__ __forceinline__ void tracer_x(Vec<T, N> &d, const T *__restrict__ q,
                                         const T *__restrict__ ud, T cu, uint32_t cb,
                                         const LineX<N> &L, int i, int nx, int order) {
    T r[N + 8], u[N + 1], fl[N + 1];
    load_row<N, true>(r, q, cb, L);
    load_next<N, true>(u, ud, cb, L, (int32_t)0);
#pragma unroll
    for (int f = 0; f <= N; f++) {
        const int m = i + f - 1;
        const Stencil6<T> w = {r[f + 1], r[f + 2], r[f + 3], r[f + 4], r[f + 5], r[f + 6]};
        fl[f] = tracer_flux<T, PER, LIN>(PER ? 0 : m, nx, u[f] * cu, w, order);
    }
#pragma unroll
    for (int c = 0; c < N; c++)
        d.v[c] = tracer_div<T, PER, LIN>(d.v[c], fl[c], fl[c + 1], i + c, order);
}
// ... and along y or z (line position m of n)
template <int N, int PER, bool LIN, typename T, typename O>
__device__ __forceinline__ void tracer_yz(Vec<T, N> &d, const T *__restrict__ q,
                                          const T *__restrict__ ud, T cu, uint32_t cb,
                                          const Line<O> &L, int m, int n, int order) {
    const Vec<T, N> m3 = ldv<N>(q, cb, L.m3), m2 = ldv<N>(q, cb, L.m2), m1 = ldv<N>(q, cb, L.m1);
    const Vec<T, N> z0 = ldv<N>(q, cb), p1 = ldv<N>(q, cb, L.p1), p2 = ldv<N>(q, cb, L.p2);
    const Vec<T, N> p3 = ldv<N>(q, cb, L.p3), u1 = ldv<N>(ud, cb), u0 = ldv<N>(ud, cb, L.m1);
#pragma unroll
    for (int c = 0; c < N; c++) {
        const Stencil6<T> hi = {m2.v[c], m1.v[c], z0.v[c], p1.v[c], p2.v[c], p3.v[c]};
        const Stencil6<T> lo = {m3.v[c], m2.v[c], m1.v[c], z0.v[c], p1.v[c], p2.v[c]};
        const T fr = tracer_flux<T, PER, LIN>(m, n, u1.v[c] * cu, hi, order);
        T fl = T(0);
        if (PER || m > 0) fl = tracer_flux<T, PER, LIN>(m - 1, n, u0.v[c] * cu, lo, order);
        d.v[c] = tracer_div<T, PER, LIN>(d.v[c], fl, fr, m, order);
    }
}

// One term of the vortex force at N cells, d -+ its flux: the vorticity
// component `om` is upwinded along axis d with the contravariant velocity
// U_d = ud*cu averaged along the target axis e (UU, UU_0 = 0. at the line
// start) and then along d (u1d).  WENO (core/fortran_vortex_force.f90:66-81,
// 145-159): q(1) = 0., q(k) = vort(k-1).  Linear (order != 0; :43-65 direc,
// :121-144 flip): (d -+ qp(md-1)*up) -+ qm(md)*um, where the vorticity is not
// shifted -- the same six values.
template <typename T, int PER, int SIGN, bool LIN>
__device__ __forceinline__ T vf_term(T d, int m, int n, T u1d, Stencil6<T> &w, int order) {
    if (LIN && order != 0) {
        T a, b;
        lin_parts<T, true, PER>(u1d, w, m - 1, n, order, a, b);
        return SIGN < 0 ? (d - a) - b : (d + a) + b;
    }
    if (!PER) {   // line position 0
        if (m == 0) w.z0 = T(0);
        else if (m == 1) w.m1 = T(0);
        else if (m == 2) w.m2 = T(0);
    }
    const T f = face_of<T, PER>(m, n, u1d, w);
    return SIGN < 0 ? d - f : d + f;
}
// Along x, averaged with the cells at offset oe:
template <int N, int PER, int SIGN, bool LIN, typename T, typename E>
__device__ __forceinline__ void vf_x(Vec<T, N> &d, const T *__restrict__ ud, T cu,
                                     const T *__restrict__ om, uint32_t cb, const LineX<N> &L,
                                     int i, int nx, E oe, int order) {
    T a[N + 1], b[N + 1], r[N + 8];
    load_next<N, true>(a, ud, cb, L, (int32_t)0);
    load_next<N, true>(b, ud, cb, L, oe);
    load_row<N, false>(r, om, cb, L);
    T uu[N + 1];
#pragma unroll
    for (int c = 0; c <= N; c++) uu[c] = T(0.5) * (a[c] * cu + b[c] * cu);
    if (!PER && i == 0) uu[0] = T(0);
#pragma unroll
    for (int c = 0; c < N; c++) {
        Stencil6<T> w = {r[c + 1], r[c + 2], r[c + 3], r[c + 4], r[c + 5], r[c + 6]};
        d.v[c] = vf_term<T, PER, SIGN, LIN>(d.v[c], i + c, nx, T(0.5) * (uu[c] + uu[c + 1]), w,
                                            order);
    }
}
// along y or z (line position m of n): uu and up, the averaged velocities at
// the cells and at the line position before
template <int N, int PER, int SIGN, bool LIN, typename T, typename O>
__device__ __forceinline__ void vf_line(Vec<T, N> &d, const T (&uu)[N], const T (&up)[N],
                                        const T *__restrict__ om, uint32_t cb, const Line<O> &L,
                                        int m, int n, int order) {
    const Vec<T, N> m3 = ldv<N>(om, cb, L.m3), m2 = ldv<N>(om, cb, L.m2), m1 = ldv<N>(om, cb, L.m1);
    const Vec<T, N> z0 = ldv<N>(om, cb), p1 = ldv<N>(om, cb, L.p1), p2 = ldv<N>(om, cb, L.p2);
#pragma unroll
    for (int c = 0; c < N; c++) {
        Stencil6<T> w = {m3.v[c], m2.v[c], m1.v[c], z0.v[c], p1.v[c], p2.v[c]};
        const T uprev = !PER && m == 0 ? T(0) : up[c];
        d.v[c] = vf_term<T, PER, SIGN, LIN>(d.v[c], m, n, T(0.5) * (uprev + uu[c]), w, order);
    }
}
// averaged with the cells at offset oe (y or z)
template <int N, int PER, int SIGN, bool LIN, typename T, typename O, typename E>
__device__ __forceinline__ void vf_yz(Vec<T, N> &d, const T *__restrict__ ud, T cu,
                                      const T *__restrict__ om, uint32_t cb, const Line<O> &L,
                                      int m, int n, E oe, int order) {
    const Vec<T, N> a = ldv<N>(ud, cb), b = ldv<N>(ud, cb, oe);
    const Vec<T, N> c = ldv<N>(ud, cb, L.m1), e = ldv2<N>(ud, cb, L.m1, oe);
    T uu[N], up[N];
#pragma unroll
    for (int q = 0; q < N; q++) {
        uu[q] = T(0.5) * (a.v[q] * cu + b.v[q] * cu);
        up[q] = T(0.5) * (c.v[q] * cu + e.v[q] * cu);
    }
    vf_line<N, PER, SIGN, LIN>(d, uu, up, om, cb, L, m, n, order);
}
// averaged with the next cells in x
template <int N, int PER, int SIGN, bool LIN, typename T, typename O>
__device__ __forceinline__ void vf_yz_x(Vec<T, N> &d, const T *__restrict__ ud, T cu,
                                        const T *__restrict__ om, uint32_t cb, const Line<O> &L,
                                        const LineX<N> &Lx, int m, int n, int order) {
    T a[N + 1], c[N + 1], uu[N], up[N];
    load_next<N, false>(a, ud, cb, Lx, (int32_t)0);
    load_next<N, false>(c, ud, cb, Lx, L.m1);
#pragma unroll
    for (int q = 0; q < N; q++) {
        uu[q] = T(0.5) * (a[q] * cu + a[q + 1] * cu);
        up[q] = T(0.5) * (c[q] * cu + c[q + 1] * cu);
    }
    vf_line<N, PER, SIGN, LIN>(d, uu, up, om, cb, L, m, n, order);
}

// One direction of core/fortran_dissipation.f90:2-34 add_laplacian at a
// cell: d + coef*(fx - fxm), fx = f(m+1) - f(m), fxm = f(m) - f(m-1); on a
// wall axis fxm = 0 at the first cell and fx = 0 at the last (no flux
// through the ends of the line).  om, op: byte offsets of the m-1 and m+1
// neighbours (wrapped on a periodic axis).
template <typename T, int P>
__device__ __forceinline__ T lap_axis(T d, const T *__restrict__ f, uint32_t cb, int m, int n,
                                      int32_t om, int32_t op, T coef) {
    const T c0 = ldb(f, cb);
    const T fx = (P || m < n - 1) ? ldb(f, cb + (uint32_t)op) - c0 : T(0);
    const T fxm = (P || m > 0) ? c0 - ldb(f, cb + (uint32_t)om) : T(0);
    return d + coef * (fx - fxm);
}

// add_viscosity (core/viscosity.py:3-9) for the three components of a cell:
// for each component, the x, y and z directions in that order
template <typename T, int PX, int PY, int PZ>
__device__ __forceinline__ void viscosity_cell(const Geo &g, const StageArgs<T> &a, uint32_t cb,
                                               int i, int j, int k, T &du, T &dv, T &dw) {
    constexpr int ES = (int)sizeof(T);
    const int32_t sx = ES, sy = (int32_t)g.sy * ES, sz = (int32_t)g.sz * ES;
    const int32_t oxm = PX ? (wrapi(i - 1, g.nx) - i) * sx : -sx;
    const int32_t oxp = PX ? (wrapi(i + 1, g.nx) - i) * sx : sx;
    const int32_t oym = PY ? (wrapi(j - 1, g.ny) - j) * sy : -sy;
    const int32_t oyp = PY ? (wrapi(j + 1, g.ny) - j) * sy : sy;
    const int32_t ozm = PZ ? (wrapi(k - 1, g.nz) - k) * sz : -sz;
    const int32_t ozp = PZ ? (wrapi(k + 1, g.nz) - k) * sz : sz;
    const T cx = T(a.vcx), cy = T(a.vcy), cz = T(a.vcz);
    auto lap3 = [&](T d, const T *__restrict__ f) -> T {
        d = lap_axis<T, PX>(d, f, cb, i, g.nx, oxm, oxp, cx);
        d = lap_axis<T, PY>(d, f, cb, j, g.ny, oym, oyp, cy);
        return lap_axis<T, PZ>(d, f, cb, k, g.nz, ozm, ozp, cz);
    };
    du = lap3(du, a.u);
    dv = lap3(dv, a.v);
    dw = lap3(dw, a.w);
}

// The stage combination of one field at N cells (core/timescheme.py) with the
// coefficients c and (LFAM3 predictor) c2: its tendency d, the current and next state, the tendency slots and the LFAM3
// 'before' state.
template <int N, int MODE, bool LIN, typename T>
__device__ __forceinline__ void stage_out(double c, double c2, uint32_t cb, const Vec<T, N> &d,
                                          const T *__restrict__ now, T *__restrict__ next,
                                          T *__restrict__ tend, const T *__restrict__ d0,
                                          const T *__restrict__ d1, T *__restrict__ before) {
    // read at a later stage; the model variants keep them at every stage
    if (MODE == 0 || MODE == 1 || MODE == 2 || LIN) stv<N, true>(tend, cb, d);
    if (MODE == 0) return;
    const T cc = T(c);
    const Vec<T, N> s = ldv<N>((MODE == 5 ? (const T *)next : now), cb);
    Vec<T, N> o, e0, e1;
    if (MODE == 2 || MODE == 3) e0 = ldv<N>(d0, cb);
    if (MODE == 3) e1 = ldv<N>(d1, cb);
    if (MODE == 4) e0 = ldv<N>((const T *)before, cb);
#pragma unroll
    for (int q = 0; q < N; q++) {
        if (MODE == 1 || MODE == 5 || MODE == 6) {   // s += dt*ds
            o.v[q] = s.v[q] + cc * d.v[q];
        } else if (MODE == 2) {                      // s += (dt/4.)*(ds1-3*ds0)
            o.v[q] = s.v[q] + cc * (d.v[q] - T(3) * e0.v[q]);
        } else if (MODE == 3) {                      // s += (dt/12.)*(8*ds2-ds0-ds1)
            o.v[q] = s.v[q] + cc * ((T(8) * d.v[q] - e0.v[q]) - e1.v[q]);
        } else {   // LFAM3 predictor: s = sb + (2.*dt)*ds; s = (1./12.)*(5.*s+8.*sn-sb); sb = sn
            const T t1 = e0.v[q] + T(c2) * d.v[q];
            o.v[q] = T(1. / 12.) * (T(5) * t1 + T(8) * s.v[q] - e0.v[q]);
        }
    }
    if (MODE == 4 || MODE == 6) stv<N, false>(before, cb, s);
    stv<N, false>(next, cb, o);
}

// Fused LES.rhs (core/model_les.py:129-144) + stage update
// (core/timescheme.py:199-220, LFAM3 :144-175 and :352-364) for N cells of a
// row.  LIN: with the model variants and the reference's linear upwind
// branches.  Y, Z: the types of the offsets along those axes.
template <typename T, int N, int MODE, int PX, int PY, int PZ, bool LIN, typename Y, typename Z>
__device__ __forceinline__ void stage_cells(const Geo &g, const StageArgs<T> &a, int i, int j,
                                            int k) {
    constexpr int ES = (int)sizeof(T);
    const int64_t cell = (int64_t)k * g.sz + (int64_t)j * g.sy + i;
    const uint32_t cb = (uint32_t)cell * (uint32_t)ES;   // the cells' byte offset
    const LineX<N> Lx = linex_of<N, PX>(i, g.nx, ES);
    const Line<Y> Ly = line_of<PY, Y>(j, g.ny, (Y)(g.sy * ES));
    const Line<Z> Lz = line_of<PZ, Z>(k, g.nz, (Z)(g.sz * ES));

    // model variants: the linear model has no vortex force
    // (core/model_les.py:135-136), Euler3d neither advects b
    // (core/model_les_euler.py:131) nor adds buoyancy (core/bernoulli.py:26-32)
    const bool vf = !LIN || !(a.flags & NYL_SF_NO_VF);
    const bool with_b = !LIN || !(a.flags & NYL_SF_NO_B);
    const bool ey = PY || j < g.ny - 1;   // loops stop at n-1 on a wall axis
    const bool ez = PZ || k < g.nz - 1;

    // tracer b: rhstrac, directions i, j, k (core/tracer.py:63-72)
    const T cx = T(a.idx2), cy = T(a.idy2), cz = T(a.idz2);
    Vec<T, N> db = {}, du = {}, dv = {}, dw = {};
    uint32_t cs = cb;
    const int oa = LIN ? a.upw_a : 0, ov = LIN ? a.upw_vf : 0;
    if (with_b) {
        tracer_x<N, PX, LIN>(db, a.b, a.u, cx, cs, Lx, i, g.nx, oa);
        if constexpr (N < 4) STAGE_SEQ(cs, db.v[0]);   // N = 4: overlapped, 3 % faster
        tracer_yz<N, PY, LIN>(db, a.b, a.v, cy, cs, Ly, j, g.ny, oa);
        if constexpr (N < 4) STAGE_SEQ(cs, db.v[0]);
        tracer_yz<N, PZ, LIN>(db, a.b, a.w, cz, cs, Lz, k, g.nz, oa);
        STAGE_SEQ(cs, db.v[0]);
    }

    // vortex force, triplets 'ikj', 'jik', 'kji' (core/vortex_force.py:69-81):
    // direc(U_i, vor_k, du_j), flip(U_j, vor_k, du_i), direc(U_j, vor_i, du_k),
    // flip(U_k, vor_i, du_j), direc(U_k, vor_j, du_i), flip(U_i, vor_j, du_k)
    if (vf) {
        if (ey) vf_x<N, PX, -1, LIN>(dv, a.u, cx, a.oz, cs, Lx, i, g.nx, Ly.p1, ov);
        STAGE_SEQ(cs, dv.v[0]);
        vf_yz_x<N, PY, +1, LIN>(du, a.v, cy, a.oz, cs, Ly, Lx, j, g.ny, ov);
        STAGE_SEQ(cs, du.v[0]);
        if (ez) vf_yz<N, PY, -1, LIN>(dw, a.v, cy, a.ox, cs, Ly, j, g.ny, Lz.p1, ov);
        STAGE_SEQ(cs, dw.v[0]);
        if (ey) vf_yz<N, PZ, +1, LIN>(dv, a.w, cz, a.ox, cs, Lz, k, g.nz, Ly.p1, ov);
        STAGE_SEQ(cs, dv.v[0]);
        vf_yz_x<N, PZ, -1, LIN>(du, a.w, cz, a.oy, cs, Lz, Lx, k, g.nz, ov);
        STAGE_SEQ(cs, du.v[0]);
        if (ez) vf_x<N, PX, +1, LIN>(dw, a.u, cx, a.oy, cs, Lx, i, g.nx, Lz.p1, ov);
    }

    // bernoulli (core/bernoulli.py:14-23, core/fortran_bernoulli.f90:2-58)
    {
        T ke[N + 1];
        load_next<N, false>(ke, a.ke, cb, Lx, (int32_t)0);
#pragma unroll
        for (int q = 0; q < N; q++) {
            du.v[q] = du.v[q] - (ke[q + 1] - ke[q]);
            if (!PX && i + q == g.nx - 1) du.v[q] = T(0);   // the wall face: no term above
        }
        if (ey) {
            const Vec<T, N> ku = ldv<N>(a.ke, cb, Ly.p1);
#pragma unroll
            for (int q = 0; q < N; q++) dv.v[q] = dv.v[q] - (ku.v[q] - ke[q]);
        }
        if (ez) {
            const T cff = T(0.5 * a.dz);
            const Vec<T, N> ku = ldv<N>(a.ke, cb, Lz.p1);
            const Vec<T, N> b0 = ldv<N>(a.b, cb), b1 = ldv<N>(a.b, cb, Lz.p1);
#pragma unroll
            for (int q = 0; q < N; q++) {
                if (with_b) dw.v[q] = dw.v[q] - (ku.v[q] - ke[q]) + cff * (b1.v[q] + b0.v[q]);
                else dw.v[q] = dw.v[q] - (ku.v[q] - ke[q]);
            }
        }
    }
    // viscosity at the last stage (core/model_les.py:140-141)
    if (a.visc) {
#pragma unroll
        for (int q = 0; q < N; q++)
            viscosity_cell<T, PX, PY, PZ>(g, a, cb + (uint32_t)(q * ES), i + q, j, k, du.v[q],
                                          dv.v[q], dw.v[q]);
    }
    stage_out<N, MODE, LIN>(a.c, a.c2, cb, db, a.b, a.bn, a.tb, a.d0b, a.d1b, a.sbb);
    stage_out<N, MODE, LIN>(a.c, a.c2, cb, du, a.u, a.un, a.tu, a.d0u, a.d1u, a.sbu);
    stage_out<N, MODE, LIN>(a.c, a.c2, cb, dv, a.v, a.vn, a.tv, a.d0v, a.d1v, a.sbv);
    stage_out<N, MODE, LIN>(a.c, a.c2, cb, dw, a.w, a.wn, a.tw, a.d0w, a.d1w, a.sbw);
}

#if defined(__HIP_DEVICE_COMPILE__)
#define WAVE_UNIFORM(x) __builtin_amdgcn_readfirstlane(x)
#else
#define WAVE_UNIFORM(x) (x)
#endif

// One cell per thread, 64 x 4 x 1 blocks: the first LFAM3 step.
template <typename T, int MODE, int PX, int PY, int PZ>
__global__ __launch_bounds__(256) void k_stage(Geo g, StageArgs<T> a) {
    const Blk3 bk = xcd_block_yslab();
    const int i = bk.x * NYL_BX + threadIdx.x;
    const int j = WAVE_UNIFORM((int)(bk.y * NYL_BY + threadIdx.y));
    const int k = bk.z;
    if (i >= g.nx || j >= g.ny) return;
    stage_cells<T, 1, MODE, PX, PY, PZ, false, int64_t, int64_t>(g, a, i, j, k);
}

// N cells per thread, the N-groups of a plane numbered along its rows: no lane
// idles whatever nx is (64-wide rows left a third of them idle at nx = 96, a
// fifth at 200).  lw > 0: tiles of 2^lw groups x 256/2^lw rows instead.
//
// What bounds it.  FP64: a load of 8 bytes per lane passes L1 at 32 B/clk, of
// 16 bytes at 64 B/clk; with one cell per thread the kernel sat at 80 % of
// that rate, with two at 43 %, and the N + 1 x faces of the group are shared.
// Now the VALU (busy 85 %) at the clock FP64 runs at (1.95 GHz).  FP32: the
// VALU (busy 93 % with one cell per thread); four cells share x faces and
// address arithmetic (944 -> 771 instructions per 64 cells).
// us per call, one cell per thread in 64-wide rows -> now: FP64 256^3
// periodic 1161 -> 970, 160x96x128 162 -> 112, 96^3 87 -> 57; FP32 256^3
// 510 -> 440, walls 256x128x64 106 -> 58, 200x120x56 72 -> 42.
#define STAGE_NT 256
#define GRID_YZ 65536   // most blocks along y and z of a launch
static inline int64_t flat_blocks(int64_t ngroup) { return (ngroup + STAGE_NT - 1) / STAGE_NT; }

template <typename T, int N, int MODE, int PX, int PY, int PZ, bool LIN = false>
__global__ __launch_bounds__(STAGE_NT) void k_stage_flat(Geo g, StageArgs<T> a, int lw) {
    const Blk3 bk = xcd_block_yslab();
    const int nxg = g.nx / N;
    int i, j;
    if (lw == 0) {
        const uint32_t q = (uint32_t)bk.y * STAGE_NT + threadIdx.x;
        j = (int)(q / (uint32_t)nxg);
        i = (int)(q - (uint32_t)j * (uint32_t)nxg);
    } else {
        i = (bk.x << lw) + (int)(threadIdx.x & ((1u << lw) - 1));
        j = bk.y * (STAGE_NT >> lw) + (int)(threadIdx.x >> lw);
        if (i >= nxg) return;
    }
    if (j >= g.ny) return;
    stage_cells<T, N, MODE, PX, PY, PZ, LIN, int32_t, int64_t>(g, a, i * N, j, bk.z);
}

template <typename T, int N, int MODE, int PX, int PY, int PZ, bool LIN>
static void stage_flat_go(const Geo &g, const StageArgs<T> &a, hipStream_t s) {
    const int nxg = g.nx / N;
    // FP64 in whole tiles of 8 pairs (one line of L2) x 32 rows: the rows that
    // neighbours in y share stay in L1, 256^3 1033 -> 978 us, 160x96x128
    // 114 -> 110; no gain in FP32, whose loads are half as long
    // (lw = 3).  Planes of more groups than the blocks along y take (2M cells in
    // a row): tiles of 64 x 4, whose blocks along x are not so limited (lw = 6).
    const int64_t nb = flat_blocks((int64_t)nxg * g.ny);
    const int lw = (N == 2 && nxg % 8 == 0 && g.ny % 32 == 0) ? 3 : (nb > GRID_YZ ? 6 : 0);
    const int cols = 1 << lw, rows = STAGE_NT >> lw;
    const dim3 grd = lw ? dim3((nxg + cols - 1) / cols, (g.ny + rows - 1) / rows, g.nz)
                        : dim3(1, (unsigned)nb, g.nz);
    NYL_LAUNCH((k_stage_flat<T, N, MODE, PX, PY, PZ, LIN>), grd, STAGE_NT, 0, s, g, a, lw);
}

// Cells per thread.  16 bytes where the row divides into such groups (an FP64
// row always does: nx is even) and the grid has enough of them to fill the
// chip (256 CUs x 4 SIMDs): in FP64 from
// two waves of pairs per SIMD (64^3: 24.8 -> 22.6 us; 64x32x32 would go
// 11.8 -> 17.3), in FP32 from six waves of fours (256x128x64: 63.5 -> 58;
// 200x120x56 would go 41.9 -> 44.2, 64x32x32 7.2 -> 15.4).  Below, one cell.
template <typename T>
static inline bool stage_wide(const Geo &g) {
    constexpr int N = 16 / (int)sizeof(T);
    return g.nx % N == 0 && (int64_t)g.nx * g.ny * g.nz >= (sizeof(T) == 8 ? 1 << 18 : 3 << 19);
}

template <typename T, int MODE, int PX, int PY, int PZ, bool LIN = false>
static void stage_go(const Geo &g, const StageArgs<T> &a, hipStream_t s) {
    if (stage_wide<T>(g)) stage_flat_go<T, 16 / (int)sizeof(T), MODE, PX, PY, PZ, LIN>(g, a, s);
    else stage_flat_go<T, 1, MODE, PX, PY, PZ, LIN>(g, a, s);
}

template <typename T, int PX, int PY, int PZ>
static hipError_t stage_les(const Geo &g, const StageArgs<T> &a, int mode, hipStream_t s) {
    switch (mode) {
    case 0: stage_go<T, 0, PX, PY, PZ>(g, a, s); break;
    case 1: stage_go<T, 1, PX, PY, PZ>(g, a, s); break;
    case 2: stage_go<T, 2, PX, PY, PZ>(g, a, s); break;
    case 3: stage_go<T, 3, PX, PY, PZ>(g, a, s); break;
    case 4: stage_go<T, 4, PX, PY, PZ>(g, a, s); break;
    case 5: stage_go<T, 5, PX, PY, PZ>(g, a, s); break;
    case 6:   // the first step of a run only
        NYL_LAUNCH((k_stage<T, 6, PX, PY, PZ>), cell_grid(g), dim3(NYL_BX, NYL_BY, 1), 0, s, g, a);
        break;
    default: return hipErrorInvalidValue;
    }
    return hipGetLastError();
}

// the model variants and the linear branches: the tendencies, or an RK3 stage
// with its tendencies stored too
template <typename T, int PX, int PY, int PZ>
static hipError_t stage_lin(const Geo &g, const StageArgs<T> &a, int mode, hipStream_t s) {
    switch (mode) {
    case 0: stage_go<T, 0, PX, PY, PZ, true>(g, a, s); break;
    case 1: stage_go<T, 1, PX, PY, PZ, true>(g, a, s); break;
    case 2: stage_go<T, 2, PX, PY, PZ, true>(g, a, s); break;
    case 3: stage_go<T, 3, PX, PY, PZ, true>(g, a, s); break;
    default: return hipErrorInvalidValue;
    }
    return hipGetLastError();
}

// fn<T, PX, PY, PZ>(g, a, mode, s) for the geometry's periodic axes
#define NYL_STAGE_GEO(fn, T)                              \
    switch (g.px + 2 * g.py + 4 * g.pz) {                 \
    case 0: return fn<T, 0, 0, 0>(g, a, mode, s);         \
    case 1: return fn<T, 1, 0, 0>(g, a, mode, s);         \
    case 2: return fn<T, 0, 1, 0>(g, a, mode, s);         \
    case 3: return fn<T, 1, 1, 0>(g, a, mode, s);         \
    case 4: return fn<T, 0, 0, 1>(g, a, mode, s);         \
    case 5: return fn<T, 1, 0, 1>(g, a, mode, s);         \
    case 6: return fn<T, 0, 1, 1>(g, a, mode, s);         \
    default: return fn<T, 1, 1, 1>(g, a, mode, s);        \
    }

}  // namespace nyl
