// nyl_api.hip -- context, workspace layout and the extern "C" entry points of
// libnyles_hip.so (declared in include/nyles_hip.h).
#include <stdarg.h>
#include <stdio.h>
#include <string.h>

#include <type_traits>
#include <utility>
#include <vector>

#include "nyl_ctx.h"
#include "nyl_march.h"
#include <algorithm>
#include <atomic>
#include <chrono>

using namespace nyl;

namespace {

thread_local char g_err[512] = "";

int fail(int code, const char *fmt, ...) {
    va_list ap;
    va_start(ap, fmt);
    vsnprintf(g_err, sizeof(g_err), fmt, ap);
    va_end(ap);
    return code;
}

}  // namespace

namespace nyl {
int set_error(int code, const char *fmt, ...) {
    va_list ap;
    va_start(ap, fmt);
    vsnprintf(g_err, sizeof(g_err), fmt, ap);
    va_end(ap);
    return code;
}
}  // namespace nyl

namespace {

#define HIPCHK(...)                                                                    \
    do {                                                                               \
        hipError_t e_ = (__VA_ARGS__);                                                 \
        if (e_ != hipSuccess)                                                          \
            return fail(NYL_E_HIP, "%s: %s (%s:%d)", #__VA_ARGS__,                    \
                        hipGetErrorString(e_), __FILE__, __LINE__);                    \
    } while (0)

}  // namespace

namespace {

uint64_t align256(uint64_t v) { return (v + 255) & ~uint64_t(255); }

Geo make_geo(int nx, int ny, int nz, int px, int py, int pz) {
    Geo g;
    g.nx = nx; g.ny = ny; g.nz = nz;
    g.px = px; g.py = py; g.pz = pz;
    g.sy = nx;
    g.sz = (int64_t)nx * ny;
    return g;
}

// core/mgfor/mg_setup.f90:225-307 on one rank: halve x and y until one of
// them equals 2; z (interior) halves alongside.  A level is restricted only
// when all its sizes are even, so that its cells pair up exactly
// (core/mgfor/basicoperators.f90:32-60).  The reference has no rule for a
// level with an odd size (its restriction drops a cell, and on one rank a
// size 3 never reaches 2): here the hierarchy stops at that level, which is
// then solved directly (nyl_coarse.hip).  Grids the reference halves down to
// x or y = 2 get exactly the reference's hierarchy.
int build_hierarchy(nyl_ctx *c) {
    int x = c->d.nx, y = c->d.ny, z = c->d.nz;
    int n = 0;
    c->exact = 0;
    c->lev[n++].g = make_geo(x, y, z, c->g.px, c->g.py, c->g.pz);
    while (!(x == 2 || y == 2)) {
        if ((x & 1) || (y & 1) || (z & 1)) {
            if (n == 1)
                return fail(NYL_E_SIZE,
                            "grid %dx%dx%d: the multigrid needs at least one halving "
                            "(nx, ny and nz even)", c->d.nx, c->d.ny, c->d.nz);
            const Geo &g = c->lev[n - 1].g;
            if (!coarse_fits(g))
                return fail(NYL_E_SIZE,
                            "grid %dx%dx%d: the coarsest multigrid level %dx%dx%d has an odd "
                            "size and more than %d cells along x or %d along y or z (direct "
                            "coarse solve)",
                            c->d.nx, c->d.ny, c->d.nz, x, y, z, CS_MAXX, CS_MAX);
            c->exact = 1;
            break;
        }
        x /= 2; y /= 2; z /= 2;
        if (n >= kMaxLevels) return fail(NYL_E_SIZE, "too many multigrid levels");
        c->lev[n++].g = make_geo(x, y, z, c->g.px, c->g.py, c->g.pz);
    }
    c->nlev = n;
    return NYL_OK;
}

void build_tabs(MGTabs &t) {
    for (int d = 0; d <= 6; d++) {
        t.diag[d] = (double)d;
        t.idiag[d] = d > 0 ? 1.0 / (double)d : 0.0;
    }
    for (int m = 0; m < 8; m++) {
        const int mx = m & 1, my = (m >> 1) & 1, mz = (m >> 2) & 1;
        t.pcoef[m] = 1.0 / (double)((3 + mx) * (3 + my) * (3 + mz));
    }
}


void build_layout(nyl_ctx *c) {
    const uint64_t es = c->mixed ? sizeof(float) : sizeof(double);
    const uint64_t fb = align256((uint64_t)c->ncell * es);
    const uint64_t fb64 = align256((uint64_t)c->ncell * sizeof(double));
    uint64_t off = 0;
    auto take = [&](uint64_t bytes) { uint64_t o = off; off += align256(bytes); return o; };
    for (int s = 0; s < 2; s++)
        for (int f = 0; f < 4; f++) c->state[s][f] = take(fb);
    for (int s = 0; s < 3; s++)
        for (int f = 0; f < 4; f++) c->ds[s][f] = take(fb);
    for (int f = 0; f < 4; f++) c->sb[f] = take(fb);
    c->ke = take(fb);
    for (int f = 0; f < 3; f++) c->vor[f] = take(fb);
    for (int f = 0; f < 3; f++) c->uc[f] = take(fb);
    c->p = take(fb64);
    for (int l = 0; l < c->nlev; l++) {
        const uint64_t lb = (uint64_t)c->lev[l].g.nx * c->lev[l].g.ny * c->lev[l].g.nz *
                            (lev64(c, l) ? sizeof(double) : sizeof(float));
        c->lev[l].x = take(lb);
        c->lev[l].b = take(lb);
        c->lev[l].y = take(lb);
    }
    if (c->mixed) {
        c->mgx = take(fb64);
        c->mgb = take(fb64);
    } else {
        c->mgx = c->lev[0].x;
        c->mgb = c->lev[0].b;
    }
    // block sums: of the reductions (capped), and of the batched march over
    // level 0, which has one per block
    c->partials = take(std::max<uint64_t>(NYL_RED_BLOCKS, b_march_blocks(c->lev[0].g)) *
                       sizeof(double));
    c->result = take(8 * sizeof(double));
    c->ctl = take(sizeof(MGCtl));
    c->ent = take(sizeof(c->cyc_ent));
    c->cs_tab = c->exact ? take(coarse_table_doubles() * sizeof(double)) : 0;
    for (int q = 0; q < c->ntr; q++) {
        c->tst[0][q] = take(fb);
        c->tst[1][q] = take(fb);
        for (int k = 0; k < 3; k++) c->tds[k][q] = take(fb);
        c->tsb[q] = take(fb);
    }
    c->ws_bytes = off;
}

int check_ready(const nyl_ctx *c) {
    if (!c) return fail(NYL_E_ARG, "null context");
    if (!c->ws) return fail(NYL_E_STATE, "workspace not bound (call nyl_bind_workspace)");
    return NYL_OK;
}

int prof_drain(nyl_ctx *c) {
    if (c->prof_used == 0) return NYL_OK;
    HIPCHK(hipEventSynchronize(c->prof_ev[2 * c->prof_used - 1]));
    for (int q = 0; q < c->prof_used; q++) {
        float ms = 0.f;
        HIPCHK(hipEventElapsedTime(&ms, c->prof_ev[2 * q], c->prof_ev[2 * q + 1]));
        c->prof_ms += ms;
    }
    c->prof_used = 0;
    return NYL_OK;
}

// Launch through `fn`; when the kernel class is being profiled, the first
// kernel `fn` launches records its start and end on a pair of events (the
// kernel's own duration) and its algorithmic bytes are counted.
constexpr int kFineLevel = 0x100;   // launch works on the finest multigrid level

template <typename Fn>
int timed_launch(nyl_ctx *c, int cls, double bytes, Fn fn) {
    // a level-1 sweep (two-sweep pass) also belongs to the NYL_K_MG_SWEEP_FINE
    // (NYL_K_MG_SWEEP2_FINE) class
    const int base = cls & 0xff;
    const bool fine = (cls & kFineLevel) != 0;
    const bool on = c->prof_cls == base ||
                    (c->prof_cls == NYL_K_MG_SWEEP_FINE && fine && base == NYL_K_MG_SWEEP) ||
                    (c->prof_cls == NYL_K_MG_SWEEP2_FINE && fine && base == NYL_K_MG_SWEEP2);
    if (on) {
        if (c->prof_used * 2 + 2 > c->prof_nev) {
            const int cap = (int)(sizeof(c->prof_ev) / sizeof(c->prof_ev[0]));
            if (c->prof_nev + 2 <= cap) {
                HIPCHK(hipEventCreate(&c->prof_ev[c->prof_nev]));
                HIPCHK(hipEventCreate(&c->prof_ev[c->prof_nev + 1]));
                c->prof_nev += 2;
            } else {
                int r = prof_drain(c);
                if (r) return r;
            }
        }
        g_launch_events = {c->prof_ev[2 * c->prof_used], c->prof_ev[2 * c->prof_used + 1]};
    }
    const hipError_t e = fn();
    const bool timed = on && g_launch_events.start == nullptr;
    g_launch_events = {nullptr, nullptr};
    HIPCHK(e);
    if (timed) {
        c->prof_used++;
        c->prof_launches++;
        c->prof_bytes += bytes;
    }
    return NYL_OK;
}

#define LAUNCH(cls, bytes, ...)                                                        \
    do {                                                                               \
        int r_ = timed_launch(c, (cls), (double)(bytes), [&]() { return (__VA_ARGS__); }); \
        if (r_) return r_;                                                             \
    } while (0)

double cells(const Geo &g) { return (double)g.nx * g.ny * g.nz; }

// The results reach the host through coherent pinned memory: a one-thread
// kernel stores them there and then a sequence number, and the host polls
// that number instead of a stream synchronisation plus a copy (each host
// round trip of the multigrid loop is on the critical path).  After a
// bounded poll the host falls back to a blocking synchronisation, which also
// reports a failed kernel.
// The final sum that writes the last of the next n results publishes them
// itself (launch_final_sum), one launch fewer per read; read_results then
// only polls.
void arm_publish(nyl_ctx *c, int n) {
    Publish &r = g_publish;
    r.src = reinterpret_cast<const double *>(c->ws + c->result);
    r.n = n;
    r.dst = c->host_dev;
    r.flag = c->host_dev ? reinterpret_cast<uint32_t *>(c->host_dev + 8) : nullptr;
    r.seq = ++c->pub_seq;
    r.consumed = 0;
}

// wait until the results with sequence number seq are in host memory
int wait_published(nyl_ctx *c, uint32_t seq) {
    volatile uint32_t *flag = reinterpret_cast<volatile uint32_t *>(c->host_out + 8);
    const auto t0 = std::chrono::steady_clock::now();
    for (uint64_t it = 1; *flag != seq; it++) {
        if ((it & 1023) == 0 &&
            std::chrono::steady_clock::now() - t0 > std::chrono::milliseconds(50)) {
            HIPCHK(hipStreamSynchronize(c->stream));
            if (*flag != seq) return fail(NYL_E_HIP, "result of the device reduction not published");
            break;
        }
    }
    std::atomic_thread_fence(std::memory_order_acquire);
    return NYL_OK;
}

int read_results(nyl_ctx *c, double *out, int n) {
    const double *src = reinterpret_cast<const double *>(c->ws + c->result);
    Publish &r = g_publish;
    const bool armed = r.consumed && r.dst && r.dst == c->host_dev && r.src == src && r.n == n;
    const uint32_t seq = armed ? r.seq : ++c->pub_seq;
    r = Publish{};
    if (!armed)
        HIPCHK(launch_publish(src, n, c->host_dev, reinterpret_cast<uint32_t *>(c->host_dev + 8),
                              seq, c->stream));
    int rc = wait_published(c, seq);
    if (rc) return rc;
    const volatile double *v = c->host_out;
    for (int q = 0; q < n; q++) out[q] = v[q];
    return NYL_OK;
}

int read_result(nyl_ctx *c, double *out) { return read_results(c, out, 1); }

template <typename T>
StageArgs<T> stage_args(nyl_ctx *c) {
    StageArgs<T> a;
    const int s = c->cur, t = 1 - c->cur;
    a.b = F<T>(c, c->state[s][0]); a.u = F<T>(c, c->state[s][1]);
    a.v = F<T>(c, c->state[s][2]); a.w = F<T>(c, c->state[s][3]);
    a.bn = F<T>(c, c->state[t][0]); a.un = F<T>(c, c->state[t][1]);
    a.vn = F<T>(c, c->state[t][2]); a.wn = F<T>(c, c->state[t][3]);
    a.ox = F<T>(c, c->vor[0]); a.oy = F<T>(c, c->vor[1]); a.oz = F<T>(c, c->vor[2]);
    a.ke = F<T>(c, c->ke);
    a.idx2 = c->d.idx2; a.idy2 = c->d.idy2; a.idz2 = c->d.idz2;
    a.d0b = F<T>(c, c->ds[0][0]); a.d0u = F<T>(c, c->ds[0][1]);
    a.d0v = F<T>(c, c->ds[0][2]); a.d0w = F<T>(c, c->ds[0][3]);
    a.d1b = F<T>(c, c->ds[1][0]); a.d1u = F<T>(c, c->ds[1][1]);
    a.d1v = F<T>(c, c->ds[1][2]); a.d1w = F<T>(c, c->ds[1][3]);
    a.tb = a.tu = a.tv = a.tw = nullptr;
    a.sbb = F<T>(c, c->sb[0]); a.sbu = F<T>(c, c->sb[1]);
    a.sbv = F<T>(c, c->sb[2]); a.sbw = F<T>(c, c->sb[3]);
    a.dz = c->d.dz;
    a.c = 0.0;
    a.c2 = 0.0;
    a.vcx = a.vcy = a.vcz = 0.0;
    a.visc = 0;
    a.flags = 0;
    a.upw_a = c->d.upwind_a;
    a.upw_vf = c->d.upwind_vf;
    return a;
}

template <typename T>
void set_tendency_out(nyl_ctx *c, StageArgs<T> &a, int slot) {
    a.tb = F<T>(c, c->ds[slot][0]); a.tu = F<T>(c, c->ds[slot][1]);
    a.tv = F<T>(c, c->ds[slot][2]); a.tw = F<T>(c, c->ds[slot][3]);
}

// ---- the levels of a V-cycle ------------------------------------------------
// How the passes of a level run:
//   cycle   from the first level whose whole remainder fits one workgroup
//           (cells <= CYC_CELLS and the LDS): k_mg_cycle, one launch
//   fused   other levels of at most NYL_FUSED_MAX_CELLS cells: k_mg_down and
//           k_mg_up, 4^3 tiles (32^3: 5.9 us each, where a march takes 7.5
//           and 10.4)
//   tiled   nx % 64 == 0, ny % 8 == 0 and one type with the level below:
//           k_mg_sweep25 + k_mg_restrict25, k_mg_prolong25 + k_mg_sweep2t
//   march   any other level: k_mg_march down and up
// Every level's first sweep is written by the restriction from the level
// above.  The correction of a level ends in its y, of a tiled level and of a
// coarsest level in its x.
#ifndef NYL_FUSED_MAX_CELLS
#define NYL_FUSED_MAX_CELLS 32768
#endif
// cells of the largest level of the cycle
#ifndef CYC_CELLS
#define CYC_CELLS 4096
#endif

bool fused_level(const nyl_ctx *c, int l) {
    return l >= 1 && l <= c->nlev - 2 && cells(c->lev[l].g) <= NYL_FUSED_MAX_CELLS &&
           fused_fits(c->lev[l].g, c->lev[l + 1].g);
}

bool tiled_level(const nyl_ctx *c, int l) {
    return l <= c->nlev - 2 && restrict25_fits(c->lev[l].g) && lev64(c, l) == lev64(c, l + 1) &&
           sweep2x_blocks(c->lev[l].g, lev64(c, l) ? 8 : 4) <= NYL_RED_BLOCKS;
}

// offset of the buffer that holds level l's correction (l >= 1)
uint64_t sol_off(const nyl_ctx *c, int l) {
    if (l == c->nlev - 1) return c->lev[l].x;
    if (l >= c->t0 || fused_level(c, l)) return c->lev[l].y;
    return tiled_level(c, l) ? c->lev[l].x : c->lev[l].y;
}

// first level of the cycle: the largest that fits (never the finest); its
// position table is uploaded when the workspace is bound
int cycle_first(nyl_ctx *c) {
    Geo g[kMaxLevels];
    for (int l = 0; l < c->nlev; l++) g[l] = c->lev[l].g;
    int t0 = c->nlev;
    for (int l = c->nlev - 1; l >= 1; l--) {
        CycleArgs a;
        CycleEnt ent[CYC_ENT];
        // A direct solve alone pays only while it is small.  us per V-cycle of a
        // two-level solve, in one workgroup / in its own three launches: 5^3
        // 28.6 / 33.9, 9^3 31.5 / 35.1, 13x9x9 33.3 / 35.4, 15x15x7 36.6 / 37.3,
        // 13^3 40.2 / 36.7, 25x15x7 46.7 / 40.2, 15^3 46.8 / 37.6.  The line is
        // at one cell per thread; up to 1600 cells the two are 1 to 2 us apart.
        if (l == c->nlev - 1 && c->exact && cells(g[l]) > 1024) break;
        if (cells(g[l]) > CYC_CELLS ||
            !cycle_layout(a, ent, g, l, c->nlev, lev64(c, l) ? 8 : 4, c->exact != 0,
                          c->d.mg_omega, c->tabs))
            break;
        t0 = l;
        c->cyc = a;
        memcpy(c->cyc_ent, ent, sizeof(ent));
    }
    return t0;
}

template <typename T, typename TC>
MarchArgs<T, TC> march_args(nyl_ctx *c, int l, uint64_t src, uint64_t dst) {
    MarchArgs<T, TC> a = {};
    const Level &f = c->lev[l], &q = c->lev[l + 1 < c->nlev ? l + 1 : l];
    a.g = f.g;
    a.gc = q.g;
    a.src = F<T>(c, src);
    a.dst = F<T>(c, dst);
    a.b = F<T>(c, f.b);
    a.omega = c->d.mg_omega;
    a.tab = c->tabs;
    return a;
}

// calls fn(T, TC) with values of the types of levels l and l + 1
template <typename Fn>
int with_types(const nyl_ctx *c, int l, Fn fn) {
    const bool f64 = lev64(c, l), c64 = lev64(c, l + 1);
    if (f64 && c64) return fn(double(), double());
    if (!f64 && c64) return fn(float(), double());
    if (!f64) return fn(float(), float());
    return fail(NYL_E_STATE, "FP64 level above an FP32 level");
}

double elem(const nyl_ctx *c, int l) { return lev64(c, l) ? sizeof(double) : sizeof(float); }

// level l's second pre-sweep (y -> x) and the restriction into level l + 1
int level_down(nyl_ctx *c, int l) {
    const Level &f = c->lev[l], &q = c->lev[l + 1];
    const double om = c->d.mg_omega, n = cells(f.g) * elem(c, l);
    return with_types(c, l, [&](auto t, auto tc) -> int {
        using T = decltype(t);
        using TC = decltype(tc);
        if (fused_level(c, l)) {
            LAUNCH(NYL_K_MG_SWEEP, 3 * n + 2 * cells(q.g) * sizeof(TC),
                   launch_mg_down<T, TC>(f.g, q.g, F<T>(c, f.y), F<T>(c, f.b), F<T>(c, f.x),
                                         F<TC>(c, q.b), F<TC>(c, q.y), om, c->tabs, c->stream));
            return NYL_OK;
        }
        if constexpr (std::is_same<T, TC>::value) {
            if (tiled_level(c, l)) {
                LAUNCH(NYL_K_MG_SWEEP, 3 * n,
                       launch_mg_sweep25<T>(f.g, F<T>(c, f.y), F<T>(c, f.x), F<T>(c, f.b), om,
                                            c->tabs, nullptr, nullptr, c->stream));
                LAUNCH(NYL_K_MG_RESTRICT, 2.25 * n,
                       launch_mg_restrict25<T, T>(f.g, q.g, F<T>(c, f.x), F<T>(c, f.b),
                                                  F<T>(c, q.b), F<T>(c, q.x), c->tabs, c->stream,
                                                  F<T>(c, q.y), om));
                return NYL_OK;
            }
        }
        MarchArgs<T, TC> a = march_args<T, TC>(c, l, f.y, f.x);
        a.bc = F<TC>(c, q.b);
        a.yc = F<TC>(c, q.y);
        LAUNCH(NYL_K_MG_SWEEP, 3 * n + 2 * cells(q.g) * sizeof(TC),
               (launch_march_down<T, TC>(a, c->stream)));
        return NYL_OK;
    });
}

// level l's prolongation from level l + 1 and both post-sweeps.  Level 0:
// from y (both pre-sweeps were done there) into x, unless the solve has
// stopped (gate).
// The march reads x and b once and writes once; the tiled form's
// prolongation writes and its two-sweep pass reads the level once more.
// At 256^3 the march takes 57 us in FP32 and 113 us in FP64 where the tiled
// launches take 68 and 148; at 128^3 they are even (18 and 17, 22 and 23),
// and below that the tiled kernels' shorter prologues win (64x32x32: 8.3
// against 10.8 us).
#ifndef NYL_UP_MARCH_CELLS
#define NYL_UP_MARCH_CELLS (1 << 22)
#endif
int level_up(nyl_ctx *c, int l, const int *gate = nullptr) {
    const Level &f = c->lev[l], &q = c->lev[l + 1];
    const double om = c->d.mg_omega, n = cells(f.g) * elem(c, l);
    const uint64_t qx = sol_off(c, l + 1);
    return with_types(c, l, [&](auto t, auto tc) -> int {
        using T = decltype(t);
        using TC = decltype(tc);
        if (l > 0 && fused_level(c, l)) {
            LAUNCH(NYL_K_MG_PROLONG, 3 * n + cells(q.g) * sizeof(TC),
                   launch_mg_up<T, TC>(f.g, q.g, F<T>(c, f.x), F<TC>(c, qx), F<T>(c, f.b),
                                       F<T>(c, f.y), om, c->tabs, c->stream));
            return NYL_OK;
        }
        const bool tiled = tiled_level(c, l);
        if constexpr (std::is_same<T, TC>::value) {
            if (tiled && (l > 0 || cells(f.g) < NYL_UP_MARCH_CELLS)) {
                // level 0: y += P(xc) in place; else y = x + P(xc)
                T *x = F<T>(c, f.x), *y = F<T>(c, f.y);
                LAUNCH(NYL_K_MG_PROLONG, 2.125 * n,
                       launch_mg_prolong25<T, T>(f.g, q.g, l > 0 ? x : y, F<T>(c, qx), c->tabs,
                                                 c->stream, l > 0 ? y : nullptr));
                LAUNCH(NYL_K_MG_SWEEP2 | (l == 0 ? kFineLevel : 0), 3 * n,
                       launch_mg_sweep2x25<T>(f.g, y, x, F<T>(c, f.b), om, c->tabs, c->stream,
                                              nullptr, nullptr, gate));
                return NYL_OK;
            }
        }
        MarchArgs<T, TC> a = march_args<T, TC>(c, l, l > 0 ? f.x : f.y, l > 0 ? f.y : f.x);
        a.xc = F<TC>(c, qx);
        a.gate = gate;
        LAUNCH(l == 0 ? (NYL_K_MG_SWEEP2 | kFineLevel) : NYL_K_MG_PROLONG,
               3 * n + cells(q.g) * sizeof(TC),
               (launch_march_up<T, TC>(a, c->stream)));
        return NYL_OK;
    });
}

// the coarsest level's step of a V-cycle outside the cycle: mgfor's smooth()
// (its second sweep, the first was written by the restriction), or the
// direct solve of a level with an odd size
int coarsest(nyl_ctx *c) {
    const int L = c->nlev - 1;
    const Level &f = c->lev[L];
    if (!c->exact) {
        if (lev64(c, L))
            LAUNCH(NYL_K_MG_SWEEP, 3 * cells(f.g) * sizeof(double),
                   launch_mg_sweep<double>(f.g, F<double>(c, f.y), F<double>(c, f.x),
                                           F<double>(c, f.b), c->d.mg_omega, c->tabs, c->stream));
        else
            LAUNCH(NYL_K_MG_SWEEP, 3 * cells(f.g) * sizeof(float),
                   launch_mg_sweep<float>(f.g, F<float>(c, f.y), F<float>(c, f.x),
                                          F<float>(c, f.b), c->d.mg_omega, c->tabs, c->stream));
        return NYL_OK;
    }
    CoarseArgs a;
    a.g = f.g;
    a.b = F<double>(c, f.b);
    a.s = F<double>(c, f.y);
    a.x = F<double>(c, f.x);
    a.tab = F<double>(c, c->cs_tab);
    LAUNCH(NYL_K_MG_COARSE, 4 * cells(f.g) * sizeof(double), launch_coarse_solve(a, c->stream));
    return NYL_OK;
}

// Levels 1 and below of a V-cycle (core/mgfor/solvers.f90:35-55), from the
// right-hand side and first sweep of level 1.  fin: the test that is waiting
// for its sum, run beside the cycle (or before, where there is no cycle).
int coarse_levels(nyl_ctx *c, const CtlArgs *fin) {
    const int L = c->nlev, t0 = c->t0;
    const int last = t0 < L ? t0 : L - 1;   // levels [1, last) run here
    int rc;
    if (fin && t0 >= L) HIPCHK(launch_ctl(*fin, c->stream));
    for (int l = 1; l < last; l++)
        if ((rc = level_down(c, l))) return rc;
    if (t0 < L) {
        const Level &f = c->lev[t0];
        double bytes = 0.0;
        for (int l = t0; l < L; l++) bytes += 3.0 * cells(c->lev[l].g) * elem(c, l);
        if (lev64(c, t0))
            LAUNCH(NYL_K_MG_COARSE, bytes,
                   launch_mg_cycle<double>(c->cyc, F<double>(c, f.b), F<double>(c, f.y),
                                           F<double>(c, f.x), fin, c->stream));
        else
            LAUNCH(NYL_K_MG_COARSE, bytes,
                   launch_mg_cycle<float>(c->cyc, F<float>(c, f.b), F<float>(c, f.y),
                                          F<float>(c, f.x), fin, c->stream));
    } else if ((rc = coarsest(c))) {
        return rc;
    }
    for (int l = last - 1; l >= 1; l--)
        if ((rc = level_up(c, l))) return rc;
    return NYL_OK;
}

// Level 0's pre-smoothing as one march with the restriction in it (x, b read
// and y written once), or as the tiled two-sweep pass and the tiled
// restriction (y and b read once more).  One march: levels that do not tile,
// FP64 from 4M cells, and FP32 whose three fields exceed the 256 MB cache.
// us of pre-smoothing + restriction + post-smoothing, two passes / one: FP64
// 256^3 270 / 253, 128x128x256 75 / 71, 128^3 45.7 / 48.1; FP32 256x256x512
// 323 / 279, 256x256x384 210 / 207, 320x256x256 163 / 181, 256^3 131 / 135;
// not tiled (two marches / one) FP64 160^3 78 / 72, 96^3 36 / 35, FP32
// 200x120x56 39.3 / 38.1, 240^3 125 / 124.
bool pre_tiled(const nyl_ctx *c) {
    const double n = cells(c->lev[0].g);
    return tiled_level(c, 0) &&
           (lev64(c, 0) ? n < (1 << 22) : 3.0 * n * sizeof(float) <= 256.0 * (1 << 20));
}

// The block sums of level 0's residual norm: those of the pre-smoothing pass
// with a norm.  The norm alone (resid_norm) sums the same cells in the same
// order, so a test gives the same bits whichever of the two the guess of a
// solve chose.  That fixes its blocks: at 256^3 it takes 59.4 us in FP64 where
// blocks of its own choice took 53.1, and 27.8 in FP32 as before.  capped: more
// blocks than partial sums, k_resnorm2 instead.
struct NormForm {
    MarchGrid grid;
    bool tiled, capped;
    int np;
};
NormForm norm_form(const nyl_ctx *c) {
    const Geo &g = c->lev[0].g;
    const int es = lev64(c, 0) ? 8 : 4;
    NormForm f = {};
    f.tiled = pre_tiled(c);
    if (f.tiled) {
        const int kz = sweep2x_kz(g, es);
        f.grid = {64, g.nx / 64, g.ny / 8, g.nz / kz, kz};
    } else {
        f.grid = march_pre_grid(g, es);
    }
    f.capped = f.grid.blocks() > NYL_RED_BLOCKS;
    f.np = f.capped ? red_blocks((int64_t)cells(g)) : f.grid.blocks();
    return f;
}

// Both pre-smoothing sweeps of level 0 into its y and the restriction into
// level 1.  zero: from a zero solution; else from x, with the block sums of
// its residual norm in the partials (their number in *np).
int pre_smooth(nyl_ctx *c, bool zero, int *np) {
    const Level &f = c->lev[0], &q = c->lev[1];
    const double om = c->d.mg_omega, n = cells(f.g) * elem(c, 0);
    double *part = F<double>(c, c->partials);
    const NormForm nf = norm_form(c);
    if (!zero) *np = nf.np;
    return with_types(c, 0, [&](auto t, auto tc) -> int {
        using T = decltype(t);
        using TC = decltype(tc);
        if constexpr (std::is_same<T, TC>::value) {
            if (nf.tiled) {
                if (zero) {
                    // (not in the fine-level class of the roofline: it reads one field)
                    LAUNCH(NYL_K_MG_SWEEP2, 2 * n,
                           launch_mg_sweep2x25<T>(f.g, nullptr, F<T>(c, f.y), F<T>(c, f.b), om,
                                                  c->tabs, c->stream));
                } else {
                    LAUNCH(NYL_K_MG_SWEEP2 | kFineLevel, 3 * n,
                           launch_mg_sweep2x25<T>(f.g, F<T>(c, f.x), F<T>(c, f.y), F<T>(c, f.b),
                                                  om, c->tabs, c->stream, part));
                }
                LAUNCH(NYL_K_MG_RESTRICT, 2.25 * n,
                       launch_mg_restrict25<T, T>(f.g, q.g, F<T>(c, f.y), F<T>(c, f.b),
                                                  F<T>(c, q.b), F<T>(c, q.x), c->tabs, c->stream,
                                                  F<T>(c, q.y), om));
                return NYL_OK;
            }
        }
        MarchArgs<T, TC> a = march_args<T, TC>(c, 0, f.x, f.y);
        if (zero) a.src = nullptr;
        else a.partials = part;
        a.bc = F<TC>(c, q.b);
        a.yc = F<TC>(c, q.y);
        if (!zero && nf.capped) {
            if constexpr (std::is_same<T, double>::value) {
                LAUNCH(NYL_K_RESNORM, 2 * n,
                       launch_resnorm2<double>(f.g, a.src, a.b, c->tabs, part, nullptr, c->stream));
                a.partials = nullptr;
            } else {
                return fail(NYL_E_SIZE, "level 1 is too wide for the residual norm");
            }
        }
        LAUNCH(NYL_K_MG_SWEEP2 | (zero ? 0 : kFineLevel),
               (zero ? 2 : 3) * n + 2 * cells(q.g) * sizeof(TC),
               (launch_march_pre<T, TC>(a, c->stream)));
        return NYL_OK;
    });
}

// the residual norm of level 0's x alone, block sums in the partials
template <typename T>
int resid_norm(nyl_ctx *c, int *np) {
    const Level &f = c->lev[0];
    MarchArgs<T, T> a = march_args<T, T>(c, 0, f.x, f.y);
    a.partials = F<double>(c, c->partials);
    const NormForm nf = norm_form(c);
    *np = nf.np;
    if (nf.capped)
        LAUNCH(NYL_K_RESNORM, 2 * cells(f.g) * sizeof(T),
               launch_resnorm2<T>(f.g, a.src, a.b, c->tabs, a.partials, nullptr, c->stream));
    else
        LAUNCH(NYL_K_RESNORM, 2 * cells(f.g) * sizeof(T),
               launch_march_norm<T>(a, nf.grid, nf.tiled, c->stream));
    return NYL_OK;
}

void fill_stats(nyl_ctx *c, nyl_mg_stats *st, int nite, double res, double normb) {
    c->total_cycles += nite;
    if (st) {
        st->nite = nite;
        st->res = res;
        st->normb = normb;
        st->total_cycles = c->total_cycles;
    }
}

// ---- the solve loops ---------------------------------------------------------
// mgfor tests the residual after every V-cycle (core/mgfor/solvers.f90:8-33).
// Waiting for each test on the host left the GPU idle for 10 to 20 us per
// V-cycle.  Here the tests run on the device (CtlArgs): the V-cycles that the
// last solves at the same place of a step needed are enqueued without a wait,
// and one that follows the stopping test leaves the solution as it is (its
// last pass is gated).  Both forms of a test sum the same cells in the same
// order (norm_form), so the result does not depend on the guess; the host
// reads the sums of all tests once and takes the same decisions from them.
// When the guess was too low, V-cycles follow one at a time.

// mixed: squared reduction of one inner solve, its most V-cycles (see mg_solve_mixed)
constexpr double kInnerRed2 = 1e-6;
constexpr int kInnerMax = 8;

CtlArgs ctl_args(nyl_ctx *c, int kind, int np) {
    CtlArgs a = {};
    a.ctl = F<MGCtl>(c, c->ctl);
    a.partials = F<double>(c, c->partials);
    a.np = np;
    a.kind = kind;
    a.slot = -1;
    a.tol = c->d.mg_tol;
    a.ncell = cells(c->lev[0].g);
    a.inner_red = kInnerRed2;
    a.inner_max = kInnerMax;
    return a;
}

// publish the first n sums of the tests with this launch
void ctl_publish(nyl_ctx *c, CtlArgs &a, int n) {
    a.dst = c->host_dev + kHostCtl;
    a.flag = reinterpret_cast<uint32_t *>(c->host_dev + 8);
    a.seq = ++c->pub_seq;
    a.nhist = n;
}

// the published results: normb and the sums of the tests
int ctl_read(nyl_ctx *c, double *normb, double *hist, int n) {
    int rc = wait_published(c, c->pub_seq);
    if (rc) return rc;
    const volatile double *v = c->host_out + kHostCtl;
    *normb = v[0];
    for (int q = 0; q < n; q++) hist[q] = v[2 + q];
    return NYL_OK;
}

// most tests between two reads
constexpr int kMaxAhead = CTL_HIST - 8;

// The guess of a solve (or of an outer step of a mixed one): the fewer of the
// V-cycles the last two at its place needed, those of the solves outside a
// step where there was none, `other` where nothing is known.  One V-cycle too
// many costs a V-cycle, one too few a host read, so the guess is low; `ends`:
// the last one stopped at the guess, so that the test there is expected to be
// the last and evaluates the norm alone.
struct Guess {
    int n;
    bool ends;
};
Guess guess_of(const nyl_ctx *c, int site, int j, int other) {
    const Pred *p = &c->pred[site][j];
    if (p->last < 0) p = &c->pred[0][j];
    if (p->last < 0) return {other, false};
    const int n = p->before >= 0 ? std::min(p->last, p->before) : p->last;
    return {n, n > 0 && p->last == n};
}
void set_guess(nyl_ctx *c, int site, int j, int n) {
    Pred &p = c->pred[site][j];
    p.before = p.last;
    p.last = n;
}

// core/mgfor/solvers.f90:8-33 with normresidual (core/mgfor/operators.f90:81-96)
int mg_solve_fp64(nyl_ctx *c, nyl_mg_stats *st, int site) {
    Level &f = c->lev[0];
    const int maxite = c->d.mg_maxite > 1 ? c->d.mg_maxite : 1;   // one V-cycle at least
    const int *gate = &F<MGCtl>(c, c->ctl)->stop;
    int rc;
    HIPCHK(launch_norm2<double>(f.g, F<double>(c, f.b), F<double>(c, c->partials), nullptr,
                                c->stream));
    HIPCHK(launch_ctl(ctl_args(c, CTL_NORMB, red_blocks((int64_t)cells(f.g))), c->stream));
    double normb = 0.0, res = 0.0, hist[CTL_HIST];
    int done = 0;    // V-cycles enqueued
    const Guess gs = guess_of(c, site, 0, 0);
    int guess = gs.n;
    bool pre = false;   // the sweeps (and test) of V-cycle done + 1 are enqueued
    for (;;) {
        const int first = done;   // V-cycles before the first test of this round
        int nt = 0;               // tests of this round
        const int to = std::min(std::min(guess, maxite), first + kMaxAhead);
        while (done < to) {
            CtlArgs t;
            if (!pre) {
                int np = 0;
                if ((rc = pre_smooth(c, false, &np))) return rc;
                t = ctl_args(c, CTL_TEST, np);
                t.slot = nt++;
            }
            if ((rc = coarse_levels(c, pre ? nullptr : &t))) return rc;
            if ((rc = level_up(c, 0, gate))) return rc;
            pre = false;
            done++;
        }
        CtlArgs t = ctl_args(c, CTL_NONE, 0);
        if (done < maxite) {
            // the test after the last V-cycle: the norm alone where the solve
            // is expected to stop, else with the next V-cycle's sweeps
            int np = 0;
            const bool ends = first == 0 && gs.ends;
            if (ends) rc = resid_norm<double>(c, &np);
            else rc = pre_smooth(c, false, &np);
            if (rc) return rc;
            pre = !ends;
            t = ctl_args(c, CTL_TEST, np);
            t.slot = nt++;
        }
        ctl_publish(c, t, nt);
        HIPCHK(launch_ctl(t, c->stream));
        if ((rc = ctl_read(c, &normb, hist, nt))) return rc;
        // the tests in order: test q follows V-cycle first + q (the first round
        // and those after a norm), or first + 1 + q when the round began with
        // the V-cycle of a test already read
        const int tests_from = done < maxite ? done - (nt - 1) : done - nt;
        int stop = -1;
        for (int q = 0; q < nt && stop < 0; q++) {
            res = normb > 0.0 ? hist[q] / normb : 0.0;
            if (res < c->d.mg_tol) stop = tests_from + q;
        }
        if (stop >= 0) {
            done = stop;
            break;
        }
        if (done >= maxite) break;
        guess = done + 1;
    }
    set_guess(c, site, 0, done);
    fill_stats(c, st, done, res, normb);
    return NYL_OK;
}

// Mixed precision: iterative refinement with the stop rule of mgfor's solve.
// The compatibility of the singular Neumann/periodic problem is enforced in
// FP64 first: one pass sums b and b**2, the mean is removed from b inside
// every outer residual and |b - mean|**2 is the norm of the stop test (the
// discrete divergence sums to zero up to rounding, so this changes nothing
// measurable, but a right-hand side with a mean could not converge).  An
// outer step computes r = (b - mean) - A x in
// FP64 and solves A e = r from e = 0 with FP32 V-cycles under mgfor's loop:
// before each further V-cycle the squared residual r - A e = b - A(x + e),
// evaluated in FP32 and summed in FP64, is tested against tol*|b|^2 (fused
// into that V-cycle's pre-smoothing, as in the FP64 path).  Then x += e in FP64
// and the FP64 residual confirms the stop (or starts another outer step).
// The V-cycle count follows mgfor's rule (nite, maxite).
// One inner solve resolves a limited reduction of r: A e of a smooth e
// cancels to ~eps32*(n/pi)^2 of its terms, so below that the FP32 residual
// norm is rounding noise and the FP32 e stops improving.  Hence an outer step
// whose tolerance asks for more than kInnerRed2*|r|^2 tests the inner
// residual against kInnerRed2*|r|^2 instead and runs at most kInnerMax
// V-cycles; the FP64 residual decides.  At mgfor's tolerance (1e-6) the
// tolerance is the target and the V-cycle count is that of the FP64 solve.
// Each outer step is enqueued whole, its V-cycles as guessed, with the add
// and the next FP64 residual: the add is gated by the inner loop's stop, so
// that a guess that was too low leaves x, and the next residual, as they
// were.
int mg_solve_mixed(nyl_ctx *c, nyl_mg_stats *st, int site) {
    Level &f = c->lev[0];
    const int maxite = c->d.mg_maxite > 1 ? c->d.mg_maxite : 1;
    MGCtl *ctl = F<MGCtl>(c, c->ctl);
    double *xo = F<double>(c, c->mgx), *bo = F<double>(c, c->mgb);
    float *e = F<float>(c, f.x);
    const double ncell = cells(f.g), tol = c->d.mg_tol;
    int rc;
    HIPCHK(launch_sum_sumsq(f.g, bo, F<double>(c, c->partials), c->stream));
    HIPCHK(launch_ctl(ctl_args(c, CTL_SHIFT, sumsq_blocks((int64_t)ncell)), c->stream));
    // FP64 residual of x into r, its test into hist[slot]
    auto outer = [&](int slot, bool publish) -> int {
        MarchArgs<double, double> a = {};
        a.g = a.gc = f.g;
        a.src = xo;
        a.b = bo;
        a.tab = c->tabs;
        a.partials = F<double>(c, c->partials);
        a.rout = F<float>(c, f.b);
        a.shift = &ctl->shift;
        LAUNCH(NYL_K_RESNORM, (2 * sizeof(double) + sizeof(float)) * ncell,
               launch_march_outer(a, c->stream));
        CtlArgs t = ctl_args(c, CTL_OUTER, march_grid(f.g, march_resident(8, MS_FIELD, 0, false), false).blocks());
        t.slot = slot;
        if (publish) ctl_publish(c, t, slot + 1);
        HIPCHK(launch_ctl(t, c->stream));
        return NYL_OK;
    };
    auto add = [&](const int *gate) -> int {
        LAUNCH(NYL_K_MG_UPDATE, (2 * sizeof(double) + sizeof(float)) * ncell,
               launch_add_correction<float>(f.g, xo, e, gate, c->stream));
        return NYL_OK;
    };
    double normb = 0.0, res = 0.0, hist[CTL_HIST];
    auto relative = [&](double s) { return normb > 0.0 ? s / normb : 0.0; };
    // the first outer residual is read with the first outer step's tests,
    // unless the solve is expected to stop at it
    bool have_res = guess_of(c, site, 0, 1).n == 0;
    if ((rc = outer(0, have_res))) return rc;
    if (have_res) {
        if ((rc = ctl_read(c, &normb, hist, 1))) return rc;
        res = relative(hist[0]);
    }
    int nite = 0;
    bool at_max = false;
    for (int j = 0;; j++) {
        if (have_res && (res < tol || at_max)) {
            if (j < kPredOuter) set_guess(c, site, j, 0);
            break;
        }
        const Guess gs = guess_of(c, site, std::min(j, kPredOuter - 1), 1);
        const int guess = std::max(gs.n, 1);
        int k = 0;            // V-cycles of this inner loop enqueued
        bool open = true;     // the inner loop has not stopped
        bool pre = false;     // the sweeps (and test) of V-cycle k + 1 are enqueued
        bool first = true, added = false;
        while (open) {
            int nt = j == 0 && !have_res ? 1 : 0;   // hist[0] is the first outer residual
            const int in0 = nt;
            int kq[CTL_HIST];                       // V-cycles before each test
            const int to = std::min(std::min(std::max(guess, k + 1), maxite - nite), k + kMaxAhead);
            while (k < to) {
                CtlArgs t;
                bool test = false;
                if (!pre) {
                    int np = 0;
                    if ((rc = pre_smooth(c, k == 0, &np))) return rc;
                    if (k > 0) {
                        test = true;
                        t = ctl_args(c, CTL_INNER, np);
                        t.k = k;
                        kq[nt] = k;
                        t.slot = nt++;
                    }
                }
                if ((rc = coarse_levels(c, test ? &t : nullptr))) return rc;
                if ((rc = level_up(c, 0, &ctl->stop))) return rc;
                pre = false;
                k++;
            }
            const bool max_now = nite + k >= maxite;
            const bool ends = max_now || (first && gs.ends);   // expected to stop here
            if (!max_now) {
                int np = 0;
                if (ends) rc = resid_norm<float>(c, &np);
                else rc = pre_smooth(c, false, &np);
                if (rc) return rc;
                pre = !ends;
                CtlArgs t = ctl_args(c, CTL_INNER, np);
                t.k = k;
                kq[nt] = k;
                t.slot = nt++;
                if (!ends) ctl_publish(c, t, nt);
                HIPCHK(launch_ctl(t, c->stream));
            }
            int last = -1;   // hist entry of the next outer residual
            if (ends) {
                if ((rc = add(max_now ? &ctl->outer_stop : &ctl->no_add))) return rc;
                last = nt++;
                if ((rc = outer(last, true))) return rc;
            }
            if ((rc = ctl_read(c, &normb, hist, nt))) return rc;
            if (!have_res) {
                res = relative(hist[0]);
                have_res = true;
                if (res < tol) {   // nothing was to be done
                    k = 0;
                    open = false;
                    break;
                }
            }
            const bool rel = res * kInnerRed2 > tol;
            const double target = rel ? res * kInnerRed2 : tol;
            for (int q = in0; q < (last >= 0 ? last : nt) && open; q++) {
                const double rin = relative(hist[q]);
                if (rin < target || (rel && kq[q] >= kInnerMax)) {
                    k = kq[q];
                    open = false;
                }
            }
            if (max_now) open = false;
            if (!open && last >= 0) {
                added = true;
                res = relative(hist[last]);
            }
            first = false;
        }
        if (k == 0) {   // the first outer residual was below the tolerance
            set_guess(c, site, 0, 0);
            break;
        }
        nite += k;
        at_max = nite >= maxite;
        if (j < kPredOuter) set_guess(c, site, j, k);
        if (!added) {
            if ((rc = add(nullptr)) || (rc = outer(0, true))) return rc;
            if ((rc = ctl_read(c, &normb, hist, 1))) return rc;
            res = relative(hist[0]);
        }
    }
    fill_stats(c, st, nite, res, normb);
    return NYL_OK;
}

// site: the place of the solve in a step (1..3), 0 outside a step
int mg_solve(nyl_ctx *c, nyl_mg_stats *st, int site) {
    return c->mixed ? mg_solve_mixed(c, st, site) : mg_solve_fp64(c, st, site);
}

template <typename T>
DiagArgs<T> diag_args(nyl_ctx *c) {
    DiagArgs<T> a;
    const int s = c->cur;
    a.u = F<T>(c, c->state[s][1]); a.v = F<T>(c, c->state[s][2]);
    a.w = F<T>(c, c->state[s][3]);
    a.Ux = F<T>(c, c->uc[0]); a.Uy = F<T>(c, c->uc[1]); a.Uz = F<T>(c, c->uc[2]);
    a.ox = F<T>(c, c->vor[0]); a.oy = F<T>(c, c->vor[1]); a.oz = F<T>(c, c->vor[2]);
    a.ke = F<T>(c, c->ke);
    a.idx2 = c->d.idx2; a.idy2 = c->d.idy2; a.idz2 = c->d.idz2;
    a.fpar = c->d.fparameter > 0.0 ? c->d.fparameter : 0.0;
    return a;
}

template <typename T>
int apply_op_t(nyl_ctx *c, int op) {
    const int s = c->cur;
    T *u = F<T>(c, c->state[s][1]), *v = F<T>(c, c->state[s][2]), *w = F<T>(c, c->state[s][3]);
    switch (op) {
    case NYL_OP_U_FROM_U:
        HIPCHK(launch_diag<T>(c->g, diag_args<T>(c), 1, c->stream));
        break;
    case NYL_OP_DIV:
        LAUNCH(NYL_K_DIV, (3 * sizeof(T) + sizeof(double)) * cells(c->g),
               launch_div<T, double>(c->g, u, v, w, c->d.idx2, c->d.idy2, c->d.idz2,
                                     F<double>(c, c->mgb), c->stream));
        break;
    case NYL_OP_CORRECT:
        LAUNCH(NYL_K_CORRECT, (6 * sizeof(T) + sizeof(double)) * cells(c->g),
               launch_correct<T, double>(c->g, u, v, w, F<double>(c, c->mgx), c->d.dx2,
                                         c->stream));
        break;
    case NYL_OP_VORTICITY:
        HIPCHK(launch_diag<T>(c->g, diag_args<T>(c), 2, c->stream));
        break;
    case NYL_OP_KINENERGY:
        HIPCHK(launch_diag<T>(c->g, diag_args<T>(c), 4, c->stream));
        break;
    case NYL_OP_PRESSURE:
        HIPCHK(launch_pressure<double, double>(c->g, F<double>(c, c->mgx), c->d.dx2,
                                               F<double>(c, c->p), c->stream));
        break;
    default:
        return fail(NYL_E_ARG, "unknown op %d", op);
    }
    return NYL_OK;
}

int apply_op(nyl_ctx *c, int op) {
    return c->mixed ? apply_op_t<float>(c, op) : apply_op_t<double>(c, op);
}

// core/model_les.py:97-127 (halo fills are implicit in the wrapped reads)
template <typename T>
int diagnose_t(nyl_ctx *c, nyl_mg_stats *st, int site) {
    int rc;
    if ((rc = apply_op_t<T>(c, NYL_OP_DIV))) return rc;
    if ((rc = mg_solve(c, st, site))) return rc;
    if ((rc = apply_op_t<T>(c, NYL_OP_CORRECT))) return rc;
    // vorticity and ke (not in the linear model, core/model_les.py:122-127);
    // U is not stored (the stage kernel recomputes it, NYL_OP_U_FROM_U fills
    // it on demand)
    if (c->d.model != NYL_MODEL_LINEAR)
        LAUNCH(NYL_K_DIAG, 7 * cells(c->g) * sizeof(T),
               launch_diag<T>(c->g, diag_args<T>(c), 6, c->stream));
    return NYL_OK;
}

int diagnose(nyl_ctx *c, nyl_mg_stats *st, int site) {
    return c->mixed ? diagnose_t<float>(c, st, site) : diagnose_t<double>(c, st, site);
}

// words of HBM traffic per cell of each stage-kernel mode: reads b,u,v,w,
// vor(3), ke plus the mode's extra inputs; writes the mode's outputs
double stage_words(int mode) {
    switch (mode) {
    case 0: return 8 + 4;            // tendencies only
    case 1: return 8 + 8;            // + next state + ds0
    case 2: return 12 + 8;           // + ds0 read
    case 3: return 16 + 4;           // + ds0, ds1 read
    case 4: return 12 + 8;           // + sb read; next state + sb written
    case 5: return 8 + 4 + 4;        // next state read and written
    case 6: return 8 + 8;            // next state + sb written
    default: return 0;
    }
}

// mode st of the stage kernel (mode tst of the passive tracers'); slot >= 0
// also writes the tendencies there
template <typename T>
int stage_t(nyl_ctx *c, int st, int tst, int slot, double coef, double coef2, bool last) {
    StageArgs<T> a = stage_args<T>(c);
    if (slot >= 0) set_tendency_out<T>(c, a, slot);
    a.c = coef;
    a.c2 = coef2;
    if (last && c->d.viscosity != 0.0) {   // core/model_les.py:140-141
        a.visc = 1;
        a.vcx = c->d.viscosity * c->d.idx2;
        a.vcy = c->d.viscosity * c->d.idy2;
        a.vcz = c->d.viscosity * c->d.idz2;
    }
    if (c->d.model == NYL_MODEL_LINEAR) a.flags |= NYL_SF_NO_VF;
    if (c->d.model == NYL_MODEL_EULER) a.flags |= NYL_SF_NO_B;
    const double words = stage_words(st) + (st == 3 && slot == 2 ? 4 : 0);
    LAUNCH(NYL_K_STAGE, words * cells(c->g) * sizeof(T), launch_stage<T>(c->g, a, st, c->stream));
    // passive tracers: the same right-hand side and update, one launch each;
    // Euler3d advects none of them (zero tendencies)
    const int s = c->cur, t = 1 - c->cur;
    for (int q = 0; q < c->ntr; q++) {
        if (c->d.model == NYL_MODEL_EULER) {
            HIPCHK(launch_zero<T>(F<T>(c, c->tds[slot][q]), c->ncell, c->stream));
            continue;
        }
        TracerArgs<T> ta;
        ta.q = F<T>(c, c->tst[s][q]);
        ta.qn = F<T>(c, c->tst[t][q]);
        ta.u = a.u; ta.v = a.v; ta.w = a.w;
        ta.d0 = F<T>(c, c->tds[0][q]);
        ta.d1 = F<T>(c, c->tds[1][q]);
        ta.tout = slot >= 0 ? F<T>(c, c->tds[slot][q]) : nullptr;
        ta.sb = F<T>(c, c->tsb[q]);
        ta.idx2 = c->d.idx2; ta.idy2 = c->d.idy2; ta.idz2 = c->d.idz2;
        ta.c = coef;
        ta.c2 = coef2;
        ta.upw = c->d.upwind_a;
        LAUNCH(NYL_K_STAGE, (stage_words(tst) / 4.0) * cells(c->g) * sizeof(T),
               launch_tracer_stage<T>(c->g, ta, tst, c->stream));
    }
    return NYL_OK;
}

// the stage combination of mode st from the stored tendencies of every
// prognostic field (b, u, v, w unless only the tracers are asked for;
// tracers): slot 0 for modes 1 and 4..6, slots 0..1 for mode 2 and 0..2 for
// mode 3
template <typename T>
int update_t(nyl_ctx *c, int st, double coef, double coef2, bool tracers_only = false) {
    const int s = c->cur, t = 1 - c->cur;
    auto one = [&](uint64_t cur, uint64_t nxt, uint64_t d0, uint64_t d1, uint64_t d2,
                   uint64_t sb) -> int {
        UpdateArgs<T> a;
        a.s = F<T>(c, cur);
        a.sn = F<T>(c, nxt);
        a.ds0 = F<T>(c, d0);
        a.ds1 = F<T>(c, d1);
        a.ds2 = F<T>(c, d2);
        a.sb = F<T>(c, sb);
        a.c = coef;
        a.c2 = coef2;
        HIPCHK(launch_update<T>(c->ncell, a, st, c->stream));
        return NYL_OK;
    };
    int rc;
    for (int f = 0; f < 4 && !tracers_only; f++)
        if ((rc = one(c->state[s][f], c->state[t][f], c->ds[0][f], c->ds[1][f], c->ds[2][f],
                      c->sb[f])))
            return rc;
    for (int q = 0; q < c->ntr; q++)
        if ((rc = one(c->tst[s][q], c->tst[t][q], c->tds[0][q], c->tds[1][q], c->tds[2][q],
                      c->tsb[q])))
            return rc;
    return NYL_OK;
}

// last: the time scheme's rhs call with last = True (RK3 stage 3, Euler
// forward, the LFAM3 corrector), which adds the viscosity
int stage(nyl_ctx *c, int st, double coef, double coef2, bool last) {
    int rc;
    if (c->d.model != NYL_MODEL_LES || c->d.upwind_a || c->d.upwind_vf) {
        // model variants and the linear upwind branches: the tendencies
        // into the slot the stage combination reads last (0 for modes 1 and
        // 4..6, 1 for mode 2, 2 for mode 3), then the combination; the stages
        // of RK3 combine b, u, v, w in the stage kernel (256x128x64 FP32,
        // order 5: 91 us and four updates of 7 became 50..59 us)
        const int slot = st == 2 ? 1 : (st == 3 ? 2 : 0);
        const bool one = st <= 3;
        rc = c->mixed ? stage_t<float>(c, one ? st : 0, 0, slot, coef, coef2, last)
                      : stage_t<double>(c, one ? st : 0, 0, slot, coef, coef2, last);
        if (rc) return rc;
        rc = c->mixed ? update_t<float>(c, st, coef, coef2, one)
                      : update_t<double>(c, st, coef, coef2, one);
        if (rc) return rc;
        if (st != 5) c->cur = 1 - c->cur;
        return NYL_OK;
    }
    const int slot = (st == 1 || st == 2) ? st - 1 : -1;
    rc = c->mixed ? stage_t<float>(c, st, st, slot, coef, coef2, last)
                  : stage_t<double>(c, st, st, slot, coef, coef2, last);
    if (rc) return rc;
    if (st != 5) c->cur = 1 - c->cur;
    return NYL_OK;
}

template <typename T>
int reduce_t(nyl_ctx *c, int what) {
    const int s = c->cur;
    double *part = F<double>(c, c->partials), *res = F<double>(c, c->result);
    T *b = F<T>(c, c->state[s][0]), *u = F<T>(c, c->state[s][1]), *v = F<T>(c, c->state[s][2]),
      *w = F<T>(c, c->state[s][3]);
    switch (what) {
    case NYL_RED_MAXU2:
        HIPCHK(launch_maxu2<T>(c->g, u, v, w, c->d.idx2, c->d.idy2, c->d.idz2, part, res,
                               c->stream));
        break;
    case NYL_RED_KE:
        HIPCHK(launch_kesum<T>(c->g, u, v, w, c->d.idx2, c->d.idy2, c->d.idz2, part, res,
                               c->stream));
        break;
    case NYL_RED_BSUM:
        HIPCHK(launch_sum<T>(c->g, b, part, res, c->stream));
        break;
    case NYL_RED_NONFINITE:
        HIPCHK(launch_nonfinite<T>(c->g, b, u, v, w, part, res, c->stream));
        break;
    default:
        return fail(NYL_E_ARG, "unknown reduction %d", what);
    }
    return NYL_OK;
}

}  // namespace

extern "C" {

int nyl_abi_version(void) { return NYL_ABI_VERSION; }

const char *nyl_last_error(void) { return g_err; }

int nyl_ctx_create(const nyl_desc *desc, nyl_ctx **out) {
    if (!desc || !out) return fail(NYL_E_ARG, "null argument");
    *out = nullptr;
    const nyl_desc &d = *desc;
    if (d.precision != NYL_PREC_FP64 && d.precision != NYL_PREC_MIXED)
        return fail(NYL_E_ARG, "unknown precision mode %d", d.precision);
    const int n3[3] = {d.nx, d.ny, d.nz};
    const int p3[3] = {d.periodic_x, d.periodic_y, d.periodic_z};
    for (int a = 0; a < 3; a++) {
        // wall axes need n >= 6 for the flux1d closures (core/weno.f90:116-150)
        if (n3[a] < 8)
            return fail(NYL_E_SIZE, "axis %d has %d cells; at least 8 are needed", a, n3[a]);
        if (p3[a] != 0 && p3[a] != 1) return fail(NYL_E_ARG, "periodic flags must be 0 or 1");
    }
    if (!(d.dx > 0 && d.dy > 0 && d.dz > 0)) return fail(NYL_E_ARG, "grid spacings must be > 0");
    // the stage kernel addresses a field with 32-bit byte offsets
    const int64_t esz = d.precision == NYL_PREC_FP64 ? 8 : 4;
    if ((int64_t)d.nx * d.ny * d.nz * esz >= ((int64_t)1 << 32))
        return fail(NYL_E_SIZE, "grid of %lld cells: a field must stay below 4 GiB "
                    "(%lld cells in FP64, %lld in mixed precision)",
                    (long long)d.nx * d.ny * d.nz, ((long long)1 << 29) - 1,
                    ((long long)1 << 30) - 1);
    if (d.mg_maxite < 0) return fail(NYL_E_ARG, "mg_maxite must be >= 0");
    if (d.n_tracers < 0 || d.n_tracers > NYL_MAX_TRACERS)
        return fail(NYL_E_ARG, "n_tracers must be 0..%d", NYL_MAX_TRACERS);
    if (!(d.viscosity >= 0.0)) return fail(NYL_E_ARG, "viscosity must be >= 0");
    if (d.model < NYL_MODEL_LES || d.model > NYL_MODEL_EULER)
        return fail(NYL_E_ARG, "model must be NYL_MODEL_LES, _LINEAR or _EULER");
    for (int o : {d.upwind_a, d.upwind_vf})
        if (o != 0 && o != 1 && o != 3 && o != 5)
            return fail(NYL_E_ARG, "linear upwind orders are 1, 3 or 5 (0: WENO)");
    if (d.upwind_a || d.upwind_vf) {
        // the reference's closures overlap (and read outside the line) on
        // wall lines shorter than 6 cells
        const int n[3] = {d.nx, d.ny, d.nz}, p[3] = {d.periodic_x, d.periodic_y, d.periodic_z};
        for (int q = 0; q < 3; q++)
            if (n[q] < 6 && !p[q])
                return fail(NYL_E_SIZE, "linear upwind needs 6 or more cells along a wall axis");
    }
    nyl_ctx *c = new nyl_ctx();
    memset(c, 0, sizeof(*c));
    c->d = d;
    c->ntr = d.n_tracers;
    c->mixed = d.precision == NYL_PREC_MIXED;
    c->g = make_geo(d.nx, d.ny, d.nz, d.periodic_x, d.periodic_y, d.periodic_z);
    if (c->mixed && !outer_resid_fits(c->g)) {
        delete c;
        return fail(NYL_E_SIZE, "grid %dx%dx%d is too wide for the mixed-precision solve",
                    d.nx, d.ny, d.nz);
    }
    c->ncell = (int64_t)d.nx * d.ny * d.nz;
    int rc = build_hierarchy(c);
    if (rc) { delete c; return rc; }
    build_tabs(c->tabs);
    build_layout(c);
    c->t0 = cycle_first(c);
    for (int q = 0; q < kSites; q++)
        for (int j = 0; j < kPredOuter; j++) c->pred[q][j] = {-1, -1};
    c->stream = nullptr;
    *out = c;
    return NYL_OK;
}

int nyl_ctx_destroy(nyl_ctx *c) {
    if (!c) return NYL_OK;
    for (int q = 0; q < c->prof_nev; q++) (void)hipEventDestroy(c->prof_ev[q]);
    if (c->host_out) (void)hipHostFree(c->host_out);
    delete c;
    return NYL_OK;
}

int nyl_workspace_bytes(const nyl_ctx *c, uint64_t *bytes) {
    if (!c || !bytes) return fail(NYL_E_ARG, "null argument");
    *bytes = c->ws_bytes;
    return NYL_OK;
}

int nyl_set_stream(nyl_ctx *c, void *stream) {
    if (!c) return fail(NYL_E_ARG, "null context");
    c->stream = (hipStream_t)stream;
    return NYL_OK;
}

int nyl_set_graphs(nyl_ctx *c, int on) {
    (void)on;   // a step enqueues its launches ahead of the GPU: nothing is replayed
    if (!c) return fail(NYL_E_ARG, "null context");
    return NYL_OK;
}

int nyl_bind_workspace(nyl_ctx *c, void *dptr, uint64_t bytes) {
    if (!c || !dptr) return fail(NYL_E_ARG, "null argument");
    if (bytes < c->ws_bytes)
        return fail(NYL_E_ARG, "workspace of %llu bytes is smaller than the %llu needed",
                    (unsigned long long)bytes, (unsigned long long)c->ws_bytes);
    if (((uintptr_t)dptr) & 255) return fail(NYL_E_ARG, "workspace must be 256-byte aligned");
    if (!c->host_out) {
        HIPCHK(hipHostMalloc((void **)&c->host_out, (kHostCtl + 2 + CTL_HIST) * sizeof(double),
                             hipHostMallocMapped | hipHostMallocCoherent));
        HIPCHK(hipHostGetDevicePointer((void **)&c->host_dev, c->host_out, 0));
        *reinterpret_cast<volatile uint32_t *>(c->host_out + 8) = 0;
        c->pub_seq = 0;
    }
    c->ws = (char *)dptr;
    HIPCHK(launch_fill((double *)c->ws, (int64_t)(c->ws_bytes / sizeof(double)), 0.0, c->stream));
    HIPCHK(hipMemcpyAsync(c->ws + c->ent, c->cyc_ent, sizeof(c->cyc_ent), hipMemcpyHostToDevice,
                          c->stream));
    c->cyc.ent = F<CycleEnt>(c, c->ent);
    if (c->exact) {
        std::vector<double> tab(coarse_table_doubles());
        coarse_tables(c->lev[c->nlev - 1].g, tab.data());
        HIPCHK(hipMemcpyAsync(c->ws + c->cs_tab, tab.data(), tab.size() * sizeof(double),
                              hipMemcpyHostToDevice, c->stream));
        c->cyc.etab = F<double>(c, c->cs_tab);
    }
    HIPCHK(hipStreamSynchronize(c->stream));
    c->cur = 0;
    c->total_cycles = 0;
    c->lf_first = 1;
    return NYL_OK;
}

int nyl_field_offset(const nyl_ctx *c, int field, uint64_t *off, int64_t *nelem, int32_t *dtype) {
    if (!c || !off) return fail(NYL_E_ARG, "null argument");
    uint64_t o;
    const int s = c->cur;
    bool f64 = !c->mixed;   // model fields follow the precision mode
    switch (field) {
    case NYL_F_B: case NYL_F_U: case NYL_F_V: case NYL_F_W: o = c->state[s][field - NYL_F_B]; break;
    case NYL_F_KE: o = c->ke; break;
    case NYL_F_VORX: case NYL_F_VORY: case NYL_F_VORZ: o = c->vor[field - NYL_F_VORX]; break;
    case NYL_F_UCX: case NYL_F_UCY: case NYL_F_UCZ: o = c->uc[field - NYL_F_UCX]; break;
    case NYL_F_P: o = c->p; f64 = true; break;
    case NYL_F_DIV: o = c->mgb; f64 = true; break;
    case NYL_F_MGX: o = c->mgx; f64 = true; break;
    case NYL_F_MGB: o = c->mgb; f64 = true; break;
    case NYL_F_MGY: o = c->lev[0].y; f64 = lev64(c, 0); break;
    default:
        if (field >= NYL_F_DS0_B && field <= NYL_F_DS2_W) {
            const int q = field - NYL_F_DS0_B;
            o = c->ds[q / 4][q % 4];
            break;
        }
        if (field >= NYL_F_TRACER(0) && field < NYL_F_TRACER(c->ntr)) {
            o = c->tst[s][field - NYL_F_TRACER(0)];
            break;
        }
        if (field >= NYL_F_DS_TRACER(0, 0) && field < NYL_F_DS_TRACER(3, 0) &&
            (field - NYL_F_DS_TRACER(0, 0)) % NYL_MAX_TRACERS < c->ntr) {
            const int q = field - NYL_F_DS_TRACER(0, 0);
            o = c->tds[q / NYL_MAX_TRACERS][q % NYL_MAX_TRACERS];
            break;
        }
        return fail(NYL_E_ARG, "unknown field %d", field);
    }
    *off = o;
    if (nelem) *nelem = c->ncell;
    if (dtype) *dtype = f64 ? NYL_DT_F64 : NYL_DT_F32;
    return NYL_OK;
}

int nyl_mg_levels(const nyl_ctx *c, int32_t *n) {
    if (!c || !n) return fail(NYL_E_ARG, "null argument");
    *n = c->nlev;
    return NYL_OK;
}

int nyl_mg_level_shape(const nyl_ctx *c, int level, int32_t *nx, int32_t *ny, int32_t *nz) {
    if (!c || !nx || !ny || !nz) return fail(NYL_E_ARG, "null argument");
    if (level < 0 || level >= c->nlev) return fail(NYL_E_ARG, "level %d out of range", level);
    *nx = c->lev[level].g.nx; *ny = c->lev[level].g.ny; *nz = c->lev[level].g.nz;
    return NYL_OK;
}

int nyl_rhs(nyl_ctx *c, int slot, int last) {
    int rc = check_ready(c);
    if (rc) return rc;
    if (slot < 0 || slot > 2) return fail(NYL_E_ARG, "slot must be 0..2");
    return c->mixed ? stage_t<float>(c, 0, 0, slot, 0.0, 0.0, last != 0)
                    : stage_t<double>(c, 0, 0, slot, 0.0, 0.0, last != 0);
}

int nyl_stage_update(nyl_ctx *c, int mode, double coef, double coef2) {
    int rc = check_ready(c);
    if (rc) return rc;
    if (mode < 1 || mode > 6) return fail(NYL_E_ARG, "mode must be 1..6");
    rc = c->mixed ? update_t<float>(c, mode, coef, coef2) : update_t<double>(c, mode, coef, coef2);
    if (rc) return rc;
    c->cur = 1 - c->cur;   // mode 5 wrote over the saved 'now' state, which becomes current
    return NYL_OK;
}

int nyl_rk3_stage(nyl_ctx *c, int st, double coef) {
    int rc = check_ready(c);
    if (rc) return rc;
    if (st < 1 || st > 3) return fail(NYL_E_ARG, "stage must be 1..3");
    return stage(c, st, coef, 0.0, st == 3);
}

int nyl_diagnose(nyl_ctx *c, nyl_mg_stats *st) {
    int rc = check_ready(c);
    if (rc) return rc;
    return diagnose(c, st, 0);
}

int nyl_step_rk3(nyl_ctx *c, double dt, nyl_mg_stats *st) {
    int rc = check_ready(c);
    if (rc) return rc;
    nyl_mg_stats s1, acc;
    memset(&acc, 0, sizeof(acc));
    const double coef[3] = {dt, dt / 4., dt / 12.};
    for (int k = 1; k <= 3; k++) {
        if ((rc = stage(c, k, coef[k - 1], 0.0, k == 3))) return rc;
        if ((rc = diagnose(c, &s1, k))) return rc;
        acc.nite += s1.nite;
        acc.res = s1.res;
        acc.normb = s1.normb;
    }
    acc.total_cycles = c->total_cycles;
    if (st) *st = acc;
    return NYL_OK;
}

int nyl_step_ef(nyl_ctx *c, double dt, nyl_mg_stats *st) {
    int rc = check_ready(c);
    if (rc) return rc;
    if ((rc = stage(c, 1, dt, 0.0, true))) return rc;
    return diagnose(c, st, 1);
}

int nyl_step_lfam3(nyl_ctx *c, double dt, nyl_mg_stats *st) {
    int rc = check_ready(c);
    if (rc) return rc;
    if (c->lf_first) {
        if ((rc = stage(c, 6, dt, 0.0, false))) return rc;
        c->lf_first = 0;
        return diagnose(c, st, 1);
    }
    nyl_mg_stats s1, s2;
    // predictor: the current buffer keeps sn, the next one receives s
    if ((rc = stage(c, 4, 0.0, 2. * dt, false))) return rc;
    if ((rc = diagnose(c, &s1, 1))) return rc;
    // corrector: rhs at n+1/2, then s = sn + dt*ds written over sn
    if ((rc = stage(c, 5, dt, 0.0, true))) return rc;
    c->cur = 1 - c->cur;
    if ((rc = diagnose(c, &s2, 2))) return rc;
    if (st) {
        *st = s2;
        st->nite = s1.nite + s2.nite;
    }
    return NYL_OK;
}

int nyl_lfam3_reset(nyl_ctx *c) {
    if (!c) return fail(NYL_E_ARG, "null context");
    c->lf_first = 1;
    return NYL_OK;
}

int nyl_mg_solve(nyl_ctx *c, nyl_mg_stats *st) {
    int rc = check_ready(c);
    if (rc) return rc;
    return mg_solve(c, st, 0);
}

int nyl_apply(nyl_ctx *c, int op) {
    int rc = check_ready(c);
    if (rc) return rc;
    return apply_op(c, op);
}

int nyl_reduce(nyl_ctx *c, int what, double *out) {
    int rc = check_ready(c);
    if (rc) return rc;
    if (!out) return fail(NYL_E_ARG, "null argument");
    arm_publish(c, 1);
    if ((rc = c->mixed ? reduce_t<float>(c, what) : reduce_t<double>(c, what))) return rc;
    return read_result(c, out);
}

int nyl_prof_start(nyl_ctx *c, int kernel_class) {
    int rc = check_ready(c);
    if (rc) return rc;
    if ((rc = prof_drain(c))) return rc;
    c->prof_cls = kernel_class;
    c->prof_ms = 0.0;
    c->prof_bytes = 0.0;
    c->prof_launches = 0;
    return NYL_OK;
}

int nyl_prof_stop(nyl_ctx *c, double *total_ms, int64_t *launches, double *alg_bytes) {
    int rc = check_ready(c);
    if (rc) return rc;
    if ((rc = prof_drain(c))) return rc;
    if (total_ms) *total_ms = c->prof_ms;
    if (launches) *launches = c->prof_launches;
    if (alg_bytes) *alg_bytes = c->prof_bytes;
    c->prof_cls = 0;
    return NYL_OK;
}

int nyl_debug_mg(nyl_ctx *c, int what) {
    int rc = check_ready(c);
    if (rc) return rc;
    if (c->mixed) return fail(NYL_E_STATE, "nyl_debug_mg works on FP64 contexts");
    Level &f = c->lev[0];
    double *x = F<double>(c, f.x), *b = F<double>(c, f.b), *y = F<double>(c, f.y);
    double *part = F<double>(c, c->partials), *res_dev = F<double>(c, c->result);
    switch (what) {
    case 0:
        HIPCHK(launch_mg_sweep<double>(f.g, x, y, b, c->d.mg_omega, c->tabs, c->stream));
        break;
    case 1:
        if (!sweep25_fits(f.g)) return fail(NYL_E_SIZE, "level 1 does not fit the tiled sweep");
        HIPCHK(launch_mg_sweep25<double>(f.g, x, y, b, c->d.mg_omega, c->tabs, nullptr, nullptr,
                                         c->stream));
        break;
    case 2:
        if (!sweep25_fits(f.g)) return fail(NYL_E_SIZE, "level 1 does not fit the tiled sweep");
        HIPCHK(launch_mg_sweep25<double>(f.g, x, y, b, c->d.mg_omega, c->tabs, part, res_dev,
                                         c->stream));
        break;
    case 3:
        HIPCHK(launch_resnorm2<double>(f.g, x, b, c->tabs, part, res_dev, c->stream));
        break;
    case 4:
    case 5:
    case 6:
        if (!sweep25_fits(f.g)) return fail(NYL_E_SIZE, "level 1 does not fit the tiled sweep");
        if (what == 5 && sweep2x_blocks(f.g, 8) > NYL_RED_BLOCKS)
            return fail(NYL_E_SIZE, "too many blocks for the residual norm");
        HIPCHK(launch_mg_sweep2x25<double>(f.g, what == 6 ? nullptr : x, y, b, c->d.mg_omega,
                                           c->tabs, c->stream, what == 5 ? part : nullptr,
                                           what == 5 ? res_dev : nullptr));
        break;
    default:
        return fail(NYL_E_ARG, "unknown debug operation %d", what);
    }
    HIPCHK(hipStreamSynchronize(c->stream));
    return NYL_OK;
}

int nyl_reduce_last(nyl_ctx *c, double *out) {
    int rc = check_ready(c);
    if (rc) return rc;
    if (!out) return fail(NYL_E_ARG, "null argument");
    return read_result(c, out);
}

int nyl_sync(nyl_ctx *c) {
    if (!c) return fail(NYL_E_ARG, "null context");
    HIPCHK(hipStreamSynchronize(c->stream));
    return NYL_OK;
}

}  // extern "C"
