// The single-workgroup cycle of the small multigrid levels (nyl_cycle.hip)
// against the per-cell multigrid kernels and the direct coarse solve, bit for
// bit in FP64, and the device-side stop rule against the host's.
#include <cstdint>
inline int __builtin_amdgcn_readfirstlane(int v) { return v; }
inline uint32_t __umulhi(uint32_t a, uint32_t b) { return (uint32_t)(((uint64_t)a * b) >> 32); }
#include "../../nyles_amd/csrc/nyl_mg.hip"
#include "../../nyles_amd/csrc/nyl_coarse.hip"
#include "../../nyles_amd/csrc/nyl_cycle.hip"
#include "emu.h"
using namespace nyl;

template <typename T>
static std::vector<T> sweep(const Geo &g, const std::vector<T> &x, const std::vector<T> &b,
                            const MGTabs &tab) {
    std::vector<T> y(x.size());
    run_blocks(mg_grid(g), dim3(MG_BX, MG_BY, 1), [&]() {
        k_mg_sweep<T>(g, x.data(), y.data(), b.data(), 0.9, tab); }, false);
    return y;
}

// levels 0 .. nl-1, the coarsest in FP64, the others of type T
template <typename T>
static int check(int nx, int ny, int nz, int nl, bool exact, int p) {
    const MGTabs tab = mktab();
    std::vector<Geo> g;
    for (int l = 0; l < nl; l++)
        g.push_back(mk(nx >> l, ny >> l, nz >> l, p & 1, (p >> 1) & 1, (p >> 2) & 1));
    std::vector<double> et(coarse_table_doubles());
    coarse_tables(g[nl - 1], et.data());
    std::vector<CycleEnt> ent(CYC_ENT);
    CycleArgs a;
    if (!cycle_layout(a, ent.data(), g.data(), 0, nl, sizeof(T), exact, 0.9, tab)) return 1;
    ent.resize(a.nent);
    a.ent = ent.data();
    a.etab = et.data();
    std::mt19937_64 rng(nx + 3 * ny + 7 * nz + p);
    auto cells = [&](int l) { return (size_t)g[l].nx * g[l].ny * g[l].nz; };
    const int c = nl - 1;
    std::vector<std::vector<T>> b(nl), y(nl), x(nl);
    std::vector<double> bc(cells(c)), yc(cells(c)), xc(cells(c));
    b[0] = rnd<T>(cells(0), rng);
    y[0] = rnd<T>(cells(0), rng);
    const auto b0 = b[0], y0 = y[0];
    if (nl == 1) {
        bc.assign(b0.begin(), b0.end());
        yc.assign(y0.begin(), y0.end());
    }
    for (int l = 0; l < c; l++) {
        x[l] = sweep(g[l], y[l], b[l], tab);
        if (l + 1 == c) {
            std::vector<double> xd(cells(c));
            run_blocks(mg_grid(g[c]), dim3(MG_BX, MG_BY, 1), [&]() {
                k_mg_resid_restrict<T, double>(g[l], g[c], x[l].data(), b[l].data(), bc.data(),
                                               xd.data(), tab, yc.data(), 0.9); }, false);
        } else {
            std::vector<T> xd(cells(l + 1));
            b[l + 1].resize(cells(l + 1));
            y[l + 1].resize(cells(l + 1));
            run_blocks(mg_grid(g[l + 1]), dim3(MG_BX, MG_BY, 1), [&]() {
                k_mg_resid_restrict<T, T>(g[l], g[l + 1], x[l].data(), b[l].data(),
                                          b[l + 1].data(), xd.data(), tab, y[l + 1].data(),
                                          0.9); }, false);
        }
    }
    if (exact) {
        std::vector<double> s(cells(c));
        CoarseArgs ca;
        ca.g = g[c]; ca.b = bc.data(); ca.s = s.data(); ca.x = xc.data(); ca.tab = et.data();
        run_blocks(dim3(g[c].nz), dim3(CS_T), [&]() { k_cs<0>(ca); }, true);
        run_blocks(dim3(g[c].ny), dim3(CS_T), [&]() { k_cs<1>(ca); }, true);
        run_blocks(dim3(g[c].nz), dim3(CS_T), [&]() { k_cs<2>(ca); }, true);
    } else {
        xc = sweep(g[c], yc, bc, tab);
    }
    for (int l = c - 1; l >= 0; l--) {
        run_blocks(mg_grid(g[l]), dim3(MG_BX, MG_BY, 1), [&]() {
            if (l + 1 == c) k_mg_prolong<T, double>(g[l], g[c], x[l].data(), xc.data(), tab);
            else k_mg_prolong<T, T>(g[l], g[l + 1], x[l].data(), x[l + 1].data(), tab); }, false);
        x[l] = sweep(g[l], sweep(g[l], x[l], b[l], tab), b[l], tab);
    }
    auto bb = b0, yy = y0;
    std::vector<T> xx(cells(0), T(3));
    CtlArgs fin = {};
    run_blocks(dim3(1), dim3(CYC_T), [&]() {
        if (a.n0 <= CYC_T) k_mg_cycle<T, 1>(a, bb.data(), yy.data(), xx.data(), fin);
        else if (a.n0 <= 2 * CYC_T) k_mg_cycle<T, 2>(a, bb.data(), yy.data(), xx.data(), fin);
        else k_mg_cycle<T, CYC_R>(a, bb.data(), yy.data(), xx.data(), fin); }, true);
    int bad = ndiff(bb, b0);
    if (nl > 1) bad += ndiff(yy, x[0]);
    else for (size_t q = 0; q < cells(0); q++) bad += (double)xx[q] != xc[q];
    printf("cycle<%d> %dx%dx%d levels %d exact %d p=%d: %d mismatches\n", (int)sizeof(T), nx, ny,
           nz, nl, exact, p, bad);
    return bad != 0;
}

static int check_ctl() {
    std::mt19937_64 rng(5);
    int bad = 0;
    for (int np : {1, 255, 257, 3000, 16384}) {
        auto part = rnd<double>(2 * np, rng);
        for (double &v : part) v = std::fabs(v);
        double want = 0, got = 0;
        run_blocks(dim3(1), dim3(RED_T), [&]() {
            k_final_sum(part.data(), np, &want, Publish{}); }, true);
        MGCtl m = {};
        double host[2 + CTL_HIST] = {};
        uint32_t flag = 0;
        CtlArgs c = {};
        c.ctl = &m; c.partials = part.data(); c.np = np; c.slot = 0;
        auto go = [&](int nt) { run_blocks(dim3(1), dim3(nt), [&]() {
            static double sh[RED_T];
            ctl_body(c, sh, threadIdx.x); }, true); };
        for (int nt : {RED_T, CYC_T}) {
            c.kind = CTL_NORMB;
            go(nt);
            bad += m.normb != want || m.stop != 0;
        }
        c.kind = CTL_TEST; c.slot = 1; c.tol = 1.0; c.dst = host; c.flag = &flag; c.seq = 7; c.nhist = 2;
        go(RED_T);                       // res = 1: not below the tolerance
        bad += m.stop != 0 || host[3] != want || flag != 7;
        c.tol = 2.0;
        go(RED_T);
        bad += m.stop != 1;
        // mixed: a tight tolerance asks the inner loop for inner_red only, at
        // most inner_max V-cycles
        c.kind = CTL_OUTER; c.tol = 1e-20; c.inner_red = 1e-6; c.inner_max = 8; c.slot = -1;
        go(RED_T);
        bad += m.rel != 1 || m.target != 1e-6 || m.outer_stop != 0 || m.stop != 0 || m.no_add != 1;
        c.kind = CTL_INNER; c.k = 7;
        go(RED_T);
        bad += m.stop != 0 || m.no_add != 1;
        c.k = 8;
        go(RED_T);
        bad += m.stop != 1 || m.no_add != 0;
        c.kind = CTL_SHIFT; c.ncell = 10.0;
        go(RED_T);
        double s2 = 0;
        run_blocks(dim3(1), dim3(RED_T), [&]() {
            k_final_sum(part.data() + np, np, &got, Publish{}); }, true);
        s2 = got - 10.0 * (want / 10.0) * (want / 10.0);
        bad += m.shift != want / 10.0 || m.normb != (s2 < 0 ? 0 : s2);
    }
    printf("control: %d mismatches\n", bad);
    return bad != 0;
}

int main() {
    int fails = check_ctl();
    for (int p : {0, 1, 3, 7, 4}) {
        fails += check<double>(16, 16, 16, 4, false, p) + check<float>(16, 16, 16, 4, false, p);
        fails += check<double>(12, 12, 12, 3, true, p) + check<float>(20, 12, 6, 2, true, p);
        fails += check<double>(4, 2, 2, 1, false, p) + check<double>(7, 5, 1, 1, true, p);
        fails += check<float>(8, 4, 4, 3, false, p);
        if (p < 2) fails += check<double>(32, 16, 8, 4, false, p) + check<double>(25, 15, 7, 1, true, p);
    }
    // levels that do not fit one workgroup are refused
    {
        Geo big[2] = {mk(64, 32, 4, 1, 1, 1), mk(32, 16, 2, 1, 1, 1)};
        std::vector<CycleEnt> ent(CYC_ENT);
        CycleArgs a;
        fails += cycle_layout(a, ent.data(), big, 0, 2, 8, false, 0.9, mktab());
        Geo wide[1] = {mk(500, 4, 1, 1, 1, 1)};
        fails += cycle_layout(a, ent.data(), wide, 0, 1, 8, false, 0.9, mktab());
    }
    printf(fails ? "FAIL %d\n" : "ALL OK\n", fails);
    return fails != 0;
}
