// The one-pass level kernels (nyl_march.hip) against the per-cell multigrid
// kernels, bit for bit: partial tiles, both tile widths, every periodicity,
// several march lengths, levels smaller than a tile and one-cell axes.
#include "../../nyles_amd/csrc/nyl_mg.hip"
#include "../../nyles_amd/csrc/nyl_march.hip"
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

// LONG: with the steps inside the march as a path of its own
template <typename T, typename TC, int TX, bool LONG = false>
int check(int nx, int ny, int nz, int px, int py, int pz, int kz, bool halves) {
    const Geo g = mk(nx, ny, nz, px, py, pz), gc = mk(nx / 2, ny / 2, nz / 2, px, py, pz);
    const MGTabs tab = mktab();
    const size_t nf = (size_t)nx * ny * nz, nc = halves ? nf / 8 : 1;
    std::mt19937_64 rng(nx + 3 * ny + 7 * nz + px + 2 * py + 4 * pz + 31 * kz);
    const auto x = rnd<T>(nf, rng), b = rnd<T>(nf, rng);
    const auto xc = rnd<TC>(nc, rng);
    const dim3 grd((nx + TX - 1) / TX, (ny + 512 / TX - 1) / (512 / TX), (nz + kz - 1) / kz);
    const size_t nblk = (size_t)grd.x * grd.y * grd.z;
    int bad = 0;
    MarchArgs<T, TC> a;
    memset(&a, 0, sizeof(a));
    a.g = g; a.gc = gc; a.omega = 0.9; a.tab = tab; a.kz = kz;
    a.b = b.data();
    const auto y1 = sweep(g, x, b, tab), y2 = sweep(g, y1, b, tab);
    std::vector<double> rn(NYL_RED_BLOCKS, 0.0);
    run_blocks(dim3(red_blocks((int64_t)nf)), dim3(RED_T), [&]() {
        k_resnorm2<T>(g, x.data(), b.data(), tab, rn.data()); }, true);
    double want = 0;
    for (double v : rn) want += v;
    auto norm_of = [&](const std::vector<double> &p) {
        double s = 0;
        for (double v : p) s += v;
        return std::fabs(s - want) > 1e-9 * want;
    };
    if (sizeof(T) == sizeof(TC)) {
        // two sweeps, with the residual norm of the input and from zero; the norm alone
        std::vector<T> z(nf, T(7));
        std::vector<double> p1(nblk, 0.0), p2(nblk, 0.0);
        a.src = x.data(); a.dst = z.data();
        run_blocks(grd, dim3(256), [&]() {
            k_mg_march<T, TC, TX, MS_FIELD, 2, false, false, false, LONG>(a, tab); }, true);
        bad += ndiff(z, y2);
        z.assign(nf, T(7));
        a.partials = p1.data();
        run_blocks(grd, dim3(256), [&]() {
            k_mg_march<T, TC, TX, MS_FIELD, 2, true, false, false, LONG>(a, tab); }, true);
        bad += ndiff(z, y2) + norm_of(p1);
        a.partials = p2.data();
        run_blocks(grd, dim3(256), [&]() {
            k_mg_march<T, TC, TX, MS_FIELD, 0, true, false, false>(a, tab); }, true);
        bad += ndiff(p1, p2);
        const std::vector<T> zero(nf, T(0));
        const auto s2 = sweep(g, sweep(g, zero, b, tab), b, tab);
        a.src = nullptr;
        run_blocks(grd, dim3(256), [&]() {
            k_mg_march<T, TC, TX, MS_ZERO, 2, false, false, false, LONG>(a, tab); }, true);
        bad += ndiff(z, s2);
    }
    if (halves) {
        // one sweep, residual and restriction; prolongation and two sweeps
        std::vector<T> z(nf, T(7)), xp = x;
        std::vector<TC> bc1(nc), yc1(nc), xd(nc), bc2(nc, TC(5)), yc2(nc, TC(6));
        run_blocks(mg_grid(gc), dim3(MG_BX, MG_BY, 1), [&]() {
            k_mg_resid_restrict<T, TC>(g, gc, y1.data(), b.data(), bc1.data(), xd.data(), tab,
                                       yc1.data(), 0.9); }, false);
        a.src = x.data(); a.dst = z.data(); a.bc = bc2.data(); a.yc = yc2.data();
        run_blocks(grd, dim3(256), [&]() {
            k_mg_march<T, TC, TX, MS_FIELD, 1, false, true, false, LONG>(a, tab); }, true);
        bad += ndiff(z, y1) + ndiff(bc1, bc2) + ndiff(yc1, yc2);
        run_blocks(mg_grid(g), dim3(MG_BX, MG_BY, 1), [&]() {
            k_mg_prolong<T, TC>(g, gc, xp.data(), xc.data(), tab); }, false);
        const auto u2 = sweep(g, sweep(g, xp, b, tab), b, tab);
        z.assign(nf, T(7));
        a.xc = xc.data();
        run_blocks(grd, dim3(256), [&]() {
            k_mg_march<T, TC, TX, MS_PROLONG, 2, false, false, false, LONG>(a, tab); }, true);
        bad += ndiff(z, u2);
        // the restriction alone, and in the pass of the two sweeps (from a
        // field with its residual norm, from zero)
        bc2.assign(nc, TC(5)); yc2.assign(nc, TC(6));
        a.src = y1.data();
        run_blocks(grd, dim3(256), [&]() {
            k_mg_march<T, TC, TX, MS_FIELD, 0, false, true, false>(a, tab); }, true);
        bad += ndiff(bc1, bc2) + ndiff(yc1, yc2);
        for (int zero = 0; zero < 2; zero++) {
            const std::vector<T> o(nf, T(0));
            const auto t2 = zero ? sweep(g, sweep(g, o, b, tab), b, tab) : y2;
            run_blocks(mg_grid(gc), dim3(MG_BX, MG_BY, 1), [&]() {
                k_mg_resid_restrict<T, TC>(g, gc, t2.data(), b.data(), bc1.data(), xd.data(),
                                           tab, yc1.data(), 0.9); }, false);
            std::vector<double> p3(nblk, 0.0);
            z.assign(nf, T(7)); bc2.assign(nc, TC(5)); yc2.assign(nc, TC(6));
            a.src = zero ? nullptr : x.data();
            a.partials = p3.data();
            run_blocks(grd, dim3(256), [&]() {
                if (zero) k_mg_march<T, TC, TX, MS_ZERO, 2, false, true, false, LONG>(a, tab);
                else k_mg_march<T, TC, TX, MS_FIELD, 2, true, true, false, LONG>(a, tab); }, true);
            bad += ndiff(z, t2) + ndiff(bc1, bc2) + ndiff(yc1, yc2) + (!zero && norm_of(p3));
        }
        a.src = x.data();
        // a closed gate leaves everything as it is
        const int one = 1;
        const auto z0 = z;
        a.gate = &one;
        a.src = y1.data();
        run_blocks(grd, dim3(256), [&]() {
            k_mg_march<T, TC, TX, MS_PROLONG, 2, false, false, false, LONG>(a, tab); }, true);
        bad += ndiff(z, z0);
    }
    if (sizeof(T) == 8 && sizeof(TC) == 8) {   // the mixed solve's FP64 residual
        MarchArgs<double, double> o;
        memset(&o, 0, sizeof(o));
        const std::vector<double> xd(x.begin(), x.end()), bd(b.begin(), b.end());
        std::vector<float> r1(nf), r2(nf), yd(nf);
        std::vector<double> p1(NYL_RED_BLOCKS, 0.0), p2(nblk, 0.0);
        const double shift = 0.125;
        o.g = o.gc = g; o.src = xd.data(); o.b = bd.data(); o.tab = tab; o.kz = kz;
        o.partials = p2.data(); o.rout = r2.data(); o.shift = &shift;
        run_blocks(outer_grid(g), dim3(MG_BX, MG_BY, 1), [&]() {
            k_mg_outer_resid<float>(g, xd.data(), bd.data(), shift, r1.data(), yd.data(), 0.9, tab,
                                    p1.data()); }, true);
        run_blocks(grd, dim3(256), [&]() {
            k_mg_march<double, double, TX, MS_FIELD, 0, true, false, true>(o, tab); }, true);
        double s1 = 0, s2 = 0;
        for (double v : p1) s1 += v;
        for (double v : p2) s2 += v;
        bad += ndiff(r1, r2) + (std::fabs(s1 - s2) > 1e-12 * s1);
    }
    printf("march<%d,%d,%d> %dx%dx%d p=%d%d%d kz=%d: %d mismatches\n", (int)sizeof(T),
           (int)sizeof(TC), TX, nx, ny, nz, px, py, pz, kz, bad);
    return bad != 0;
}

int main() {
    int fails = 0;
    for (int p : {0, 3, 5, 7, 2, 4}) {
        const int px = p & 1, py = (p >> 1) & 1, pz = (p >> 2) & 1;
        fails += check<double, double, 64>(70, 10, 6, px, py, pz, 2, true);
        fails += check<float, float, 32>(40, 18, 10, px, py, pz, 4, true);
        fails += check<float, double, 32>(6, 10, 14, px, py, pz, 8, true);
        fails += check<float, float, 64>(2, 2, 2, px, py, pz, 2, true);
        if (p == 0 || p == 7) {   // one march; one with a short rest
            fails += check<double, double, 64, true>(34, 10, 16, px, py, pz, 16, true);
            fails += check<float, float, 32, true>(6, 10, 22, px, py, pz, 16, true);
        }
        if (p == 0 || p == 7) {
            fails += check<double, double, 64>(64, 8, 8, px, py, pz, 8, true);
            fails += check<float, float, 64>(130, 24, 4, px, py, pz, 2, true);
            fails += check<double, double, 32>(33, 17, 5, px, py, pz, 1, false);
            fails += check<float, float, 64>(65, 9, 7, px, py, pz, 3, false);
        }
    }
    printf(fails ? "FAIL %d\n" : "ALL OK\n", fails);
    return fails != 0;
}
