// The residual norm alone (k_mg_march, STRIPS) against the norm that comes
// with the tiled two-sweep pass (k_mg_sweep2t): the same block sums, bit for
// bit, with walls and periodic axes, marches of one plane and of several.
#include "../../nyles_amd/csrc/nyl_mg.hip"
#include "../../nyles_amd/csrc/nyl_march.hip"
#include "emu.h"
using namespace nyl;

template <typename T, int PZ>
int check(int nx, int ny, int nz, int px, int py, int kz) {
    const Geo g = mk(nx, ny, nz, px, py, PZ);
    const MGTabs tab = mktab();
    const size_t nf = (size_t)nx * ny * nz;
    std::mt19937_64 rng(nx + 3 * ny + 7 * nz + px + 2 * py + 4 * PZ + 31 * kz);
    const auto x = rnd<T>(nf, rng), b = rnd<T>(nf, rng);
    const dim3 grd(nx / 64, ny / 8, nz / kz);
    const size_t nb = (size_t)grd.x * grd.y * grd.z;
    std::vector<T> y(nf);
    std::vector<double> p1(nb, -1.0), p2(nb, -2.0);
    run_blocks(grd, dim3(64, 4), [&]() {
        k_mg_sweep2t<T, false, PZ, true, false>(g, x.data(), y.data(), b.data(), 0.9, tab, kz,
                                                nullptr, p1.data()); }, true);
    MarchArgs<T, T> a;
    memset(&a, 0, sizeof(a));
    a.g = a.gc = g; a.src = x.data(); a.b = b.data(); a.omega = 0.9; a.tab = tab;
    a.kz = kz; a.partials = p2.data();
    run_blocks(grd, dim3(256), [&]() {
        k_mg_march<T, T, 64, MS_FIELD, 0, true, false, false, false, true>(a, tab); }, true);
    const int bad = ndiff(p1, p2);
    printf("norm<%d> %dx%dx%d p=%d%d%d kz=%d: %d mismatches\n", (int)sizeof(T), nx, ny, nz, px, py,
           PZ, kz, bad);
    return bad != 0;
}

int main() {
    int fails = 0;
    for (int p : {0, 1, 3})
        for (int kz : {1, 8}) {
            fails += check<double, 0>(128, 16, 8, p & 1, p >> 1, kz);
            fails += check<double, 1>(64, 8, 8, p & 1, p >> 1, kz);
            fails += check<float, 0>(64, 24, 8, p & 1, p >> 1, kz);
            fails += check<float, 1>(128, 8, 8, p & 1, p >> 1, kz);
        }
    printf(fails ? "FAIL %d\n" : "ALL OK\n", fails);
    return fails != 0;
}
