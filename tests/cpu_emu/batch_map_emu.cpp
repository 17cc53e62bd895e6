// The map from the blocks of a batched march to its items (k_b_march) with
// more items than 16 bits count: the blocks of items 65536 and 65537 work for
// those, and item 0 is left alone.
#include "../../nyles_amd/csrc/nyl_mg.hip"
#include "../../nyles_amd/csrc/nyl_march.hip"
#include "emu.h"
using namespace nyl;

template <typename I, typename M>
M map_entry(void (*)(const I *, const M *, MGTabs, const int *));

int main() {
    typedef decltype(map_entry(&k_b_march<double, double, MS_FIELD, 2, true, false, false, false>))
        Entry;
    const Geo g = mk(8, 8, 4, 1, 1, 0);
    const MGTabs tab = mktab();
    const size_t nf = 8 * 8 * 4, n = 65538;
    std::vector<MarchItem<double, double>> items(n);
    memset((void *)items.data(), 0, n * sizeof(items[0]));
    std::mt19937_64 rng(3);
    const size_t who[3] = {0, n - 2, n - 1};
    std::vector<double> x[3], b[3], y[3], want[3];
    double part[3] = {7.0, 7.0, 7.0};
    for (int r = 0; r < 3; r++) {
        x[r] = rnd<double>(nf, rng);
        b[r] = rnd<double>(nf, rng);
        y[r].assign(nf, 7.0);
        std::vector<double> t(nf);
        want[r].assign(nf, 7.0);
        if (r > 0) {
            run_blocks(mg_grid(g), dim3(MG_BX, MG_BY, 1), [&]() {
                k_mg_sweep<double>(g, x[r].data(), t.data(), b[r].data(), 0.9, tab); }, false);
            run_blocks(mg_grid(g), dim3(MG_BX, MG_BY, 1), [&]() {
                k_mg_sweep<double>(g, t.data(), want[r].data(), b[r].data(), 0.9, tab); }, false);
        }
        MarchItem<double, double> &it = items[who[r]];
        it.h.g = it.a.g = it.a.gc = g;
        it.h.member = (int)who[r];
        it.h.nblk = it.bx = it.by = 1;
        it.h.start = r == 0 ? 0 : r - 1;
        it.a.src = x[r].data();
        it.a.b = b[r].data();
        it.a.dst = y[r].data();
        it.a.omega = 0.9;
        it.a.partials = part + r;
        it.a.kz = 4;
    }
    const std::vector<Entry> map = {(Entry)who[1], (Entry)who[2]};
    run_blocks(dim3(2), dim3(256), [&]() {
        k_b_march<double, double, MS_FIELD, 2, true, false, false, false>(items.data(), map.data(),
                                                                          tab, nullptr); }, true);
    int bad = part[0] != 7.0;
    for (int r = 0; r < 3; r++) bad += ndiff(y[r], want[r]);
    printf("map of %d-byte entries: %d mismatches\n", (int)sizeof(Entry), bad);
    printf(bad ? "FAIL\n" : "ALL OK\n");
    return bad != 0;
}
