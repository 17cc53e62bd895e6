// The stage and tracer kernels with the blocks of a plane as for planes of more
// than 65536 blocks (the stage in tiles of 64 x 4 groups with partial ones, the
// tracers' along x and y) against the blocks along y alone, and
// the tendencies and the second RK3 stage of the linear branches and model
// variants with 16 bytes of cells per thread against one cell, bit for bit.
#define NYL_STAGE_SEQ 0
#include "../../nyles_amd/csrc/nyl_stage.h"
#include "../../nyles_amd/csrc/nyl_tracer.hip"
#include "emu.h"
using namespace nyl;

template <typename T>
struct Fields {
    std::vector<std::vector<T>> in, out;
    StageArgs<T> a;
    Fields(const Geo &g, unsigned seed) : in(19), out(12) {
        const size_t n = (size_t)g.nx * g.ny * g.nz;
        std::mt19937_64 rng(seed);
        for (auto &v : in) v = rnd<T>(n, rng);
        for (int f = 0; f < 12; f++) out[f] = f >= 4 && f < 8 ? std::vector<T>(n, T(5)) : in[11 + f % 4];
        memset(&a, 0, sizeof(a));
        a.b = in[0].data(); a.u = in[1].data(); a.v = in[2].data(); a.w = in[3].data();
        a.ox = in[4].data(); a.oy = in[5].data(); a.oz = in[6].data(); a.ke = in[7].data();
        a.d0b = in[8].data(); a.d0u = in[9].data(); a.d0v = in[10].data(); a.d0w = in[14].data();
        a.d1b = in[15].data(); a.d1u = in[16].data(); a.d1v = in[17].data(); a.d1w = in[18].data();
        a.bn = out[0].data(); a.un = out[1].data(); a.vn = out[2].data(); a.wn = out[3].data();
        a.tb = out[4].data(); a.tu = out[5].data(); a.tv = out[6].data(); a.tw = out[7].data();
        a.sbb = out[8].data(); a.sbu = out[9].data(); a.sbv = out[10].data(); a.sbw = out[11].data();
        a.idx2 = 1.7; a.idy2 = 2.3; a.idz2 = 0.9; a.dz = 0.37;
        a.c = 0.013; a.c2 = 0.026; a.visc = 1;
        a.vcx = 0.011; a.vcy = 0.013; a.vcz = 0.007;
    }
    TracerArgs<T> tracer() {
        TracerArgs<T> t;
        memset(&t, 0, sizeof(t));
        t.q = a.b; t.u = a.u; t.v = a.v; t.w = a.w;
        t.qn = a.bn; t.d0 = a.d0b; t.d1 = a.d1b; t.tout = a.tb; t.sb = a.sbb;
        t.idx2 = a.idx2; t.idy2 = a.idy2; t.idz2 = a.idz2; t.c = a.c; t.c2 = a.c2;
        return t;
    }
};

template <typename T, int N, int PX, int PY, int PZ>
int split(int nx, int ny, int nz, int gx) {
    const Geo g = mk(nx, ny, nz, PX, PY, PZ);
    const unsigned nb = (nx / N * ny + STAGE_NT - 1) / STAGE_NT;
    Fields<T> f1(g, nx + ny), f2(g, nx + ny);
    const dim3 one(1, nb, nz), many(gx, (nb + gx - 1) / gx, nz);
    auto stage = [&](dim3 grd, Fields<T> &f, int lw) {
        run_blocks(grd, dim3(STAGE_NT), [&]() { k_stage_flat<T, N, 3, PX, PY, PZ>(g, f.a, lw); }, false);
    };
    auto tracer = [&](dim3 grd, Fields<T> &f) {
        const TracerArgs<T> t = f.tracer();
        run_blocks(grd, dim3(STAGE_NT), [&]() { k_tracer_stage<T, N, 2, PX, PY, PZ>(g, t); }, false);
    };
    int bad = 0;
    stage(one, f1, 0);
    stage(dim3((nx / N + 63) / 64, (ny + 3) / 4, nz), f2, 6);
    for (int q = 0; q < 12; q++) bad += ndiff(f1.out[q], f2.out[q]);
    tracer(one, f1);
    tracer(many, f2);
    for (int q = 0; q < 12; q++) bad += ndiff(f1.out[q], f2.out[q]);
    printf("split<%d, %d> %dx%dx%d over %d: %d mismatches\n", (int)sizeof(T), N, nx, ny, nz, gx, bad);
    return bad != 0;
}

template <typename T, int N, int MODE, int PX, int PY, int PZ>
int lin(int nx, int ny, int nz) {
    const int orders[][3] = {{1, 1, 0}, {3, 5, 0}, {5, 3, 0}, {5, 0, NYL_SF_NO_B}, {0, 0, NYL_SF_NO_VF}};
    const Geo g = mk(nx, ny, nz, PX, PY, PZ);
    int bad = 0;
    for (auto &o : orders) {
        Fields<T> f1(g, nx + ny), f2(g, nx + ny);
        for (auto *f : {&f1, &f2}) { f->a.upw_a = o[0]; f->a.upw_vf = o[1]; f->a.flags = o[2]; }
        auto grd = [&](int n) { return dim3(1, (nx / n * ny + STAGE_NT - 1) / STAGE_NT, nz); };
        run_blocks(grd(1), dim3(STAGE_NT), [&]() {
            k_stage_flat<T, 1, MODE, PX, PY, PZ, true>(g, f1.a, 0); }, false);
        run_blocks(grd(N), dim3(STAGE_NT), [&]() {
            k_stage_flat<T, N, MODE, PX, PY, PZ, true>(g, f2.a, 0); }, false);
        for (int q = 0; q < 12; q++) bad += ndiff(f1.out[q], f2.out[q]);
    }
    printf("lin<%d, %d> mode %d %dx%dx%d p=%d%d%d: %d mismatches\n", (int)sizeof(T), N, MODE, nx, ny,
           nz, PX, PY, PZ, bad);
    return bad != 0;
}

template <int PX, int PY, int PZ>
int lin_all() {
    return lin<double, 2, 0, PX, PY, PZ>(8, 8, 8) + lin<double, 2, 2, PX, PY, PZ>(30, 9, 8) +
           lin<float, 4, 0, PX, PY, PZ>(12, 9, 8) + lin<float, 4, 2, PX, PY, PZ>(8, 8, 8);
}

int main() {
    int fails = lin_all<0, 0, 0>() + lin_all<1, 0, 0>() + lin_all<0, 1, 0>() + lin_all<0, 0, 1>() +
                lin_all<1, 1, 1>();
    for (int gx : {2, 3}) {
        fails += split<double, 2, 0, 1, 0>(66, 40, 8, gx);
        fails += split<double, 1, 1, 0, 0>(33, 40, 8, gx);
        fails += split<float, 4, 1, 1, 1>(64, 90, 8, gx);
    }
    printf(fails ? "FAIL %d\n" : "ALL OK\n", fails);
    return fails != 0;
}
