// Stage kernel with one or 16 bytes of cells per thread (k_stage_flat)
// against the per-cell kernel (k_stage), bit for bit: every mode and
// periodicity, rows of one group to several tiles, planes that leave a block
// partly filled, the smallest wall axes (8 cells); with the model variants
// and the linear branches, 16 bytes of cells against one.  And the FP64 WENO5 with
// its short division against the reference's expression, over magnitudes
// that leave the short division's range (zeros, subnormals, overflow, inf,
// NaN).
#define NYL_STAGE_SEQ 0
#include "../../nyles_amd/csrc/nyl_stage.h"
#include "emu.h"
#include <cmath>
#include <limits>
using namespace nyl;

// core/weno.f90:25-54 as written
static double weno5_ref(double qmm, double qm, double q0, double qp, double qpp) {
    const double eps = 1e-16f;
    const double c13 = 1.0f / 3.0f, c76 = 7.0f / 6.0f, c116 = 11.0f / 6.0f;
    const double c16 = 1.0f / 6.0f, c56 = 5.0f / 6.0f, k1 = 13.0f / 12.0f, k2 = 0.25;
    const double qi1 = c13 * qmm - c76 * qm + c116 * q0;
    const double qi2 = -(c16 * qm) + c56 * q0 + c13 * qp;
    const double qi3 = c13 * q0 + c56 * qp - c16 * qpp;
    const double t1 = qmm - 2.0 * qm + q0, t2 = qmm - 4.0 * qm + 3.0 * q0;
    const double beta1 = k1 * (t1 * t1) + k2 * (t2 * t2);
    const double t3 = qm - 2.0 * q0 + qp, t4 = qm - qp;
    const double beta2 = k1 * (t3 * t3) + k2 * (t4 * t4);
    const double t5 = q0 - 2.0 * qp + qpp, t6 = 3.0 * q0 - 4.0 * qp + qpp;
    const double beta3 = k1 * (t5 * t5) + k2 * (t6 * t6);
    const double tau5 = (float)fabs(beta1 - beta3);
    const double w1 = 1.0 + tau5 / (beta1 + eps);
    const double w2 = 6.0 * (1.0 + tau5 / (beta2 + eps));
    const double w3 = 3.0 * (1.0 + tau5 / (beta3 + eps));
    return (w1 * qi1 + w2 * qi2 + w3 * qi3) / (w1 + w2 + w3);
}

static int check_weno5() {
    std::mt19937_64 rng(7);
    std::normal_distribution<double> nd;
    std::uniform_int_distribution<int> kind(0, 11);
    const int ex[] = {-1074, -1022, -600, -300, -60, -27, 0, 20, 62, 64, 126, 200, 511, 900, 1022};
    std::uniform_int_distribution<int> pick(0, (int)(sizeof(ex) / sizeof(ex[0])) - 1);
    int bad = 0;
    for (int r = 0; r < 400000; r++) {
        const int e = ex[pick(rng)], mix = kind(rng);
        const double base = mix == 1 ? ldexp(nd(rng), e) : 0.0;   // a constant plus small differences
        double q[5];
        for (double &x : q) {
            x = ldexp(nd(rng), mix == 2 ? ex[pick(rng)] : e);
            if (mix == 1) x = base + ldexp(x, -40);
            if (mix == 3 && kind(rng) < 6) x = kind(rng) & 1 ? 0.0 : -0.0;
            if (mix == 4 && kind(rng) == 0) x = std::numeric_limits<double>::infinity();
            if (mix == 5 && kind(rng) == 0) x = std::numeric_limits<double>::quiet_NaN();
        }
        const double a = weno5<double>(q[0], q[1], q[2], q[3], q[4]);
        const double b = weno5_ref(q[0], q[1], q[2], q[3], q[4]);
        if (a != a && b != b) continue;
        if (memcmp(&a, &b, 8) != 0) {
            if (bad++ < 5) printf("weno5(%a %a %a %a %a) = %a, want %a\n", q[0], q[1], q[2], q[3], q[4], a, b);
        }
    }
    printf("weno5: %d mismatches\n", bad);
    return bad != 0;
}

template <typename T, int N, int MODE, int PX, int PY, int PZ>
int check_mode(const Geo &g, StageArgs<T> a1, StageArgs<T> a2, std::vector<std::vector<T>> &o1,
               std::vector<std::vector<T>> &o2, int lw) {
    run_blocks(cell_grid(g), dim3(NYL_BX, NYL_BY, 1),
               [&]() { k_stage<T, MODE, PX, PY, PZ>(g, a1); }, false);
    const int nxg = g.nx / N, rows = STAGE_NT >> lw;
    const dim3 grd = lw ? dim3((nxg + (1 << lw) - 1) >> lw, (g.ny + rows - 1) / rows, g.nz)
                        : dim3(1, (nxg * g.ny + STAGE_NT - 1) / STAGE_NT, g.nz);
    run_blocks(grd, dim3(STAGE_NT, 1, 1),
               [&]() { k_stage_flat<T, N, MODE, PX, PY, PZ>(g, a2, lw); }, false);
    int b = 0;
    for (int f = 0; f < 12; f++) b += ndiff(o1[f], o2[f]);
    return b;
}

// the linear branches and the model variants: N cells per thread against one
template <typename T, int N, int MODE, int PX, int PY, int PZ>
int check_lin(const Geo &g, StageArgs<T> a1, StageArgs<T> a2, std::vector<std::vector<T>> &o1,
              std::vector<std::vector<T>> &o2, int k) {
    const int orders[][3] = {{1, 1, 0}, {3, 5, 0}, {5, 3, 0}, {5, 0, NYL_SF_NO_B}, {0, 0, NYL_SF_NO_VF}};
    const int *o = orders[k];
    for (StageArgs<T> *a : {&a1, &a2}) { a->upw_a = o[0]; a->upw_vf = o[1]; a->flags = o[2]; }
    auto grd = [&](int n) { return dim3(1, (g.nx / n * g.ny + STAGE_NT - 1) / STAGE_NT, g.nz); };
    run_blocks(grd(1), dim3(STAGE_NT, 1, 1),
               [&]() { k_stage_flat<T, 1, MODE, PX, PY, PZ, true>(g, a1, 0); }, false);
    run_blocks(grd(N), dim3(STAGE_NT, 1, 1),
               [&]() { k_stage_flat<T, N, MODE, PX, PY, PZ, true>(g, a2, 0); }, false);
    int b = 0;
    for (int f = 0; f < 12; f++) b += ndiff(o1[f], o2[f]);
    return b;
}

template <typename T, int N, int PX, int PY, int PZ>
int check(int nx, int ny, int nz, int lw, int visc) {
    const Geo g = mk(nx, ny, nz, PX, PY, PZ);
    const size_t n = (size_t)nx * ny * nz;
    std::mt19937_64 rng(3 * nx + 5 * ny + 7 * nz + PX + 2 * PY + 4 * PZ);
    std::vector<std::vector<T>> in(19);
    for (auto &v : in) v = rnd<T>(n, rng);
    for (int f = 1; f <= 3; f++)   // exact zeros: the u > 0 / u <= 0 split
        for (size_t q = 0; q < n; q += 7) in[f][q] = T(0);
    int bad = 0;
    for (int run = 0; run <= 5 + (N > 1 && PX == PY ? 10 : 0); run++) {
        const int mode = run <= 5 ? run : (run <= 10 ? 1 : 3);
        std::vector<std::vector<T>> o1(12), o2;
        for (int f = 0; f < 12; f++) o1[f] = f < 4 ? in[11 + f] : (f < 8 ? std::vector<T>(n, T(5)) : in[15 + f - 8]);
        o2 = o1;
        auto args = [&](std::vector<std::vector<T>> &o) {
            StageArgs<T> a;
            memset(&a, 0, sizeof(a));
            a.b = in[0].data(); a.u = in[1].data(); a.v = in[2].data(); a.w = in[3].data();
            a.bn = o[0].data(); a.un = o[1].data(); a.vn = o[2].data(); a.wn = o[3].data();
            a.ox = in[4].data(); a.oy = in[5].data(); a.oz = in[6].data(); a.ke = in[7].data();
            a.d0b = in[8].data(); a.d0u = in[9].data(); a.d0v = in[10].data(); a.d0w = in[14].data();
            a.d1b = in[11].data(); a.d1u = in[12].data(); a.d1v = in[13].data(); a.d1w = in[18].data();
            a.tb = o[4].data(); a.tu = o[5].data(); a.tv = o[6].data(); a.tw = o[7].data();
            a.sbb = o[8].data(); a.sbu = o[9].data(); a.sbv = o[10].data(); a.sbw = o[11].data();
            a.idx2 = 1.7; a.idy2 = 2.3; a.idz2 = 0.9; a.dz = 0.37;
            a.c = 0.013; a.c2 = 0.026; a.visc = visc;
            a.vcx = 0.011; a.vcy = 0.013; a.vcz = 0.007;
            return a;
        };
        const StageArgs<T> a1 = args(o1), a2 = args(o2);
        int b = 0;
        if (run > 5) {
            if constexpr (N > 1 && PX == PY)
                b = run > 10 ? check_lin<T, N, 3, PX, PY, PZ>(g, a1, a2, o1, o2, run - 11)
                             : check_lin<T, N, 1, PX, PY, PZ>(g, a1, a2, o1, o2, run - 6);
        } else switch (mode) {
        case 0: b = check_mode<T, N, 0, PX, PY, PZ>(g, a1, a2, o1, o2, lw); break;
        case 1: b = check_mode<T, N, 1, PX, PY, PZ>(g, a1, a2, o1, o2, lw); break;
        case 2: b = check_mode<T, N, 2, PX, PY, PZ>(g, a1, a2, o1, o2, lw); break;
        case 3: b = check_mode<T, N, 3, PX, PY, PZ>(g, a1, a2, o1, o2, lw); break;
        case 4: b = check_mode<T, N, 4, PX, PY, PZ>(g, a1, a2, o1, o2, lw); break;
        default: b = check_mode<T, N, 5, PX, PY, PZ>(g, a1, a2, o1, o2, lw); break;
        }
        if (b) printf("  run %d mode %d: %d mismatches\n", run, mode, b);
        bad += b;
    }
    printf("stage_flat<%s, %d> %dx%dx%d p=%d%d%d lw=%d visc=%d: %d mismatches\n",
           sizeof(T) == 8 ? "f64" : "f32", N, nx, ny, nz, PX, PY, PZ, lw, visc, bad);
    return bad != 0;
}

template <int PX, int PY, int PZ>
int all() {
    int f = 0;
    f += check<double, 2, PX, PY, PZ>(8, 8, 8, 0, 1);     // the smallest axes, four pairs a row
    f += check<double, 2, PX, PY, PZ>(30, 9, 8, 0, 0);    // 135 pairs: rows across waves
    f += check<double, 2, PX, PY, PZ>(32, 32, 9, 3, 0);   // whole tiles
    f += check<double, 1, PX, PY, PZ>(33, 8, 8, 0, 1);    // an odd row
    f += check<float, 4, PX, PY, PZ>(8, 8, 8, 0, 1);      // two groups a row
    f += check<float, 4, PX, PY, PZ>(12, 9, 8, 0, 0);     // three
    f += check<float, 4, PX, PY, PZ>(72, 17, 8, 0, 0);    // past one block
    f += check<float, 1, PX, PY, PZ>(22, 13, 8, 0, 1);
    return f;
}

int main() {
    int fails = check_weno5();
    fails += all<0, 0, 0>() + all<1, 0, 0>() + all<0, 1, 0>() + all<1, 1, 0>();
    fails += all<0, 0, 1>() + all<1, 0, 1>() + all<0, 1, 1>() + all<1, 1, 1>();
    printf(fails ? "FAIL %d\n" : "ALL OK\n", fails);
    return fails != 0;
}
