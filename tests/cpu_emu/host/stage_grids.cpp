// The launch grids of the explicit stages stay within the device's limit of
// 65536 blocks along y and z, for planes of many cells (a long row of 2M
// cells: more than 65536 blocks of pairs).  The library's host code runs as
// it is; launches are recorded.
#include "../../../nyles_amd/csrc/nyl_api.hip"
#include <sys/mman.h>
#include <cstdio>

static int check(int nx, int ny, int nz, int prec, int order) {
    nyl_desc d;
    memset(&d, 0, sizeof(d));
    d.nx = nx; d.ny = ny; d.nz = nz;
    d.periodic_x = 1;
    d.dx = d.dy = d.dz = d.idx2 = d.idy2 = d.idz2 = d.dx2 = 1.0;
    d.precision = prec;
    d.mg_maxite = 20; d.mg_tol = 1e-6; d.mg_omega = 0.9;
    d.n_tracers = 1;
    d.upwind_a = d.upwind_vf = order;
    nyl_ctx *c = nullptr;
    uint64_t n = 0;
    if (nyl_ctx_create(&d, &c) || nyl_workspace_bytes(c, &n)) return 1;
    void *w = mmap(nullptr, n, PROT_READ | PROT_WRITE, MAP_PRIVATE | MAP_ANONYMOUS | MAP_NORESERVE,
                   -1, 0);
    if (w == MAP_FAILED || nyl_bind_workspace(c, w, n)) return 1;
    emu_launches.clear();
    int bad = nyl_rhs(c, 0, 0) != NYL_OK;
    for (int st = 1; st <= 3; st++) bad += nyl_rk3_stage(c, st, 0.1) != NYL_OK;
    for (const EmuLaunch &l : emu_launches)
        if (l.grid.y > 65536 || l.grid.z > 65536) {
            if (bad++ < 3) printf("  %s: grid %u x %u x %u\n", l.name.c_str(), l.grid.x, l.grid.y, l.grid.z);
        }
    printf("%dx%dx%d precision %d order %d: %d launches, %d faults\n", nx, ny, nz, prec, order,
           (int)emu_launches.size(), bad);
    munmap(w, n);
    nyl_ctx_destroy(c);
    return bad != 0;
}

int main() {
    int fails = 0;
    for (int order : {0, 3}) {
        fails += check(2097216, 16, 8, NYL_PREC_FP64, order);
        fails += check(262144, 16, 8, NYL_PREC_MIXED, order);
        fails += check(64, 32, 32, NYL_PREC_FP64, order);
    }
    printf(fails ? "FAIL %d\n" : "ALL OK\n", fails);
    return fails != 0;
}
