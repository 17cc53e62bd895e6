// The item tables of a batch (nyl_batch.hip) against the members' workspaces:
// every block of a pass with block sums, and every final sum, stays inside
// the member's partials, for members from the smallest to very wide shallow
// ones.  The library's host code runs as it is; launches do nothing, and the
// members' workspaces are reserved addresses of which the host code touches
// only the tables.
#include "../../../nyles_amd/csrc/nyl_batch.hip"
#include <sys/mman.h>
#include <cstdio>

static nyl_ctx *member(int nx, int ny, int nz, int prec, int per) {
    nyl_desc d;
    memset(&d, 0, sizeof(d));
    d.nx = nx; d.ny = ny; d.nz = nz;
    d.periodic_x = per & 1; d.periodic_y = (per >> 1) & 1; d.periodic_z = (per >> 2) & 1;
    d.dx = d.dy = d.dz = d.idx2 = d.idy2 = d.idz2 = d.dx2 = 1.0;
    d.precision = prec;
    d.mg_maxite = 20; d.mg_tol = 1e-6; d.mg_omega = 0.9;
    nyl_ctx *c = nullptr;
    uint64_t n = 0;
    if (nyl_ctx_create(&d, &c) || nyl_workspace_bytes(c, &n)) return nullptr;
    void *w = mmap(nullptr, n, PROT_READ | PROT_WRITE, MAP_PRIVATE | MAP_ANONYMOUS | MAP_NORESERVE,
                   -1, 0);
    if (w == MAP_FAILED || nyl_bind_workspace(c, w, n)) return nullptr;
    return c;
}

// the member whose partials start at p, and how many there are
static uint64_t room(const nyl_batch *b, const double *p) {
    for (nyl_ctx *c : b->m)
        if (F<double>(c, c->partials) == p) return (c->result - c->partials) / sizeof(double);
    return 0;
}

template <typename T, typename TC>
static int marches(const nyl_batch *b, const Launch &L) {
    int bad = 0;
    for (int q = 0; q < L.nitems; q++) {
        const MarchItem<T, TC> &it = ((const MarchItem<T, TC> *)(b->blob.data() + L.off))[q];
        const int64_t cover = (int64_t)it.bx * it.by * ((it.a.g.nz + it.a.kz - 1) / it.a.kz);
        bad += cover != it.h.nblk;
        const bool sums = L.arg == MK_PRE || L.arg == MK_PRE_RESTRICT || L.arg == MK_OUTER;
        if (sums && (uint64_t)it.h.nblk > room(b, it.a.partials)) {
            printf("  %dx%dx%d: %d block sums, room for %llu\n", it.a.g.nx, it.a.g.ny, it.a.g.nz,
                   it.h.nblk, (unsigned long long)room(b, it.a.partials));
            bad++;
        }
    }
    return bad;
}

static int plan(const nyl_batch *b, const std::vector<Launch> &p) {
    int bad = 0;
    for (const Launch &L : p) {
        if (L.kind == L_MARCH)
            bad += L.type == T_F ? marches<float, float>(b, L)
                                 : (L.type == T_FD ? marches<float, double>(b, L)
                                                   : marches<double, double>(b, L));
        if (L.kind == L_RED)
            for (int q = 0; q < L.nitems; q++) {
                const RedItem &it = ((const RedItem *)(b->blob.data() + L.off))[q];
                bad += (uint64_t)it.h.nblk * (L.arg == 2 ? 2 : 1) > room(b, it.partials);
            }
        if (L.kind == L_FINAL)
            for (int q = 0; q < L.nitems; q++) {
                const FinalItem &it = ((const FinalItem *)(b->blob.data() + L.off))[q];
                bad += (uint64_t)it.nparts > room(b, it.partials);
            }
    }
    return bad;
}

int main() {
    struct { int n[3], prec; } cases[] = {
        {{8, 8, 8}, NYL_PREC_FP64}, {{96, 96, 96}, NYL_PREC_FP64}, {{128, 128, 80}, NYL_PREC_FP64},
        {{64, 32, 32}, NYL_PREC_MIXED}, {{128, 128, 80}, NYL_PREC_MIXED},
        {{256, 256, 512}, NYL_PREC_FP64},     // 8-plane marches just inside the room
        {{8, 262160, 8}, NYL_PREC_FP64},      // 16385 tiles of 32 x 16 columns
        {{131136, 64, 32}, NYL_PREC_FP64},    // 16392
        {{16, 524288, 8}, NYL_PREC_FP64},     // 32768
        {{8, 65536, 8}, NYL_PREC_MIXED},      // the widest mixed member
    };
    int fails = 0;
    for (auto &k : cases) {
        nyl_ctx *c = member(k.n[0], k.n[1], k.n[2], k.prec, 3);
        nyl_ctx *small = member(16, 16, 16, k.prec, 0);
        if (!c || !small) {
            printf("%dx%dx%d: no member\n", k.n[0], k.n[1], k.n[2]);
            fails++;
            continue;
        }
        nyl_ctx *both[2] = {small, c};
        nyl_batch *b = nullptr;
        if (nyl_batch_create(both, 2, &b)) {
            printf("%dx%dx%d: no batch\n", k.n[0], k.n[1], k.n[2]);
            fails++;
            continue;
        }
        int bad = plan(b, b->vcyc);
        for (int p = 0; p < 2; p++)
            for (int s = 0; s < 3; s++) bad += plan(b, b->pre[p][s]);
        printf("%dx%dx%d precision %d: %d faults\n", k.n[0], k.n[1], k.n[2], k.prec, bad);
        fails += bad != 0;
        nyl_batch_destroy(b);
    }
    printf(fails ? "FAIL %d\n" : "ALL OK\n", fails);
    return fails != 0;
}
