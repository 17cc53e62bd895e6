// nyl_march.hip -- the passes of a multigrid V-cycle over one level: sweeps,
// prolongation, residual and restriction fused into one 2.5-D march, for
// levels of any size.
#include "nyl_march.h"

#include <type_traits>

namespace nyl {

// periodic wrap of any offset
__device__ __forceinline__ int wrap_any(int m, int n) {
    const int r = m % n;
    return r < 0 ? r + n : r;
}

// A block owns a TX x TY tile of columns (TY = 512 / TX) and marches up kz
// planes.  Thread (tx, ty) owns rows 2 ty and 2 ty + 1 of column tx, and one
// cell of each of the R rings around the tile (R = the number of in-plane
// stencils applied one after another: sweeps, and the residual of a
// restriction).  Stage 0 is the input, stage s the s-th sweep; stage s is
// evaluated on the tile and its first R - s rings.  A position keeps the
// planes m-1, m, m+1 of a stage in registers (z neighbours) and its in-plane
// neighbours come from LDS, two slots per stage: in step p the block stores
// plane p of stage 0, passes one barrier, evaluates stage 1 of plane p, stage
// 2 of plane p-1 (whose neighbours were stored in step p-1) and the residual
// one plane later still.  A slot is written again two steps after it was
// read, with a barrier between.  Loads are issued two steps ahead of their
// use, from valid addresses (clamped or wrapped), and values outside a wall
// are replaced by zero when they enter the window.
// PROLONG: the input is src + P(xc); a coarse plane is staged in LDS every
// second step and every position keeps the planar sums (9,3,3,1) of the two
// latest ones, so each is evaluated once for the two fine planes that use it.
// Every value is the per-cell kernel's expression (sweep_cell, residual_at,
// restrict_cell, prolong_term) in its order, so the results are bitwise those
// of the separate launches.
// STRIPS (the norm alone): thread (tx, ty) owns rows ty and ty + TY/2, so that
// its sum runs over the cells, in the order, of a thread of k_mg_sweep2t.
template <typename T, typename TC, int TX, int SRC, int NSW, bool RESN, bool RESTR, bool OUTER,
          bool XADD = false, bool LONG = false, bool STRIPS = false>
__device__ __forceinline__ void march_body(const MarchArgs<T, TC> &a, const MGTabs &tab,
                                           const Blk3 &bk, int nb) {
    static_assert(!STRIPS || (SRC == MS_FIELD && NSW == 0 && RESN && !RESTR), "the norm alone");
    constexpr int TY = 512 / TX;
    constexpr int R = RESTR ? NSW + 1 : (NSW > 0 ? NSW : 1);
    constexpr int NP = 2 + R;                       // own cells, then one per ring
    constexpr int N1 = NSW > 0 ? 1 + R : 0;         // positions of stage 1
    constexpr int N2 = NSW == 2 ? R : 0;            // ... and of stage 2
    constexpr int NB = NSW > 0 ? N1 : 2;            // positions that read b
    constexpr int W0 = TX + 2 * R, H0 = TY + 2 * R;
    constexpr int W1 = W0 - 2, H1 = H0 - 2, W2 = W0 - 4, H2 = H0 - 4;
    constexpr bool LDS1 = NSW == 2 || (RESTR && NSW == 1), LDS2 = NSW == 2 && RESTR;
    constexpr int CW = TX / 2 + 4, CH = TY / 2 + 4, NC = CW * CH;   // coarse footprint (R = 2)
    constexpr int CR = (NC + 255) / 256;
    __shared__ T s0[SRC == MS_ZERO ? 1 : 2 * W0 * H0];
    __shared__ T s1[LDS1 ? 2 * W1 * H1 : 1];
    __shared__ T s2[LDS2 ? 2 * W2 * H2 : 1];
    __shared__ T sc[SRC == MS_PROLONG ? 3 * NC : 1];
    __shared__ T sid[8], spc[8];
    __shared__ TC sidc[8];
    const Geo &g = a.g, &gc = a.gc;
    const int tid = threadIdx.x, tx = tid % TX, ty = tid / TX;
    const int i0 = bk.x * TX, j0 = bk.y * TY, k0 = bk.z * a.kz;
    const int nz = g.nz, k1 = k0 + a.kz < nz ? k0 + a.kz : nz;
    const bool pz = g.pz != 0;
    const T om = T(a.omega), cff1 = T(1.0 - a.omega);
    if (tid < 7) {
        sid[tid] = T(tab.idiag[tid]);
        sidc[tid] = TC(tab.idiag[tid]);
    }
    if (tid < 8) spc[tid] = T(tab.pcoef[tid]);

    // positions: in-plane offset, domain test, in-plane neighbour count, place
    // in the stage-0 plane; own cells: also whether the cell is stored
    int off[NP], nxy[NP], at[NP], ay[NP];
    bool in[NP], has[NP], st[2];
    int cb[NP], cdx[NP], cdy[NP], mxy[NP];          // PROLONG: coarse cell, its neighbours
#pragma unroll
    for (int p = 0; p < NP; p++) {
        int lx, ly;
        has[p] = true;
        if (p < 2) {
            lx = tx + R;
            ly = (STRIPS ? ty + p * (TY / 2) : 2 * ty + p) + R;
        } else {
            const int q = p - 1, W = TX + 2 * q, H = TY + 2 * q;
            // rings 1 and 3 belong to the first threads, ring 2 to the last
            const int t = q == 2 ? 255 - tid : tid;
            has[p] = t < 2 * W + 2 * (H - 2);
            const int u = t - 2 * W;
            lx = t < W ? t : (t < 2 * W ? t - W : ((u & 1) ? W - 1 : 0));
            ly = t < W ? 0 : (t < 2 * W ? H - 1 : 1 + (u >> 1));
            lx += R - q;
            ly += R - q;
            if (!has[p]) lx = ly = 0;
        }
        at[p] = ly * W0 + lx;
        ay[p] = ly;
        const int ui = i0 - R + lx, uj = j0 - R + ly;   // unwrapped
        int gi = ui, gj = uj;
        bool ok = has[p];
        if (g.px) gi = wrap_any(ui, g.nx); else ok = ok && ui >= 0 && ui < g.nx;
        if (g.py) gj = wrap_any(uj, g.ny); else ok = ok && uj >= 0 && uj < g.ny;
        in[p] = ok;
        off[p] = ok ? gj * (int)g.sy + gi : 0;
        nxy[p] = (g.px || gi > 0) + (g.px || gi < g.nx - 1) + (g.py || gj > 0) +
                 (g.py || gj < g.ny - 1);
        if (!ok) nxy[p] = 0;
        if (p < 2) st[p] = ok && ui < g.nx && uj < g.ny;
        if (SRC == MS_PROLONG) {
            const int ic = ui >> 1, jc = uj >> 1;
            cdx[p] = (ui & 1) ? 1 : -1;
            cdy[p] = (uj & 1) ? CW : -CW;
            const int icn = ic + cdx[p], jcn = jc + ((uj & 1) ? 1 : -1);
            mxy[p] = ((gc.px || (icn >= 0 && icn < gc.nx)) ? 1 : 0) +
                     ((gc.py || (jcn >= 0 && jcn < gc.ny)) ? 2 : 0);
            cb[p] = (jc - ((j0 >> 1) - 2)) * CW + ic - ((i0 >> 1) - 2);
        }
    }
    __syncthreads();   // sid, spc
    T id2[NP], pc1[NP];   // the coefficients of planes with both z neighbours
#pragma unroll
    for (int p = 0; p < NP; p++) {
        id2[p] = sid[nxy[p] + 2];
        if (SRC == MS_PROLONG) pc1[p] = spc[mxy[p] + 4];
    }

    auto zin = [&](int m) { return pz || (m >= 0 && m < nz); };
    auto nzw = [&](int m) { return pz ? 2 : (m > 0) + (m < nz - 1); };
    // a plane that can be loaded for plane m: the wrapped one, or the nearest
    auto pl = [&](int m, int n, bool per) {
        return per ? wrap_any(m, n) : (m < 0 ? 0 : (m < n ? m : n - 1));
    };
    auto next = [&](int q, int m, int n, bool per) {   // pl(m + 1) from q = pl(m)
        return per ? (q + 1 == n ? 0 : q + 1) : (m + 1 < 0 ? 0 : (m + 1 < n ? m + 1 : n - 1));
    };
    auto ldx = [&](int q, T (&v)[NP]) {
        if (SRC == MS_ZERO) return;
        const T *s = a.src + (int64_t)q * g.sz;
#pragma unroll
        for (int p = 0; p < NP; p++) v[p] = s[off[p]];
    };
    auto ldb = [&](int q, T (&v)[NB]) {
        const T *s = a.b + (int64_t)q * g.sz;
#pragma unroll
        for (int p = 0; p < NB; p++) v[p] = s[off[p]];
    };

    // ---- coarse planes (PROLONG)
    int coff[CR];
    bool cin[CR];
    T A0[NP] = {}, A1[NP] = {}, craw[CR] = {};
    if (SRC == MS_PROLONG) {
#pragma unroll
        for (int r = 0; r < CR; r++) {
            const int t = tid + 256 * r;
            const int lx = t % CW, ly = t / CW;
            int gi = (i0 >> 1) - 2 + lx, gj = (j0 >> 1) - 2 + ly;
            bool ok = t < NC;
            if (gc.px) gi = wrap_any(gi, gc.nx); else ok = ok && gi >= 0 && gi < gc.nx;
            if (gc.py) gj = wrap_any(gj, gc.ny); else ok = ok && gj >= 0 && gj < gc.ny;
            cin[r] = ok;
            coff[r] = ok ? gj * (int)gc.sy + gi : 0;
        }
    }
    auto czin = [&](int m) { return pz || (m >= 0 && m < gc.nz); };
    auto ldc = [&](int m) {
        const TC *s = a.xc + (int64_t)pl(m, gc.nz, pz) * gc.sz;
#pragma unroll
        for (int r = 0; r < CR; r++) craw[r] = T(s[coff[r]]);
    };
    auto putc = [&](int m, int slot) {   // zero outside the domain
        const bool zi = czin(m);
#pragma unroll
        for (int r = 0; r < CR; r++)
            if (tid + 256 * r < NC) sc[slot * NC + tid + 256 * r] = (zi && cin[r]) ? craw[r] : T(0);
    };
    auto planar = [&](int slot, T (&A)[NP]) {
        const T *c = sc + slot * NC;
#pragma unroll
        for (int p = 0; p < NP; p++) {
            if (p >= 2 && !has[p]) continue;
            A[p] = T(9) * c[cb[p]] + T(3) * c[cb[p] + cdx[p]] + T(3) * c[cb[p] + cdy[p]] +
                   c[cb[p] + cdx[p] + cdy[p]];
        }
    };
    // stage-0 values of plane m from the raw loads; PROLONG: lo, hi the planar
    // sums of the coarse planes around it (lo the lower one), par the parity of m
    auto enter = [&](auto par, auto inner, int m, const T (&v)[NP], const T (&lo)[NP],
                     const T (&hi)[NP], T (&out)[NP]) {
        constexpr bool odd = decltype(par)::value != 0, FAST = decltype(inner)::value;
        const bool zi = FAST || zin(m);
        const bool mz = FAST || (SRC == MS_PROLONG && czin(odd ? (m >> 1) + 1 : (m >> 1) - 1));
#pragma unroll
        for (int p = 0; p < NP; p++) {
            T t = v[p];
            if (SRC == MS_PROLONG) {
                const T bmid = odd ? lo[p] : hi[p], aside = odd ? hi[p] : lo[p];
                T pc = pc1[p];
                if (!mz) pc = spc[mxy[p]];
                t = t + pc * (T(3) * bmid + aside);
            }
            out[p] = (zi && in[p]) ? t : T(0);
        }
    };
    using Even = std::integral_constant<int, 0>;
    using Odd = std::integral_constant<int, 1>;
    using Edge = std::false_type;
    using Inner = std::true_type;

    const int p0 = k0 - (R - 1), p1 = k1 - 1 + (R - 1);
    // windows: stage 0 planes p-1, p, p+1; stage 1 planes p-2, p-1, p; stage 2
    // planes p-3, p-2, p-1; b of planes p, p-1, p-2
    T I0[NP] = {}, I1[NP] = {}, I2[NP] = {};
    T M0[N1 > 0 ? N1 : 2] = {}, M1[N1 > 0 ? N1 : 2] = {}, M2[N1 > 0 ? N1 : 2] = {};
    T K0[2] = {}, K1[2] = {}, K2[N2 > 0 ? N2 : 2] = {};
    T B0[NB] = {}, B1[NB] = {}, B2[2] = {};
    T xa[NP] = {}, xb[NP] = {}, ba[NB] = {}, bb[NB] = {};
    T racc = T(0);
    double acc = 0.0;
    const double shift = OUTER && a.shift ? *a.shift : 0.0;
    {
        T x0[NP] = {}, x1[NP] = {}, x2[NP] = {};
        ldx(pl(p0 - 1, nz, pz), x0);
        ldx(pl(p0, nz, pz), x1);
        ldx(pl(p0 + 1, nz, pz), x2);
        ldx(pl(p0 + 2, nz, pz), xa);
        ldb(pl(p0, nz, pz), B0);
        ldb(pl(p0 + 1, nz, pz), ba);
        if (SRC == MS_PROLONG) {
            // p0 - 1 = 2 kc, so the three planes use the coarse planes kc-1, kc, kc+1
            const int kc = (p0 - 1) >> 1;
            ldc(kc - 1);
            putc(kc - 1, 0);
            ldc(kc);
            putc(kc, 1);
            ldc(kc + 1);
            putc(kc + 1, 2);
            __syncthreads();
            T Am[NP] = {};
            planar(0, Am);
            planar(1, A0);
            planar(2, A1);
            enter(Even(), Edge(), p0 - 1, x0, Am, A0, I0);
            enter(Odd(), Edge(), p0, x1, A0, A1, I1);
            enter(Even(), Edge(), p0 + 1, x2, A0, A1, I2);
            ldc(kc + 2);
            __syncthreads();   // slot 0 is written again in the first step
        } else if (SRC == MS_FIELD) {
            enter(Even(), Edge(), p0 - 1, x0, A0, A1, I0);
            enter(Even(), Edge(), p0, x1, A0, A1, I1);
            enter(Even(), Edge(), p0 + 1, x2, A0, A1, I2);
        }
    }
    int qx = pl(p0 + 3, nz, pz), qb = pl(p0 + 2, nz, pz);

    // place of position p in the plane of stage e
    auto place = [&](int p, int e) { return at[p] - e * (W0 + 1) - 2 * e * (ay[p] - e); };
    // sum of the x-, x+, y-, y+, z-, z+ neighbours of position p in the plane P
    // of stage e; the two own cells are each other's y neighbours (not in STRIPS)
    auto six = [&](const T *P, int e, int p, const T (&c)[2], T zm, T zp) -> T {
        const int q = place(p, e), W = W0 - 2 * e;
        const T xm = P[q - 1], xp = P[q + 1];
        const T ym = !STRIPS && p == 1 ? c[0] : P[q - W];
        const T yp = !STRIPS && p == 0 ? c[1] : P[q + W];
        return xm + xp + ym + yp + zm + zp;
    };

    // One step; ph alternates 0, 1 from the first one.  The march of a
    // restriction or prolongation starts on an even plane k0, so there ph = 0
    // is an odd p of a prolongation (p0 = k0 - 1) and an even residual plane.
    // inner: a step whose planes all have both z neighbours and are all the
    // block's own, so that nothing depends on z (the march is latency-bound:
    // two waves per SIMD, and a branch per position and stage costs as much as
    // its arithmetic).
    auto step = [&](auto ph, auto inner, int p, T (&xu)[NP], T (&xn)[NP], T (&bu)[NB], T (&bn)[NB]) {
        constexpr int A = decltype(ph)::value, B = 1 - A;   // slots of planes p, p - 1
        constexpr bool FAST = decltype(inner)::value;
        constexpr bool pair = SRC == MS_PROLONG && A == 0;  // a new coarse plane this step
        if (SRC != MS_ZERO) {
            T *P = s0 + A * (W0 * H0);
#pragma unroll
            for (int q = 0; q < NP; q++)
                if (q < 2 || has[q]) P[at[q]] = I1[q];
        }
        if (pair) {
            putc((p + 3) >> 1, 0);
            if (p + 2 <= p1 + 1) ldc(((p + 3) >> 1) + 1);
        }
        // (always issued, past the end from the last plane again: behind a
        // condition the compiler waits for the loads of this step where it
        // needs those of the one before)
        ldx(qx, xn);
        ldb(qb, bn);
        __syncthreads();
        // residual of the input, and stage 1 of plane p
        const T *P0 = s0 + A * (W0 * H0);
        const bool z0 = FAST || zin(p);
        const int n0 = FAST ? 2 : nzw(p);
        T *P1 = s1 + A * (W1 * H1);
#pragma unroll
        for (int q = 0; q < (NSW > 0 ? N1 : 2); q++) {
            if (q >= 2 && !has[q]) continue;
            T S = T(0);
            if (SRC != MS_ZERO) {
                const T own[2] = {I1[0], I1[1]};
                S = six(P0, 0, q, own, I0[q], I2[q]);
            }
            if (RESN && q < 2 && (FAST || (p >= k0 && p < k1)) && st[q]) {
                const T d = T(nxy[q] + n0);
                if constexpr (OUTER) {
                    const double rr = (B0[q] - shift) + d * I1[q] - S;
                    acc = acc + rr * rr;
                    if (a.rout) a.rout[(int64_t)p * g.sz + off[q]] = float(rr);
                } else {
                    const double rr = (double)(B0[q] + d * I1[q] - S);
                    acc = acc + rr * rr;
                }
            }
            if constexpr (NSW > 0) {
                T id = id2[q];
                if (!FAST && n0 != 2) id = sid[nxy[q] + n0];
                const T v = cff1 * I1[q] + om * (S - B0[q]) * id;
                M2[q] = (z0 && in[q]) ? v : T(0);
                if (LDS1) P1[place(q, 1)] = M2[q];
                if (NSW == 1 && q < 2 && (FAST || (p >= k0 && p < k1)) && st[q])
                    a.dst[(int64_t)p * g.sz + off[q]] = M2[q];
            }
        }
        // stage 2 of plane p - 1
        const int m = p - 1;
        const T *Q1 = s1 + B * (W1 * H1);
        const int n1 = FAST ? 2 : nzw(m);
        const bool z1 = FAST || zin(m);
        if constexpr (NSW == 2) {
            if (FAST || (m >= p0 && m >= k0 - (R - 2))) {
                T *P2 = s2 + B * (W2 * H2);
#pragma unroll
                for (int q = 0; q < N2; q++) {
                    if (q >= 2 && !has[q]) continue;
                    const T own[2] = {M1[0], M1[1]};
                    const T S = six(Q1, 1, q, own, M0[q], M2[q]);
                    T id = id2[q];
                    if (!FAST && n1 != 2) id = sid[nxy[q] + n1];
                    const T v = cff1 * M1[q] + om * (S - B1[q]) * id;
                    if (RESTR) {
                        K2[q] = (z1 && in[q]) ? v : T(0);
                        P2[place(q, 2)] = K2[q];
                    }
                    if (q < 2 && (FAST || (m >= k0 && m < k1)) && st[q]) {
                        const int64_t c = (int64_t)m * g.sz + off[q];
                        if (XADD) a.xadd[c] = a.xadd[c] + (double)v;
                        else a.dst[c] = v;
                    }
                }
            }
        }
        // residual of the last stage and its restriction
        if constexpr (RESTR) {
            const int k = p - NSW;
            if (FAST || (k >= k0 && k < k1)) {
                const T *Q = NSW == 2 ? s2 + A * (W2 * H2) : (NSW == 1 ? Q1 : P0);
                const int nk = FAST ? 2 : nzw(k);
                T r[2];
#pragma unroll
                for (int q = 0; q < 2; q++) {
                    const T own[2] = {NSW == 2 ? K1[0] : (NSW == 1 ? M1[0] : I1[0]),
                                      NSW == 2 ? K1[1] : (NSW == 1 ? M1[1] : I1[1])};
                    const T zm = NSW == 2 ? K0[q] : (NSW == 1 ? M0[q] : I0[q]);
                    const T zp = NSW == 2 ? K2[q] : (NSW == 1 ? M2[q] : I2[q]);
                    const T S = six(Q, NSW, q, own, zm, zp);
                    const T bv = NSW == 2 ? B2[q] : (NSW == 1 ? B1[q] : B0[q]);
                    r[q] = bv + T(nxy[q] + nk) * own[q] - S;
                }
                const T rx0 = __shfl_down(r[0], 1), rx1 = __shfl_down(r[1], 1);
                if constexpr (A == 0) {
                    racc = ((r[0] + rx0) + r[1]) + rx1;
                } else {
                    racc = (((racc + r[0]) + rx0) + r[1]) + rx1;
                    const int ic = (i0 + tx) >> 1, jc = (j0 >> 1) + ty, kc = k >> 1;
                    if ((tx & 1) == 0 && ic < gc.nx && jc < gc.ny) {
                        const int64_t cc = (int64_t)kc * gc.sz + (int64_t)jc * gc.sy + ic;
                        const TC bv = TC(T(0.5) * racc);
                        const int nw = (gc.px || ic > 0) + (gc.px || ic < gc.nx - 1) +
                                       (gc.py || jc > 0) + (gc.py || jc < gc.ny - 1) +
                                       (gc.pz || kc > 0) + (gc.pz || kc < gc.nz - 1);
                        a.bc[cc] = bv;
                        // the coarse level's first sweep from x = 0
                        const TC omc = TC(a.omega), c1 = TC(1.0 - a.omega);
                        a.yc[cc] = c1 * TC(0) + omc * (TC(0) - bv) * sidc[nw];
                    }
                }
            }
        }
        // the next plane
        if (pair) {
#pragma unroll
            for (int q = 0; q < NP; q++) A0[q] = A1[q];
            planar(0, A1);
        }
        T In[NP];
        // (p + 2 is odd in the steps that bring a coarse plane)
        if (SRC != MS_ZERO)
            enter(std::integral_constant<int, B>(), inner, p + 2, xu, A0, A1, In);
#pragma unroll
        for (int q = 0; q < NP; q++) {
            I0[q] = I1[q];
            I1[q] = I2[q];
            if (SRC != MS_ZERO) I2[q] = In[q];
        }
#pragma unroll
        for (int q = 0; q < N1; q++) {
            M0[q] = M1[q];
            M1[q] = M2[q];
        }
#pragma unroll
        for (int q = 0; q < 2; q++) {
            if (NSW == 2 && RESTR) {
                K0[q] = K1[q];
                K1[q] = K2[q];
            }
            B2[q] = B1[q];
        }
#pragma unroll
        for (int q = 0; q < NB; q++) {
            B1[q] = B0[q];
            B0[q] = bu[q];
        }
        if (p + 3 <= p1) qx = next(qx, p + 3, nz, pz);
        if (p + 2 < p1) qb = next(qb, p + 2, nz, pz);
    };
    auto inside = [&](int p) {
        return p - 2 >= k0 && p < k1 && (pz || (p > 2 && p + 3 < nz));
    };
    for (int p = p0; p <= p1; p += 2) {
        if constexpr (LONG) {
            if (inside(p) && inside(p + 1)) {
                step(Even(), Inner(), p, xa, xb, ba, bb);
                step(Odd(), Inner(), p + 1, xb, xa, bb, ba);
                continue;
            }
        }
        step(Even(), Edge(), p, xa, xb, ba, bb);
        if (p + 1 <= p1) step(Odd(), Edge(), p + 1, xb, xa, bb, ba);
    }
    if (RESN) {
        __syncthreads();
        block_sum_store(acc, a.partials + nb, tid);
    }
}

// LONG: with the steps inside the march as a path of its own, and the
// registers held to the residency that march_grid counts on.  For marches of
// 16 planes or more with sweeps: pre-smoothing with restriction + post-
// smoothing FP64 256^3 252 -> 238 us, FP32 256^3 136 -> 126, 256x256x512
// 279 -> 271; in short marches the second copy of the code costs more than
// its few steps gain (96^3: 35.5 -> 36.6).  The limit costs a few spills: 6 of
// the 128 registers of the FP32 prolongation march (28 bytes of scratch per
// lane, 2 and 12 with 32 columns), 1 of the 256 of the FP64 pre-smoothing with
// restriction and norm; the times above include them.
template <typename T, int SRC, int NSW, bool RESTR, bool LONG>
constexpr int march_waves() {
    return LONG ? march_resident(sizeof(T), SRC, NSW, RESTR) : 1;
}
constexpr int MARCH_LONG = 16;

template <typename T, typename TC, int TX, int SRC, int NSW, bool RESN, bool RESTR, bool OUTER,
          bool LONG = false, bool STRIPS = false>
__global__ __launch_bounds__(256, (march_waves<T, SRC, NSW, RESTR, LONG>())) void k_mg_march(
    MarchArgs<T, TC> a, MGTabs tab) {
    if (a.gate && *a.gate) return;
    march_body<T, TC, TX, SRC, NSW, RESN, RESTR, OUTER, false, LONG, STRIPS>(
        a, tab, xcd_block(), blockIdx.x + gridDim.x * (blockIdx.y + gridDim.y * blockIdx.z));
}

// The pass over one level of every member of a batch: block b works for item
// map[b], on its block number b - start (x fastest, then y, then z).
template <typename T, typename TC, int SRC, int NSW, bool RESN, bool RESTR, bool OUTER, bool XADD>
__global__ __launch_bounds__(256) void k_b_march(const MarchItem<T, TC> *__restrict__ items,
                                                 const uint32_t *__restrict__ map, MGTabs tab,
                                                 const int *__restrict__ active) {
    const MarchItem<T, TC> &it = items[map[blockIdx.x]];
    if (active && !active[it.h.member]) return;
    const MarchArgs<T, TC> a = it.a;
    const int lb = (int)((int64_t)blockIdx.x - it.h.start);
    Blk3 bk;
    bk.x = lb % it.bx;
    const int t = lb / it.bx;
    bk.y = t % it.by;
    bk.z = t / it.by;
    march_body<T, TC, 32, SRC, NSW, RESN, RESTR, OUTER, XADD>(a, tab, bk, lb);
}

// Tile width and march length of a level.  The width (64 or 32 columns, rows
// to match) is the one that pads the level less.  The march is the shortest
// whose blocks are all resident at once (res per CU): a second round of
// blocks waits for the first and repeats its prologue, a longer march leaves
// SIMDs idle.  Measured (us, planes per block: time): prolongation and two
// sweeps FP32 256^3 16: 66, 32: 57, 64: 83; 256x256x512 32: 126, 64: 119;
// FP64 256^3 32: 120, 64: 113; 96^3 2: 23, 4: 16, 8: 19; two sweeps FP64
// 96^3 2: 17, 4: 13, 8: 15.
MarchGrid march_grid(const Geo &g, int res, bool even) {
    auto up = [](int64_t n, int64_t t) { return (int)((n + t - 1) / t); };
    MarchGrid m;
    const int64_t a64 = (int64_t)up(g.nx, 64) * up(g.ny, 8), a32 = (int64_t)up(g.nx, 32) * up(g.ny, 16);
    m.tx = a32 < a64 ? 32 : 64;
    m.bx = up(g.nx, m.tx);
    m.by = up(g.ny, 512 / m.tx);
    const int64_t cols = (int64_t)m.bx * m.by;
    int64_t bz = 256 * (int64_t)res / cols;
    if (bz < 1) bz = 1;
    int kz = up(g.nz, bz);
    if (even && (kz & 1)) kz++;
    if (kz < 2) kz = 2;
    m.kz = kz;
    m.bz = up(g.nz, kz);
    return m;
}

#define MARCH_GO(T, TC, SRC, NSW, RESN, RESTR, OUTER)                                          \
    do {                                                                                      \
        MarchArgs<T, TC> m = a;                                                               \
        const MarchGrid gr = march_grid(a.g, march_resident(sizeof(T), SRC, NSW, RESTR),      \
                                        (RESTR) || (SRC) == MS_PROLONG);                      \
        m.kz = gr.kz;                                                                         \
        const dim3 grd(gr.bx, gr.by, gr.bz), blk(256);                                        \
        const bool lng = (NSW) > 0 && gr.kz >= MARCH_LONG;                                    \
        if (gr.tx == 64 && lng)                                                               \
            NYL_LAUNCH((k_mg_march<T, TC, 64, SRC, NSW, RESN, RESTR, OUTER, (NSW) != 0>), grd, blk, 0, \
                       s, m, a.tab);                                                          \
        else if (gr.tx == 64)                                                                 \
            NYL_LAUNCH((k_mg_march<T, TC, 64, SRC, NSW, RESN, RESTR, OUTER>), grd, blk, 0, s, m, \
                       a.tab);                                                                \
        else if (lng)                                                                         \
            NYL_LAUNCH((k_mg_march<T, TC, 32, SRC, NSW, RESN, RESTR, OUTER, (NSW) != 0>), grd, blk, 0, \
                       s, m, a.tab);                                                          \
        else                                                                                  \
            NYL_LAUNCH((k_mg_march<T, TC, 32, SRC, NSW, RESN, RESTR, OUTER>), grd, blk, 0, s, m, \
                       a.tab);                                                                \
    } while (0)

template <typename T, typename TC>
hipError_t launch_march_up(const MarchArgs<T, TC> &a, hipStream_t s) {
    if (a.src == a.dst || !a.xc) return hipErrorInvalidValue;
    MARCH_GO(T, TC, MS_PROLONG, 2, false, false, false);
    return hipGetLastError();
}

template <typename T, typename TC>
hipError_t launch_march_down(const MarchArgs<T, TC> &a, hipStream_t s) {
    if (a.src == a.dst || !a.bc || !a.yc) return hipErrorInvalidValue;
    MARCH_GO(T, TC, MS_FIELD, 1, false, true, false);
    return hipGetLastError();
}

template <typename T, typename TC>
hipError_t launch_march_pre(const MarchArgs<T, TC> &a, hipStream_t s) {
    if (a.src == a.dst || (!a.src && a.partials) || !a.bc || !a.yc) return hipErrorInvalidValue;
    if (!a.src) MARCH_GO(T, TC, MS_ZERO, 2, false, true, false);
    else if (a.partials) MARCH_GO(T, TC, MS_FIELD, 2, true, true, false);
    else MARCH_GO(T, TC, MS_FIELD, 2, false, true, false);
    return hipGetLastError();
}

MarchGrid march_pre_grid(const Geo &g, int es) {
    return march_grid(g, march_resident(es, MS_FIELD, 2, true), true);
}

template <typename T>
hipError_t launch_march_norm(const MarchArgs<T, T> &a, const MarchGrid &gr, bool strips,
                             hipStream_t s) {
    if (!a.partials || (strips && (gr.tx != 64 || a.g.nx % 64 || a.g.ny % 8)))
        return hipErrorInvalidValue;
    MarchArgs<T, T> m = a;
    m.kz = gr.kz;
    const dim3 grd(gr.bx, gr.by, gr.bz), blk(256);
    if (strips)
        NYL_LAUNCH((k_mg_march<T, T, 64, MS_FIELD, 0, true, false, false, false, true>), grd, blk,
                   0, s, m, a.tab);
    else if (gr.tx == 64)
        NYL_LAUNCH((k_mg_march<T, T, 64, MS_FIELD, 0, true, false, false>), grd, blk, 0, s, m, a.tab);
    else
        NYL_LAUNCH((k_mg_march<T, T, 32, MS_FIELD, 0, true, false, false>), grd, blk, 0, s, m, a.tab);
    return hipGetLastError();
}

hipError_t launch_march_outer(const MarchArgs<double, double> &a, hipStream_t s) {
    if (!a.partials || !a.rout) return hipErrorInvalidValue;
    MARCH_GO(double, double, MS_FIELD, 0, true, false, true);
    return hipGetLastError();
}

static int64_t b_march_tiles(const Geo &g) {
    return (int64_t)((g.nx + 31) / 32) * ((g.ny + 15) / 16);
}

int b_march_kz(const Geo &g) {
    int kz = (int64_t)g.nx * g.ny * g.nz < (1 << 18) ? 4 : 8;
    while (b_march_tiles(g) * ((g.nz + kz - 1) / kz) > NYL_RED_BLOCKS && kz < g.nz) kz *= 2;
    return kz;
}

int64_t b_march_blocks(const Geo &g) {
    const int kz = b_march_kz(g);
    return b_march_tiles(g) * ((g.nz + kz - 1) / kz);
}

template <typename T, typename TC>
hipError_t launch_b_march(const MarchItem<T, TC> *items, const uint32_t *map, int64_t nblk,
                          MarchKind kind, const MGTabs &tab, const int *active, hipStream_t s) {
    const dim3 grd((unsigned)nblk), blk(256);
#define B_GO(SRC, NSW, RESN, RESTR)                                                      \
    NYL_LAUNCH((k_b_march<T, TC, SRC, NSW, RESN, RESTR, false, false>), grd, blk, 0, s, items, \
               map, tab, active)
    switch (kind) {
    case MK_UP: B_GO(MS_PROLONG, 2, false, false); break;
    case MK_UP_ADD:
        if constexpr (sizeof(T) == 4)
            NYL_LAUNCH((k_b_march<T, TC, MS_PROLONG, 2, false, false, false, true>), grd, blk, 0,
                       s, items, map, tab, active);
        else return hipErrorInvalidValue;
        break;
    case MK_DOWN: B_GO(MS_FIELD, 1, false, true); break;
    case MK_RESTRICT: B_GO(MS_FIELD, 0, false, true); break;
    case MK_PRE: B_GO(MS_FIELD, 2, true, false); break;
    case MK_PRE_RESTRICT: B_GO(MS_FIELD, 2, true, true); break;
    case MK_ZERO: B_GO(MS_ZERO, 2, false, false); break;
    case MK_ZERO_RESTRICT: B_GO(MS_ZERO, 2, false, true); break;
    case MK_OUTER:
        if constexpr (sizeof(T) == 8)
            NYL_LAUNCH((k_b_march<T, TC, MS_FIELD, 0, true, false, true, false>), grd, blk, 0, s, items,
                       map, tab, active);
        else return hipErrorInvalidValue;
        break;
    }
#undef B_GO
    return hipGetLastError();
}
template hipError_t launch_b_march<double, double>(const MarchItem<double, double> *,
                                                   const uint32_t *, int64_t, MarchKind,
                                                   const MGTabs &, const int *, hipStream_t);
template hipError_t launch_b_march<float, float>(const MarchItem<float, float> *,
                                                 const uint32_t *, int64_t, MarchKind,
                                                 const MGTabs &, const int *, hipStream_t);
template hipError_t launch_b_march<float, double>(const MarchItem<float, double> *,
                                                  const uint32_t *, int64_t, MarchKind,
                                                  const MGTabs &, const int *, hipStream_t);

#define NYL_MARCH_INST(T, TC)                                                              \
    template hipError_t launch_march_up<T, TC>(const MarchArgs<T, TC> &, hipStream_t);     \
    template hipError_t launch_march_down<T, TC>(const MarchArgs<T, TC> &, hipStream_t);   \
    template hipError_t launch_march_pre<T, TC>(const MarchArgs<T, TC> &, hipStream_t);
NYL_MARCH_INST(double, double)
NYL_MARCH_INST(float, float)
NYL_MARCH_INST(float, double)
template hipError_t launch_march_norm<double>(const MarchArgs<double, double> &, const MarchGrid &,
                                              bool, hipStream_t);
template hipError_t launch_march_norm<float>(const MarchArgs<float, float> &, const MarchGrid &,
                                             bool, hipStream_t);

}  // namespace nyl
