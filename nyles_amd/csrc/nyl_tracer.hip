// nyl_tracer.hip -- passive tracers: the b part of the stage kernel for another
// scalar, with the stage update of the mode (the same expressions as b's).
#include "nyl_stage.h"

namespace nyl {

// N cells per thread as in k_stage_flat, whose rule chooses N: the tracer of
// 128x64x64 FP64 in a closed box took 23 us with one cell per thread in
// 64-wide rows, 19.7 with two (bound by VALU issue, as the stage kernel).  The
// blocks of a plane lie along y, and along x past the GRID_YZ that y takes.
template <typename T, int N, int MODE, int PX, int PY, int PZ>
__global__ __launch_bounds__(STAGE_NT) void k_tracer_stage(Geo g, TracerArgs<T> a) {
    constexpr int ES = (int)sizeof(T);
    constexpr bool LIN = MODE == 0;   // the linear upwind branch too
    const Blk3 bk = xcd_block_yslab();
    const uint32_t nxg = (uint32_t)g.nx / N;
    const uint32_t q = ((uint32_t)bk.y * gridDim.x + bk.x) * STAGE_NT + threadIdx.x;
    const int j = (int)(q / nxg), i = (int)(q - (uint32_t)j * nxg) * N, k = bk.z;
    if (j >= g.ny) return;
    const uint32_t cb = (uint32_t)((int64_t)k * g.sz + (int64_t)j * g.sy + i) * (uint32_t)ES;
    const int oa = LIN ? a.upw : 0;
    const LineX<N> Lx = linex_of<N, PX>(i, g.nx, ES);
    const Line<int32_t> Ly = line_of<PY, int32_t>(j, g.ny, (int32_t)(g.sy * ES));
    const Line<int64_t> Lz = line_of<PZ, int64_t>(k, g.nz, g.sz * ES);
    Vec<T, N> d = {};
    tracer_x<N, PX, LIN>(d, a.q, a.u, T(a.idx2), cb, Lx, i, g.nx, oa);
    tracer_yz<N, PY, LIN>(d, a.q, a.v, T(a.idy2), cb, Ly, j, g.ny, oa);
    tracer_yz<N, PZ, LIN>(d, a.q, a.w, T(a.idz2), cb, Lz, k, g.nz, oa);
    stage_out<N, MODE, false>(a.c, a.c2, cb, d, a.q, a.qn, a.tout, a.d0, a.d1, a.sb);
}

template <typename T, int N, int PX, int PY, int PZ>
static void tracer_modes(const Geo &g, const TracerArgs<T> &a, int mode, hipStream_t s) {
    const int64_t nb = flat_blocks((int64_t)(g.nx / N) * g.ny), bx = (nb + GRID_YZ - 1) / GRID_YZ;
    const dim3 grd((unsigned)bx, (unsigned)((nb + bx - 1) / bx), g.nz);
#define NYL_TRACER_MODE(M) \
    case M: NYL_LAUNCH((k_tracer_stage<T, N, M, PX, PY, PZ>), grd, STAGE_NT, 0, s, g, a); break;
    switch (mode) {
        NYL_TRACER_MODE(0)
        NYL_TRACER_MODE(1)
        NYL_TRACER_MODE(2)
        NYL_TRACER_MODE(3)
        NYL_TRACER_MODE(4)
        NYL_TRACER_MODE(5)
        NYL_TRACER_MODE(6)
    default: break;
    }
#undef NYL_TRACER_MODE
}

template <typename T, int PX, int PY, int PZ>
static hipError_t tracer_go(const Geo &g, const TracerArgs<T> &a, int mode, hipStream_t s) {
    if (stage_wide<T>(g)) tracer_modes<T, 16 / (int)sizeof(T), PX, PY, PZ>(g, a, mode, s);
    else tracer_modes<T, 1, PX, PY, PZ>(g, a, mode, s);
    return hipGetLastError();
}

template <typename T>
hipError_t launch_tracer_stage(const Geo &g, const TracerArgs<T> &a, int mode, hipStream_t s) {
    if (mode < 0 || mode > 6) return hipErrorInvalidValue;
    NYL_STAGE_GEO(tracer_go, T)
}
template hipError_t launch_tracer_stage<double>(const Geo &, const TracerArgs<double> &, int,
                                                hipStream_t);
template hipError_t launch_tracer_stage<float>(const Geo &, const TracerArgs<float> &, int,
                                               hipStream_t);

}  // namespace nyl
