"""The residual a solve reports does not depend on the solves before it: the
test that is expected to be the last evaluates the norm alone, any other one
in the pass of the next V-cycle's sweeps, and both sum the same cells in the
same order (GPU)."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

# tiled two-sweep pass; marches of 64 and of 32 columns, with partial tiles;
# one march with the restriction (4M cells).  A sum in another order differs
# for one right-hand side in six.
SIZES = [(64, 16, 16, 24), (128, 64, 64, 24), (200, 120, 56, 12), (96, 96, 96, 12),
         (128, 128, 256, 6)]


@pytest.mark.parametrize("geometry", ["closed", "perio_xyz"])
@pytest.mark.parametrize("nx,ny,nz,draws", SIZES, ids=["%dx%dx%d" % s[:3] for s in SIZES])
def test_residual_does_not_depend_on_earlier_solves(nx, ny, nz, draws, geometry):
    import compare as cmp
    from nyles_amd import _lib as L
    from nyles_amd.device import DeviceModel
    print("case residual", nx, ny, nz, geometry, flush=True)
    rng = np.random.default_rng(31)
    zero = np.zeros((nz, ny, nx))
    m = DeviceModel(nx, ny, nz, cmp.GEOMETRY_XYZ[geometry], 1 / nx, 1 / ny, 1 / nz)

    def solve(again):
        if not again:
            m.upload(L.NYL_F_MGX, zero)
        s = m.mg_solve()
        return s["nite"], s["res"], s["normb"]

    for draw in range(draws):
        b = rng.standard_normal((nz, ny, nx))
        m.upload(L.NYL_F_MGB, b - b.mean())
        solve(False)
        solve(True)                  # from the solution: the next guess is too low
        low = solve(False)
        solve(False)
        right = solve(False)         # the guess is right: the norm alone at its end
        assert right == low, draw
    m.close()
