"""A finest level past the size from which its pre-smoothing and restriction
run as one march (4M cells in FP64), on the GPU: the solve against the oracle,
element by element, from a cold start and from a warm one (powers of two: the
oracle has no rule for levels of odd size)."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("size", [(128, 64, 512), (32, 256, 512)], ids=["tiles", "rows of half a tile"])
def test_large_level_solve_matches_the_oracle(size):
    import compare as cmp
    from nyles_amd import _lib as L
    print("case large level", size, flush=True)
    nx, ny, nz = size
    orc, dev = cmp.make_pair(nx, ny, nz, "perio_xy")
    mg = orc.mg
    rng = np.random.default_rng(23)
    for rep in range(2):
        r = rng.standard_normal((nz, ny, nx))
        r -= r.mean()
        sub = np.zeros(orc.shape)
        orc.set_interior(sub, r)
        orc.fill(sub)
        mg.b[...] = 0.0
        mg.b[mg.idx] = sub
        nite = mg.solve()
        dev.upload(L.NYL_F_MGB, r)
        s = dev.mg_solve()
        assert s["nite"] == nite, "solve %d" % rep
        bad = cmp.mismatches(dev.download(L.NYL_F_MGX), mg.x[3:-3, 3:-3, 3:-3])
        assert bad == 0, "solve %d: %d elements differ" % (rep, bad)
    dev.close()
