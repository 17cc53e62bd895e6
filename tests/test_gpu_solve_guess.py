"""The V-cycles a solve enqueues before it reads their tests are a guess from
the last solve; its result must not depend on that guess (GPU)."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("precision", [0, 1], ids=["fp64", "mixed"])
@pytest.mark.parametrize("shape,geometry", [((64, 16, 16), "perio_x"), ((48, 40, 24), "closed"),
                                            ((40, 24, 8), "perio_xyz")])
@pytest.mark.parametrize("tol,maxite", [(1e-6, 20), (1e-18, 20), (1e-18, 3)])
def test_solve_does_not_depend_on_the_guess(precision, shape, geometry, tol, maxite):
    import compare as cmp
    import torch
    from nyles_amd import _lib as L
    print("case guess", precision, shape, geometry, tol, maxite, flush=True)
    nx, ny, nz = shape

    def make():
        orc, m = cmp.make_pair(nx, ny, nz, geometry, Lx=nx / 16, Ly=ny / 16, Lz=nz / 16,
                               precision=precision, mg_tol=tol, mg_maxite=maxite)
        return orc, m

    orc, m = make()
    st = cmp.random_state(orc, seed=5)
    rng = np.random.default_rng(6)
    x0 = 1e-3 * rng.standard_normal((nz, ny, nx))

    def load(model, zero):
        for k, f in (("u_i", L.NYL_F_U), ("u_j", L.NYL_F_V), ("u_k", L.NYL_F_W)):
            model.upload(f, st[k])
        model.apply(L.NYL_OP_DIV)
        model.upload(L.NYL_F_MGX, np.zeros_like(x0) if zero else x0)

    def fresh(zero):
        _, f = make()
        load(f, zero)
        s = f.mg_solve()
        x = f.download(L.NYL_F_MGX)
        again = f.mg_solve()          # from the solution: fewer V-cycles
        y = f.download(L.NYL_F_MGX)
        f.close()
        return s["nite"], x, again["nite"], y

    want = {z: fresh(z) for z in (True, False)}
    # a model whose guesses come from other solves: right, too high, too low
    for z in (True, True, False, True):
        load(m, z)
        s = m.mg_solve()
        assert s["nite"] == want[z][0]
        assert cmp.mismatches(m.download(L.NYL_F_MGX), want[z][1]) == 0
        s = m.mg_solve()              # the guess is the longer solve's
        assert s["nite"] == want[z][2]
        assert cmp.mismatches(m.download(L.NYL_F_MGX), want[z][3]) == 0
    torch.cuda.synchronize()
    m.close()
