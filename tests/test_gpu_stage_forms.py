"""The stage kernel's forms (one cell or 16 bytes of cells per thread, whole
tiles or planes numbered along their rows) on the GPU: the FP64 tendencies
against the oracle, element by element, also for magnitudes whose
reconstruction weights leave the range of the kernel's short division."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

# pairs in whole 16-cell x 32-row tiles; pairs along the rows of a plane, the
# last block partly filled; one cell per thread (odd nx or ny is refused)
SHAPES = [(64, 64, 64), (90, 52, 60), (34, 16, 10)]


@pytest.mark.parametrize("scale", [1.0, 1e-170, 1e60, 1e155])
@pytest.mark.parametrize("geometry", ["closed", "perio_x", "perio_xyz"])
@pytest.mark.parametrize("shape", SHAPES, ids=["%dx%dx%d" % s for s in SHAPES])
def test_rhs_forms_match_the_oracle(shape, geometry, scale):
    import compare as cmp
    import oracle as O
    from nyles_amd import _lib as L
    print("case stage form", shape, geometry, scale, flush=True)
    nx, ny, nz = shape
    orc, dev = cmp.make_pair(nx, ny, nz, geometry)
    rng = np.random.default_rng(17)
    metric = {"u_i": orc.idx2, "u_j": orc.idy2, "u_k": orc.idz2}
    for name, arr, fid in (("b", orc.b, L.NYL_F_B), ("u_i", orc.U["i"], L.NYL_F_U),
                           ("u_j", orc.U["j"], L.NYL_F_V), ("u_k", orc.U["k"], L.NYL_F_W),
                           ("vor_i", orc.vor["i"], L.NYL_F_VORX),
                           ("vor_j", orc.vor["j"], L.NYL_F_VORY),
                           ("vor_k", orc.vor["k"], L.NYL_F_VORZ), ("ke", orc.ke, L.NYL_F_KE)):
        vals = rng.standard_normal((nz, ny, nx))
        vals.flat[::7] = 0.0
        if name == "b" or name.startswith("vor"):   # the reconstructed quantities
            vals *= scale
            vals[nz // 2:, : ny // 2, :] = 0.0       # and a region at rest
        dev.upload(fid, vals)
        orc.set_interior(arr, vals * metric.get(name, 1.0))
        O.halo_fill(arr, geometry, orc.nh)
    with np.errstate(all="ignore"):
        orc.rhs(orc.ds[1])
    dev.rhs(1)
    want = {"b": orc.ds[1]["b"], "u_i": orc.ds[1]["u"]["i"], "u_j": orc.ds[1]["u"]["j"],
            "u_k": orc.ds[1]["u"]["k"]}
    ids = {"b": L.NYL_F_DS1_B, "u_i": L.NYL_F_DS1_U, "u_j": L.NYL_F_DS1_V, "u_k": L.NYL_F_DS1_W}
    for k in want:
        bad = cmp.mismatches(dev.download(ids[k]), orc.interior(want[k]))
        assert bad == 0, "d%s: %d elements differ" % (k, bad)
    dev.close()


@pytest.mark.parametrize("scheme", ["rk3", "lfam3"])
@pytest.mark.parametrize("geometry", ["closed", "perio_xy"])
def test_tracers_in_pairs_match_the_oracle(scheme, geometry):
    """two steps with passive tracers on a grid that takes two cells per thread"""
    import compare as cmp
    print("case tracer pairs", scheme, geometry, flush=True)
    orc, dev = cmp.make_pair(64, 64, 64, geometry, n_tracers=2)
    st = cmp.random_state(orc, seed=19, amp_u=3e-3)
    rng = np.random.default_rng(20)
    for q in range(2):
        st["t%d" % q] = rng.standard_normal(st["b"].shape)
    cmp.load_state(orc, dev, st)
    orc.diagnose_var()
    dev.diagnose()
    for n in range(2):
        dt = orc.compute_dt(cfl=0.5, dt_max=0.1)
        if scheme == "rk3":
            orc.rk3_ssp(dt)
            dev.step_rk3(dt)
        else:
            orc.lfam3(dt)
            dev.step_lfam3(dt)
    want, got = cmp.oracle_fields(orc), cmp.device_fields(dev)
    for k in want:
        bad = cmp.mismatches(got[k], want[k])
        assert bad == 0, "%s: %d elements differ" % (k, bad)
    dev.close()
