"""The forms that a grid's size selects, past their thresholds (GPU): the
stage kernel's 16 bytes of cells per thread with the linear branches and the
model variants (two FP64 cells from 2^18 cells on) and in single precision
(four cells from 1.5M on) with walls in x or y; batches with members of more
than 1M cells, whose level-0 sweeps and restriction are two passes.

FP64: the oracle's or the single member's bits.  Mixed: within 1e-5 relative
(L2) of the FP64 oracle or of the single member, the mixed path's target."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def cmp():
    import compare
    return compare


def _start(cmp, size, geometry, **opts):
    n_tracers = opts.get("n_tracers", 0)
    orc, dev = cmp.make_pair(*size, geometry, Lx=size[0] / 32, Ly=size[1] / 32, Lz=size[2] / 32,
                             **opts)
    st = cmp.random_state(orc, seed=37, amp_u=3e-3)
    rng = np.random.default_rng(38)
    for q in range(n_tracers):
        st["t%d" % q] = rng.standard_normal(st["b"].shape)
    cmp.load_state(orc, dev, st)
    orc.diagnose_var()
    dev.diagnose()
    return orc, dev


VARIANTS = [dict(upwind_a=5, upwind_vf=5), dict(upwind_a=3, upwind_vf=1),
            dict(upwind_a=1, upwind_vf=3), dict(model="linear"), dict(model="Euler3d")]


@pytest.mark.parametrize("scheme", ["rk3", "lfam3"])
@pytest.mark.parametrize("geometry", ["closed", "perio_x", "perio_xyz"])
@pytest.mark.parametrize("variant", VARIANTS, ids=["5-5", "3-1", "1-3", "linear", "Euler3d"])
def test_wide_variants_match_the_oracle(cmp, variant, geometry, scheme):
    print("case wide variant", variant, geometry, scheme, flush=True)
    orc, dev = _start(cmp, (64, 64, 64), geometry, viscosity=1e-3, n_tracers=1, **variant)
    for n in range(1 if scheme == "rk3" else 2):   # LFAM3 starts with an Euler step
        dt = orc.compute_dt(cfl=0.5, dt_max=0.1)
        getattr(orc, "rk3_ssp" if scheme == "rk3" else "lfam3")(dt)
        getattr(dev, "step_" + scheme)(dt)
    want, got = cmp.oracle_fields(orc), cmp.device_fields(dev)
    for k in want:
        bad = cmp.mismatches(got[k], want[k])
        assert bad == 0, "%s: %d elements differ" % (k, bad)
    dev.close()


@pytest.mark.parametrize("variant", [{}, dict(upwind_a=5, upwind_vf=5)], ids=["weno", "linear"])
@pytest.mark.parametrize("geometry", ["closed", "perio_x", "perio_y"])
def test_four_cells_with_walls_close_to_the_oracle(cmp, geometry, variant):
    print("case four cells", geometry, variant, flush=True)
    orc, dev = _start(cmp, (128, 128, 96), geometry, precision=1, **variant)
    dt = orc.compute_dt(cfl=0.5, dt_max=0.1)
    orc.rk3_ssp(dt)
    dev.step_rk3(dt)
    want, got = cmp.oracle_fields(orc), cmp.device_fields(dev)
    for k in ("b", "u_i", "u_j", "u_k"):
        e = cmp.rel_l2(got[k], want[k])
        print("  %s rel err %.2e" % (k, e), flush=True)
        assert e < 1e-5, (k, e)
    dev.close()


# a tiled and a ragged member above 1M cells, one at the limit, a small one
LARGE = [((128, 128, 80), "perio_xy"), ((120, 104, 88), "closed"), ((128, 128, 64), "perio_x"),
         ((32, 32, 32), "perio_xyz")]


def _member(size, geometry, seed, precision):
    from nyles_amd import _lib as L
    from nyles_amd.device import DeviceModel
    import compare
    d = 1.0 / 32
    m = DeviceModel(*size, compare.GEOMETRY_XYZ[geometry], d, d, d, precision=precision)
    rng = np.random.default_rng(seed)
    nx, ny, nz = size
    per = compare.GEOMETRY_XYZ[geometry]
    for f, amp, ax in ((L.NYL_F_B, 1.0, None), (L.NYL_F_U, 3e-3 * d, 2), (L.NYL_F_V, 3e-3 * d, 1),
                       (L.NYL_F_W, 3e-3 * d, 0)):
        a = amp * rng.standard_normal((nz, ny, nx))
        if ax is not None and not per[2 - ax]:   # the wall face
            a[tuple(-1 if q == ax else slice(None) for q in range(3))] = 0.0
        m.upload(f, a)
    m.diagnose()
    return m


def _fields(m):
    from nyles_amd import _lib as L
    return {k: m.download(f) for k, f in (("b", L.NYL_F_B), ("u", L.NYL_F_U), ("v", L.NYL_F_V),
                                          ("w", L.NYL_F_W))}


@pytest.mark.parametrize("precision", [0, 1], ids=["fp64", "mixed"])
def test_large_members_match_single_members(cmp, precision):
    from nyles_amd.device import DeviceBatch
    print("case large members", precision, flush=True)
    single = [_member(s, g, 50 + q, precision) for q, (s, g) in enumerate(LARGE)]
    mixed = [_member(s, g, 50 + q, precision) for q, (s, g) in enumerate(LARGE)]
    alone = _member(*LARGE[0], 50, precision)
    dts = [0.01] * len(LARGE)
    bn, b1 = DeviceBatch(mixed, tile=256), DeviceBatch([alone], tile=256)
    for n in range(2):
        want = [m.step_rk3(dt) for m, dt in zip(single, dts)]
        got = bn.step_rk3(dts)
        one = b1.step_rk3(dts[:1])
        assert one[0]["nite"] == got[0]["nite"]
        if precision == 0:
            assert [s["nite"] for s in got] == [s["nite"] for s in want]
    for q in range(len(LARGE)):
        a, b = _fields(mixed[q]), _fields(single[q])
        for k in a:
            if precision == 0:
                bad = cmp.mismatches(a[k], b[k])
                assert bad == 0, "member %d %s: %d elements differ" % (q, k, bad)
            else:
                e = cmp.rel_l2(a[k], b[k])
                print("  member %d %s rel %.2e" % (q, k, e), flush=True)
                assert e < 1e-5, (q, k, e)
    a, b = _fields(mixed[0]), _fields(alone)
    for k in a:
        bad = cmp.mismatches(a[k], b[k])
        assert bad == 0, "alone %s: %d elements differ" % (k, bad)
    bn.close()
    b1.close()
    for m in single + mixed + [alone]:
        m.close()
