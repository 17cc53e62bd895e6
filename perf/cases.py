"""The work a user of this framework has it do, as measurable cases.

A case is a dict of plain values.  ``listed()`` names the fixed ones,
``draw(rng)`` gives one more case of the ranges they stand for, ``prepare``
builds what a program holds before the call (the model or batch with its
projected initial state on the GPU), ``run`` is one pass through the public
entry points (``nyles_amd.device``), ``work`` counts the bytes and operations
one pass cannot do without, and ``exact`` evaluates the same pass in 64 bits
with plain torch: the scheme's own arithmetic (WENO or linear upwind
reconstructions with their single-precision literals, the multigrid iteration
with its stop rule), without this repository's kernels.

Kinds of case:

  step      one time step (RK3_SSP, Euler forward or LFAM3) of a model whose
            state stays on the GPU; ``adapt`` takes dt from the CFL reduction
            before every step, as the time loop of a run does
  batch     one RK3_SSP step of an ensemble of models of uneven sizes
  rhs       the tendencies of a state (a program with its own time scheme or
            forcing calls this once per stage)
  solve     one pressure solve from a zero first guess
  monitor   the scalar diagnostics a run prints: max U^2, kinetic energy, sum
            of b, count of non-finite values
"""
import math
import random

import torch

from nyles_amd import _lib as L
from nyles_amd.device import DeviceBatch, DeviceModel

PERIODIC = {"closed": (0, 0, 0), "perio_x": (1, 0, 0), "perio_y": (0, 1, 0),
            "perio_xy": (1, 1, 0), "perio_xyz": (1, 1, 1)}       # (x, y, z)
PRECISION = {"fp64": L.NYL_PREC_FP64, "mixed": L.NYL_PREC_MIXED}
DEVICE = "cuda"
STATE = (("b", L.NYL_F_B), ("u_i", L.NYL_F_U), ("u_j", L.NYL_F_V), ("u_k", L.NYL_F_W))
TEND = (("b", L.NYL_F_DS0_B), ("u_i", L.NYL_F_DS0_U), ("u_j", L.NYL_F_DS0_V),
        ("u_k", L.NYL_F_DS0_W))

# defaults of the keys a case may leave out
DEFAULT = {"scheme": "rk3", "adapt": False, "tol": 1e-6, "maxite": 20, "viscosity": 0.0,
           "coriolis": 0.0, "tracers": 0, "upwind": 0}


def listed():
    return [
        # the scalar diagnostics of a small run, printed at every step: the
        # smallest calls, one launch pair and one host read each
        {"name": "monitor_64x32x32", "kind": "monitor", "nx": 64, "ny": 32, "nz": 32,
         "geometry": "perio_x", "flow": "lock", "precision": "fp64"},
        # the lock exchange at the size of the experiment scripts, stepped by
        # the time loop (dt from the CFL reduction): bound by latency
        {"name": "lock_64x32x32_fp64", "kind": "step", "nx": 64, "ny": 32, "nz": 32,
         "geometry": "perio_x", "flow": "lock", "precision": "fp64", "adapt": True},
        # a stratified shear layer of the ensemble's and server's upper sizes,
        # stepped on its own; 96 is not a multiple of the 64-wide tiles
        {"name": "shear_96_fp64", "kind": "step", "nx": 96, "ny": 96, "nz": 96,
         "geometry": "perio_xy", "flow": "shear", "precision": "fp64", "adapt": True},
        # a basin of ragged size in mixed precision (the multigrid stops at
        # 25 x 15 x 7 and solves that level directly)
        {"name": "lock_200x120x56_mixed", "kind": "step", "nx": 200, "ny": 120, "nz": 56,
         "geometry": "perio_x", "flow": "lock", "precision": "mixed", "adapt": True},
        # LFAM3 in a closed rotating box with viscosity and two passive tracers
        {"name": "lfam3_closed_128x64x64_fp64", "kind": "step", "nx": 128, "ny": 64, "nz": 64,
         "geometry": "closed", "flow": "lock", "precision": "fp64", "scheme": "lfam3",
         "viscosity": 1e-4, "coriolis": 1.0, "tracers": 2},
        # the linear upwind branches of orders 5/5
        {"name": "linear5_256x128x64_mixed", "kind": "step", "nx": 256, "ny": 128, "nz": 64,
         "geometry": "perio_xyz", "flow": "vortex", "precision": "mixed", "upwind": 5},
        # the headline workload: Taylor-Green vortex 256^3, both precisions
        {"name": "vortex_256_mixed", "kind": "step", "nx": 256, "ny": 256, "nz": 256,
         "geometry": "perio_xyz", "flow": "vortex", "precision": "mixed"},
        {"name": "vortex_256_fp64", "kind": "step", "nx": 256, "ny": 256, "nz": 256,
         "geometry": "perio_xyz", "flow": "vortex", "precision": "fp64"},
        # Rayleigh-Taylor 256 x 256 x 512 with the projection converged to
        # |r|/|b| <= 1e-10: the largest call, nearly all multigrid
        {"name": "rt_256x256x512_tight_mixed", "kind": "step", "nx": 256, "ny": 256, "nz": 512,
         "geometry": "perio_xy", "flow": "rt", "precision": "mixed", "tol": 1e-20, "maxite": 50},
        # an ensemble of uneven members advanced together
        {"name": "ensemble_16_mixed", "kind": "batch", "members": 16, "lo": 32, "hi": 96,
         "sizes": 7, "geometry": "perio_xy", "flow": "shear", "precision": "mixed"},
        # tendencies alone, walls in z, for a program with its own scheme
        {"name": "rhs_160x96x128_fp64", "kind": "rhs", "nx": 160, "ny": 96, "nz": 128,
         "geometry": "perio_xy", "flow": "shear", "precision": "fp64"},
        # one pressure solve in a closed basin from a zero first guess
        {"name": "solve_closed_192x128x96_fp64", "kind": "solve", "nx": 192, "ny": 128, "nz": 96,
         "geometry": "closed", "flow": "noise", "precision": "fp64"},
    ]


def _size(rng, most):
    """(nx, ny, nz), each 16..256 and every one halving evenly 1 to 4 times
    down to a level the direct solve takes (or further), ragged ones among
    them; at most ``most`` cells"""
    while True:
        k = rng.randint(1, 4)
        n = []
        for cmax in (64, 32, 32):
            lo, hi = max(4, 16 >> k), min(cmax, 256 >> k)
            n.append(int(round(math.exp(rng.uniform(math.log(lo), math.log(hi))))) << k)
        if n[0] * n[1] * n[2] <= most:
            return n


def draw(rng):
    kind = rng.choice(["step"] * 6 + ["batch", "rhs", "solve", "monitor"])
    precision = rng.choice(["fp64", "mixed"])
    if kind == "batch":
        return {"kind": "batch", "members": rng.randint(4, 16), "lo": 32,
                "hi": rng.choice([48, 64, 80, 96]), "sizes": rng.randint(0, 999),
                "geometry": "perio_xy", "flow": "shear", "precision": precision}
    nx, ny, nz = _size(rng, 1 << 23)
    geometry = rng.choice(sorted(PERIODIC))
    c = {"kind": kind, "nx": nx, "ny": ny, "nz": nz, "geometry": geometry,
         "precision": "fp64" if kind == "solve" else precision}
    if kind == "solve":
        return dict(c, flow="noise")
    c["flow"] = {"perio_xyz": "vortex", "perio_xy": rng.choice(["shear", "rt"])}.get(geometry,
                                                                                   "lock")
    if kind == "step":
        c["scheme"] = rng.choice(["rk3", "rk3", "rk3", "lfam3", "ef"])
        c["adapt"] = c["scheme"] == "rk3" and rng.random() < 0.5
        if geometry == "perio_xyz" and c["scheme"] == "rk3" and rng.random() < 0.3:
            c["upwind"] = rng.choice([1, 3, 5])
        if rng.random() < 0.3:
            c["viscosity"] = 1e-4
        if rng.random() < 0.3:
            c["tracers"] = rng.randint(1, 3)
        if geometry != "perio_xyz" and rng.random() < 0.3:
            c["coriolis"] = 1.0
        if rng.random() < 0.15:
            c["tol"], c["maxite"] = 1e-14, 40
    return c


# --------------------------------------------------------------------------
# grids and initial states

class _Grid:
    """cubic cells, the longest side of length 1"""

    def __init__(self, case, shape=None):
        self.nx, self.ny, self.nz = shape or (case["nx"], case["ny"], case["nz"])
        self.shape = (self.nz, self.ny, self.nx)
        self.d = 1.0 / max(self.nx, self.ny, self.nz)
        self.Lx, self.Ly, self.Lz = self.nx * self.d, self.ny * self.d, self.nz * self.d
        self.periodic = PERIODIC[case["geometry"]]
        self.i2 = 1 / self.d ** 2
        self.fpar = case["coriolis"] * self.d * self.d
        self.ncell = self.nx * self.ny * self.nz


def _full(case):
    return dict(DEFAULT, **case)


def _initial(case, g, seed):
    """the fields of a flow in 64 bits on the GPU: b, covariant u, v, w
    (physical velocity times the spacing) and the tracers"""
    dev, f64 = torch.device(DEVICE), torch.float64
    gen = torch.Generator(device=dev)
    gen.manual_seed(seed)

    def noise(a):
        return a * torch.randn(g.shape, generator=gen, device=dev, dtype=f64)

    def line(n, L_, shape, at):
        return ((torch.arange(n, device=dev, dtype=f64) + at) * (L_ / n)).view(shape)

    x, xf = (line(g.nx, g.Lx, (1, 1, -1), a) for a in (0.5, 1.0))
    y, yf = (line(g.ny, g.Ly, (1, -1, 1), a) for a in (0.5, 1.0))
    z, zf = (line(g.nz, g.Lz, (-1, 1, 1), a) for a in (0.5, 1.0))
    zero = torch.zeros(g.shape, device=dev, dtype=f64)
    flow, tau, sin, cos = case["flow"], 2 * math.pi, torch.sin, torch.cos
    kx, ky, kz = tau / g.Lx, tau / g.Ly, tau / g.Lz
    if flow == "vortex":        # Taylor-Green vortex and one of half its strength across it
        u = sin(kx * xf) * cos(ky * y) * cos(kz * z) * (tau / kx)
        v = (0.5 * cos(kx * x) * sin(ky * yf) * cos(kz * z)
             - cos(kx * x) * sin(ky * yf) * cos(kz * z)) * (tau / ky)
        w = -0.5 * cos(kx * x) * cos(ky * y) * sin(kz * zf) * (tau / kz)
        u, v, w = u + noise(1e-4), v + noise(1e-4), w + noise(1e-4)
        b = 0.1 * cos(kx * x) * cos(ky * y) + noise(1e-4)
    elif flow == "shear":       # stratified shear layer
        u = torch.tanh((z - g.Lz / 2) / (0.05 * g.Lz)) + noise(1e-3)
        v = 0.05 * sin(kx * x) + noise(1e-3)
        w = 0.05 * sin(ky * y) * sin(0.5 * kz * zf) + noise(1e-3)
        b = 0.1 * z + zero
    elif flow == "lock":        # heavy and light fluid side by side, at rest
        b = torch.where(x < g.Lx / 2 + 0.15 * g.Lx * cos(2 * ky * y), 0.5, -0.5) + noise(1e-3)
        u, v, w = zero, zero, noise(1e-5)
    elif flow == "rt":          # heavy fluid above a wavy interface, at rest
        r = random.Random(seed)
        eta = torch.zeros((1, g.ny, g.nx), device=dev, dtype=f64)
        for _ in range(16):
            p, q, ph = r.randint(1, 8), r.randint(1, 8), r.uniform(0, tau)
            eta = eta + cos(p * kx * x + q * ky * y + ph)
        b = torch.where(z > g.Lz / 2 + 0.01 * g.Lz / 4 * eta, -0.5, 0.5) + zero
        u, v, w = zero, zero, noise(1e-5)
    else:                       # "noise": a random velocity
        b, u, v, w = zero, noise(1e-2), noise(1e-2), noise(1e-2)
    st = {"b": b, "u_i": u * g.d, "u_j": v * g.d, "u_k": w * g.d}
    for name, axis in (("u_i", 0), ("u_j", 1), ("u_k", 2)):      # no flow through walls
        if not g.periodic[axis]:
            st[name] = st[name].clone()
            st[name].select(2 - axis, -1).zero_()
    for q in range(case["tracers"]):
        st["t%d" % q] = cos((q + 1) * kx * x) * cos(ky * y) + noise(1e-2)
    if case["precision"] == "mixed":    # what the model holds
        st = {k: v.float().double() for k, v in st.items()}
    return st


def _rest_dt(case, g):
    """dt of a flow that starts at rest from the buoyancy jump (1) and depth,
    of a moving one from its largest velocity"""
    if case["flow"] in ("lock", "rt"):
        return 0.5 * g.d / math.sqrt(1.0 * g.Lz)
    return 0.5 * g.d / {"vortex": 1.5 * max(g.Lx, g.Ly, g.Lz)}.get(case["flow"], 1.1)


def _model(case, g, seed):
    m = DeviceModel(g.nx, g.ny, g.nz, g.periodic, g.d, g.d, g.d, idx2=g.i2, idy2=g.i2, idz2=g.i2,
                    dx2=g.d ** 2, fparameter=g.fpar, precision=PRECISION[case["precision"]],
                    mg_maxite=case["maxite"], mg_tol=case["tol"], viscosity=case["viscosity"],
                    n_tracers=case["tracers"], upwind_a=case["upwind"], upwind_vf=case["upwind"])
    st = _initial(case, g, seed)
    torch.cuda.current_stream().synchronize()
    ids = list(STATE) + [("t%d" % q, L.NYL_F_TRACER(q)) for q in range(case["tracers"])]
    with torch.cuda.stream(m.stream):
        for name, fid in ids:
            m.field(fid).copy_(st[name])
    m.sync()
    return m


def _members(case):
    r = random.Random(case["sizes"])
    lo, hi = math.log(case["lo"]), math.log(case["hi"])
    return [8 * int(round(math.exp(r.uniform(lo, hi)) / 8)) for _ in range(case["members"])]


def prepare(case, seed):
    case = _full(case)
    if case["kind"] == "batch":
        grids = [_Grid(case, (n, n, n)) for n in _members(case)]
        models = [_model(case, g, seed * 1000 + q) for q, g in enumerate(grids)]
        for m in models:
            m.diagnose()
        return {"case": case, "models": models, "batch": DeviceBatch(models),
                "dts": [_rest_dt(case, g) for g in grids]}
    g = _Grid(case)
    m = _model(case, g, seed)
    s = {"case": case, "model": m, "dt": _rest_dt(case, g)}
    if case["kind"] == "solve":
        m.apply(L.NYL_OP_DIV)
    else:
        m.diagnose()
        if case["scheme"] == "lfam3" and case["kind"] == "step":
            m.step_lfam3(s["dt"])        # the starting step of the scheme
    m.sync()
    return s


def _state(m, tracers=0):
    out = {name: m.field(fid) for name, fid in STATE}
    for q in range(tracers):
        out["t%d" % q] = m.field(L.NYL_F_TRACER(q))
    return out


def run(s):
    case = s["case"]
    kind = case["kind"]
    if kind == "batch":
        s["batch"].step_rk3(s["dts"])
        return [_state(m) for m in s["models"]]
    m = s["model"]
    if kind == "step":
        dt = s["dt"]
        if case["adapt"]:
            umax2 = m.reduce(L.NYL_RED_MAXU2)
            if umax2 > 0.0:
                dt = min(dt, 0.5 / math.sqrt(umax2))
        {"rk3": m.step_rk3, "ef": m.step_ef, "lfam3": m.step_lfam3}[case["scheme"]](dt)
        return _state(m, case["tracers"])
    if kind == "rhs":
        m.rhs(0)
        return {name: m.field(fid) for name, fid in TEND}
    if kind == "solve":
        with torch.cuda.stream(m.stream):
            m.field(L.NYL_F_MGX).zero_()
        m.mg_solve()
        return {"x": m.field(L.NYL_F_MGX)}
    return {"maxu2": m.reduce(L.NYL_RED_MAXU2), "ke": m.reduce(L.NYL_RED_KE),
            "bsum": m.reduce(L.NYL_RED_BSUM), "nonfinite": int(m.reduce(L.NYL_RED_NONFINITE))}


def work(case):
    """Each stage of a step reads the state, the vorticity and ke once and
    writes them once (the tendencies of earlier stages are read too), and
    each projection reads and writes the velocity and the FP64 pressure; the
    multigrid's passes in between are not counted.  Operations: the six
    tracer and six vortex-force reconstructions of a cell, about 70 each."""
    case = _full(case)
    w = 8 if case["precision"] == "fp64" else 4
    if case["kind"] == "batch":
        cells = sum(n ** 3 for n in _members(case))
    else:
        cells = case["nx"] * case["ny"] * case["nz"]
    if case["kind"] == "solve":
        return {"bytes": 2 * 8 * cells, "flops": 200 * cells}
    if case["kind"] == "monitor":
        return {"bytes": 11 * w * cells, "flops": 40 * cells}
    if case["kind"] == "rhs":
        return {"bytes": 12 * w * cells, "flops": 900 * cells}
    stages = {"rk3": 3, "lfam3": 2, "ef": 1}[case["scheme"]]
    more = 2 * case["tracers"]
    stage = 8 + 4 + 4 + more             # state, vorticity, ke in; state out; tendencies
    project = 3 + 3 + 4                  # velocity in and out, vorticity and ke out
    return {"bytes": stages * ((stage + project) * w + 16) * cells,
            "flops": stages * 1100 * cells}


# --------------------------------------------------------------------------
# the same passes in 64 bits with plain torch

def _f32(v):
    """a single-precision literal of the scheme, widened"""
    return float(torch.tensor(v, dtype=torch.float32))


_C13, _C76, _C116 = _f32(1 / 3), _f32(7 / 6), _f32(11 / 6)
_C16, _C56, _K1 = _f32(1 / 6), _f32(5 / 6), _f32(13 / 12)
_EPS3, _EPS5 = _f32(1e-14), _f32(1e-16)
_C26 = _f32(2 / 6)
_B1, _B2, _B3, _B4, _B5 = (_f32(v / 60) for v in (2, -13, 47, 27, -3))


def _weno3(qm, q0, qp):
    b1, b2 = (q0 - qm) ** 2, (qp - q0) ** 2
    tau = (b2 - b1).abs()
    w1, w2 = 1 + tau / (b1 + _EPS3), 2 * (1 + tau / (b2 + _EPS3))
    return (w1 * (3 * q0 - qm) * 0.5 + w2 * (q0 + qp) * 0.5) / (w1 + w2)


def _weno5(a, b, c, d, e):
    b1 = _K1 * (a - 2 * b + c) ** 2 + 0.25 * (a - 4 * b + 3 * c) ** 2
    b2 = _K1 * (b - 2 * c + d) ** 2 + 0.25 * (b - d) ** 2
    b3 = _K1 * (c - 2 * d + e) ** 2 + 0.25 * (3 * c - 4 * d + e) ** 2
    tau = (b1 - b3).abs().float().double()
    w1, w2 = 1 + tau / (b1 + _EPS5), 6 * (1 + tau / (b2 + _EPS5))
    w3 = 3 * (1 + tau / (b3 + _EPS5))
    return (w1 * (_C13 * a - _C76 * b + _C116 * c) + w2 * (_C56 * c + _C13 * d - _C16 * b)
            + w3 * (_C13 * c + _C56 * d - _C16 * e)) / (w1 + w2 + w3)


def _sh(a, axis, s, per):
    """the value s cells further along a tensor axis: wrapped, or zero
    beyond a wall"""
    r = torch.roll(a, -s, axis)
    if not per and s:
        n = a.shape[axis]
        r.narrow(axis, n - s if s > 0 else 0, abs(s)).zero_()
    return r


def _pos(a, axis):
    v = [1, 1, 1]
    v[axis] = -1
    return torch.arange(a.shape[axis], device=a.device).view(v)


def _face(u, q, axis, per):
    """u times the upwinded reconstruction of q at the face after each cell;
    near a wall the order drops 5, 3, 1, and nothing passes the last face"""
    m2, m1, p1, p2, p3 = (_sh(q, axis, s, per) for s in (-2, -1, 1, 2, 3))
    right, left = _weno5(m2, m1, q, p1, p2), _weno5(p3, p2, p1, q, m1)
    if not per:
        f, n = _pos(q, axis), q.shape[axis]
        right = torch.where((f == 1) | (f == n - 2), _weno3(m1, q, p1), right)
        right = torch.where(f == 0, q, right)
        left = torch.where((f == 0) | (f == n - 3), _weno3(p2, p1, q), left)
        left = torch.where(f == n - 2, p1, left)
    r = u * torch.where(u > 0, right, left)
    return r if per else torch.where(f == n - 1, 0.0, r)


def _linear(q, axis, order, right):
    """linear reconstruction on a periodic axis: left-biased, or right-biased"""
    s = [_sh(q, axis, k, True) for k in (-2, -1, 0, 1, 2)]
    if order == 1:
        return q
    s = s[::-1] if right else s
    if order == 3:
        return -_C16 * s[1] + _C56 * s[2] + _C26 * s[3]
    return _B1 * s[0] + _B2 * s[1] + _B3 * s[2] + _B4 * s[3] + _B5 * s[4]


def _ahead(a, ax):
    """difference to the next value along a tensor axis"""
    return _sh(a, ax, 1, True) - a


class _Exact:
    """one model in 64 bits"""

    def __init__(self, case, g, seed):
        self.case, self.g = case, g
        self.s = _initial(case, g, seed)
        self.per = tuple(reversed(g.periodic))          # by tensor axis (z, y, x)
        self.x = torch.zeros(g.shape, device=DEVICE, dtype=torch.float64)
        self.levels = self._hierarchy()
        self.eig = None

    def _hierarchy(self):
        nz, ny, nx = self.g.shape
        lev = [(nz, ny, nx)]
        self.direct = False
        while not (nx == 2 or ny == 2):
            if (nx | ny | nz) & 1:
                self.direct = True
                break
            nz, ny, nx = nz // 2, ny // 2, nx // 2
            lev.append((nz, ny, nx))
        return lev

    # ---- pressure
    def _sum6(self, a):
        r = 0
        for ax in (2, 1, 0):
            r = r + _sh(a, ax, -1, self.per[ax]) + _sh(a, ax, 1, self.per[ax])
        return r

    def _diag(self, shape):
        if not hasattr(self, "_nw"):
            self._nw = {}
        if shape not in self._nw:
            self._nw[shape] = self._sum6(torch.ones(shape, device=DEVICE, dtype=torch.float64))
        return self._nw[shape]

    def _smooth(self, x, b):
        for _ in range(2):
            x = (1.0 - 0.9) * x + 0.9 * (self._sum6(x) - b) / self._diag(tuple(x.shape))
        return x

    def _resid(self, x, b):
        return b + self._diag(tuple(x.shape)) * x - self._sum6(x)

    def _restrict(self, r):
        nz, ny, nx = r.shape
        return 0.5 * r.view(nz // 2, 2, ny // 2, 2, nx // 2, 2).sum(dim=(1, 3, 5))

    def _prolong(self, c):
        for ax in (2, 1, 0):
            per = self.per[ax]
            one = torch.ones_like(c)
            parts = [(3 * c + _sh(c, ax, s, per)) / (3 + _sh(one, ax, s, per)) for s in (-1, 1)]
            shape = list(c.shape)
            shape[ax] *= 2
            c = torch.stack(parts, dim=ax + 1).reshape(shape)
        return c

    def _coarsest(self, b):
        if not self.direct:
            return self._smooth(torch.zeros_like(b), b)
        if self.eig is None:
            self.eig = []
            for ax in range(3):
                n = b.shape[ax]
                one = torch.eye(n, device=DEVICE, dtype=torch.float64)
                m = torch.roll(one, 1, 0) + torch.roll(one, -1, 0) - 2 * one
                if not self.per[ax]:
                    if n > 1:
                        m[0, n - 1] -= 1
                        m[n - 1, 0] -= 1
                        m[0, 0] += 1
                        m[n - 1, n - 1] += 1
                    else:
                        m.zero_()
                self.eig.append(torch.linalg.eigh(m))
        (lz, ez), (ly, ey), (lx, ex) = self.eig
        lam = lz.view(-1, 1, 1) + ly.view(1, -1, 1) + lx.view(1, 1, -1)

        def apply(a, mz, my, mx):
            a = torch.tensordot(a, mx, dims=([2], [0]))
            a = torch.tensordot(a, my, dims=([1], [0])).permute(0, 2, 1)
            return torch.tensordot(a, mz, dims=([0], [0])).permute(2, 0, 1)

        t = apply(b, ez, ey, ex)
        t = torch.where(lam.abs() > 1e-9, t / torch.where(lam.abs() > 1e-9, lam, 1.0), 0.0)
        return apply(t, ez.T, ey.T, ex.T).contiguous()

    def _cycle(self, l, x, b):
        if l == len(self.levels) - 1:
            return self._coarsest(b)
        x = self._smooth(x, b)
        bc = self._restrict(self._resid(x, b))
        return self._smooth(x + self._prolong(self._cycle(l + 1, torch.zeros_like(bc), bc)), b)

    def solve(self, b):
        if self.case["precision"] == "mixed":
            b = b - b.mean()
        normb = float((b * b).sum())

        def res():
            return float((self._resid(self.x, b) ** 2).sum()) / normb if normb > 0 else 0.0

        r, nite = res(), 0
        while not r < self.case["tol"]:
            self.x = self._cycle(0, self.x, b)
            nite += 1
            if nite >= self.case["maxite"]:
                break
            r = res()

    def div(self):
        r = 0
        for name, ax in (("u_i", 2), ("u_j", 1), ("u_k", 0)):
            U = self.s[name] * self.g.i2
            r = r + (U - _sh(U, ax, -1, self.per[ax]))
        return r

    def _inside(self, a, *axes):
        """zero at the last position of the wall axes among `axes`"""
        for ax in axes:
            if not self.per[ax]:
                a = torch.where(_pos(a, ax) == a.shape[ax] - 1, 0.0, a)
        return a

    def diagnose(self):
        self.solve(self.div())
        s, p = self.s, self.x * self.g.d ** 2
        for name, ax in (("u_i", 2), ("u_j", 1), ("u_k", 0)):
            s[name] = s[name] - self._inside(_sh(p, ax, 1, True) - p, ax)
        u, v, w = s["u_i"], s["u_j"], s["u_k"]
        self.oz = self._inside(_ahead(v, 2) - _ahead(u, 1) + self.g.fpar, 2, 1)
        self.ox = self._inside(_ahead(w, 1) - _ahead(v, 0), 1, 0)
        self.oy = self._inside(_ahead(u, 0) - _ahead(w, 2), 0, 2)
        self.ke = 0
        for a, ax in ((u, 2), (v, 1), (w, 0)):
            t = 0.25 * self.g.i2 * (a * a + _sh(a, ax, -1, True) ** 2)
            if not self.per[ax]:
                t = torch.where(_pos(a, ax) == 0, 0.0, t)
            self.ke = self.ke + t

    # ---- tendencies
    def _advect(self, q):
        order, d = self.case["upwind"], 0
        for name, ax in (("u_i", 2), ("u_j", 1), ("u_k", 0)):
            U, per = self.s[name] * self.g.i2, self.per[ax]
            if order:
                f = (0.5 * (U + U.abs()) * _linear(q, ax, order, False)
                     + 0.5 * (U - U.abs()) * _sh(_linear(q, ax, order, True), ax, 1, True))
            else:
                f = _face(U, q, ax, per)
            d = d + (_sh(f, ax, -1, per) - f)
        return d

    def _vortex(self, name, om, ax, e):
        """the flux of vorticity om along ax by the velocity of that axis
        averaged along the target axis e"""
        U, per, order = self.s[name] * self.g.i2, self.per[ax], self.case["upwind"]
        UU = 0.5 * (U + _sh(U, e, 1, True))
        u1 = 0.5 * (_sh(UU, ax, -1, per) + UU)
        if order:
            return (0.5 * (u1 + u1.abs()) * _sh(_linear(om, ax, order, False), ax, -1, True)
                    + 0.5 * (u1 - u1.abs()) * _linear(om, ax, order, True))
        return _face(u1, _sh(om, ax, -1, per), ax, per)

    def rhs(self, last=False):
        s, X, Y, Z = self.s, 2, 1, 0
        out = {k: self._advect(s[k]) for k in s if k == "b" or k[0] == "t"}
        dv = -self._vortex("u_i", self.oz, X, Y) + self._vortex("u_k", self.ox, Z, Y)
        du = self._vortex("u_j", self.oz, Y, X) - self._vortex("u_k", self.oy, Z, X)
        dw = -self._vortex("u_j", self.ox, Y, Z) + self._vortex("u_i", self.oy, X, Z)
        du = self._inside(du - _ahead(self.ke, X), X)
        dv = self._inside(dv - _ahead(self.ke, Y), Y)
        buoyancy = 0.5 * self.g.d * (_sh(s["b"], Z, 1, True) + s["b"])
        dw = self._inside(dw - _ahead(self.ke, Z) + buoyancy, Z)
        out.update(u_i=du, u_j=dv, u_k=dw)
        if last and self.case["viscosity"]:
            for name in ("u_i", "u_j", "u_k"):
                for ax in (X, Y, Z):
                    fx = self._inside(_ahead(s[name], ax), ax)
                    out[name] = out[name] + self.case["viscosity"] * self.g.i2 * (
                        fx - _sh(fx, ax, -1, self.per[ax]))
        return out

    # ---- schemes
    def _set(self, fn):
        self.s = {k: fn(k) for k in self.s}
        self.diagnose()

    def rk3(self, dt):
        d0 = self.rhs()
        self._set(lambda k: self.s[k] + dt * d0[k])
        d1 = self.rhs()
        self._set(lambda k: self.s[k] + dt / 4 * (d1[k] - 3 * d0[k]))
        d2 = self.rhs(True)
        self._set(lambda k: self.s[k] + dt / 12 * (8 * d2[k] - d0[k] - d1[k]))

    def ef(self, dt):
        d = self.rhs(True)
        self._set(lambda k: self.s[k] + dt * d[k])

    def lfam3_start(self, dt):
        d = self.rhs()
        self.before = dict(self.s)
        self._set(lambda k: self.s[k] + dt * d[k])

    def lfam3(self, dt):
        now, d = dict(self.s), self.rhs()
        old = self.before
        self._set(lambda k: (5 * (old[k] + 2 * dt * d[k]) + 8 * now[k] - old[k]) / 12)
        d = self.rhs(True)
        self.before = now
        self._set(lambda k: now[k] + dt * d[k])

    def maxu2(self):
        return float(sum((self.s[k] * self.g.i2) ** 2 for k in ("u_i", "u_j", "u_k")).max())


def exact(case, seed):
    case = _full(case)
    if case["kind"] == "batch":
        ends = []
        for q, n in enumerate(_members(case)):
            e = _Exact(case, _Grid(case, (n, n, n)), seed * 1000 + q)
            e.diagnose()
            e.rk3(_rest_dt(case, e.g))
            ends.append(e.s)
        return ends
    g = _Grid(case)
    e = _Exact(case, g, seed)
    dt = _rest_dt(case, g)
    if case["kind"] == "solve":
        e.solve(e.div())
        return {"x": e.x}
    e.diagnose()
    if case["kind"] == "rhs":
        t = e.rhs()
        return {name: t[name] for name, _ in TEND}
    if case["kind"] == "monitor":
        return {"maxu2": e.maxu2(), "ke": float(e.ke.sum()), "bsum": float(e.s["b"].sum()),
                "nonfinite": 0}
    if case["scheme"] == "lfam3":
        e.lfam3_start(dt)
        e.lfam3(dt)
    else:
        if case["adapt"]:
            umax2 = e.maxu2()
            if umax2 > 0.0:
                dt = min(dt, 0.5 / math.sqrt(umax2))
        {"rk3": e.rk3, "ef": e.ef}[case["scheme"]](dt)
    return {k: e.s[k] for k in e.s}
