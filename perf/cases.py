"""The work a user of porturb_amd has it do, as cases that can be prepared, run, priced and checked.

    listed()              the listed cases (dicts of plain values)
    draw(rng)             one more case of the same ranges
    prepare(case, seed)   the state, contexts, networks and buffers a program holds before the call
    run(state)            one pass through the public entry points; its outputs whole
    work(case)            bytes and floating-point operations a pass cannot do without
    exact(case, seed)     what run() returns, from plain torch in 64 bits (None where not given)

Kinds of case:
    step      one physics step: Dycore.time_step, and with a closure surface_apply and les_apply,
              on coupler fields that the caller holds
    farm      one physics step of the C++ driver (core::Coupler and modules) of the wind-farm
              case with actuator disks
    closure   les_apply alone (plain, or with the learned closure)
    forcing   geostrophic_forcing and sponge_layer
    filter    pu_sgs_filter: box filter of a fine run into training targets
    train     Mlp.train_step, ten Adam steps, then the parameters

The flow fields are a sheared boundary layer (log law) with turbulence that decays with height,
smooth motion above it, buildings, moisture, subgrid TKE and passive tracers that fill only part
of the air, so that the limiter meets rough, smooth and uniform stencils as in a developed run.
Coupler fields are double in both precisions; a program that runs the FP32 mode hands them on in
single precision (the accuracy they are computed to), and so do the FP32 cases here.
"""
import ctypes
import math
import os
from fractions import Fraction

import torch

import porturb_amd as pa

DEV = "cuda"
F64 = torch.float64
MODEL = os.path.join(os.path.dirname(os.path.abspath(pa.__file__)), "data", "sgs_abl_urban_dx2.bin")
TURBINE = os.path.join(os.path.dirname(os.path.abspath(pa.__file__)), "data", "turbine_disk_ct075_d120.yaml")
FIELDS = ("density_dry", "uvel", "vvel", "wvel", "temp")
EXACT_CELLS = 36e6            # larger grids take plain torch too long


def _step(name, flow, nx, ny, nz, dx, order, precision, closure, bc="periodic", cycles=1.0, latitude=0.0):
    c = dict(kind="step", flow=flow, nx=nx, ny=ny, nz=nz, dx=dx, order=order, precision=precision,
             closure=closure, bc=bc, cycles=cycles, latitude=latitude)
    return dict(c, name=name) if name else c


def listed():
    return [
        # the dry warm bubble of the examples: 64^3, WENO-5, dycore only; a step of many small launches
        _step("bubble_64_fp64", "bubble", 64, 64, 64, 156.25, 5, "fp64", "none"),
        # a debugging or teaching run of the urban case: every module of the step at its smallest
        _step("urban_small_fp64", "urban", 48, 40, 32, 4.0, 9, "fp64", "tke"),
        # the benchmark workload: neutral urban boundary layer, WENO-9, 4 tracers, double
        _step("urban_1024_fp64", "urban", 1024, 1024, 128, 2.0, 9, "fp64", "tke"),
        # the same physics in the FP32 mode on a quarter of the domain
        _step("urban_512_fp32", "urban", 512, 512, 128, 2.0, 9, "fp32", "tke"),
        # FP32 with the learned closure on a ragged grid (sizes from a site plan, not powers of two)
        _step("urban_ragged_learned", "urban", 500, 310, 90, 2.0, 9, "fp32", "learned"),
        # an inflow-driven box at an odd size: precursor x, WENO-7, Coriolis, several dynamics cycles a step
        _step("inflow_ragged_fp64", "urban", 150, 70, 51, 8.0, 7, "fp64", "none", "precursor", 2.5, 43.0),
        # wind farm through the C++ driver: precursor inflow, actuator disks, learned closure, FP32
        dict(name="farm_driver_fp32", kind="farm", nx=640, ny=320, nz=96, dx=5.0, order=9, precision="fp32",
             closure="learned", columns=2, rows=1),
        # the closure by itself (a program that couples its own dynamics): double, TKE closure
        dict(name="closure_tke_fp64", kind="closure", nx=384, ny=250, nz=100, dx=2.0, precision="fp64", closure="tke"),
        # the learned closure by itself in the FP32 mode
        dict(name="closure_learned_fp32", kind="closure", nx=512, ny=256, nz=128, dx=2.0, precision="fp32", closure="learned"),
        # column forcing of a boundary-layer run, done once a step: geostrophic wind and the sponge
        dict(name="forcing_512", kind="forcing", nx=512, ny=512, nz=128, dx=2.0),
        # training data of the learned closure: a fine snapshot filtered by 2
        dict(name="filter_fine_by_2", kind="filter", nx=384, ny=256, nz=128, dx=1.0, ratio=2),
        # training of the learned closure: ten Adam steps of the shipped recipe's batch
        dict(name="train_batch_8192", kind="train", samples=200000, batch=8192, steps=10),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["step"] * 5 + ["farm", "closure", "closure", "forcing", "filter", "train"])
    nx, ny = _log_int(rng, 24, 700), _log_int(rng, 24, 700)
    nz = rng.randint(24, 144)
    if kind == "step":
        flow = rng.choice(["urban", "urban", "urban", "bubble"])
        closure = "none" if flow == "bubble" else rng.choice(["none", "tke", "tke", "learned"])
        return _step(None, flow, nx, ny, nz, 156.25 if flow == "bubble" else rng.choice([2.0, 4.0, 10.0]), rng.choice([3, 5, 5, 7, 9, 9, 9, 11]),
                     rng.choice(["fp64", "fp64", "fp32"]), closure, rng.choice(["periodic", "periodic", "precursor"]),
                     rng.choice([1.0, 1.0, 1.0, 2.0, 2.5]), rng.choice([0.0, 0.0, 43.0]))
    if kind == "farm":
        return dict(kind="farm", nx=rng.randint(160, 640), ny=rng.randint(120, 400), nz=rng.randint(56, 112), dx=5.0,
                    order=rng.choice([5, 9]), precision=rng.choice(["fp32", "fp64"]),
                    closure=rng.choice(["tke", "learned"]), columns=rng.randint(1, 2), rows=1)
    if kind == "closure":
        return dict(kind="closure", nx=nx, ny=ny, nz=nz, dx=2.0, precision=rng.choice(["fp64", "fp32"]),
                    closure=rng.choice(["tke", "learned"]))
    if kind == "forcing":
        return dict(kind="forcing", nx=nx, ny=ny, nz=nz, dx=rng.choice([2.0, 10.0]))
    if kind == "filter":
        r = rng.choice([2, 2, 3, 4])
        return dict(kind="filter", nx=r * _log_int(rng, 16, 190), ny=r * _log_int(rng, 16, 120), nz=r * rng.randint(8, 32),
                    dx=1.0, ratio=r)
    return dict(kind="train", samples=_log_int(rng, 20000, 400000), batch=_log_int(rng, 256, 16384), steps=rng.randint(4, 10))


# ------------------------------------------------------------------------------------------
# inputs
# ------------------------------------------------------------------------------------------
def _tracers(case):
    if case.get("flow") == "bubble":
        return [("water_vapor", True, True, True)]
    return [("water_vapor", True, True, True), ("TKE", True, False, False),
            ("passive_1", True, False, True), ("passive_2", True, False, True)]


def _config(case):
    n = (case["nx"], case["ny"], case["nz"])
    return pa.make_config(*n, *(m * case["dx"] for m in n), ord=case.get("order", 9), tracers=_tracers(case),
                          bc_x=pa.PU_BC_PRECURSOR if case.get("bc") == "precursor" else pa.PU_BC_PERIODIC,
                          precision=pa.PU_FP32 if case.get("precision") == "fp32" else pa.PU_FP64,
                          latitude=case.get("latitude", 0.0))


def _constants():
    R_d, cp_d, R_v, p0, grav = 287.0, 1003.0, 461.0, 1.0e5, 9.81
    gamma = cp_d / (cp_d - R_d)
    return R_d, cp_d, R_v, p0, grav, gamma, (R_d * p0 ** (-R_d / cp_d)) ** gamma


def _inputs(case, seed):
    """(fields [5], tracer masses, immersed_proportion) of the case as double tensors [nz][ny][nx]."""
    nx, ny, nz, dx = case["nx"], case["ny"], case["nz"], case["dx"]
    g = torch.Generator(DEV)
    g.manual_seed(int(seed) * 7919 + 11)
    R_d, cp_d, R_v, p0, grav, gamma, C0 = _constants()
    x = ((torch.arange(nx, device=DEV, dtype=F64) + 0.5) / nx)[None, None, :]
    y = ((torch.arange(ny, device=DEV, dtype=F64) + 0.5) / ny)[None, :, None]
    z = ((torch.arange(nz, device=DEV, dtype=F64) + 0.5) * dx)[:, None, None]
    height = nz * dx

    def rand(*shape):
        return torch.rand(shape, generator=g, device=DEV, dtype=F64)

    def smooth():                          # motion on the scale of the domain: a few modes
        f = torch.zeros((nz, ny, nx), device=DEV, dtype=F64)
        for m in range(3):
            p, a = rand(3) * 2 * math.pi, 0.3 + rand(1)
            f += a * (torch.sin(2 * math.pi * (m + 1) * x + p[0]) * torch.sin(2 * math.pi * y * (m + 1) + p[1])
                      * torch.cos(math.pi * (m + 1) * z / height + p[2]))
        return f

    def rough():                           # turbulence: noise on the grid scale and on eight cells
        f = torch.randn((nz, ny, nx), generator=g, device=DEV, dtype=F64)
        for ax in range(3):
            f = 0.25 * torch.roll(f, 1, ax) + 0.5 * f + 0.25 * torch.roll(f, -1, ax)
        c = torch.randn((1, 1, max(2, nz // 8), max(2, ny // 8), max(2, nx // 8)), generator=g, device=DEV, dtype=torch.float32)
        return f + torch.nn.functional.interpolate(c, (nz, ny, nx), mode="trilinear")[0, 0].double()

    def background(theta):
        exner = 1.0 - grav * z / (cp_d * theta)
        return ((p0 * exner ** (cp_d / R_d)) / C0) ** (1 / gamma) / theta

    rho = background(300.0).expand(nz, ny, nx).clone()
    imm = torch.zeros((nz, ny, nx), device=DEV, dtype=F64)
    if case.get("flow") == "bubble":
        # warm bubble in air with weak smooth motion
        r2 = ((x - 0.5) * nx * dx / 2000) ** 2 + ((y - 0.5) * ny * dx / 2000) ** 2 + ((z - 0.2 * height) / 2000) ** 2
        d = r2.sqrt() * (math.pi / 2)
        theta = 300.0 + torch.where(d <= math.pi / 2, (2 + rand(1)) * torch.cos(d) ** 2, torch.zeros_like(d))
        u, v, w = (0.5 * smooth() for _ in range(3))
        masses = [torch.zeros_like(rho)]
    else:
        layer = torch.exp(-z / (0.35 * height))
        u = 8.0 * torch.log((z + 0.1) / 0.1) / math.log(900.0) + 0.8 * layer * rough() + 0.02 * smooth()
        v = 0.5 * layer * rough() + 0.02 * smooth()
        w = 0.4 * layer * rough() * (z / (z + 10.0)) + 0.01 * smooth()
        deep = torch.where(z < 0.5 * height, layer, torch.zeros_like(layer))   # mixed below, neutral above
        theta = 300.0 + 0.2 * deep * rough()
        rho = rho * (1 + 1e-5 * smooth())
        wet = rho * (5e-3 * (1 + 0.1 * deep * rough()))
        tke = rho * (0.1 + 0.2 * layer * rough().abs())
        low = torch.where(z < 0.25 * height, torch.ones_like(z), torch.zeros_like(z))
        masses = [wet.clamp_min(0), tke, rho * low * (1 + 0.3 * rough()).clamp_min(0), rho * torch.where(x < 0.125, torch.ones_like(x), torch.zeros_like(x))]
        if case["kind"] != "farm" and case["kind"] != "filter":
            # up to eight by eight cuboid buildings, 10 to 40 m high or a third of the domain
            nb = max(1, min(8, nx // 12, ny // 12))
            tall = rand(nb, nb) * min(30.0, 0.2 * height) + min(10.0, 0.1 * height)
            bi, bj = (x * nb).long().clamp_max(nb - 1), (y * nb).long().clamp_max(nb - 1)
            fx, fy = (x * nb - bi - 0.5).abs(), (y * nb - bj - 0.5).abs()
            top = tall[bj.expand(1, ny, nx), bi.expand(1, ny, nx)]
            imm[(fx < 0.25) & (fy < 0.25) & (z < top)] = 1.0
            for f in (u, v, w):
                f[imm > 0] = 0.0
    full = rho + masses[0]
    temp = C0 * (full * theta) ** gamma / (rho * R_d + masses[0] * R_v)
    return [rho, u, v, w, temp], masses, imm


class Coupled:
    """Coupler fields of a program that holds them as torch tensors."""

    def __init__(self, cfg, fields, masses, imm):
        self.cfg, self.fields, self.masses, self.imm = cfg, [f.contiguous() for f in fields], [m.contiguous() for m in masses], imm.contiguous()
        self.c = pa.PuCouplerState()
        for name, f in zip(FIELDS, self.fields):
            setattr(self.c, name, f.data_ptr())
        for i, m in enumerate(self.masses):
            self.c.tracers[i] = m.data_ptr()
        self.c.immersed_proportion = self.imm.data_ptr()


class _Memory:
    """Device memory of the library as torch sees it; keeps `owner` alive."""

    def __init__(self, ptr, shape, kind, owner):
        self.owner = owner
        self.__cuda_array_interface__ = {"shape": tuple(shape), "typestr": kind, "data": (ptr, False), "version": 2}


def _view(ptr, shape, kind, owner):
    return torch.as_tensor(_Memory(ptr, shape, kind, owner), device=DEV)


def _network_inputs(case, seed):
    g = torch.Generator(DEV)
    g.manual_seed(int(seed) * 104729 + 5)
    n = case["samples"]
    x = torch.randn((n, 112), generator=g, device=DEV)
    x[:, 108:] = 0
    x = x.bfloat16()
    mix = torch.randn((108, 9), generator=g, device=DEV) / 10
    t = torch.tanh(x[:, :108].float() @ mix) + 0.05 * torch.randn((n, 9), generator=g, device=DEV)
    rows = torch.stack([torch.randint(0, n, (case["batch"],), generator=g, device=DEV, dtype=torch.int32) for _ in range(case["steps"])])
    shapes = ((64, 108), (64,), (64, 64), (64,), (9, 64), (9,))
    params = torch.cat([(torch.randn(s, generator=g, device=DEV) / math.sqrt(s[1])).reshape(-1) if len(s) == 2 else torch.zeros(s, device=DEV) for s in shapes])
    return x, t, rows, params


class _Buffer:
    def __init__(self, t):
        self.t, self.ptr = t, t.data_ptr()


def prepare(case, seed):
    kind, s = case["kind"], {"case": case}
    if kind == "train":
        x, t, rows, params = _network_inputs(case, seed)
        s["mlp"] = pa.Mlp(params.cpu().numpy())
        s["x"], s["t"], s["rows"] = _Buffer(x), _Buffer(t), [_Buffer(r) for r in rows]
        return s
    fields, masses, imm = _inputs(case, seed)
    s["single"] = case.get("precision") == "fp32"
    if kind == "farm":
        d = pa.Driver(pa.PU_CASE_WINDFARM, case["nx"], case["ny"], case["nz"], case["dx"], ord=case["order"],
                      precision=pa.PU_FP32 if s["single"] else pa.PU_FP64, seed=int(seed) & 0x7fffffff,
                      sgs_model=MODEL if case["closure"] == "learned" else None)
        d.set_turbines(TURBINE, case["columns"], case["rows"], orig_C_T=True)
        shape = (case["nz"], case["ny"], case["nx"])
        views = {n: _view(p, shape, "<f8", d) for n, p in d.field_pointers().items()}
        for n, f in zip(FIELDS, fields):
            views[n].copy_(f)
        for (n, _, _, _), m in zip(_tracers(case), masses):
            views[n].copy_(m)
        s["driver"], s["views"] = d, views
        torch.cuda.synchronize()
        return s
    cfg = _config(case)
    cs = Coupled(cfg, fields, masses, imm)
    d = pa.Dycore(cfg)
    s["coupled"], s["dycore"] = cs, d
    d.init(cs)
    s["dt"] = d.compute_time_step() * case.get("cycles", 1.0)
    closure = case.get("closure", "none")
    if closure == "learned":
        s["mlp"] = pa.Mlp.load(MODEL)
        d.set_sgs_model(s["mlp"])
    if kind == "filter":                   # the program's buffers for a filtered snapshot
        n = [case[k] // case["ratio"] for k in ("nz", "ny", "nx")]
        box = [m + 2 for m in n]
        s["filtered"] = [torch.zeros([6] + box, device=DEV, dtype=F64), torch.zeros(box, device=DEV, dtype=F64), torch.zeros([9] + n, device=DEV)]
    if kind == "step" and closure != "none":
        rough = torch.full_like(imm, 0.1)
        warm = torch.zeros_like(imm)
        pa.check(pa.lib().pu_surface_fluxes_init(d.ctx, rough.data_ptr(), warm.data_ptr(), rough[0].data_ptr(), warm[0].data_ptr()))
    torch.cuda.synchronize()
    return s


def run(s):
    case = s["case"]
    kind = case["kind"]
    if kind == "train":
        for rows in s["rows"]:
            s["mlp"].train_step(s["x"], s["t"], rows, case["batch"], 1e-3)
        return s["mlp"].get_params()
    if kind == "farm":
        s["driver"].step(1)
        return {n: v.float() if s["single"] else v for n, v in s["views"].items()}
    d, cs, dt = s["dycore"], s["coupled"], s["dt"]
    if kind == "filter":
        r = case["ratio"]
        les, imm, targets = s["filtered"]
        pa.check(pa.lib().pu_sgs_filter(d.ctx, ctypes.byref(cs.c), r, les.data_ptr(), imm.data_ptr(), targets.data_ptr()))
        return s["filtered"]
    if kind == "forcing":
        d.geostrophic_forcing(cs, dt, 43.3, 10.0, 0.0)
        d.sponge_layer(cs, dt, 10 * dt, 0.1)
        return cs.fields[1:]
    if kind == "step":
        d.time_step(cs, dt)
        if case["closure"] != "none":
            d.surface_apply(cs, dt)
    if case["closure"] != "none":
        d.les_apply(cs, dt)
    out = cs.fields + cs.masses
    return [f.float() for f in out] if s["single"] else out


# ------------------------------------------------------------------------------------------
# work
# ------------------------------------------------------------------------------------------
def _reconstruction(order, sides):
    """Operations of one limited reconstruction: total variations, then weights, map and combination a side."""
    n = (order + 1) // 2
    variation = order - 1 + n * ((n - 1) * (n - 2) + 3 * (n - 1)) + n
    return variation + 4 * n + sides * n * (2 * n + 22)


def work(case):
    kind = case["kind"]
    if kind == "train":
        n = case["batch"] * case["steps"]
        weights = 108 * 64 + 64 * 64 + 64 * 9
        return {"bytes": n * (224 + 36 + 4) + 4 * 11721, "flops": 6.0 * n * weights}
    cells = case["nx"] * case["ny"] * case["nz"]
    if kind == "forcing":
        return {"bytes": cells * (4 * 8 + 0.1 * 8 * 8), "flops": cells * 6.0}
    if kind == "filter":
        coarse = cells / case["ratio"] ** 3
        return {"bytes": 6 * 8 * cells + coarse * (7 * 8 + 9 * 4), "flops": 60.0 * cells}
    ntr = len(_tracers(case))
    closure = case.get("closure", "none")
    flops = {"none": 0, "tke": 500, "learned": 24000}[closure]
    if kind == "closure":
        return {"bytes": cells * (8 * (5 + ntr) + 8 * (4 + ntr) + 1), "flops": float(flops * cells)}
    # a step: the pressure, density and normal velocity on both sides of a face, the transported
    # quantities on its upwind side
    nf = 6 + ntr
    stage = 3 * (3 * _reconstruction(case["order"], 2) + (nf - 3) * _reconstruction(case["order"], 1) + 16 + 5 * nf) + 40
    cycles = math.ceil(case.get("cycles", 1.0) - 1e-9)
    return {"bytes": cells * (16.0 * (5 + ntr) + 10), "flops": float(cells) * (3 * cycles * stage + flops)}


# ------------------------------------------------------------------------------------------
# the same in plain torch, 64 bits
# ------------------------------------------------------------------------------------------
def _solve(rows, rhs):
    """Exact solution of a small linear system (Fractions); rhs: list of columns."""
    n = len(rows)
    a = [list(r) + list(b) for r, b in zip(rows, rhs)]
    for c in range(n):
        p = next(r for r in range(c, n) if a[r][c])
        a[c], a[p] = a[p], a[c]
        a[c] = [v / a[c][c] for v in a[c]]
        for r in range(n):
            if r != c and a[r][c]:
                a[r] = [v - a[r][c] * w for v, w in zip(a[r], a[c])]
    return [r[n:] for r in a]


def _polynomial(offsets):
    """Coefficients (rows) from cell averages (columns) at the given offsets from the cell."""
    n = len(offsets)
    half = Fraction(1, 2)
    rows = [[((o + half) ** (k + 1) - (o - half) ** (k + 1)) / (k + 1) for k in range(n)] for o in offsets]
    return _solve(rows, [[Fraction(int(i == j)) for j in range(n)] for i in range(n)])


class _Weno:
    def __init__(self, order):
        self.order, self.hs = order, (order - 1) // 2
        n = self.hs + 1
        half = Fraction(1, 2)
        at = lambda c, x: [sum(c[k][i] * x ** k for k in range(len(c))) for i in range(len(c[0]))]  # noqa: E731
        sub = [_polynomial([m + r - self.hs for r in range(n)]) for m in range(n)]
        whole = _polynomial([i - self.hs for i in range(order)])
        self.coef = [[[float(v) for v in row] for row in c] for c in sub]
        self.face, self.ideal = [], []
        for x in (-half, half):
            rows = [at(c, x) for c in sub]
            full, d = at(whole, x), []
            for c in range(n):            # cell c is covered by the sub-stencils 0 .. c
                d.append((full[c] - sum(d[m] * rows[m][c - m] for m in range(c))) / rows[c][0])
            self.face.append([[float(v) for v in r] for r in rows])
            self.ideal.append([float(v) for v in d])
        # total variation: squares of the derivatives, powers below n, over the cell
        self.tv = {}
        for l in range(1, n):
            for a in range(l, n):
                for b in range(l, n):
                    q = a + b - 2 * l
                    if q < n and q % 2 == 0:
                        fall = lambda k: Fraction(math.factorial(k), math.factorial(k - l))  # noqa: E731,B023
                        key = (min(a, b), max(a, b))
                        self.tv[key] = self.tv.get(key, 0) + float(fall(a) * fall(b) * 2 * half ** (q + 1) / (q + 1))

    def edges(self, s, mapped, imm_left, imm_right):
        """Both interface values from the stencil s [order]."""
        n = self.hs + 1
        tv = []
        for m in range(n):
            a = [None] + [sum(self.coef[m][k][i] * (s[m + i] - s[self.hs]) for i in range(n)) for k in range(1, n)]
            tv.append(sum(c * a[p] * a[q] for (p, q), c in self.tv.items()))
        total = sum(tv)
        scale = torch.where(total > 1e-20, 1 / total, torch.ones_like(total))
        tv = [t * scale for t in tv]
        largest = tv[0]
        for t in tv[1:]:
            largest = torch.maximum(largest, t)
        tv[n - 1] = torch.where(imm_left, largest, tv[n - 1])
        tv[0] = torch.where(imm_right, largest, tv[0])
        inverse = [1 / (t * t + 1e-20) for t in tv]
        out = []
        for side in (0, 1):
            d = self.ideal[side]
            w = [d[m] * inverse[m] for m in range(n)]
            total = sum(w)
            w = [v / total for v in w]
            if self.order == 3:
                h = [v * (q + q * q - 3 * q * v + v * v) / (q * q + (1 - 2 * q) * v) for v, q in zip(w, d)]
            else:
                h = [q + (v - q) ** 7 / ((v - q) ** 6 + 2000 * (v * (1 - v)) ** 3) for v, q in zip(w, d)]
            total = sum(h)
            w = [torch.where(mapped, v / total, u) for v, u in zip(h, w)]
            out.append(sum(w[m] * sum(self.face[side][m][i] * s[m + i] for i in range(n)) for m in range(n)))
        return out


class _Flow:
    """The dycore step, surface fluxes and TKE closure of a case in plain torch."""

    def __init__(self, case, fields, masses, imm):
        self.R_d, _, self.R_v, _, self.grav, self.gamma, self.C0 = _constants()
        self.case, self.imm = case, imm
        self.names = _tracers(case)
        self.n = (case["nz"], case["ny"], case["nx"])
        self.dx = case["dx"]
        self.weno = _Weno(case.get("order", 9))
        self.hs = self.weno.hs
        self.inflow = case.get("bc") == "precursor"
        self.fcor = 2 * 7.2921e-5 * math.sin(case.get("latitude", 0.0) / 180 * math.pi)
        self.background(fields, masses)
        self.masks()

    # hydrostatic levels with isentropic halo, and their interface values
    def background(self, fields, masses):
        state = self.conserved(fields, masses, relax=False)
        nz, hs, g, gm = self.n[0], self.hs, self.grav, self.gamma
        mean = lambda f: [float(v) for v in f.mean((1, 2))]  # noqa: E731
        r, t, p = mean(state[0]), mean(state[4] / state[0]), mean(self.C0 * state[4] ** gm)
        for end in (0, 1):
            r0, t0 = (r[-1], t[-1]) if end else (r[0], t[0])
            for k in range(1, hs + 1):
                rk = (r0 ** (gm - 1) + (-1 if end else 1) * g * (gm - 1) * self.dx * k / (gm * self.C0 * t0 ** gm)) ** (1 / (gm - 1))
                new = (rk, t0, self.C0 * (rk * t0) ** gm)
                for col, v in zip((r, t, p), new):
                    col.append(v) if end else col.insert(0, v)
        self.re, self.te = [], []
        for k in range(nz + 1):
            at = hs + k
            if self.weno.order < 5:
                w = ((-1, 0.5), (0, 0.5))
            else:
                w = ((-2, -1 / 12), (-1, 7 / 12), (0, 7 / 12), (1, -1 / 12))
            self.re.append(math.exp(sum(c * math.log(r[at + o]) for o, c in w)))
            self.te.append(sum(c * t[at + o] for o, c in w))
        col = lambda v: torch.tensor(v, device=DEV, dtype=F64)[:, None, None]  # noqa: E731
        self.r, self.t, self.p = (col(v[hs:hs + nz]) for v in (r, t, p))
        self.re, self.te = col(self.re), col(self.te)

    def wrap(self, f, pad, low, high):
        """f with `pad` periodic cells in x and y, and levels of `low` below and `high` above."""
        f = torch.cat([torch.full_like(f[:1], low)] * pad + [f] + [torch.full_like(f[:1], high)] * pad, 0)
        for ax in (1, 2):
            n = f.shape[ax]
            idx = torch.arange(-pad, n + pad, device=DEV) % n
            f = f.index_select(ax, idx)
        return f

    def spread(self, mask, rad, low, high):
        """Whether any cell of the cube of the given radius is set."""
        m = self.wrap(mask.float(), rad, low, high)[None, None]
        return torch.nn.functional.max_pool3d(m, 2 * rad + 1, 1)[0, 0] > 0

    def masks(self):
        solid = self.imm > 0
        self.near = self.spread(solid, 10, 0.0, 0.0)
        tau = torch.ones_like(self.imm)
        for rad, v in ((3, 2.0), (2, 4.0), (1, 8.0)):
            tau = torch.where(self.spread(self.imm == 0, rad, 0.0, 0.0), torch.full_like(tau, v), tau)
        self.relax = self.imm ** 5 / tau
        self.stencils = []
        hs, order = self.hs, self.weno.order
        box = self.wrap(solid.float(), hs, 1.0, 1.0) > 0
        for ax in range(3):             # z, y, x
            f = []
            for q in range(order):
                v = box
                for a in range(3):
                    v = v.narrow(a, q if a == ax else hs, self.n[a])
                f.append(v)
            lo, hi = torch.zeros(self.n, device=DEV, dtype=torch.long), torch.full(self.n, order - 1, device=DEV)
            for q in range(order - 1, hs, -1):
                hi = torch.where(f[q], torch.full_like(hi, q - 1), hi)
            for q in range(hs):
                lo = torch.where(f[q], torch.full_like(lo, q + 1), lo)
            lo, hi = torch.where(f[hs], torch.zeros_like(lo), lo), torch.where(f[hs], torch.full_like(hi, order - 1), hi)
            any_window = bool(((lo > 0) | (hi < order - 1)).any())
            self.stencils.append((lo.to(torch.int8), hi.to(torch.int8), f[hs - 1].clone(), f[hs + 1].clone(), any_window))

    # conversions
    def settle(self, state):
        target = [self.r, 0.0, 0.0, 0.0, self.r * self.t] + [0.0] * (len(state) - 5)
        out = [v + (w - v) * self.relax for v, w in zip(state, target)]
        return self.clip(out)

    def clip(self, state):
        return state[:5] + [v.clamp_min(0) if t[1] else v for v, t in zip(state[5:], self.names)]

    def conserved(self, fields, masses, relax=True):
        rho_d, u, v, w, temp = fields
        press = rho_d * self.R_d * temp + masses[0] * self.R_v * temp
        rho = rho_d + sum(m for m, t in zip(masses, self.names) if t[2])
        state = [rho, rho * u, rho * v, rho * w, (press / self.C0) ** (1 / self.gamma)] + list(masses)
        return self.settle(state) if relax else state

    def coupled(self, state):
        rho, masses = state[0], state[5:]
        rho_d = rho - sum(m for m, t in zip(masses, self.names) if t[2])
        temp = self.C0 * state[4] ** self.gamma / (rho_d * self.R_d + masses[0] * self.R_v)
        return [rho_d] + [state[k] / rho for k in (1, 2, 3)] + [temp], masses

    # one direction
    def halo(self, f, ax, zero):
        n, p = f.shape[ax], self.hs
        idx = torch.arange(-p, n + p, device=DEV)
        if ax == 0 or (ax == 2 and self.inflow):
            out = f.index_select(ax, idx.clamp(0, n - 1))
            if ax == 0 and zero:
                out[:p], out[-p:] = 0, 0
            return out
        return f.index_select(ax, idx % n)

    def edges(self, f, ax, window, zero=False):
        box = self.halo(f, ax, zero)
        lo, hi, left, right, some = self.stencils[ax]
        s = [box.narrow(ax, q, f.shape[ax]) for q in range(self.weno.order)]
        if window and some:
            wide, s = s, []
            for q in range(self.weno.order):
                at = torch.clamp(torch.full_like(lo, q), lo, hi)
                v = wide[q]
                for k in range(self.weno.order):
                    if k != q:
                        v = torch.where(at == k, wide[k], v)
                s.append(v)
        return self.weno.edges(s, ~self.near, left, right)

    def faces(self, pair, ax, wall=None):
        """Values left and right of every interface (n + 1 of them) from the cells' two edges."""
        low, high = pair
        n = low.shape[ax]
        first, last = low.narrow(ax, 0, 1), high.narrow(ax, n - 1, 1)
        if ax == 0 or (ax == 2 and self.inflow):
            a, b = first, last
        else:
            a, b = last, first
        left, right = torch.cat([a, high], ax), torch.cat([low, b], ax)
        if ax == 0 and wall is not None:
            for f in (left, right):
                f[0], f[-1] = wall, wall
        return left, right

    def direction(self, prim, ax, tend):
        normal = {0: 3, 1: 2, 2: 1}[ax]                  # state index of the normal velocity
        hr, ht = (self.re, self.te) if ax == 0 else (self.r, self.t)
        rl, rr = self.faces(self.edges(prim["rho"], ax, False), ax)
        ul, ur = self.faces(self.edges(prim[normal], ax, False, normal == 3), ax, 0.0 if ax == 0 else None)
        pl, pr = self.faces(self.edges(prim["p"], ax, True), ax)
        ml, mr = ul * (rl + hr), ur * (rr + hr)
        p_up = 0.5 * (pl + pr - 350.0 * (mr - ml))
        flow = 0.5 * (ml + mr - (pr - pl) / 350.0)
        from_left = flow > 0
        diff = lambda f: (f.narrow(ax, 0, f.shape[ax] - 1) - f.narrow(ax, 1, f.shape[ax] - 1)) / self.dx  # noqa: E731
        tend[0] += diff(flow)
        tend[normal] += diff(flow * torch.where(from_left, ul, ur) + p_up)
        for k in range(1, 5 + len(self.names)):
            if k == normal:
                continue
            l, r = self.faces(self.edges(prim[k], ax, k < 4, k in (3, 4)), ax, 0.0 if k == 4 else None)
            if k == 4:
                l, r = l + ht, r + ht
            tend[k] += diff(flow * torch.where(from_left, l, r))

    def tendencies(self, state):
        rho = state[0]
        prim = {"rho": rho - self.r, "p": self.C0 * state[4] ** self.gamma - self.p}
        for k in range(1, len(state)):
            prim[k] = state[k] / rho
        prim[4] = prim[4] - self.t
        tend = [torch.zeros_like(rho) for _ in state]
        for ax in (0, 1, 2):
            self.direction(prim, ax, tend)
        tend[3] -= self.grav * (rho - self.r)
        if self.fcor:
            tend[1] += self.fcor * state[2]
            tend[2] -= self.fcor * state[1]
        return tend

    def time_step(self, fields, masses, dt, cycles):
        state = self.conserved(fields, masses)
        for c in range(cycles):
            if c:
                state = self.settle(state)
            h = dt / cycles
            new = self.settle([a + h * t for a, t in zip(state, self.tendencies(state))])
            new = self.settle([0.75 * a + 0.25 * b + 0.25 * h * t for a, b, t in zip(state, new, self.tendencies(new))])
            new = [a / 3 + 2 * b / 3 + 2 * h * t / 3 for a, b, t in zip(state, new, self.tendencies(new))]
            state = self.settle(self.clip(new))
        return self.coupled(state)

    # the rough wall: log-law drag against every solid neighbour
    def surface(self, fields, dt):
        rho_d, u, v, w, temp = fields
        box = self.wrap((self.imm > 0).float(), 1, 1.0, 0.0) > 0
        drag = 0.16 / math.log((self.dx / 2 + 0.1) / 0.1) ** 2 / self.dx
        vel, tend = {2: u, 1: v, 0: w}, {a: torch.zeros_like(u) for a in range(3)}
        for ax in range(3):
            a, b = [q for q in range(3) if q != ax]
            speed = (vel[a] ** 2 + vel[b] ** 2).sqrt()
            for side in (0, 2):
                solid = box
                for q in range(3):
                    solid = solid.narrow(q, side if q == ax else 1, self.n[q])
                for q in (a, b):
                    tend[q] -= torch.where(solid, drag * vel[q] * speed, torch.zeros_like(u))
        return [rho_d, u + dt * tend[2], v + dt * tend[1], w + dt * tend[0], temp]

    # the TKE closure
    def closure(self, fields, masses, dt):
        rho_d, u, v, w, temp = fields
        tke = next(i for i, t in enumerate(self.names) if t[0] == "TKE")
        theta = (rho_d * self.R_d * temp / self.C0) ** (1 / self.gamma) / rho_d
        mixed = [i for i, t in enumerate(self.names) if t[3]]
        n, d, g = self.n, self.dx, self.grav
        solid = self.wrap(self.imm, 1, 1.0, 0.0)

        def box(f, level):
            f = torch.cat([f[:1], f, f[-1:]], 0)
            if level == "zero":
                f[0], f[-1] = 0, 0
            for ax in (1, 2):
                m = f.shape[ax]
                idx = torch.arange(-1, m + 1, device=DEV)
                inner = f.index_select(ax, idx % m)
                if ax == 2 and self.inflow:        # the faces copy the edge cells, the corners wrap
                    edge = f.index_select(ax, idx.clamp(0, m - 1))
                    inner[:, 1:-1] = edge[:, 1:-1]
                f = inner
            return f

        R, U, V, W, T, K = (box(f, level) for f, level in ((rho_d, ""), (u, ""), (v, ""), (w, "zero"), (theta, ""), ((masses[tke] / rho_d).clamp_min(0), "")))
        gm = self.gamma
        for k, sgn in ((0, 1.0), (-1, -1.0)):
            R[k] = (R[k] ** (gm - 1) + sgn * g * (gm - 1) * d / (gm * self.C0 * T[k] ** gm)) ** (1 / (gm - 1))
        Q = [box(masses[i] / rho_d, "") for i in mixed]

        def at(f, off, faces=None):
            for ax in range(3):
                f = f.narrow(ax, 1 + off[ax], n[ax] + (1 if ax == faces else 0))
            return f

        unit = ((1, 0, 0), (0, 1, 0), (0, 0, 1))
        minus = lambda a: tuple(-x for x in a)  # noqa: E731
        add = lambda a, b: tuple(x + y for x, y in zip(a, b))  # noqa: E731
        vel = {0: W, 1: V, 2: U}
        tend = {key: torch.zeros(n, device=DEV, dtype=F64) for key in (0, 1, 2, "t", "k")}
        qtend = [torch.zeros(n, device=DEV, dtype=F64) for _ in Q]
        cap = 0.25 * d * d / dt
        for ax in range(3):
            m, c = minus(unit[ax]), (0, 0, 0)
            F = lambda f, off: at(f, off, ax)  # noqa: E731,B023
            across = lambda f, e: 0.25 / d * (F(f, add(m, unit[e])) - F(f, add(m, minus(unit[e]))) + F(f, unit[e]) - F(f, minus(unit[e])))  # noqa: E731,B023
            slope = lambda f, e: (F(f, c) - F(f, m)) / d if e == ax else across(f, e)  # noqa: E731,B023
            mid = lambda f: 0.5 * (F(f, m) + F(f, c))  # noqa: E731,B023
            rho, k, t = mid(R), mid(K), mid(T)
            dtdz = slope(T, 0)
            N = torch.where(dtdz >= 0, (g / t * dtdz).clamp_min(0).sqrt(), torch.zeros_like(t))
            ell = (0.76 * k.sqrt() / (N + 1e-20)).clamp_max(d)
            km = 0.1 * ell * k.sqrt()
            visc, visc_t = km.clamp_max(0.5 * cap), (km * (1 + 2 * ell) / d).clamp_max(0.5 * cap)
            open_ = ~((F(solid, m) == 1) | (F(solid, c) == 1))
            div = sum(slope(vel[e], e) for e in range(3))
            diff = lambda f: (f.narrow(ax, 0, n[ax]) - f.narrow(ax, 1, n[ax])) / d  # noqa: E731,B023
            shut = lambda f: torch.where(open_, f, torch.zeros_like(f))  # noqa: E731,B023
            for e in range(3):
                s = slope(vel[e], ax) + slope(vel[ax], e) - (2.0 / 3.0 * div if e == ax else 0.0)
                tend[e] += diff(shut(-rho * visc * s))
            tend["t"] += diff(shut(-rho * visc_t * slope(T, ax)))
            tend["k"] += diff(shut(-rho * visc * 2 * slope(K, ax)))
            for q in range(len(Q)):
                qtend[q] += diff(shut(-rho * visc * slope(Q[q], ax)))
        c = (0, 0, 0)
        rho, k, t = at(R, c), at(K, c), at(T, c)
        dtdz = (at(T, unit[0]) - at(T, minus(unit[0]))) / (2 * d)
        N = torch.where(dtdz >= 0, (g / t * dtdz).clamp_min(0).sqrt(), torch.zeros_like(t))
        ell = (0.76 * k.sqrt() / (N + 1e-20)).clamp_max(d)
        km = 0.1 * ell * k.sqrt()
        grad = {}
        for e in range(3):
            for ax in range(3):
                up, dn = at(vel[e], unit[ax]), at(vel[e], minus(unit[ax]))
                if e != ax:                       # tangential velocities do not reach into solid cells
                    up = torch.where(at(solid, unit[ax]) > 0, at(vel[e], c), up)
                    dn = torch.where(at(solid, minus(unit[ax])) > 0, at(vel[e], c), dn)
                grad[e, ax] = (up - dn) / (2 * d)
        shear = sum((grad[e, ax] + grad[ax, e]) * grad[e, ax] for e in range(3) for ax in range(3))
        src = -g * rho * km * (1 + 2 * ell) / d / t * dtdz - rho * (0.19 + 0.51 * ell / d) / d * k * k.sqrt() + rho * km * shear
        src = torch.where(at(solid, c) == 1, torch.zeros_like(src), src)
        out = [rho_d] + [f + dt * tend[e] / rho for f, e in ((u, 2), (v, 1), (w, 0))]
        out.append(self.C0 * (theta * rho + dt * tend["t"]) ** self.gamma / (rho * self.R_d))
        masses = list(masses)
        masses[tke] = (k * rho + dt * (tend["k"] + src)).clamp_min(0)
        for i, q in zip(mixed, qtend):
            masses[i] = masses[i] + dt * q
        return out, masses


def _exact_train(case, seed):
    x, t, rows, params = _network_inputs(case, seed)
    p = params.double().requires_grad_(True)
    first, second = torch.zeros_like(p), torch.zeros_like(p)
    cuts = (64 * 108, 64, 64 * 64, 64, 9 * 64, 9)
    for step, r in enumerate(rows, 1):
        w1, b1, w2, b2, w3, b3 = torch.split(p, cuts)
        a = torch.relu(x[r.long(), :108].double() @ w1.view(64, 108).T + b1)
        a = torch.relu(a @ w2.view(64, 64).T + b2)
        loss = ((a @ w3.view(9, 64).T + b3 - t[r.long()].double()) ** 2).mean()
        (g,) = torch.autograd.grad(loss, p)
        first, second = 0.9 * first + 0.1 * g, 0.999 * second + 0.001 * g * g
        with torch.no_grad():
            p = p - 1e-3 * (first / (1 - 0.9 ** step)) / ((second / (1 - 0.999 ** step)).sqrt() + 1e-8)
        p.requires_grad_(True)
    return p.detach()


def _exact_filter(case, fields, imm):
    R_d, _, _, _, _, gamma, C0 = _constants()
    r = case["ratio"]
    n = tuple(case[k] // r for k in ("nz", "ny", "nx"))
    mean = lambda f: f.view(n[0], r, n[1], r, n[2], r).mean((1, 3, 5))  # noqa: E731
    rho, u, v, w, temp = fields
    theta = (rho * R_d * temp / C0) ** (1 / gamma) / rho
    m = [mean(f) for f in (rho, u, v, w, theta)]
    vel = (u, v, w)
    pairs = ((0, 0), (0, 1), (0, 2), (1, 1), (1, 2), (2, 2))
    tau = [mean(vel[a] * vel[b]) - m[1 + a] * m[1 + b] for a, b in pairs]
    heat = [mean(vel[a] * theta) - m[1 + a] * m[4] for a in range(3)]
    k = 0.5 * (tau[0] + tau[3] + tau[5])

    def box(f, level=None):
        f = torch.cat([f[:1], f, f[-1:]], 0)
        if level is not None:
            f[0], f[-1] = level, level
        for ax in (1, 2):
            f = f.index_select(ax, torch.arange(-1, f.shape[ax] + 1, device=DEV) % f.shape[ax])
        return f

    solid = imm.view(n[0], r, n[1], r, n[2], r).amax((1, 3, 5))
    les = torch.stack([box(m[0]), box(m[1]), box(m[2]), box(m[3], 0.0), box(m[4]), box(k)])
    return [les, box(solid, 1.0), torch.stack(tau + heat)]


def exact(case, seed):
    kind = case["kind"]
    if kind == "train":
        return _exact_train(case, seed)
    if kind == "farm" or case.get("closure") == "learned" or case["nx"] * case["ny"] * case["nz"] > EXACT_CELLS:
        return None
    fields, masses, imm = _inputs(case, seed)
    if kind == "filter":
        return _exact_filter(case, fields, imm)
    dt = 0.6 * case["dx"] / 450.0
    if kind == "forcing":
        f = 2 * 7.2921e-5 * math.sin(43.3 / 180 * math.pi)
        _, u, v, w, temp = fields
        mu, mv = u.mean((1, 2), keepdim=True), v.mean((1, 2), keepdim=True)
        u, v = u + dt * f * mv, v - dt * f * (mu - 10.0)
        height = case["nz"] * case["dx"]
        z = ((torch.arange(case["nz"], device=DEV, dtype=F64) + 0.5) * case["dx"])[:, None, None]
        z1 = 0.9 * height
        a = torch.where(z > z1, ((z - z1) / (height - z1)) ** 3 * 0.1, torch.zeros_like(z))
        ease = lambda q, to: a * to + (1 - a) * q  # noqa: E731
        return [ease(u, u.mean((1, 2), keepdim=True)), ease(v, v.mean((1, 2), keepdim=True)), ease(w, 0.0),
                ease(temp, temp.mean((1, 2), keepdim=True))]
    flow = _Flow(case, fields, masses, imm)
    if kind == "step":
        dt *= case["cycles"]
        fields, masses = flow.time_step(fields, masses, dt, math.ceil(case["cycles"] - 1e-9))
        if case["closure"] != "none":
            fields = flow.surface(fields, dt)
    if case["closure"] != "none":
        fields, masses = flow.closure(fields, masses, dt)
    return list(fields) + list(masses)
