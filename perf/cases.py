"""The work that performance of this framework is measured on.

Every case is a run, or a part of one, as a program drives it through `fdtd3d_amd.engine`: the
handle is created and given its materials in `prepare`, and a pass advances it by the case's time
steps and reads the fields back as numpy arrays, which is how results leave the engine.  Handles
keep advancing from pass to pass, as a long run does; the adjoint starts over with every forward.

`exact` restates the update in 64 bits with plain torch (whole arrays, no kernel of this
repository): curl, PML D / B stage, Drude recursion, TF/SF correction, sources, far field; the
adjoint's gradient comes from torch's autograd over that restatement.
"""
import math

import numpy as np
import torch

from fdtd3d_amd.config import (Config, SCHEME_DIM3, SCHEME_EXHY, SCHEME_EYHZ, SCHEME_EZHX, SCHEME_TEX, SCHEME_TEZ,
                               SCHEME_TMY, SCHEME_TMZ)
from fdtd3d_amd.engine import Batch, Engine

DX, WAVELENGTH, COURANT = 0.0005, 0.02, 0.5   # 40 cells a wavelength
PERIOD = 80.0                                 # steps a period of the source

SCHEMES = {"3d": SCHEME_DIM3, "tmz": SCHEME_TMZ, "tez": SCHEME_TEZ, "tex": SCHEME_TEX, "tmy": SCHEME_TMY,
           "exhy": SCHEME_EXHY, "eyhz": SCHEME_EYHZ, "ezhx": SCHEME_EZHX}


def grid(name, scheme, size, precision, steps, **more):
    """A single simulation: `size` along the scheme's axes, inset PML and TF/SF borders."""
    case = {"name": name, "kind": "grid", "scheme": scheme, "precision": precision, "steps": steps,
            "x": size[0], "y": size[1], "z": size[2], "pml": 10, "tfsf": 16, "teta": 30.0, "phi": 45.0, "psi": 90.0,
            "eps": "blocks", "mu": False, "source": False, "drude": 0, "layout": 0}
    case.update(more)
    return case


def listed():
    return [
        # a 1D validation run of the test suite: ExHy, 600 cells, PML 50, the wave enters at cell
        # 150 and meets a dielectric half-space; thousands of tiny steps, all launches and latency
        grid("line-exhy-600", "exhy", (1, 1, 600), 8, 400, pml=50, tfsf=150, tfsf_right=0, teta=0.0, phi=0.0,
             eps="half"),
        # the reference's default size and step count as a 2D run with a hard source in FP64
        grid("tmz-100", "tmz", (100, 100, 1), 8, 100, tfsf=0, source=True, teta=90.0, phi=0.0),
        # one simulation of the 2D sweep on its own, ragged, with an oblique plane wave
        grid("tmz-1403x977", "tmz", (1403, 977, 1), 4, 200, pml=12, tfsf=24, teta=90.0, phi=30.0),
        # the accurate-sphere validation grid: 80^3 FP64, PML 10, TF/SF 20, normal incidence
        grid("sphere-80", "3d", (80, 80, 80), 8, 100, tfsf=20, teta=0.0, phi=0.0, psi=0.0, eps="sphere"),
        # an ordinary ragged 3D run: oblique wave, hard source, a mu grid besides eps
        grid("3d-251x187x301", "3d", (251, 187, 301), 4, 120, source=True, mu=True),
        # the headline family: 512^3 FP32, PML 16, TF/SF 24, oblique incidence, eps in 8^3 blocks
        grid("3d-512", "3d", (512, 512, 512), 4, 200, pml=16, tfsf=24),
        # the same in FP64, the reference's default value type
        grid("3d-320-fp64", "3d", (320, 320, 320), 8, 150, pml=16, tfsf=24),
        # metamaterial slab: Drude terms in the central 128^3
        grid("drude-256", "3d", (256, 256, 256), 4, 120, pml=16, tfsf=24, drude=128),
        # the other Yee layout
        grid("h-centered-192", "3d", (192, 192, 192), 4, 120, pml=16, tfsf=24, layout=1),
        # a sweep: sixteen 2D simulations of different sizes advanced together
        {"name": "batch-16", "kind": "batch", "sims": 16, "lo": 256, "hi": 1024, "pml": 12, "steps": 1000, "shape": 11},
        # inverse design: J and dJ/deps over a design box, state checkpoints every 50 steps
        {"name": "adjoint-128", "kind": "adjoint", "n": 128, "precision": 4, "steps": 160, "pml": 16, "tfsf": 24,
         "design": 32, "window": 40, "every": 50},
        # complex fields and their far field: 64^3 FP64, a diagram of 37 azimuths
        {"name": "complex-ntff-64", "kind": "ntff", "n": 64, "precision": 8, "steps": 60, "pml": 8, "tfsf": 14,
         "step_angle": 10.0},
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["line", "2d", "2d", "3d", "3d", "3d", "3d", "drude", "batch", "adjoint", "ntff"])
    prec = rng.choice([4, 8])
    if kind == "line":
        scheme = rng.choice(["exhy", "eyhz", "ezhx"])
        n = _log(rng, 200, 4000)
        size = {"exhy": (1, 1, n), "eyhz": (n, 1, 1), "ezhx": (1, n, 1)}[scheme]
        ang = {"exhy": (0.0, 0.0), "eyhz": (90.0, 0.0), "ezhx": (90.0, 90.0)}[scheme]
        c = grid("", scheme, size, prec, rng.randint(100, 400), pml=rng.randint(8, 50), tfsf=rng.randint(60, 80),
                 tfsf_right=0, teta=ang[0], phi=ang[1])
    elif kind == "2d":
        scheme = rng.choice(["tmz", "tmz", "tez", "tex", "tmy"])
        a, b = _log(rng, 64, 1500), _log(rng, 64, 1500)
        tfsf = rng.choice([0, rng.randint(18, 28)])
        size = {"tmz": (a, b, 1), "tez": (a, b, 1), "tex": (1, a, b), "tmy": (a, 1, b)}[scheme]
        c = grid("", scheme, size, prec, rng.randint(60, 200), pml=rng.randint(5, 16),
                 tfsf=tfsf, teta=90.0 if scheme in ("tmz", "tez") else 40.0,
                 phi=rng.choice([0.0, 30.0, 45.0]) if scheme in ("tmz", "tez") else (90.0 if scheme == "tex" else 0.0),
                 source=tfsf == 0 or rng.random() < 0.3)
    elif kind == "3d":
        long = rng.random() < 0.3   # rows of up to 1024 cells
        size = tuple(_log(rng, 32, 320) for _ in range(2)) + (_log(rng, 300, 1024) if long else _log(rng, 32, 320),)
        pml = rng.choice([0, 8, 10, 16])
        if min(size) < 48:
            pml = min(pml, 8)
        while size[0] * size[1] * size[2] * (prec // 4) > 32 << 20:
            size = (max(32, size[0] * 3 // 4), max(32, size[1] * 3 // 4), size[2])
        tfsf = rng.choice([0, min(pml + rng.randint(2, 8), min(size) // 2 - 4)])
        c = grid("", "3d", size, prec, rng.randint(40, 120), pml=pml, tfsf=max(0, tfsf),
                 teta=rng.choice([0.0, 30.0, 75.0]), phi=rng.choice([0.0, 45.0, 20.0]), psi=rng.choice([0.0, 90.0]),
                 source=tfsf <= 0 or rng.random() < 0.3, mu=rng.random() < 0.25, layout=int(rng.random() < 0.2))
    elif kind == "drude":
        n = _log(rng, 72, 220)
        c = grid("", "3d", (n, n + rng.randint(-7, 7), n + rng.randint(-7, 7)), prec, rng.randint(40, 120), pml=10,
                 teta=rng.choice([15.0, 30.0, 60.0]), phi=20.0, psi=rng.choice([40.0, 90.0]),
                 drude=rng.randint(8, n // 2))
    elif kind == "batch":
        lo = _log(rng, 64, 512)
        c = {"kind": "batch", "sims": rng.randint(2, 20), "lo": lo, "hi": rng.randint(lo, 1100), "pml": rng.choice([0, 12]),
             "steps": rng.randint(200, 1000), "shape": rng.randint(0, 1 << 20)}
    elif kind == "adjoint":
        n = rng.randint(64, 136)
        c = {"kind": "adjoint", "n": n, "precision": prec, "steps": rng.randint(80, 160), "pml": 10, "tfsf": 16,
             "design": rng.randint(8, n // 2 - 20), "window": rng.randint(10, 60), "every": rng.choice([0, 30, 50])}
    else:
        c = {"kind": "ntff", "n": 2 * rng.randint(24, 40), "precision": prec, "steps": rng.randint(40, 80), "pml": 6,
             "tfsf": 12, "step_angle": rng.choice([5.0, 10.0, 30.0])}
    c.pop("name", None)
    return c


# ---------------------------------------------------------------------------------------
# inputs
# ---------------------------------------------------------------------------------------
def _size(case):
    if case["kind"] == "grid":
        return (case["x"], case["y"], case["z"])
    return (case["n"],) * 3


def _config(case):
    if case["kind"] == "grid":
        size = _size(case)
        c = Config(scheme=SCHEMES[case["scheme"]], precision=case["precision"], time_steps=case["steps"], size=list(size),
                   pml=[case["pml"]] * 3, dx=DX, wavelength=WAVELENGTH, courant=COURANT,
                   angle_deg=[case["teta"], case["phi"], case["psi"]], use_pml=case["pml"] > 0,
                   use_tfsf=case["tfsf"] > 0, use_metamaterials=case["drude"] > 0, layout=case["layout"])
        if c.use_tfsf:
            c.tfsf_left = [case["tfsf"]] * 3
            c.tfsf_right = [case.get("tfsf_right", case["tfsf"])] * 3
        if case["source"]:
            c.point_source = [c.components[0] if "Ez" not in c.components else "Ez"]
            c.point_source_pos = [n // 3 if n > 1 else 0 for n in size]
        return c
    n = case["n"]
    c = Config(scheme=SCHEME_DIM3, precision=case["precision"], time_steps=case["steps"], size=[n] * 3,
               pml=[case["pml"]] * 3, tfsf_left=[case["tfsf"]] * 3, tfsf_right=[case["tfsf"]] * 3, dx=DX,
               wavelength=WAVELENGTH, courant=COURANT, use_pml=True, use_tfsf=True,
               complex_fields=case["kind"] == "ntff")
    return c


def _blocks(shape, seed, lo, hi, block=8):
    """Piecewise constant over cubes of 8 cells, i.i.d. U[lo, hi] per cube (FP32 values)."""
    v = np.random.default_rng(seed).uniform(lo, hi, [-(-s // block) for s in shape]).astype(np.float32)
    t = torch.from_numpy(v)
    for ax, s in enumerate(shape):
        t = t.index_select(ax, torch.arange(s) // block)
    return np.ascontiguousarray(t.numpy())


def _materials(case, cfg, seed):
    """Material arrays of the grid, FP32 values, from the seed alone."""
    shape = tuple(cfg.shape)
    rng = np.random.default_rng([seed, 1])
    if case["kind"] == "ntff" or case.get("eps") == "sphere":
        n = shape[0]
        x = np.arange(n) + 0.5 - n / 2
        r2 = x[:, None, None] ** 2 + x[None, :, None] ** 2 + x[None, None, :] ** 2
        return {"eps": np.where(r2 < (n / 5) ** 2, rng.uniform(2.0, 6.0), 1.0).astype(np.float32)}
    out = {}
    eps = case.get("eps")
    if eps == "blocks":
        out["eps"] = _blocks(shape, [seed, 2], 1.0, 12.0)
    elif eps == "half":
        v = np.ones(shape, dtype=np.float32)
        v[shape[0] // 2:] = rng.uniform(2.0, 6.0)
        out["eps"] = v
    if case.get("mu"):
        out["mu"] = _blocks(shape, [seed, 3], 1.0, 3.0)
    if case.get("drude"):
        w0 = 2 * math.pi * 299792458.0 / cfg.wavelength
        d = case["drude"]
        box = tuple(slice(n // 2 - d // 2, n // 2 - d // 2 + d) for n in shape)
        om, ga = np.zeros(shape, dtype=np.float32), np.zeros(shape, dtype=np.float32)
        om[box] = rng.uniform(1.2, 1.8) * w0
        ga[box] = rng.uniform(0.005, 0.02) * w0
        out.update(omegape=om, omegapm=om, gammae=ga, gammam=ga)
    return out


def _batch(case, seed):
    """(configurations, eps maps, source times) of a sweep; its shapes belong to the case."""
    shapes, rng = np.random.default_rng(case["shape"]), np.random.default_rng(seed)
    cfgs, eps = [], []
    for _ in range(case["sims"]):
        nx, ny = (int(round(math.exp(shapes.uniform(math.log(case["lo"]), math.log(case["hi"] + 1))))) for _ in range(2))
        px, py = int(shapes.integers(14, nx - 14)), int(shapes.integers(14, ny - 14))
        cfgs.append(Config(scheme=SCHEME_TMZ, precision=4, time_steps=case["steps"], size=[nx, ny, 1],
                           pml=[case["pml"], case["pml"], 0], use_pml=case["pml"] > 0, point_source=["Ez"],
                           point_source_pos=[px, py, 0], dx=DX, wavelength=WAVELENGTH, courant=COURANT))
        x, y = torch.arange(nx, dtype=torch.float64), torch.arange(ny, dtype=torch.float64)
        e = torch.ones(nx, ny, dtype=torch.float64)
        for _ in range(int(rng.integers(4, 10))):
            cx, cy, r = rng.uniform(0, nx), rng.uniform(0, ny), rng.uniform(8, 40)
            e += 8 * torch.outer(torch.exp(-(x - cx) ** 2 / (2 * r * r)), torch.exp(-(y - cy) ** 2 / (2 * r * r)))
        eps.append(e.clamp_(1, 9).float().numpy())
    return cfgs, eps


def _design(case, seed):
    d = case["design"]
    return np.random.default_rng([seed, 4]).uniform(1.0, 4.0, size=(d, d, d)).astype(np.float32).astype(np.float64)


def _design_box(case):
    lo = case["n"] // 2 - case["design"] // 2
    return lo, lo + case["design"]


def _monitor(case):
    n = case["n"]
    return n // 2, (n // 4, n // 4), (n - n // 4, n - n // 4)


def _ntff_box(case):
    return [case["pml"] + 2] * 3, [case["n"] - case["pml"] - 1] * 3


def _phis(case):
    return np.arange(0.0, 360.0 + 1e-9, case["step_angle"]) * math.pi / 180.0


def prepare(case, seed):
    if case["kind"] == "batch":
        cfgs, eps = _batch(case, seed)
        b = Batch(cfgs)
        for s, e in enumerate(eps):
            b.set_material(s, "eps", e)
            b.set_point_source_gaussian(s, 4 * PERIOD, PERIOD)
        b.prepare()
        return {"case": case, "batch": b}
    cfg = _config(case)
    eng = Engine(cfg)
    for name, v in _materials(case, cfg, seed).items():
        eng.set_material(name, v)
    eng.prepare()
    state = {"case": case, "eng": eng, "comps": list(cfg.components)}
    if case["kind"] == "adjoint":
        lo, hi = _design_box(case)
        z, mlo, mhi = _monitor(case)
        eng.adjoint_setup((lo,) * 3, (hi,) * 3, z, mlo, mhi, case["window"], checkpoint_every=case["every"])
        state["design"] = _design(case, seed)
    return state


def run(state):
    case = state["case"]
    if case["kind"] == "batch":
        b = state["batch"]
        b.step(case["steps"])
        return {"%02d" % s: [b.field(s, c) for c in ("Ez", "Hx", "Hy")] for s in range(case["sims"])}
    eng = state["eng"]
    if case["kind"] == "adjoint":
        return {"J": eng.forward(state["design"]), "grad": eng.backward(1.0)}
    if case["kind"] == "ntff":
        left, right = _ntff_box(case)
        eng.step(case["steps"] - 1)
        eng.ntff_snapshot()
        eng.step(1)
        im = eng.imag()
        return {"far": eng.ntff(math.pi / 2, _phis(case), left, right),
                "re": {c: eng.field_raw(c) for c in state["comps"]}, "im": {c: im.field_raw(c) for c in state["comps"]}}
    eng.step(case["steps"])
    return {c: eng.field_raw(c) for c in state["comps"]}


def work(case):
    """A time step reads and writes every field word of a cell (and its D / B word in the PML, its
    Drude history in the box) and reads its eps; the fields then leave the card once."""
    def cells_pml(size, pml):
        n, inner = 1, 1
        for s in size:
            n *= s
            inner *= s if s == 1 else max(0, s - 2 * pml)
        return n, n - inner

    if case["kind"] == "batch":
        total = [0.0, 0.0]
        shapes = np.random.default_rng(case["shape"])
        for _ in range(case["sims"]):
            nx, ny = (int(round(math.exp(shapes.uniform(math.log(case["lo"]), math.log(case["hi"] + 1))))) for _ in range(2))
            shapes.integers(14, nx - 14), shapes.integers(14, ny - 14)
            n, p = cells_pml((nx, ny), case["pml"])
            total[0] += 4.0 * ((7 * n + 6 * p) * case["steps"] + 3 * n)
            total[1] += 25.0 * n * case["steps"]
        return {"bytes": total[0], "flops": total[1]}
    size, w = _size(case), case["precision"]
    n, p = cells_pml(size, case["pml"])
    comps = 6 if min(size) > 1 else (2 if sorted(size)[1] == 1 else 3)
    steps, fields = case["steps"], comps * n * w
    per_step = w * (2 * comps * (n + p) + n + (n if case.get("mu") else 0) + 36 * case.get("drude", 0) ** 3)
    flops = (comps * 8.0 * n) * steps
    if case["kind"] == "ntff":
        steps, fields, flops = 2 * steps, 2 * fields, 2 * flops
    if case["kind"] == "adjoint":   # forward and reverse sweep
        fields, per_step, flops = 8.0 * case["design"] ** 3, 2 * per_step + 6 * w * case["design"] ** 3, 2 * flops
    return {"bytes": float(per_step * steps + fields), "flops": float(flops)}


# ---------------------------------------------------------------------------------------
# the same in 64 bits, plain torch
# ---------------------------------------------------------------------------------------
C0 = 299792458.0
MU0 = 4 * math.pi * 1e-7
EPS0 = 1 / (MU0 * C0 * C0)
E, H = (0, 1, 2), (3, 4, 5)
NAMES = ["Ex", "Ey", "Ez", "Hx", "Hy", "Hz"]


def _wave_number(a1, a2):
    """Numerical wave number of the Yee grid along the angles (times the wavelength)."""
    nd = DX / WAVELENGTH
    a, b, c = (nd / 2 * v for v in (math.sin(a1) * math.cos(a2), math.sin(a1) * math.sin(a2), math.cos(a1)))
    rhs = (math.sin(math.pi * COURANT * nd) / COURANT) ** 2
    k = 2 * math.pi
    for _ in range(60):
        f = math.sin(a * k) ** 2 + math.sin(b * k) ** 2 + math.sin(c * k) ** 2 - rhs
        k -= f / (a * math.sin(2 * a * k) + b * math.sin(2 * b * k) + c * math.sin(2 * c * k))
    return k


def _newton_wave_number(a1, a2):
    """The engine's (and the reference's) wave number: closed forms on axes and diagonals, else
    Newton's iteration stopped where two iterates differ by less than sqrt (1e-7)."""
    axial = [0, math.pi / 2, math.pi, 3 * math.pi / 2]
    diagonal = [math.pi / 4, 3 * math.pi / 4, 5 * math.pi / 4, 7 * math.pi / 4]
    if (a1 in axial and a2 in axial + diagonal) or (a1 in diagonal and a2 in axial):
        return _wave_number(a1, a2)
    nd = DX / WAVELENGTH
    a, b, c = (nd * v / 2 for v in (math.sin(a1) * math.cos(a2), math.sin(a1) * math.sin(a2), math.cos(a1)))
    rhs = (math.sin(math.pi * COURANT * nd) / COURANT) ** 2
    k, last = 2 * math.pi, 1e9
    while (last - k) ** 2 >= 1e-7:
        last = k
        f = math.sin(a * k) ** 2 + math.sin(b * k) ** 2 + math.sin(c * k) ** 2 - rhs
        k -= f / (a * math.sin(2 * a * k) + b * math.sin(2 * b * k) + c * math.sin(2 * c * k))
    return k


class Restated:
    """One real-valued simulation on whole FP64 torch arrays (part: 0 real run, 1 / 2 the real /
    imaginary part of a complex one)."""

    def __init__(self, cfg, mats, part=0, gauss=None):
        self.cfg, self.part, self.gauss = cfg, part, gauss
        self.dev = "cuda" if torch.cuda.is_available() else "cpu"
        self.act = list(cfg.active_axes)
        self.n = [int(cfg.size[a]) if a in self.act else 1 for a in range(3)]
        self.comps = [NAMES.index(c) for c in cfg.components]
        self.dt, self.freq = DX * COURANT / C0, C0 / WAVELENGTH
        self.lay = cfg.layout
        one = lambda v: torch.as_tensor(np.asarray(v, np.float64).reshape(self.n), device=self.dev)  # noqa: E731
        self.mats = {k: one(v) for k, v in mats.items()}
        zero = lambda: torch.zeros(self.n, dtype=torch.float64, device=self.dev)  # noqa: E731
        self.f = {c: zero() for c in self.comps}
        self.d = {c: zero() for c in self.comps} if cfg.use_pml else {}
        self.t = 0
        self._pml()
        self._incident()
        self.set_media(self.mats.get("eps"), self.mats.get("mu"))
        if cfg.use_metamaterials:
            self._drude()

    def hlike(self, c):
        return (c >= 3) != (self.lay == 1)

    def off2(self, c, ax):
        """Twice the coordinate offset of component c along ax."""
        return (1 if ax == c % 3 else 2) if self.hlike(c) else (2 if ax == c % 3 else 1)

    def along(self, v, ax):
        shape = [1, 1, 1]
        shape[ax] = -1
        return torch.as_tensor(np.asarray(v), device=self.dev).reshape(shape)

    def next(self, a, ax):
        return torch.roll(a, -1, ax)

    def mean(self, m, c):
        """Average of a cell-centred grid at the points of component c."""
        if not isinstance(m, torch.Tensor):
            return m
        axes = [ax for ax in self.act if (ax != c % 3) == self.hlike(c)]
        for ax in axes:
            m = (m + self.next(m, ax)) / 2
        return m

    def set_media(self, eps, mu):
        self.mod = {c: (EPS0 * self.mean(eps if eps is not None else 1.0, c) if c < 3
                        else MU0 * self.mean(mu if mu is not None else 1.0, c)) for c in self.comps}
        self.co = {}
        for c in self.comps:
            inner = torch.ones([1, 1, 1], dtype=torch.float64, device=self.dev)
            for ax in self.act:
                v = np.ones(self.n[ax])
                v[0] = v[-1] = 0.0
                inner = inner * self.along(v, ax)
            if self.cfg.use_pml:
                cac, cbc, p4, m4, ca5, dd5 = self.tab[c]
                # d' = cac d + cbc curl; f' = ca5 f + (p4 d' - m4 d) / mod / dd5, interior only
                self.co[c] = (1 + inner * (cac - 1), inner * cbc, p4 / dd5 * inner / self.mod[c],
                              m4 / dd5 * inner / self.mod[c], 1 + inner * (ca5 - 1))
            else:
                self.co[c] = (inner * (self.dt / DX) / self.mod[c],)

    def _pml(self):
        self.tab = {}
        if not self.cfg.use_pml:
            return
        prof = {}
        for ax in self.act:
            n, P = self.n[ax], float(self.cfg.pml[ax])
            smax = -math.log(1e-16) * 7.0 / (2 * math.sqrt(MU0 / EPS0) * P * DX)
            factor = smax / (DX * (P * DX) ** 6 * 7)
            first = ax == self.act[0]
            v = np.zeros(n + 1)
            for p in range(n):
                pos, edge = p + 0.5, n + (0.0 if first else 0.5)
                dist = P - pos if pos < P else (pos - (edge - P) if pos >= edge - P else None)
                if dist is not None:
                    dist = dist if first else float(int(dist))
                    v[p] = factor * (((dist + 1) * DX) ** 7 - (dist * DX) ** 7)
            prof[ax] = v

        def sigma(c, ax):
            if ax not in self.act:
                return torch.zeros([1, 1, 1], dtype=torch.float64, device=self.dev)
            v = prof[ax]
            return self.along((v[:-1] + v[1:]) / 2 if self.off2(c, ax) == 2 else v[:-1], ax)

        for c in self.comps:
            a = c % 3
            cu, s4, s5 = [(1, 0, 2), (2, 1, 0), (0, 2, 1)][a]
            sc, sp, sq = (sigma(c, ax) * self.dt for ax in (cu, s4, s5))
            e2 = 2 * EPS0
            self.tab[c] = ((e2 - sc) / (e2 + sc), e2 * (self.dt / DX) / (e2 + sc), e2 + sp, e2 - sp,
                           (e2 - sq) / (e2 + sq), e2 + sq)

    def _incident(self):
        self.tf = []
        if not self.cfg.use_tfsf:
            return
        a1, a2, a3 = (v * math.pi / 180.0 for v in self.cfg.angle_deg)
        rel = _newton_wave_number(a1, a2) / _newton_wave_number(math.pi / 2, 0.0)
        self.modE, self.modH = (self.dt / (rel * m * DX) for m in (EPS0, MU0))
        s1, c1, s2, c2, s3, c3 = (f(v) for v in (a1, a2, a3) for f in (math.sin, math.cos))
        dirs = [s1 * c2, s1 * s2, c1]
        if len(self.act) == 3:
            proj = [c3 * s2 - s3 * c1 * c2, -c3 * c2 - s3 * c1 * s2, s3 * s1,
                    s3 * s2 + c3 * c1 * c2, -s3 * c2 + c3 * c1 * s2, -c3 * s1]
        elif len(self.act) == 1:
            dirs = [1.0 if a in self.act else 0.0 for a in range(3)]
            proj = {"ExHy": [-1, 0, 0, 0, -1, 0], "EyHz": [0, -1, 0, 0, 0, -1], "EzHx": [0, 0, 1, 1, 0, 0]}[
                "".join(self.cfg.components)]
        elif 2 not in self.act:   # TMz, TEz
            dirs = [c2, s2, 0.0]
            proj = [s2, -c2, 1, s2, -c2, -1]
        elif 0 not in self.act:   # TEx
            dirs = [0.0, s1, c1]
            proj = [0, -c1, s1, 1, 0, 0]
        else:                     # TMy
            dirs = [s1, 0.0, c1]
            proj = [0, -1, 0, c1, 0, -s1]
        L = [int(v) for v in self.cfg.tfsf_left]
        R = [int(self.cfg.size[a]) - int(self.cfg.tfsf_right[a]) for a in range(3)]
        self.len = 500 * self.n[self.act[0]]
        for c in self.comps:
            own, h = c % 3, self.hlike(c)
            for b in self.act:
                if b == own:
                    continue
                opp = (3 - own - b) + (0 if c >= 3 else 3)   # the field differenced along b
                if opp not in self.comps:
                    continue
                # curl = + d_b (opp) or - d_b (opp)
                sign = 1.0 if (own, b) in ((0, 1), (1, 2), (2, 0)) else -1.0
                sign = sign if c < 3 else -sign
                for low in (True, False):
                    p = L[b] - 1 if low else (R[b] - 1 if h else R[b])
                    if not 1 <= p < self.n[b] - 1:
                        continue
                    idx = []
                    for ax in range(3):
                        if ax == b:
                            idx.append(np.array([p]))
                        elif ax not in self.act:
                            idx.append(np.array([0]))
                        else:
                            q = np.arange(1, self.n[ax] - 1)
                            q2 = 2 * q + self.off2(c, ax)
                            wide = (ax == own) != h
                            lo, hi = (2 * L[ax], 2 * R[ax]) if wide else (2 * L[ax] + 1, 2 * R[ax] - 1)
                            idx.append(q[(q2 >= lo) & (q2 <= hi)])
                    if min(len(v) for v in idx) == 0:
                        continue
                    # operands at slots (lo, hi): differences backward at E-like points, forward at H-like
                    hi_slot = low if not h else not low
                    shift = (0 if hi_slot else -1) if not h else (1 if hi_slot else 0)
                    amount = (1.0 if hi_slot else -1.0) * sign * (1.0 if h else -1.0)
                    d = 0.0
                    for ax in range(3):
                        if ax in self.act:
                            x = idx[ax] + (shift if ax == b else 0)
                            zinc = L[ax] - 2.5 * dirs[ax]
                            d = d + self.along((0.5 * (2 * x + self.off2(opp, ax)) - zinc) * dirs[ax], ax)
                    d = d - (0.5 if c < 3 else 0.0)
                    i1 = d.long()
                    w2 = d - i1
                    box = tuple(slice(int(v[0]), int(v[-1]) + 1) for v in idx)
                    self.tf.append((c, box, i1, amount * proj[opp] * (1 - w2), amount * proj[opp] * w2))
        self.einc = torch.zeros(min(self.len, 4096 + 4 * sum(self.n)), dtype=torch.float64, device=self.dev)
        self.hinc = torch.zeros_like(self.einc)

    def _drude(self):
        om, ga = self.mats["omegape"], self.mats["gammae"]
        nz = torch.nonzero(om)
        self.box = tuple(slice(int(nz[:, a].min()) - 1, int(nz[:, a].max()) + 2) for a in range(3))
        self.ade = {}
        for c in self.comps:
            M = EPS0 if c < 3 else MU0
            m = self.mod[c] / M
            m = m[self.box] if isinstance(m, torch.Tensor) else m
            w = (self.dt * self.mean(om, c)[self.box]) ** 2
            g = self.dt * self.mean(ga, c)[self.box]
            a = 4 * M * m + 2 * M * m * g + M * w
            z = torch.zeros_like(w)
            # increments of D and D1: dd1' = b0 dd' - b2 dd - c D1 + a2 dd1
            self.ade[c] = ((4 + 2 * g) / a, (4 - 2 * g) / a, 4 * M * w / a, (4 * M * m - 2 * M * m * g + M * w) / a,
                           {"dd": z, "d1": z, "dd1": z})

    def curl(self, c):
        own = c % 3
        b1, b2 = (own + 1) % 3, (own + 2) % 3   # curl_own = d_b1 F_b2 - d_b2 F_b1, H negated
        opp = 0 if c >= 3 else 3
        total = None
        for b, o, s in ((b1, b2, 1.0), (b2, b1, -1.0)):
            o += opp
            if b not in self.act or o not in self.comps:
                continue
            s = s if c < 3 else -s
            a = self.f[o]
            d = self.next(a, b) - a if self.hlike(c) else a - torch.roll(a, 1, b)
            total = s * d if total is None else total + s * d
        return total

    def half(self, comps, inc):
        new, newd = {}, {}
        for c in comps:
            cu = self.curl(c)
            for k, box, i1, w1, w2 in self.tf:
                if k == c:
                    cu[box] = cu[box] + inc[i1] * w1 + inc[i1 + 1] * w2
            if not self.cfg.use_pml:
                new[c] = self.f[c] + self.co[c][0] * cu
                continue
            cac, cbc, kp, km, ca5 = self.co[c]
            newd[c] = cac * self.d[c] + cbc * cu
            new[c] = ca5 * self.f[c] + kp * newd[c] - km * self.d[c]
            if self.cfg.use_metamaterials:
                b0, b2, cc, a2, s = self.ade[c]
                dd = newd[c][self.box] - self.d[c][self.box]
                dd1 = b0 * dd - b2 * s["dd"] - cc * s["d1"] + a2 * s["dd1"]
                s["d1"], s["dd1"], s["dd"] = s["d1"] + dd1, dd1, dd
                new[c][self.box] = self.f[c][self.box] + dd1
        for c in comps:
            self.f[c] = new[c]
            if newd:
                self.d[c] = newd[c]

    def sources(self, comps, ts):
        arg = self.dt * ts * 2 * math.pi * self.freq
        v = math.cos(arg) if self.part == 2 else math.sin(arg)
        if self.gauss:
            v *= math.exp(-((ts - self.gauss[0]) / self.gauss[1]) ** 2)
        for name in self.cfg.point_source:
            c = NAMES.index(name)
            if c in comps:
                self.f[c][tuple(p if a in self.act else 0 for a, p in enumerate(self.cfg.point_source_pos))] = v

    def step(self):
        t, es, hs = self.t, [c for c in self.comps if c < 3], [c for c in self.comps if c >= 3]
        hprev = None
        if self.cfg.use_tfsf:
            arg = self.dt * t * 2 * math.pi * self.freq
            hprev = self.hinc
            self.einc = torch.cat([torch.full((1,), math.cos(arg) if self.part == 2 else math.sin(arg),
                                              dtype=torch.float64, device=self.dev),
                                   self.einc[1:] + (hprev[:-1] - hprev[1:]) * self.modE])
            self.hinc = torch.cat([hprev[:-1] + (self.einc[:-1] - self.einc[1:]) * self.modH, hprev[-1:]])
        if t > 0:
            self.half(es, hprev)
        self.sources(es, t + 0.5)
        if t > 0:
            self.half(hs, self.einc if self.cfg.use_tfsf else None)
        self.sources(hs, t + 1.0)
        self.t += 1

    def field(self, c):
        return self.f[c].reshape(self.cfg.shape).cpu().numpy()


def _far(cfg, re, im, old, case):
    """Pointing_scat / Pointing_inc of the complex fields `re` + i `im` (dicts of FP64 arrays by
    component) with `old` = H one step before, at elevation 90 degrees."""
    left, right = _ntff_box(case)
    phis = torch.as_tensor(_phis(case), device=re[0].device)
    st, ct = math.sin(math.pi / 2), math.cos(math.pi / 2)
    k = 2 * math.pi / WAVELENGTH
    f = {c: torch.complex(re[c], im[c]) for c in range(6)}
    for c in H:
        f[c] = (f[c] + old[c]) / 2

    def at(c, pos):   # values at coordinates pos (a list of three 1D arrays)
        ix = []
        for ax in range(3):
            low = (1.0 if ax == c % 3 else 0.5) if c < 3 else (0.5 if ax == c % 3 else 1.0)
            ix.append(torch.as_tensor((pos[ax] - low).astype(np.int64), device=re[0].device))
        return f[c][ix[0][:, None, None], ix[1][None, :, None], ix[2][None, None, :]]

    sums = {(kind, w): torch.zeros(len(phis), dtype=torch.complex128, device=re[0].device) for kind in (0, 1) for w in "tf"}
    cp, sp = torch.cos(phis), torch.sin(phis)
    for ax in range(3):
        u, v = [a for a in range(3) if a != ax]
        for side in (0, 1):
            base = [np.arange(left[a], right[a]) + 0.5 for a in range(3)]
            base[ax] = np.array([float(right[ax] if side else left[ax])])
            sign = 1.0 if side else -1.0
            rel = [torch.as_tensor(base[a] - case["n"] // 2, device=re[0].device).reshape([-1 if b == a else 1 for b in range(3)])
                   for a in range(3)]
            for kind in (0, 1):
                def mid(c, d):
                    total = 0
                    for s in (-0.5, 0.5):
                        pos = list(base)
                        pos[d] = base[d] + s
                        if kind == 0:
                            total = total + at(c, pos)
                        else:   # across the face
                            for q in (-0.5, 0.5):
                                pp = list(pos)
                                pp[ax] = pos[ax] + q
                                total = total + at(c, pp) / 2
                    return total / 2
                c1 = (4 if ax == 2 else 5) if kind == 0 else (1 if ax == 0 else 0)
                c2 = (4 if ax == 0 else 3) if kind == 0 else (1 if ax == 2 else 2)
                a, b = mid(c1, u), mid(c2, v)
                ts = (-1.0 if ax == 0 else 1.0) if kind == 0 else (-1.0 if ax == 1 else 1.0)
                fs = (1.0 if ax == 2 else -1.0) if kind == 0 else (-1.0 if ax == 2 else 1.0)
                p, q = (a, b) if kind == 0 else (b, a)
                for i in range(len(phis)):
                    C, S = cp[i], sp[i]
                    phase = torch.exp(1j * k * DX * (rel[0] * st * C + rel[1] * st * S + rel[2] * ct))
                    if ax == 0:
                        te, fi = p * ct * S + q * st, p * C
                    elif ax == 1:
                        te, fi = p * ct * C + q * st, p * S
                    elif kind == 0:
                        te, fi = -a * ct * C + b * ct * S, a * S + b * C
                    else:
                        te, fi = b * ct * C - a * ct * S, b * S + a * C
                    sums[(kind, "t")][i] += (te * phase).sum() * DX * DX * ts * sign
                    sums[(kind, "f")][i] += (fi * phase).sum() * DX * DX * fs * sign
    n0 = math.sqrt(MU0 / EPS0)
    scat = k * k / (8 * math.pi * n0) * ((sums[(1, "f")] + sums[(0, "t")] * n0).abs() ** 2
                                         + (sums[(1, "t")] - sums[(0, "f")] * n0).abs() ** 2)
    return (scat / (math.sqrt(EPS0 / MU0) / 2)).cpu().numpy()


def exact(case, seed):
    with torch.no_grad():
        if case["kind"] == "batch":
            cfgs, eps = _batch(case, seed)
            if sum(c.size[0] * c.size[1] for c in cfgs) * case["steps"] > 6e9 or case["sims"] * case["steps"] > 17000:
                return None   # over 20 seconds
            out = {}
            for s, (c, e) in enumerate(zip(cfgs, eps)):
                r = Restated(c, {"eps": e}, gauss=(4 * PERIOD, PERIOD))
                for _ in range(case["steps"]):
                    r.step()
                out["%02d" % s] = [r.field(k) for k in (2, 3, 4)]
            return out
        cfg = _config(case)
        if case["kind"] == "grid":
            r = Restated(cfg, _materials(case, cfg, seed))
            for _ in range(case["steps"]):
                r.step()
            return {NAMES[c]: r.field(c) for c in r.comps}
        if case["kind"] == "ntff":
            parts = [Restated(cfg, _materials(case, cfg, seed), part=p) for p in (1, 2)]
            for t in range(case["steps"]):
                if t == case["steps"] - 1:
                    old = {c: torch.complex(parts[0].f[c], parts[1].f[c]) for c in H}
                for r in parts:
                    r.step()
            re, im = parts
            return {"far": _far(cfg, re.f, im.f, old, case), "re": {NAMES[c]: re.field(c) for c in range(6)},
                    "im": {NAMES[c]: im.field(c) for c in range(6)}}
    # the adjoint: J by the restated run, dJ/deps by autograd, a step at a time
    n, (lo, hi) = case["n"], _design_box(case)
    r = Restated(cfg, {})
    design = torch.tensor(_design(case, seed), device=r.dev, requires_grad=True)
    eps = torch.ones([n] * 3, dtype=torch.float64, device=r.dev)
    eps[lo:hi, lo:hi, lo:hi] = design
    r.set_media(eps, None)
    z, mlo, mhi = _monitor(case)
    J = torch.zeros((), dtype=torch.float64, device=r.dev)
    for t in range(case["steps"]):
        r.step()
        if t >= case["steps"] - case["window"]:
            J = J + (r.f[2][mlo[0]:mhi[0], mlo[1]:mhi[1], z] ** 2).sum()
    J.backward()
    return {"J": float(J.detach()), "grad": design.grad.cpu().numpy()}
