"""How the work of a time step is cut into launches must not show in its results (needs the GPU).

One launch updates every box around the fused kernel (PML slabs, TF/SF faces, source cells): the
fields are bit-identical to the half-step kernels over the whole grid (YEE_KERNEL=split), with the
hard source on a face plane, an edge of two faces, in a slab, inside the fused box and on the grid
border (never updated: the source alone writes it), and with boxes of one cell along an axis.
"""
import numpy as np
import pytest

from fdtd3d_amd.config import parse_args
from fdtd3d_amd.engine import Batch, Engine

pytestmark = pytest.mark.gpu


def _run(args, precision, monkeypatch, kernel, eps, steps):
    monkeypatch.setenv("YEE_KERNEL", kernel)
    cfg = parse_args(args.split(), precision=precision)
    eng = Engine(cfg)
    eng.set_material("eps", eps)
    eng.prepare()
    eng.step(steps)
    names = list(cfg.components) + (["D" + c[1] if c[0] == "E" else "B" + c[1] for c in cfg.components] if cfg.use_pml else [])
    out = {n: eng.field_raw(n) for n in names}
    eng.close()
    return out


BOXES = "--3d --size x:19,y:21,z:70 --use-pml --pml-size x:3,y:1,z:4 --use-tfsf --tfsf-size-left x:6,y:5,z:7 " \
        "--tfsf-size-right x:6,y:5,z:7 --angle-teta 30 --angle-phi 45 --angle-psi 90 --point-source-ez --point-source-hx "


@pytest.mark.parametrize("precision", [4, 8])
@pytest.mark.parametrize("pos", ["x:5,y:9,z:30", "x:5,y:4,z:30", "x:9,y:9,z:66", "x:9,y:10,z:31", "x:0,y:9,z:30",
                                 "x:9,y:20,z:69"])
def test_boxes_in_one_launch(pos, precision, engine_lib, monkeypatch):
    args = BOXES + f"--point-source {pos} --time-steps 20"
    print(f"[gpu] boxes, source {pos}, precision {precision}", flush=True)
    eps = np.random.default_rng(3).uniform(1.0, 4.0, size=(19, 21, 70))
    ref = _run(args, precision, monkeypatch, "split", eps, 20)
    got = _run(args, precision, monkeypatch, "fused", eps, 20)
    for n, v in ref.items():
        assert np.array_equal(got[n], v), n
    assert np.abs(ref["Ez"]).max() > 0


@pytest.mark.parametrize("precision", [4, 8])
@pytest.mark.parametrize("args", [
    "--1d-exhy --size z:40 --use-pml --pml-size z:5 --use-tfsf --tfsf-size-left z:12 --tfsf-size-right z:0 --angle-teta 0 "
    "--angle-phi 0",
    "--2d-tmz --size x:40,y:33 --use-tfsf --tfsf-size-left x:8,y:7 --tfsf-size-right x:8,y:7 --angle-teta 90 --angle-phi 30",
    "--3d --size x:14,y:13,z:15 --use-tfsf --tfsf-size-left x:4,y:4,z:4 --tfsf-size-right x:4,y:4,z:4 --angle-teta 140 "
    "--angle-phi 200 --angle-psi 10",
])
def test_incident_steps_in_groups(args, precision, engine_lib):
    """The incident grid advances up to 32 steps a launch: calls of 1, 31, 32, 33 and 70 steps give
    the fields and the exported incident grids of single steps (beyond one workgroup's 448 cells)."""
    cfg = parse_args((args + " --time-steps 1200").split(), precision=precision)
    out = []
    for calls in ([1] * 1167, [1, 31, 32, 33, 70, 1000]):
        eng = Engine(cfg)
        eng.prepare()
        for n in calls:
            eng.step(n)
        einc, hinc = eng.incident(500 * cfg.size[cfg.active_axes[0]])
        assert np.count_nonzero(einc) > 448
        out.append({"einc": einc, "hinc": hinc, **{c: eng.field_raw(c) for c in cfg.components}})
        eng.close()
    for n, v in out[0].items():
        assert np.array_equal(out[1][n], v), n


@pytest.mark.parametrize("precision", [4, 8])
@pytest.mark.parametrize("size", [(90, 91, 92), (100, 128, 131), (181, 257, 199)])
def test_large_fields_read_back_in_chunks(size, precision, engine_lib):
    """Fields on both sides of the least size of the chunked read, with a ragged last chunk: every
    value of yee_get_field_raw and of yee_get_field (widened from FP32) is the device's."""
    cfg = parse_args(f"--3d --size x:{size[0]},y:{size[1]},z:{size[2]} --point-source x:40,y:41,z:42 --point-source-ez "
                     "--time-steps 60".split(), precision=precision)
    eng = Engine(cfg)
    eng.prepare()
    eng.step(60)
    raw, wide = eng.field_raw("Ez"), eng.field("Ez")
    assert raw.shape == size and wide.dtype == np.float64
    assert np.array_equal(raw.astype(np.float64), wide)
    # the vacuum pattern is mirror symmetric about the source in x: every plane is in its place
    assert np.count_nonzero(raw) > 1000
    assert np.allclose(raw[40 + 5, 30:50, 30:50], raw[40 - 5, 30:50, 30:50], rtol=1e-4, atol=1e-9)
    small = np.array([eng.field_raw("Ez").sum() for _ in range(3)])
    assert np.all(small == small[0])
    eng.close()


# 2D schemes by the option, their two axes; sizes around the owned part of a tile (48 x 48 cells in
# FP32, 32 x 48 in FP64 with the full margin of 8) and the smallest grids
PLANES = {"tmz": "xy", "tez": "xy", "tex": "yz", "tmx": "yz", "tey": "xz", "tmy": "xz"}


def _plane_args(scheme, na, nb, pml, tfsf, source):
    a, b = PLANES[scheme]
    s = f"--2d-{scheme} --size {a}:{na},{b}:{nb} --angle-teta {90 if scheme in ('tmz', 'tez') else 40} "
    s += {"tmz": "--angle-phi 30 ", "tez": "--angle-phi 30 ", "tex": "--angle-phi 90 ", "tmx": "--angle-phi 90 ",
          "tey": "--angle-phi 0 ", "tmy": "--angle-phi 0 "}[scheme]
    s += "--angle-psi 0 " if scheme in ("tez", "tex", "tmy") else "--angle-psi 90 "
    if pml:
        s += f"--use-pml --pml-size {a}:{pml},{b}:{pml + 1} "
    if tfsf:
        s += f"--use-tfsf --tfsf-size-left {a}:{tfsf},{b}:{tfsf + 2} --tfsf-size-right {a}:{tfsf + 1},{b}:{tfsf} "
    if source:
        s += f"--point-source {a}:{na // 2},{b}:{nb // 3} --point-source-{source} "
    return s + "--time-steps 60"


@pytest.mark.parametrize("precision", [4, 8])
@pytest.mark.parametrize("scheme,na,nb,pml,tfsf,source", [
    ("tmz", 98, 99, 6, 12, ""), ("tmz", 50, 50, 0, 0, "ez"), ("tmz", 34, 147, 5, 0, "hx"), ("tmz", 3, 60, 0, 0, "ez"),
    ("tez", 67, 98, 4, 9, "hz"), ("tez", 131, 49, 0, 11, "ex"), ("tex", 51, 97, 5, 13, "ey"), ("tmx", 66, 51, 6, 0, "hy"),
    ("tey", 35, 100, 3, 10, "ez"), ("tmy", 99, 66, 7, 13, "hz"), ("tmy", 52, 3, 0, 0, "ey"),
])
def test_plane_steps_in_one_launch(scheme, na, nb, pml, tfsf, source, precision, engine_lib, monkeypatch):
    """Up to 8 steps a launch on register tiles: the fields and D / B of the half-step kernels, bit
    for bit, however the steps are split into calls, with eps and mu grids."""
    cfg = parse_args(_plane_args(scheme, na, nb, pml, tfsf, source).split(), precision=precision)
    rng = np.random.default_rng(11)
    eps, mu = rng.uniform(1.0, 5.0, size=cfg.shape), rng.uniform(1.0, 2.0, size=cfg.shape)
    print(f"[gpu] plane {scheme} {na}x{nb} pml {pml} tfsf {tfsf} source {source or '-'} precision {precision}", flush=True)
    out = []
    for kernel, calls in (("split", [60]), ("plane", [60]), ("plane", [1, 1, 2, 7, 9, 17, 23])):
        monkeypatch.setenv("YEE_KERNEL", kernel)
        eng = Engine(cfg)
        eng.set_material("eps", eps)
        eng.set_material("mu", mu)
        eng.prepare()
        for n in calls:
            eng.step(n)
        names = list(cfg.components) + ([("D" if c[0] == "E" else "B") + c[1] for c in cfg.components] if pml else [])
        out.append({n: eng.field_raw(n) for n in names})
        eng.close()
    for n, v in out[0].items():
        assert np.array_equal(out[1][n], v), n
        assert np.array_equal(out[2][n], v), n
    assert any(np.abs(v).max() > 0 for v in out[0].values())


LINES = {"exhy": ("z", 0, 0), "exhz": ("y", 90, 90), "eyhx": ("z", 0, 90), "eyhz": ("x", 90, 0), "ezhx": ("y", 90, 90),
         "ezhy": ("x", 90, 0)}


@pytest.mark.parametrize("precision", [4, 8])
@pytest.mark.parametrize("scheme,n,pml,tfsf,right,source", [
    ("exhy", 600, 50, 150, 0, ""), ("exhz", 193, 7, 20, 15, ""), ("eyhx", 194, 0, 0, 0, "ey"), ("eyhz", 195, 6, 0, 0, "hz"),
    ("ezhx", 386, 9, 190, 3, "ez"), ("ezhy", 3, 0, 0, 0, "ez"), ("ezhy", 421, 5, 30, 200, ""),
])
def test_line_steps_in_one_launch(scheme, n, pml, tfsf, right, source, precision, engine_lib, monkeypatch):
    """Up to 32 steps a launch of a 1D line, a wave to 192 cells: the half-step kernels' fields and
    D / B bit for bit, however the steps are split into calls."""
    ax, teta, phi = LINES[scheme]
    s = f"--1d-{scheme} --size {ax}:{n} --angle-teta {teta} --angle-phi {phi} --angle-psi 90 "
    if pml:
        s += f"--use-pml --pml-size {ax}:{pml} "
    if tfsf:
        s += f"--use-tfsf --tfsf-size-left {ax}:{tfsf} --tfsf-size-right {ax}:{right} "
    if source:
        s += f"--point-source {ax}:{max(1, n // 2 - 1)} --point-source-{source} "
    cfg = parse_args((s + "--time-steps 300").split(), precision=precision)
    rng = np.random.default_rng(13)
    eps, mu = rng.uniform(1.0, 5.0, size=cfg.shape), rng.uniform(1.0, 2.0, size=cfg.shape)
    out = []
    for kernel, calls in (("split", [300]), ("line", [300]), ("line", [1, 1, 30, 31, 32, 33, 64, 108])):
        monkeypatch.setenv("YEE_KERNEL", kernel)
        eng = Engine(cfg)
        eng.set_material("eps", eps)
        eng.set_material("mu", mu)
        eng.prepare()
        for k in calls:
            eng.step(k)
        names = list(cfg.components) + ([("D" if c[0] == "E" else "B") + c[1] for c in cfg.components] if pml else [])
        out.append({c: eng.field_raw(c) for c in names})
        eng.close()
    for c, v in out[0].items():
        assert np.array_equal(out[1][c], v), c
        assert np.array_equal(out[2][c], v), c
    assert any(np.abs(v).max() > 0 for v in out[0].values())


@pytest.mark.parametrize("precision", [4, 8])
@pytest.mark.parametrize("shapes,mu", [(((42, 50), (43, 98), (3, 64), (121, 57)), False), (((81, 49), (30, 33)), True)])
def test_batch_register_tiles(shapes, mu, precision, engine_lib, monkeypatch):
    """The batch's register tiles (40 x 48 owned cells in FP32, 40 x 56 in FP64) against single runs,
    bit for bit: edges of tiles, a mu grid, calls that are no multiple of a launch's steps."""
    sims = [f"--2d-tmz --size x:{a},y:{b} --point-source x:{a // 2},y:{b // 2} --point-source-ez --point-source-hy "
            + ("--use-pml --pml-size x:4,y:5 " if min(a, b) > 20 and k != 1 else "--pml-size x:0,y:0 ")
            + "--time-steps 80"
            for k, (a, b) in enumerate(shapes)]
    cfgs = [parse_args(s.split(), precision=precision) for s in sims]
    rng = np.random.default_rng(17)
    eps = [rng.uniform(1.0, 5.0, size=c.shape) for c in cfgs]
    mus = [rng.uniform(1.0, 2.0, size=c.shape) for c in cfgs]
    monkeypatch.setenv("YEE_BATCH_CAND", "12")
    b = Batch(cfgs)
    for s, c in enumerate(cfgs):
        b.set_material(s, "eps", eps[s])
        if mu:
            b.set_material(s, "mu", mus[s])
        b.set_point_source_gaussian(s, 30.0, 10.0)
    b.prepare()
    for n in (1, 3, 64, 5, 7):
        b.step(n)
    monkeypatch.setenv("YEE_KERNEL", "split")
    for s, c in enumerate(cfgs):
        e = Engine(c)
        e.set_material("eps", eps[s])
        if mu:
            e.set_material("mu", mus[s])
        e.set_point_source_gaussian(30.0, 10.0)
        e.prepare()
        e.step(80)
        for f in ("Ez", "Hx", "Hy") + (("Dz", "Bx", "By") if c.use_pml else ()):
            assert np.array_equal(b.field(s, f), e.field(f)), f"sim {s} {f}"
        e.close()
    b.close()


@pytest.mark.parametrize("precision,y", [(4, 128), (8, 64)])
@pytest.mark.parametrize("z", [1017, 1018])
def test_sweep_and_half_steps_meet(z, y, precision, engine_lib, monkeypatch):
    """Grids whose E and H fill at most 200 MB run by whole-grid half steps, larger ones by the
    fused sweep: the fields on both sides of that line are those of the sweep."""
    args = f"--3d --size x:64,y:{y},z:{z} --use-pml --pml-size x:5,y:5,z:5 --use-tfsf --tfsf-size-left x:9,y:9,z:9 " \
           "--tfsf-size-right x:9,y:9,z:9 --angle-teta 30 --angle-phi 45 --angle-psi 90 --time-steps 8"
    print(f"[gpu] line between sweep and half steps, z {z}, precision {precision}", flush=True)
    eps = np.kron(np.random.default_rng(4).uniform(1.0, 4.0, size=(8, y // 8, 128)), np.ones((8, 8, 8)))[:, :, :z]
    ref = _run(args, precision, monkeypatch, "fused", eps, 8)
    got = _run(args, precision, monkeypatch, "", eps, 8)
    for n, v in ref.items():
        assert np.array_equal(got[n], v), n
    assert np.abs(ref["Ez"]).max() > 0


@pytest.mark.parametrize("precision", [4, 8])
@pytest.mark.parametrize("dims", [(1, 1, 1), (16, 16, 1), (1, 1, 17), (8, 4, 8), (7, 6, 7)])
def test_gradient_in_the_next_reverse_step(dims, precision, engine_lib):
    """A reverse step's gradient is added in the next one's H launch (1 to 294 voxels: one block, one
    full block, a block of rest): bit-identical to the gradient in a launch of its own, which segments
    of one step take, with the monitor rectangle through the design box."""
    args = "--3d --size x:28,y:27,z:29 --use-pml --pml-size x:3,y:3,z:3 --point-source x:5,y:6,z:7 --point-source-ez " \
           "--wavelength 0.004 --time-steps 24"
    print(f"[gpu] gradient in the next reverse step, design {dims}, precision {precision}", flush=True)
    rng = np.random.default_rng(6)
    eps = rng.uniform(1.0, 4.0, size=(28, 27, 29))
    design = rng.uniform(1.0, 4.0, size=dims)
    out = []
    for every in (0, 1, 5):
        eng = Engine(parse_args(args.split(), precision=precision))
        eng.set_material("eps", eps)
        eng.prepare()
        eng.adjoint_setup((5, 5, 6), tuple(lo + n for lo, n in zip((5, 5, 6), dims)), 6, (4, 4), (20, 19), 9, every)
        out.append((eng.forward(design), eng.backward(1.0)))
        eng.close()
    for J, g in out[1:]:
        assert J == out[0][0] and np.array_equal(g, out[0][1])
    assert np.abs(out[0][1]).max() > 0


@pytest.mark.parametrize("precision", [4, 8])
@pytest.mark.parametrize("args,one_launch", [
    ("--1d-exhy --size z:600 --use-pml --pml-size z:50 --use-tfsf --tfsf-size-left z:150 --tfsf-size-right z:0 --angle-teta 0 "
     "--angle-phi 0", True),
    ("--2d-tmz --size x:160,y:140 --use-pml --pml-size x:6,y:6 --use-tfsf --tfsf-size-left x:12,y:12 --tfsf-size-right "
     "x:12,y:12 --angle-teta 90 --angle-phi 30", True),
    ("--3d --size x:40,y:40,z:40 --use-pml --pml-size x:5,y:5,z:5 --use-tfsf --tfsf-size-left x:9,y:9,z:9 --tfsf-size-right "
     "x:9,y:9,z:9 --angle-teta 30 --angle-phi 45 --angle-psi 90", False),
])
def test_profile_is_per_step(args, one_launch, precision, engine_lib):
    """The groups of yee_profile_steps are milliseconds per step however many steps a launch takes:
    their intervals follow one another on one stream inside the measured run, so their sum is at most
    the step's own time (5 % for the resolution of the time stamps)."""
    eng = Engine(parse_args((args + " --time-steps 300").split(), precision=precision))
    eng.prepare()
    eng.step(70)
    p = eng.profile_steps(70)
    eng.close()
    groups = [p[k] for k in ("incident_ms", "e_half_ms", "h_half_ms", "fused_ms")]
    print(f"[gpu] profile {args.split()[0]} precision {precision}: {p}", flush=True)
    assert p["incident_ms"] > 0 and (p["fused_ms"] > 0) == one_launch and (p["e_half_ms"] > 0) != one_launch
    assert sum(groups) <= 1.05 * p["step_ms"]


@pytest.mark.parametrize("precision", [4, 8])
@pytest.mark.parametrize("mu", [False, True])
def test_batch_steps_past_a_full_launch(mu, precision, engine_lib, monkeypatch):
    """The steps of a call past the last full launch of the register tiles may take another launch
    shape: 3.3e6 cells (where one or two steps do without the tuner's times), calls of every remainder of
    4 and 8 steps before the tuner has run and after it, against single runs, bit for bit."""
    calls = [1, 1, 2, 3, 4, 5, 6, 7, 9, 10, 62, 1, 2, 3, 4, 5, 6, 7, 9]
    sims = [f"--2d-tmz --size x:{a},y:{b} --use-pml --pml-size x:6,y:7 --point-source x:{a // 2},y:{b // 2} --point-source-ez "
            f"--time-steps {sum(calls)}" for a, b in ((1303, 1250), (1290, 1301))]
    cfgs = [parse_args(s.split(), precision=precision) for s in sims]
    print(f"[gpu] batch remainders, mu {mu}, precision {precision}", flush=True)
    rng = np.random.default_rng(23)
    eps = [rng.uniform(1.0, 5.0, size=c.shape) for c in cfgs]
    mus = [rng.uniform(1.0, 2.0, size=c.shape) for c in cfgs]
    b = Batch(cfgs)
    for s in range(2):
        b.set_material(s, "eps", eps[s])
        if mu:
            b.set_material(s, "mu", mus[s])
    b.prepare()
    for n in calls:
        b.step(n)
    assert b.time == sum(calls)
    monkeypatch.setenv("YEE_KERNEL", "split")
    for s, c in enumerate(cfgs):
        e = Engine(c)
        e.set_material("eps", eps[s])
        if mu:
            e.set_material("mu", mus[s])
        e.prepare()
        e.step(sum(calls))
        for f in ("Ez", "Hx", "Hy", "Dz", "Bx", "By"):
            assert np.array_equal(b.field(s, f), e.field(f)), f"sim {s} {f}"
        e.close()
    b.close()


@pytest.mark.parametrize("precision,nb", [(4, 2886), (8, 2041)])
@pytest.mark.parametrize("fits", [True, False])
def test_single_steps_of_2d_runs(fits, precision, nb, engine_lib, monkeypatch):
    """A single step takes the tiles where two buffers of E and H fill at most 200 MB and half steps in
    place above; both sides of that line, mixed with calls of several steps: the half-step kernels'
    fields and D / B, bit for bit."""
    na = int(200e6 / (6 * precision) / nb) + (0 if fits else 1)
    assert (6 * precision * na * nb <= 200e6) == fits
    cfg = parse_args(f"--2d-tmz --size x:{na},y:{nb} --use-pml --pml-size x:7,y:6 --point-source x:{na // 2},y:{nb // 2} "
                     "--point-source-ez --time-steps 60".split(), precision=precision)
    eps = np.random.default_rng(29).uniform(1.0, 5.0, size=cfg.shape)
    calls = [1, 1, 1, 9, 1, 2, 17, 1]
    print(f"[gpu] single steps {na}x{nb} precision {precision}", flush=True)
    out = []
    for kernel in ("split", ""):
        monkeypatch.setenv("YEE_KERNEL", kernel)
        eng = Engine(cfg)
        eng.set_material("eps", eps)
        eng.prepare()
        for n in calls:
            eng.step(n)
        out.append({c: eng.field_raw(c) for c in ("Ez", "Hx", "Hy", "Dz", "Bx", "By")})
        eng.close()
    for c, v in out[0].items():
        assert np.array_equal(out[1][c], v), c
    assert np.abs(out[0]["Ez"]).max() > 0


@pytest.mark.parametrize("precision", [4, 8])
@pytest.mark.parametrize("args", [
    "--2d-tmz --size x:98,y:67 --use-pml --pml-size x:6,y:5 --use-tfsf --tfsf-size-left x:12,y:12 --tfsf-size-right x:12,y:12 "
    "--angle-teta 90 --angle-phi 30",
    "--2d-tex --size y:51,z:99 --use-pml --pml-size y:5,z:6 --point-source y:25,z:50 --point-source-ey",
    "--2d-tmy --size x:66,z:52 --point-source x:30,z:20 --point-source-ey",
    "--1d-exhy --size z:421 --use-pml --pml-size z:9 --use-tfsf --tfsf-size-left z:60 --tfsf-size-right z:0 --angle-teta 0 "
    "--angle-phi 0",
    "--1d-eyhz --size x:195 --point-source x:90 --point-source-ey",
])
def test_double_material_precision_in_one_launch(args, precision, engine_lib, monkeypatch):
    """Runs with double material precision take the tiles and lines as well, with the 8-cell averages
    of each component: the half-step kernels' fields and D / B, bit for bit."""
    cfg = parse_args((args + " --use-double-material-precision --time-steps 70").split(), precision=precision)
    assert cfg.double_material
    rng = np.random.default_rng(31)
    eps, mu = rng.uniform(1.0, 5.0, size=cfg.material_shape), rng.uniform(1.0, 2.0, size=cfg.material_shape)
    print(f"[gpu] double material precision {args.split()[0]} precision {precision}", flush=True)
    out = []
    for kernel, calls in (("split", [70]), ("", [70]), ("", [1, 2, 7, 33, 27])):
        monkeypatch.setenv("YEE_KERNEL", kernel)
        eng = Engine(cfg)
        eng.set_material("eps", eps)
        eng.set_material("mu", mu)
        eng.prepare()
        for n in calls:
            eng.step(n)
        names = list(cfg.components) + ([("D" if c[0] == "E" else "B") + c[1] for c in cfg.components] if cfg.use_pml else [])
        out.append({c: eng.field_raw(c) for c in names})
        eng.close()
    for c, v in out[0].items():
        assert np.array_equal(out[1][c], v), c
        assert np.array_equal(out[2][c], v), c
    assert any(np.abs(v).max() > 0 for v in out[0].values())


@pytest.mark.parametrize("precision", [4, 8])
@pytest.mark.parametrize("x,y,z", [(31, 40, 257), (24, 560, 260), (12, 1100, 320), (203, 30, 330)])
def test_sweep_chunks_of_long_rows(x, y, z, precision, engine_lib, monkeypatch):
    """Rows of five and six waves with fewer strips than compute units, one to two strips a unit and
    more than two: however the sweep is cut into chunks, the half steps' fields, bit for bit."""
    args = f"--3d --size x:{x},y:{y},z:{z} --use-pml --pml-size x:3,y:4,z:5 --point-source x:{x // 2},y:{y // 2},z:{z // 2} " \
           "--point-source-ez --time-steps 12"
    print(f"[gpu] chunks {x}x{y}x{z} precision {precision}", flush=True)
    eps = np.random.default_rng(37).uniform(1.0, 4.0, size=(x, y, z))
    ref = _run(args, precision, monkeypatch, "split", eps, 12)
    got = _run(args, precision, monkeypatch, "fused", eps, 12)
    for n, v in ref.items():
        assert np.array_equal(got[n], v), n
    assert np.abs(ref["Ez"]).max() > 0
