"""Every form of the step's plan and of the adjoint's gather, in every storage mode,
against the two-pass kernels, cell by cell (plan_grids.py names grids by form)."""
import time

import numpy as np
import pytest

from conftest import W, feq, moments, random_state
from dugks_amd import (KERNEL_AUTO, KERNEL_TWOPASS, PREC_FP16N, PREC_FP16S, PREC_FP32, PREC_FP64, configs)
from plan_grids import GATHER_GRIDS, STEP_GRIDS
from test_gpu_adjoint import _flow_grad, _flow_J, _flow_problem
from test_gpu_adjoint import _engine as _stream_engine
from test_gpu_step import _engine

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu

MODES = {"fp64": PREC_FP64, "fp32": PREC_FP32, "fp16": PREC_FP16S, "fp16n": PREC_FP16N}
WALLS = {"periodic": {}, "walls_y": dict(periods_y=0, mesh_y="tanh:0.85", dt_rule="min"),
         "walls_x": dict(periods_x=0, mesh_x="tanh:0.8", dt_rule="min"),
         "walls_xy": dict(periods_x=0, periods_y=0)}


def _text(n, walls, recon="tri"):
    kw = {k: v for k, v in WALLS[walls].items() if recon == "tri" or not k.startswith(("mesh", "dt"))}
    return configs.base(nx=n[0], ny=n[1], nz=n[2], xwidth=n[0] / 10, ywidth=n[1] / 10, zwidth=n[2] / 10, visc=0.02,
                        CFL=0.5, recon=recon, ambient_fx=2e-4, ambient_fz=1e-4, **kw)


STEP_CASES = [(form, mode, n, walls) for form in STEP_GRIDS for mode in MODES for n in STEP_GRIDS[form][mode]
              for walls in WALLS if n[0] * n[1] * n[2] < 200000 or walls == "walls_y"]


@pytest.mark.parametrize("form,mode,n,walls", STEP_CASES,
                         ids=lambda v: "-".join(map(str, v)) if isinstance(v, tuple) else v)
def test_step_forms_match_twopass(rng, form, mode, n, walls):
    """With a force in every cell.  Both paths' distances from the oracle, as tested
    on whole tiles: 1e-13 a step in FP64 (three steps here), 2e-6 in FP32
    arithmetic, and for FP16 storage one rounding each."""
    text = _text(n, walls, form[0])
    f0 = random_state(n, rng)
    G = 1e-4 * rng.standard_normal((3,) + f0.shape[:3])
    got = []
    for kernel in (KERNEL_AUTO, KERNEL_TWOPASS):
        eng = _engine(text, precision=MODES[mode], kernel=kernel)
        eng.set_f(f0)
        eng.set_cell_force(*G)
        eng.step(3 if mode == "fp64" else 1)
        got.append(eng.get_f())
    a, b = got
    big = np.abs(b).max()
    if mode == "fp64":
        tol = 2 * 3e-13 * big
    elif mode == "fp32":
        tol = 2 * 2e-6 * big
    elif mode == "fp16":
        tol = 2 * (W * np.maximum(2.0 ** -11 * np.abs(b / W - eng.params["rho0"]), 2.0 ** -25) + 4e-6 * big)
    else:
        rho, j = moments(b)
        tol = 2 * (2.0 ** -11 * np.abs(b - feq(rho, j / rho[..., None])) + 2.0 ** -25 * W / 1024 + 4e-6 * big)
    assert np.all(np.abs(a - b) <= tol)


GATHER_CASES = [(rows, mode, n, lam) for rows in GATHER_GRIDS for mode in GATHER_GRIDS[rows]
                for n in GATHER_GRIDS[rows][mode] for lam in (("f64",) if mode == "fp64" else ("f64", "f32"))]


@pytest.mark.parametrize("walls", ["periodic", "walls_y", "walls_x"])
@pytest.mark.parametrize("rows,mode,n,lam", GATHER_CASES,
                         ids=lambda v: "-".join(map(str, v)) if isinstance(v, tuple) else str(v))
def test_gather_forms_match_twopass(rng, rows, mode, n, lam, walls):
    """lam and the force gradient, added to what the array holds, against the FP64
    two-pass adjoint about the same stored state: the bounds of one adjoint step
    against the oracle, 1e-12 (FP64) and 2e-5 (FP32 arithmetic) of the largest
    value.  A row of cells taken twice or not at all is off by that value."""
    text = _text(n, walls)
    nz, ny, nx = n[2], n[1], n[0]
    lam0 = torch.randn((19, nz, ny, nx), dtype=torch.float32, device="cuda",
                       generator=torch.Generator("cuda").manual_seed(3)).double()
    G = 1e-4 * rng.standard_normal((3, nz, ny, nx))
    eng = _stream_engine(text, precision=MODES[mode], kernel=KERNEL_AUTO)
    eng.set_f(random_state(n, rng))
    ref = _stream_engine(text, precision=PREC_FP64, kernel=KERNEL_TWOPASS)
    ref.set_f(eng.get_f())
    out = []
    for e, dtype in ((eng, torch.float32 if lam == "f32" else torch.float64), (ref, torch.float64)):
        e.set_cell_force(*G)
        lp = torch.full((19, nz, ny, nx), float("nan"), dtype=dtype, device="cuda")
        g = torch.full((3, nz, ny, nx), 0.5, dtype=torch.float64, device="cuda")
        e.adjoint_step(lam0.to(dtype), lp, g)
        torch.cuda.synchronize()
        out.append((lp.double(), g - 0.5))
    tol = 1e-12 if mode == "fp64" else 2e-5
    for got, want in zip(*out):
        assert float((got - want).abs().max()) <= tol * float(want.abs().max())


@pytest.mark.parametrize("n", [GATHER_GRIDS[12]["fp64"][0], (32, 16, 1)], ids=["rows12", "one_plane"])
def test_controller_sweep_over_gather_forms(rng, n):
    """The gather that adds the controller's term, on overlapping tiles of 12 rows
    and on one plane: FP64 against central differences (the bar of the 8-row sweep,
    1e-7)."""
    eng, f0, F0, G, T = _flow_problem(PREC_FP64, *n, T=8)
    J, grad, dF0 = _flow_grad(eng, f0, F0, G, T)
    for trial in range(3):
        v = rng.standard_normal(G.shape) * 1e-6
        fd = (_flow_J(eng, f0, F0, G + v, T) - _flow_J(eng, f0, F0, G - v, T)) / 2
        an = float((grad * v).sum())
        assert abs(fd - an) <= 1e-7 * abs(an), (trial, fd, an)


@pytest.mark.parametrize("n,images", [((32, 16, 1), 3), ((96, 40, 1), 4), ((256, 200, 2), 2), ((512, 200, 2), 2)],
                         ids=str)
def test_controller_sweep_on_periodic_images(rng, n, images):
    """One and two planes in forms of their own against the general one: a state that
    repeats along z has the same J per cell, so with `images` copies J and dJ/dF^0
    are the same and the gradient in a cell is the 1/images part.  Eight FP64 steps
    of 1e-13, forward and back, and sums of 1e5 terms: 1e-11."""
    got = []
    f0 = G = None
    for m in (1, images):
        text = configs.adjoint_channel(nx=n[0], ny=n[1], nz=n[2] * m, zwidth=0.13 * n[2] * m, xwidth=0.13 * n[0],
                                       flow_rate=0.06, flow_axis=0)
        eng = _stream_engine(text, precision=PREC_FP64)
        if m == 1:
            f0 = eng.get_f() * (1 + 1e-3 * rng.standard_normal(eng.fshape))
            G = 1e-6 * rng.standard_normal((3,) + eng.fshape[:3])
        got.append(_flow_grad(eng, np.tile(f0, (m, 1, 1, 1)), eng.ambient_force(), np.tile(G, (1, m, 1, 1)), 8))
    (Ja, ga, da), (Jb, gb, db) = got
    assert abs(Ja - Jb) <= 1e-11 * abs(Ja)
    assert abs(da - db) <= 1e-11 * abs(da)
    assert np.abs(np.tile(ga, (1, images, 1, 1)) - images * gb).max() <= 1e-11 * np.abs(ga).max()


@pytest.mark.parametrize("n", [GATHER_GRIDS[12]["fp32"][0], (32, 16, 1)], ids=["rows12", "one_plane"])
@pytest.mark.parametrize("mode,tol", [("fp32", 1e-5), ("fp16", 2e-4)])
def test_reduced_precision_controller_sweep_over_gather_forms(mode, tol, n):
    """Against the FP64 sweep, with the bars of the 8-row one."""
    got = []
    for precision in (MODES[mode], PREC_FP64):
        eng, f0, F0, G, T = _flow_problem(precision, *n, T=8)
        got.append(_flow_grad(eng, f0, F0, G, T))
    (Ja, ga, da), (Jb, gb, db) = got
    assert abs(Ja - Jb) <= tol * abs(Jb)
    assert np.abs(ga - gb).max() <= tol * np.abs(gb).max()
    assert abs(da - db) <= tol * abs(db)


def test_one_plane_adjoint_takes_the_plane_once():
    """On one plane the gather's three neighbouring planes are the same.  Taken once,
    an adjoint step costs 0.6 of one on two planes, taken three times as much as
    that one; the least time of many runs of each, in turn, must stay below 0.85."""
    best = {}
    runs = {}
    for nz in (1, 2):
        eng = _stream_engine(_text((64, 64, nz), "periodic"), precision=PREC_FP32)
        lam = torch.randn((19, nz, 64, 64), dtype=torch.float64, device="cuda")
        runs[nz] = (eng, lam, torch.empty_like(lam))
    for _ in range(40):
        for nz, (eng, lam, out) in runs.items():
            torch.cuda.synchronize()
            t = time.perf_counter()
            for _ in range(20):
                eng.adjoint_step(lam, out)
            torch.cuda.synchronize()
            best[nz] = min(best.get(nz, 1.0), time.perf_counter() - t)
    assert best[1] <= 0.85 * best[2], best
