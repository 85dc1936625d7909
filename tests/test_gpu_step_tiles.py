"""Edges of the step kernel's tiles: grids that the tile does not divide (the
last tile of an axis overlaps the one before it), lower or narrower than one
tile, one to three planes, and uneven z-chunks, against the oracle.

Tolerances, as for the tile-sized grids: five FP64 steps differ from the
oracle by round-off (1e-15 relative per operation and about 100 operations
deep: 1e-13 a step), one FP32 step by 2e-6 of the largest population.
"""
import numpy as np
import pytest

from conftest import W, feq, moments, random_state
from dugks_amd import (KERNEL_AUTO, KERNEL_FUSED, KERNEL_TWOPASS, LOSS_KINETIC_ENERGY, PREC_FP16N, PREC_FP16S,
                       PREC_FP32, PREC_FP64, configs)
from test_gpu_step import _engine, _oracle_for, _relerr

pytestmark = pytest.mark.gpu

# (nx, ny, nz): 32 x 12 tiles in FP32, 16 x 12 in FP64
EDGES = [
    (16, 12, 1),    # one plane; narrower than an FP32 tile
    (32, 4, 2),     # lower than a tile
    (32, 16, 3),    # the last tile overlaps 8 rows
    (48, 36, 2),    # the last FP32 tile overlaps 16 columns
    (64, 20, 37),   # one-plane and two-plane chunks
]
WALLS = {
    "periodic": {},
    "walls_y": dict(periods_y=0, mesh_y="tanh:0.85", dt_rule="min"),
    "walls_xy": dict(periods_x=0, periods_y=0),
}


def _text(n, walls, recon="tri"):
    kw = {k: v for k, v in WALLS[walls].items() if recon == "tri" or k not in ("mesh_y", "dt_rule")}
    return configs.base(nx=n[0], ny=n[1], nz=n[2], xwidth=n[0] / 10, ywidth=n[1] / 10, zwidth=n[2] / 10, visc=0.02,
                        CFL=0.5, recon=recon, ambient_fx=2e-4, ambient_fz=1e-4, **kw)


@pytest.mark.parametrize("recon", ["tri", "grad"])
@pytest.mark.parametrize("walls", list(WALLS))
@pytest.mark.parametrize("n", EDGES, ids=str)
def test_tile_edges_match_oracle(rng, n, walls, recon):
    text = _text(n, walls, recon)
    for precision, steps, tol in ((PREC_FP64, 5, 5e-13), (PREC_FP32, 1, 2e-6)):
        eng = _engine(text, precision=precision, kernel=KERNEL_FUSED)
        ora = _oracle_for(eng, text)
        eng.set_f(random_state(eng.shape, rng))
        ora.set_f(eng.get_f())
        eng.step(steps)
        ora.step(steps)
        assert _relerr(eng.get_f(), ora.get_f()) <= tol


# Grids that are not whole tiles, which the automatic choice takes to the step
# kernel: odd rows and columns, narrower and lower than a tile, one row, one
# column, overlaps of all but one row or column.
RAGGED = [(13, 40, 1), (31, 33, 3), (50, 11, 2), (17, 13, 5), (8, 64, 8), (33, 25, 4)]
RAGGED_WALLS = {**WALLS, "walls_x": dict(periods_x=0, mesh_x="tanh:0.8", dt_rule="min")}


@pytest.mark.parametrize("recon", ["tri", "grad"])
@pytest.mark.parametrize("walls,n", [(w, n) for w in RAGGED_WALLS for n in RAGGED] +
                         [("periodic", (1, 520, 1)), ("periodic", (520, 1, 2)), ("walls_y", (171, 3, 1)),
                          ("walls_xy", (3, 3, 60))], ids=str)
def test_ragged_grids_match_twopass(rng, n, walls, recon):
    """All storage modes against the two-pass kernels.  Tolerances: both paths'
    distances from the oracle as tested for whole tiles, 1e-13 (FP64) and
    2e-6 (FP32 arithmetic) a step, and for FP16 storage one rounding each."""
    kw = {k: v for k, v in RAGGED_WALLS[walls].items() if recon == "tri" or not k.startswith(("mesh", "dt"))}
    text = configs.base(nx=n[0], ny=n[1], nz=n[2], xwidth=n[0] / 10, ywidth=n[1] / 10, zwidth=n[2] / 10, visc=0.02,
                        CFL=0.5, recon=recon, ambient_fx=2e-4, ambient_fz=1e-4, **kw)
    for precision in (PREC_FP64, PREC_FP32, PREC_FP16S, PREC_FP16N):
        got = []
        f0 = random_state(n, rng)
        for kernel in (KERNEL_AUTO, KERNEL_TWOPASS):
            eng = _engine(text, precision=precision, kernel=kernel)
            eng.set_f(f0)
            eng.step(3 if precision == PREC_FP64 else 1)
            got.append(eng.get_f())
        a, b = got
        big = np.abs(b).max()
        if precision == PREC_FP64:
            tol = 2 * 3e-13 * big
        elif precision == PREC_FP32:
            tol = 2 * 2e-6 * big
        elif precision == PREC_FP16S:
            tol = 2 * (W * np.maximum(2.0 ** -11 * np.abs(b / W - eng.params["rho0"]), 2.0 ** -25) + 4e-6 * big)
        else:
            rho, j = moments(b)
            tol = 2 * (2.0 ** -11 * np.abs(b - feq(rho, j / rho[..., None])) + 2.0 ** -25 * W / 1024 + 4e-6 * big)
        assert np.all(np.abs(a - b) <= tol)


def test_automatic_choice_of_ragged_grids():
    def launches(**kw):
        base = dict(nx=20, ny=17, nz=5, xwidth=2.0, ywidth=1.7, zwidth=0.5, visc=0.02)
        return _engine(configs.base(**{**base, **kw}), kernel=KERNEL_AUTO).time_steps(1)["launches_per_step"]
    assert launches() == 1
    assert launches(periods_y=0, flow_rate=0.01, ambient_fx=1e-4) == 1  # the controller runs in the step
    assert launches(nz=1) == 5       # fewer than 512 cells
    assert launches(periods_z=0) == 5


@pytest.mark.parametrize("precision,tol", [(PREC_FP64, 1e-12), (PREC_FP32, 5e-5)], ids=["fp64", "fp32"])
def test_ragged_flow_rate_matches_twopass(precision, tol):
    """The controller's force over 10 steps: FP64 to round-off; FP32 to ten
    roundings of the velocity (6e-8 of 0.1) over the time step's share of the
    gain, 1e-5 of the force, times a margin of 5."""
    text = configs.base(nx=45, ny=29, nz=11, xwidth=4.5, ywidth=2.9, zwidth=1.1, periods_y=0, visc=0.02,
                        flow_rate=0.05, ambient_fx=2e-4)
    got = []
    for kernel in (KERNEL_AUTO, KERNEL_TWOPASS):
        eng = _engine(text, precision=precision, kernel=kernel)
        eng.step(10)
        got.append(np.array(eng.get_f(), dtype=np.float64))
    assert _relerr(got[0], got[1]) <= tol


@pytest.mark.parametrize("nx", [1, 28, 29, 300], ids=lambda v: f"rows{v}")
def test_planar_statistics_over_row_counts(rng, nx):
    """Row sums and the global mean, minimum and maximum where the last block of
    row sums is nearly full (9 x 28 of 256 threads), just over, and with several
    slots per thread (300 rows).  Means of O(1) values in FP64: 1e-12."""
    eng = _engine(configs.base(nx=nx, ny=3, nz=200, xwidth=0.1 * nx, ywidth=0.3, zwidth=20.0, visc=0.02))
    eng.set_f(random_state(eng.shape, rng))
    prof, diag = eng.statistics()
    rho, ux, uy, uz = eng.macro()
    mean = lambda a: a.mean(axis=(0, 1))
    U, V, Wv = mean(ux), mean(uy), mean(uz)
    expect = np.stack([U, V, Wv, mean(ux * uz) - U * Wv, mean(ux * uy) - U * V, mean(uy * uz) - V * Wv,
                       mean(ux * ux) - U * U, mean(uy * uy) - V * V, mean(uz * uz) - Wv * Wv], axis=1)
    assert np.abs(prof - expect).max() <= 1e-12
    fields = (rho, ux, uy, uz)
    assert np.abs(diag[0:4] - [a.mean() for a in fields]).max() <= 1e-12
    assert np.abs(diag[4:8] - [a.min() for a in fields]).max() <= 1e-15
    assert np.abs(diag[8:12] - [a.max() for a in fields]).max() <= 1e-15


@pytest.mark.parametrize("n", [(32, 24, 1), (32, 24, 3), (64, 8, 32), (32, 40, 67), (64, 16, 5)], ids=str)
@pytest.mark.parametrize("walls", ["periodic", "walls_y", "walls_x"])
@pytest.mark.parametrize("precision", [PREC_FP64, PREC_FP32], ids=["fp64", "fp32"])
def test_adjoint_step_over_tiles_and_chunks(rng, precision, walls, n):
    """lam.(df) = lam_prev.(df0) for the adjoint step over chunks of one plane,
    of a few, and of unequal length, and over tiles that overlap, that fill the
    grid's height and that exceed it, against the finite difference of the FP64
    step (central, 1e-6 of a unit perturbation: truncation and cancellation
    1e-8 of the sums of 1e4 terms)."""
    torch = pytest.importorskip("torch")
    text = configs.base(nx=n[0], ny=n[1], nz=n[2], xwidth=n[0] / 10, ywidth=n[1] / 10, zwidth=n[2] / 10, visc=0.02,
                        CFL=0.5, ambient_fx=2e-4, **RAGGED_WALLS[walls])
    eng = _engine(text, precision=precision, kernel=KERNEL_AUTO)
    ref = _engine(text, precision=PREC_FP64, kernel=KERNEL_AUTO)
    f0 = random_state(eng.shape, rng)
    df = rng.standard_normal(f0.shape)
    lam = rng.standard_normal(f0.shape)
    eng.set_f(f0)
    f0 = np.array(eng.get_f())
    dev = torch.tensor(np.ascontiguousarray(np.moveaxis(lam, -1, 0)), device="cuda")
    out = torch.empty_like(dev)
    eng.adjoint_step(dev, out)
    got = float((np.moveaxis(out.cpu().numpy(), 0, -1) * df).sum())
    J = []
    for s in (1, -1):
        ref.set_f(f0 + s * 1e-6 * df)
        ref.step(1)
        J.append(float((ref.get_f() * lam).sum()))
    want = (J[0] - J[1]) / 2e-6
    size = np.linalg.norm(lam) * np.linalg.norm(df)
    assert abs(got - want) <= (1e-8 if precision == PREC_FP64 else 1e-6) * size


@pytest.mark.parametrize("precision,n,tol", [
    (PREC_FP64, (82, 39, 41), 6e-13), (PREC_FP64, (51, 50, 49), 6e-13),      # chunks of 4 planes, runs over the rest
    (PREC_FP32, (102, 61, 41), 4e-6), (PREC_FP32, (38, 54, 126), 4e-6),
    (PREC_FP64, (48, 40, 20), 6e-13), (PREC_FP64, (64, 64, 32), 6e-13),      # tiles of 12 and of 8 rows
    (PREC_FP32, (64, 64, 32), 4e-6), (PREC_FP32, (20, 20, 20), 4e-6)])       # of 8 rows, of 4 rows
@pytest.mark.parametrize("walls", ["periodic", "walls_y", "walls_x"])
def test_plans_match_twopass(rng, precision, n, tol, walls):
    """Every form of the step's plan, with the flow-rate controller where there
    are walls (its sums run over the same tiles), against the two-pass kernels:
    3 FP64 steps of 1e-13, one FP32 step of 2e-6, on both sides."""
    kw = dict(RAGGED_WALLS[walls], **({"flow_rate": 0.02} if walls != "periodic" else {}))
    text = configs.base(nx=n[0], ny=n[1], nz=n[2], xwidth=n[0] / 10, ywidth=n[1] / 10, zwidth=n[2] / 10, visc=0.02,
                        CFL=0.5, ambient_fz=1e-4, flow_axis=2, **kw)
    f0 = random_state(n, rng)
    got = []
    for kernel in (KERNEL_AUTO, KERNEL_TWOPASS):
        eng = _engine(text, precision=precision, kernel=kernel)
        eng.set_f(f0)
        eng.step(3 if precision == PREC_FP64 else 1)
        got.append(eng.get_f())
    assert _relerr(*got) <= tol


@pytest.mark.parametrize("n", [(3, 4, 2), (16, 16, 1), (257, 1, 1), (64, 64, 65)], ids=str)
def test_loss_over_grid_sizes(rng, n):
    """The kinetic-energy loss on fewer cells than a block has threads, exactly
    one block, one more, and more than the largest grid of blocks, against the
    fields; the same bits on a second call.  FP64 sums of like terms: 1e-13."""
    eng = _engine(configs.base(nx=n[0], ny=n[1], nz=n[2], xwidth=n[0] / 10, ywidth=n[1] / 10, zwidth=n[2] / 10,
                               visc=0.02, ambient_fx=2e-4))
    eng.set_f(random_state(n, rng))
    rho, ux, uy, uz = eng.macro()
    want = (0.5 * rho * (ux ** 2 + uy ** 2 + uz ** 2)).mean()
    got = eng.loss(LOSS_KINETIC_ENERGY)
    assert abs(got - want) <= 1e-13 * want
    assert eng.loss(LOSS_KINETIC_ENERGY) == got
