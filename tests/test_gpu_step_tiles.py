"""Edges of the step kernel's tiles: grids that the tile does not divide (the
last tile of an axis overlaps the one before it), lower or narrower than one
tile, one to three planes, and uneven z-chunks, against the oracle.

Tolerances, as for the tile-sized grids: five FP64 steps differ from the
oracle by round-off (1e-15 relative per operation and about 100 operations
deep: 1e-13 a step), one FP32 step by 2e-6 of the largest population.
"""
import pytest

from conftest import random_state
from dugks_amd import KERNEL_FUSED, PREC_FP32, PREC_FP64, configs
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
