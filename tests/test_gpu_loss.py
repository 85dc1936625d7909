"""The losses on both sides of the rule that gives small grids one launch (up to
32 blocks of 256 cells) and larger ones two, and their cost beside a reduction
that reads the same state."""
import time

import numpy as np
import pytest

from conftest import random_state
from dugks_amd import (LOSS_KINETIC_ENERGY, LOSS_WALL_SHEAR, PREC_FP16N, PREC_FP16S, PREC_FP32, PREC_FP64, configs)
from test_gpu_step import _engine

pytestmark = pytest.mark.gpu


def _text(n, **kw):
    return configs.base(nx=n[0], ny=n[1], nz=n[2], xwidth=n[0] / 10, ywidth=n[1] / 10, zwidth=n[2] / 10, visc=0.02,
                        ambient_fx=2e-4, periods_y=0, **kw)


# cells of a kinetic-energy call: 32 blocks, one cell more, 33 blocks and a rest;
# of a wall-shear call (two planes of nx nz cells): 32 blocks, 33 blocks
@pytest.mark.parametrize("n", [(32, 16, 16), (8193, 3, 1), (43, 14, 14), (64, 3, 64), (64, 3, 65)], ids=str)
@pytest.mark.parametrize("precision", [PREC_FP64, PREC_FP32, PREC_FP16S, PREC_FP16N],
                         ids=["fp64", "fp32", "fp16", "fp16n"])
def test_losses_on_both_sides_of_the_launch_rule(rng, precision, n):
    """Against the fields of the stored state; FP64 sums of like terms: 1e-12 (the
    wall shear's terms differ in sign: of the sum of their sizes), and the same
    bits on a second call."""
    eng = _engine(_text(n), precision=precision)
    eng.set_f(random_state(n, rng))
    rho, ux, uy, uz = eng.macro()
    got = eng.loss(LOSS_KINETIC_ENERGY)
    want = (0.5 * rho * (ux ** 2 + uy ** 2 + uz ** 2)).mean()
    assert abs(got - want) <= 1e-12 * want
    assert eng.loss(LOSS_KINETIC_ENERGY) == got
    got = eng.loss(LOSS_WALL_SHEAR)
    walls = (rho * ux)[:, [0, n[1] - 1], :]
    coef = eng.params["visc"] / (0.5 * eng.spacing(1)[0] * 2 * n[0] * n[2])
    assert abs(got - coef * walls.sum()) <= 1e-12 * coef * np.abs(walls).sum()
    assert eng.loss(LOSS_WALL_SHEAR) == got


def test_loss_costs_no_more_than_a_reduction_over_the_state():
    """A kinetic-energy call reads the state once, as global_sums does, which
    forms more sums: it may take 1.5 times its time (2.1 times when 1024 blocks
    counted themselves in).  The least of many calls in turn, both with the copy
    back and the wait."""
    eng = _engine(_text((64, 64, 64)), precision=PREC_FP32)
    best = {}
    for _ in range(200):
        for name, call in (("loss", lambda: eng.loss(LOSS_KINETIC_ENERGY)), ("sums", eng.global_sums)):
            t = time.perf_counter()
            call()
            best[name] = min(best.get(name, 1.0), time.perf_counter() - t)
    assert best["loss"] <= 1.5 * best["sums"], best
