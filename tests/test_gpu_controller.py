"""What the flow-rate controller reads: the bulk velocity <j/rho> of the state
that the step leaves, summed in FP64 in every storage mode and on every form of
the step's plan, so that the force it sets follows from the state."""
import numpy as np
import pytest

from conftest import C, W, feq, moments, random_state
from dugks_amd import KERNEL_AUTO, KERNEL_TWOPASS, PREC_FP16N, PREC_FP16S, PREC_FP32, PREC_FP64, configs
from test_gpu_step import _engine

pytestmark = pytest.mark.gpu

TARGET = 0.02


def _bulk(eng, f, axis):
    """Bulk velocity along an axis and, for FP16 storage, how far the rounding of
    the populations can move it (half an FP16 ulp of the deviation, or of the
    non-equilibrium part, each population; the latter keeps u to FP32)."""
    rho, j = moments(f)
    u = j / rho[..., None]
    w = [eng.spacing(a) for a in range(3)]
    dV = w[2][:, None, None] * w[1][None, :, None] * w[0][None, None, :]
    prec = int(eng.params["precision"])
    if prec == PREC_FP16S:
        codec = W * np.maximum(2.0 ** -11 * np.abs(f / W - eng.params["rho0"]), 2.0 ** -25)
    elif prec == PREC_FP16N:
        codec = 2.0 ** -11 * np.abs(f - feq(rho, u)) + 2.0 ** -25 * W / 1024 + 2.0 ** -23 * np.abs(f)
    else:
        codec = np.zeros_like(f)
    moved = (np.einsum("...q,q->...", codec, np.abs(C[:, axis])) + np.abs(u[..., axis]) * codec.sum(-1)) / rho
    return (u[..., axis] * dV).sum() / dV.sum(), 1.01 * (moved * dV).sum() / dV.sum(), np.abs(u).max()


# one-plane tiles, lower tiles, 12-row tiles that overlap, chunks and runs
GRIDS = [(16, 12, 1), (20, 20, 20), (45, 29, 11), (64, 64, 32), (102, 61, 41), (51, 50, 49), (150, 97, 83)]


@pytest.mark.parametrize("kernel", [KERNEL_AUTO, KERNEL_TWOPASS], ids=["auto", "twopass"])
@pytest.mark.parametrize("walls,axis", [("y", 0), ("x", 2)], ids=["walls_y", "walls_x"])
@pytest.mark.parametrize("n", GRIDS, ids=str)
@pytest.mark.parametrize("precision", [PREC_FP64, PREC_FP32, PREC_FP16S, PREC_FP16N],
                         ids=["fp64", "fp32", "fp16", "fp16n"])
def test_force_follows_from_the_state(rng, precision, n, walls, axis, kernel):
    """F1 = F0 + gain (target - U1) / dt, then F2 = F1 - (U2 - U1) / dt + gain
    (target - U2) / dt, U of the states after each step.  FP64 sums of N like
    terms and a reciprocal: U to 2e-14 of the largest velocity (FP32 sums: about
    1e-8 a cell, 3e-12 and more of the mean over up to 1e7 terms); FP16 storage
    may move U by its rounding on top."""
    _force_follows(rng, precision, n, axis, kernel,
                   {f"periods_{walls}": 0, f"mesh_{walls}": "tanh:0.85", "dt_rule": "min"})


@pytest.mark.parametrize("n", [(16, 12, 1), (256, 300, 1), (45, 29, 11), (64, 64, 32), (41, 21, 44)], ids=str)
@pytest.mark.parametrize("precision", [PREC_FP64, PREC_FP32, PREC_FP16S, PREC_FP16N],
                         ids=["fp64", "fp32", "fp16", "fp16n"])
def test_force_follows_from_the_state_with_gradient_reconstruction(rng, precision, n):
    """The same on the gradient step's tiles and on one plane."""
    _force_follows(rng, precision, n, 0, KERNEL_AUTO, {"periods_y": 0, "recon": "grad"})


def _force_follows(rng, precision, n, axis, kernel, kw):
    text = configs.base(nx=n[0], ny=n[1], nz=n[2], xwidth=n[0] / 10, ywidth=n[1] / 10, zwidth=n[2] / 10, visc=0.02,
                        CFL=0.5, ambient_fx=2e-4, ambient_fz=1e-4, flow_rate=TARGET, flow_axis=axis, **kw)
    eng = _engine(text, precision=precision, kernel=kernel)
    eng.set_f(random_state(n, rng))
    dt = eng.params["dt"]
    F0 = eng.ambient_force()[axis]
    eng.step(1)
    F1 = eng.ambient_force()[axis]
    U1, moved1, big = _bulk(eng, eng.get_f(), axis)
    assert abs(F1 - (F0 + (TARGET - U1) / dt)) <= (2e-14 * big + moved1) / dt
    eng.step(1)
    F2 = eng.ambient_force()[axis]
    U2, moved2, big = _bulk(eng, eng.get_f(), axis)
    want = F1 - (U2 - U1) / dt + (TARGET - U2) / dt
    assert abs(F2 - want) <= (6e-14 * big + moved1 + 2 * moved2) / dt
