"""CPU tests of how the step kernel and the adjoint's gather divide a grid: every
form of a plan deals every plane of every tile once, and the grids that the GPU
tests name for a form take it."""
import pytest

import dugks_amd
from dugks_amd import PREC_FP16N, PREC_FP16S, PREC_FP32, PREC_FP64, configs
from plan_grids import GATHER_GRIDS, STEP_GRIDS

MODES = {"fp64": PREC_FP64, "fp32": PREC_FP32, "fp16": PREC_FP16S, "fp16n": PREC_FP16N}


def _plan(n, precision, recon="tri"):
    return dugks_amd.config_plan(configs.base(nx=n[0], ny=n[1], nz=n[2], recon=recon), precision)


def _tiles(n, precision, rows):
    tx = 16 if precision == PREC_FP64 else 32
    return -(-n[0] // tx) * -(-n[1] // rows)


@pytest.mark.parametrize("recon", ["tri", "grad"])
@pytest.mark.parametrize("precision", list(MODES.values()), ids=list(MODES))
def test_step_plans_deal_every_plane_once(precision, recon):
    seen = set()
    for nx in (1, 8, 16, 33, 64, 150, 256):
        for ny in (1, 4, 11, 12, 40, 97, 192):
            for nz in (1, 2, 5, 32, 83, 128):
                n = (nx, ny, nz)
                p = _plan(n, precision, recon)
                tiles = _tiles(n, precision, p["rows"])
                seen.add((p["rows"], p["chunk_planes"] > 0))
                assert 1 <= p["chunks"] <= nz
                if p["chunk_planes"] == 0:
                    assert p["blocks"] == tiles * p["chunks"]
                else:  # whole chunks, and runs of at least one plane over the rest
                    assert p["rows"] == 12 and recon == "tri"
                    left = nz - p["chunks"] * p["chunk_planes"]
                    runs = p["blocks"] - tiles * p["chunks"]
                    assert left > 0 and 0 < runs <= 256 and p["blocks"] == 256
                    assert runs <= left * tiles
    assert seen == {(12, False), (8, False), (4, False)} | ({(12, True)} if recon == "tri" else set())


def test_plans_need_a_grid_and_a_precision():
    assert _plan((128, 128, 128), -1) == _plan((128, 128, 128), PREC_FP64)  # the config's
    with pytest.raises(dugks_amd.DugksError):
        dugks_amd.config_plan(configs.base(), 4)
    with pytest.raises(dugks_amd.DugksError):
        dugks_amd.config_plan("nx=8\n", PREC_FP64)


@pytest.mark.parametrize("form", list(STEP_GRIDS))
def test_step_grids_take_the_form_they_are_named_for(form):
    recon, rows, runs = form
    for mode, grids in STEP_GRIDS[form].items():
        for n in grids:
            p = _plan(n, MODES[mode], recon)
            assert (p["rows"], p["chunk_planes"] > 0) == (rows, runs), (mode, n, p)


@pytest.mark.parametrize("rows", list(GATHER_GRIDS))
def test_gather_grids_take_the_rows_they_are_named_for(rows):
    for mode, grids in GATHER_GRIDS[rows].items():
        for n in grids:
            p = _plan(n, MODES[mode])
            assert p["gather_rows"] == rows and n[0] % 32 == 0 and n[1] % 8 == 0, (mode, n, p)
    # tiles of 12 rows that overlap, and ones that do not
    if rows == 12:
        assert all({n[1] % 12 != 0 for n in GATHER_GRIDS[rows][m]} == {True, False} for m in ("fp64", "fp32"))
