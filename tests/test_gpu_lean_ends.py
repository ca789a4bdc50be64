"""The lean fluid sweep (fluid_lean_impl.h) with boundary ghosts, on every tile it is compiled
for, and with cell differences at the low end of the FP64 range.

Large grids take four and eight cells per thread, in tiles that a test-sized grid would not
choose: the tiles are pinned, on x pencils that fill whole chunks (vector loads and stores)
and on ones that do not.  FP64 against the oracle: <= 1e-12 relative L-inf per iteration
(expected 0).  FP32 against FP64 from the same state: <= 1e-5 relative L1.
"""
import numpy as np
import pytest

from imogen_amd import autotune, iteration, problems
from imogen_amd.ensemble import Ensemble

from .helpers import FLUID_FIELDS, MAG_FIELDS, compare, make_gpu, make_oracle, rel_l1, rel_linf

pytestmark = pytest.mark.gpu

TOL = 1e-12
ENDS = ["trans", "wall", {"x": ["circ", "trans"], "y": ["wall", "circ"], "z": ["mirror", "zero"]}]


def box(grid, bc, limiter, magnet=False, seed=1):
    h = 1.0 / max(grid)
    ini = {"grid": grid, "dGrid": (h, h, h), "gamma": 1.4, "cfl": 0.4, "bcMode": bc,
           "bcInfinity": 20, "fluxLimiter": limiter, "minMass": 1e-5,
           "mode": {"fluid": True, "magnet": magnet}, "iterMax": 100, "timeMax": 1e9}
    return ini, problems.random_state(grid, seed=seed, magnet=magnet)


def tiles(esz, grid):
    """Tiles that hold the longest pencil of the grid: of the lean sweep, and with 32 pencils
    (more than it takes) of the general one."""
    return sorted({(bs, k, px) for e, bs, k in autotune._build.fluid_variants() if e == esz
                   for px in (1, 2, 8, 16, 32) if bs // px * k >= max(grid)})


def pin(run, grid, tile):
    for X in (1, 2, 3):
        if grid[X - 1] >= 3:
            run.set_fluid_tile(X, *tile)


@pytest.mark.parametrize("grid", [(16, 35, 1), (40, 3, 1), (37, 24, 1), (8, 6, 13)])
@pytest.mark.parametrize("bc", ENDS, ids=["trans", "wall", "mixed"])
@pytest.mark.parametrize("magnet", [False, True])
def test_every_tile_fp64(grid, bc, magnet):
    ini, st = box(grid, bc, "vanleer", magnet, seed=sum(grid))
    fields = FLUID_FIELDS + (MAG_FIELDS if magnet else [])
    for tile in tiles(8, grid):
        orc, run = make_oracle(ini, st), make_gpu(ini, st)
        pin(run, grid, tile)
        for it in range(3):
            orc.iteration()
            iteration(run)
            try:
                compare(run, orc, fields, TOL)
            except AssertionError as e:
                raise AssertionError("tile %s, iteration %d: %s" % (tile, it + 1, e))
        run.close()
        orc.close()


@pytest.mark.parametrize("grid", [(16, 35, 1), (37, 24, 1), (8, 6, 13)])
@pytest.mark.parametrize("bc", ["const"] + ENDS, ids=["const", "trans", "wall", "mixed"])
@pytest.mark.parametrize("magnet", [False, True])
def test_every_tile_fp32(grid, bc, magnet):
    """Every FP32 tile, against the FP64 run and against the first tile's bits."""
    ini, st = box(grid, bc, "vanleer", magnet, seed=sum(grid) + 1)
    fields = FLUID_FIELDS + (MAG_FIELDS if magnet else [])
    ref = make_gpu(ini, st)
    for _ in range(4):
        iteration(ref)
    want = {f: ref.download(f) for f in fields}
    ref.close()
    first = None
    for tile in tiles(4, grid):
        run = make_gpu(ini, st, "fp32")
        pin(run, grid, tile)
        for _ in range(4):
            iteration(run)
        got = {f: run.download(f) for f in fields}
        run.close()
        first = first or got
        for f in fields:
            if np.any(want[f] != 0):
                assert rel_l1(got[f], want[f]) <= 1e-5, (tile, f)
            np.testing.assert_array_equal(got[f], first[f], err_msg="%s %s" % (tile, f))


@pytest.mark.parametrize("scale", [1e-200, 1e-300, 3e-307, 1e-308])
def test_differences_below_the_normal_range(scale):
    """A passive momentum that decays towards transparent ends: the ghosts' slopes divide by
    differences of its cells, whose quotients overflow (and with them the slope is 0): 3050 of
    10091 in the oracle at the two smallest scales.  The circular x side leaves the trackers of
    the y side unused, so that the far node is 0."""
    grid = (24, 30, 1)
    ini, st = box(grid, {"x": "circ", "y": "trans"}, "vanleer", seed=5)
    y = np.arange(grid[1], dtype=float)[None, :, None]
    r = 1.0 + np.abs(np.asarray(st["mom"][2])).reshape(1, grid[1], grid[0])
    decay = np.exp(-np.abs(y - grid[1] / 2.0) / 4.0).reshape(1, grid[1], 1)
    st["mom"][2] = (scale * 0.5 * r * decay).reshape(np.shape(st["mom"][2]))
    orc, run = make_oracle(ini, st), make_gpu(ini, st)
    for _ in range(4):
        orc.iteration()
        iteration(run)
        for f in FLUID_FIELDS:
            assert np.all(np.isfinite(orc.get(f))) and np.all(np.isfinite(run.download(f))), f
        compare(run, orc, FLUID_FIELDS, TOL)
    run.close()
    orc.close()


@pytest.mark.parametrize("precision", ["fp64", "fp32"])
def test_batch_with_neumann_richtmyer(precision):
    """Simulations with the viscosity in a batch, beside ones without, against each alone:
    the same bodies on the same argument blocks."""
    sims = [box((40, 33, 1), "trans", "vanleer", seed=3), box((130, 9, 1), "circ", "superbee", seed=4),
            box((9, 14, 11), {"x": "wall", "y": "circ", "z": "const"}, "minmond", seed=5),
            box((24, 20, 1), "circ", "vanleer", True, seed=6), box((300, 1, 1), "trans", "vanleer", seed=7)]
    viscous = [0, 2, 3, 4]
    ens = Ensemble(sims, precision)
    for i in viscous:
        ens.set_viscosity(i, "neumann_richtmyer", 0.2, 0.4)
    ens.step(5)
    for i, (ini, st) in enumerate(sims):
        run = make_gpu(ini, st, precision)
        if i in viscous:
            run.set_viscosity("neumann_richtmyer", 0.2, 0.4)
        run.run_iterations(6)
        assert ens.time(i)[2] == run.time.iteration, i
        for f in FLUID_FIELDS + (MAG_FIELDS if ini["mode"]["magnet"] else []):
            assert rel_linf(ens.download(i, f), run.download(f)) <= TOL, (i, f)
        run.close()
    ens.close()
