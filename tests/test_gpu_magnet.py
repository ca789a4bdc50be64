"""The lean magnetic sweep (magnet_lean_impl.h) against the oracle, in lockstep.

FP64 reproduces the .m text's operations in their order, so every field stays within
1e-12 relative L-inf of the oracle each iteration (the bound of the parity tests).  The cases sit
where the sweep's windows and tiles can go wrong: pencils of 8 cells (the shortest it takes;
7 go to the general form), one to three cells past a whole chunk of four, a second round of
chunks per thread, pencil groups with padding; every boundary mode along the sweep and
across it, grids of one and two cells across, and a circular end opposite another mode (the
general form).
"""
import pytest

from imogen_amd import iteration, problems

from .helpers import FLUID_FIELDS, MAG_FIELDS, compare, make_gpu, make_oracle

pytestmark = pytest.mark.gpu

TOL = 1e-12

MODES = ["circ", "const", "trans", "mirror", "flip", "wall", "zero"]


def lockstep(grid, bc, limiter, iterations, seed):
    st = problems.random_state(grid, seed=seed, magnet=True)
    h = 1.0 / max(grid)
    ini = {"grid": grid, "dGrid": (h, h, h), "gamma": 5.0 / 3.0, "cfl": 0.3, "bcMode": bc,
           "bcInfinity": 20, "fluxLimiter": limiter, "minMass": 1e-5,
           "mode": {"fluid": True, "magnet": True}, "iterMax": 100, "timeMax": 1e9}
    orc = make_oracle(ini, st)
    run = make_gpu(ini, st)
    for it in range(iterations):
        orc.iteration()
        iteration(run)
        try:
            compare(run, orc, FLUID_FIELDS + MAG_FIELDS, TOL)
        except AssertionError as e:
            raise AssertionError("%s %s iteration %d: %s" % (grid, bc, it + 1, e))
    run.close()
    orc.close()


@pytest.mark.parametrize("mode", MODES)
@pytest.mark.parametrize("grid", [(8, 9, 1), (11, 10, 8)])
def test_modes(grid, mode):
    lockstep(grid, {"x": mode, "y": mode, "z": mode}, "vanleer", 5, 3)


@pytest.mark.parametrize("grid", [(7, 12, 1), (13, 16, 3), (21, 5, 35), (70, 18, 1), (9, 67, 9)])
def test_lengths(grid):
    lockstep(grid, {"x": "circ", "y": "trans", "z": "const"},
             {"x": "superbee", "y": "minmond", "z": "vanleer"}, 5, 7)


@pytest.mark.parametrize("grid,mode", [(g, m) for g in [(19, 1, 1), (10, 2, 1), (9, 2, 3)]
                                       for m in MODES if m != "mirror" or g[1] > 1])
def test_thin_across(grid, mode):
    lockstep(grid, {"x": "trans", "y": mode, "z": mode}, "vanleer", 4, 5)


@pytest.mark.parametrize("grid", [(1030, 4, 1), (4, 1029, 1)])
def test_several_chunks_per_thread(grid):
    lockstep(grid, {"x": "trans", "y": "circ", "z": "circ"}, "vanleer", 4, 9)


@pytest.mark.parametrize("bc", [
    {"x": ["circ", "trans"], "y": ["wall", "const"], "z": "circ"},
    {"x": ["zero", "mirror"], "y": ["flip", "trans"], "z": ["trans", "zero"]},
    {"x": "fade", "y": "trans", "z": "mirror"},
])
def test_mixed_ends(bc):
    lockstep((24, 22, 21) if bc["x"] == "fade" else (12, 10, 9), bc, "minmond", 4, 13)
