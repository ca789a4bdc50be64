"""The lean fluid sweep (fluid_lean_impl.h) at the edges of its tiles, against the oracle.

The first iteration of a run is the general form's, the following ones are the lean
form's.  Pencil lengths at, one below and one above multiples of the cells per thread and
of a wave's cells, the shortest pencils that are swept, tiles with padding pencils and
every tile the sweep is compiled for; every boundary mode it evaluates, mixed modes
included, and the transparent ghost whose argument is the far node (bcInfinity 4).  FP64
keeps the operations and their order: <= 1e-12 relative L-inf per iteration (expected 0).
FP32 against FP64 from the same state: <= 1e-5 relative L1 over 6 iterations.
"""
import numpy as np
import pytest

from imogen_amd import autotune, iteration, problems

from .helpers import FLUID_FIELDS, MAG_FIELDS, compare, make_gpu, make_oracle, rel_l1

pytestmark = pytest.mark.gpu

TOL = 1e-12


def box(grid, bc, limiter, magnet=False, seed=1, inf=20):
    h = 1.0 / max(grid)
    ini = {"grid": grid, "dGrid": (h, h, h), "gamma": 1.4, "cfl": 0.4, "bcMode": bc,
           "bcInfinity": inf, "fluxLimiter": limiter, "minMass": 1e-5,
           "mode": {"fluid": True, "magnet": magnet}, "iterMax": 100, "timeMax": 1e9}
    return ini, problems.random_state(grid, seed=seed, magnet=magnet)


def lockstep(ini, st, tile=None, iterations=4, magnet=False):
    orc, run = make_oracle(ini, st), make_gpu(ini, st)
    for X in (1, 2, 3):
        if tile is not None and ini["grid"][X - 1] >= 3:
            run.set_fluid_tile(X, *tile)
    for _ in range(iterations):
        orc.iteration()
        iteration(run)
        compare(run, orc, FLUID_FIELDS + (MAG_FIELDS if magnet else []), TOL)
    run.close()
    orc.close()


@pytest.mark.parametrize("n", [3, 4, 5, 8, 15, 17, 33, 63, 65, 127, 129, 255, 257, 511, 513])
@pytest.mark.parametrize("bc", ["circ", "trans", {"x": ["const", "mirror"], "y": ["wall", "zero"]}])
def test_pencil_lengths(n, bc):
    lockstep(*box((n, 6, 1), bc, "vanleer", seed=n))
    lockstep(*box((5, n, 1), bc, "superbee", seed=n + 1))


@pytest.mark.parametrize("grid", [(9, 35, 1), (37, 3, 1), (11, 6, 13)])
@pytest.mark.parametrize("magnet", [False, True])
def test_every_tile(grid, magnet):
    tiles = sorted({(bs, k, px) for e, bs, k in autotune._build.fluid_variants() if e == 8
                    for px in (1, 4, 16) if bs // px * k >= max(grid)})
    for tile in tiles:
        lockstep(*box(grid, "const", "minmond", magnet, seed=sum(grid)), tile=tile, iterations=2,
                 magnet=magnet)


@pytest.mark.parametrize("lo,hi", [("circ", "trans"), ("trans", "circ"), ("flip", "const"),
                                   ("zero", "flip"), ("mirror", "trans"), ("wall", "wall")])
def test_mixed_ends(lo, hi):
    m = [lo, hi]
    lockstep(*box((21, 18, 1), {"x": m, "y": m}, "vanleer", seed=3))
    lockstep(*box((7, 10, 6), {"x": m, "y": m, "z": m}, "minmond", seed=4), iterations=3)


def test_transparent_far_node():
    lockstep(*box((19, 14, 1), "trans", "vanleer", seed=6, inf=4))
    lockstep(*box((19, 14, 1), "trans", "vanleer", seed=6, inf=5))


@pytest.mark.parametrize("grid", [(7, 130, 1), (33, 65, 1), (17, 9, 12)])
@pytest.mark.parametrize("magnet", [False, True])
def test_fp32(grid, magnet):
    ini, st = box(grid, "trans" if not magnet else "circ", "vanleer", magnet, seed=8)
    a, b = make_gpu(ini, st), make_gpu(ini, st, "fp32")
    for _ in range(6):
        iteration(a)
        iteration(b)
    for f in FLUID_FIELDS:
        ref = a.download(f)
        if np.any(ref != 0):
            assert rel_l1(b.download(f), ref) <= 1e-5, f
    a.close()
    b.close()


@pytest.mark.parametrize("bc", ["circ", "trans", "wall", "mirror", ["const", "flip"], ["trans", "zero"]])
@pytest.mark.parametrize("magnet", [False, True])
def test_neumann_richtmyer(bc, magnet):
    """The viscosity's shifted momentum at chunk ends, and its upper ghost in every mode;
    pencils whose last chunk holds one to four cells."""
    for n, tile in [(3, None), (9, (256, 4, 16)), (10, (256, 4, 8)), (23, (256, 2, 4)), (259, None)]:
        ini, st = box((n, 5, 1) if n > 100 else (n, 6, 4), {"x": bc, "y": bc, "z": bc}, "vanleer",
                      magnet, seed=n)
        orc, run = make_oracle(ini, st), make_gpu(ini, st)
        orc.set_viscosity("neumann_richtmyer", 0.2, 0.4)
        run.set_viscosity("neumann_richtmyer", 0.2, 0.4)
        if tile:
            run.set_fluid_tile(1, *tile)
        for _ in range(3):
            orc.iteration()
            iteration(run)
            compare(run, orc, FLUID_FIELDS + (MAG_FIELDS if magnet else []), TOL)
        run.close()
        orc.close()
