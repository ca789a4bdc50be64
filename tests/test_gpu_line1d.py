"""The 1-D iteration kernel (line1d_variant.hip: many iterations per launch) against the
launches of one iteration at a time.

Both run the same bodies in the same order, so fields, time, dt and iteration agree bit for
bit: at pencil lengths around its chunk sizes (1, 2, 4 and 8 cells for each of 512 threads),
the shortest and the longest it takes; hydro, a magnetic field carried along and magnetic
sweeps; transparent, circular and wall ends; two time updates per iteration; more iterations
than one launch holds, and a run that ends within a launch.
"""
import numpy as np
import pytest

from imogen_amd import iteration, problems

from .helpers import FLUID_FIELDS, MAG_FIELDS, make_gpu

pytestmark = pytest.mark.gpu


def box(n, bc, magnet, **more):
    ini = {"grid": (n, 1, 1), "dGrid": (1.0 / n, 1.0 / n, 1.0 / n), "gamma": 1.4, "cfl": 0.4,
           "bcMode": {"x": bc, "y": "circ", "z": "circ"}, "bcInfinity": 20,
           "fluxLimiter": "vanleer", "minMass": 1e-5,
           "mode": {"fluid": True, "magnet": magnet}, "iterMax": 1000, "timeMax": 1e9}
    ini.update(more)
    return ini, problems.random_state((n, 1, 1), seed=n, magnet=magnet)


def agree(ini, st, prec, n, fields, calls=None):
    a, b = make_gpu(ini, st, prec), make_gpu(ini, st, prec)
    for k in calls or [n]:
        a.run_iterations(k)
    b.set_graphs(False)
    b.run_iterations(n)
    assert (a.time.time, a.time.dTime, a.time.iteration) == (b.time.time, b.time.dTime,
                                                             b.time.iteration)
    for f in fields:
        np.testing.assert_array_equal(a.download(f), b.download(f), err_msg=f)
    a.close()
    b.close()


@pytest.mark.parametrize("prec", ["fp64", "fp32"])
@pytest.mark.parametrize("magnet", [False, True])
@pytest.mark.parametrize("n", [3, 8, 257, 511, 513, 1024, 1500, 2049, 4096])
def test_lengths(n, magnet, prec):
    agree(*box(n, "trans", magnet), prec, 5, FLUID_FIELDS + (MAG_FIELDS if magnet else []))


@pytest.mark.parametrize("bc", ["circ", "wall", ["const", "mirror"], ["circ", "trans"]])
@pytest.mark.parametrize("magnet", [False, True])
def test_ends(bc, magnet):
    agree(*box(300, bc, magnet), "fp64", 6, FLUID_FIELDS + (MAG_FIELDS if magnet else []))


@pytest.mark.parametrize("prec", ["fp64", "fp32"])
def test_two_time_updates(prec):
    agree(*box(300, "trans", True, timeUpdateMode=0), prec, 6, FLUID_FIELDS + MAG_FIELDS)


def test_many_iterations_and_an_end():
    ini, st = problems.sod(257)
    agree(ini, st, "fp32", 150, FLUID_FIELDS, calls=[1, 70, 79])
    agree(dict(ini, timeMax=0.05), st, "fp64", 400, FLUID_FIELDS)
    agree(dict(ini, iterMax=40), st, "fp64", 200, FLUID_FIELDS)
