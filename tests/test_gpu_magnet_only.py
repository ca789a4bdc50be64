"""Runs whose flux objects are not all made by a first eager fluid sweep: the magnetic field alone
(fluid off), and a run after a direct fluid sweep.  Eighteen iterations, three times each captured
iteration order, against the oracle at <= 1e-12 relative L-inf; transparent ends, whose
edge stores a replayed first assignment would reset."""
import pytest

import imogen_amd
from imogen_amd import problems

from .helpers import FLUID_FIELDS, MAG_FIELDS, compare, make_gpu, make_oracle

pytestmark = pytest.mark.gpu


def case(grid, fluid):
    h = 1.0 / max(grid)
    ini = {"grid": grid, "dGrid": (h, h, h), "gamma": 5.0 / 3.0, "cfl": 0.3, "bcMode": "trans",
           "bcInfinity": 20, "fluxLimiter": "vanleer", "minMass": 1e-5,
           "mode": {"fluid": fluid, "magnet": True}, "iterMax": 100, "timeMax": 1e9}
    return ini, problems.random_state(grid, seed=sum(grid), magnet=True)


@pytest.mark.parametrize("grid", [(40, 1, 1), (24, 20, 1), (7, 12, 9)])
@pytest.mark.parametrize("fluid", [False, True])
def test_run(grid, fluid):
    ini, st = case(grid, fluid)
    orc, run = make_oracle(ini, st), make_gpu(ini, st)
    if fluid:
        mass, mom, ener, mag = run._arrays
        orc.dtime = run.time.dTime = 1e-3
        orc.relaxing_fluid(1)
        imogen_amd.relaxingFluid(run, mass, mom, ener, mag, None, 1)
    for n in (1, 6, 11):
        for _ in range(n):
            orc.iteration()
        run.run_iterations(n)
        compare(run, orc, FLUID_FIELDS + MAG_FIELDS, 1e-12)
    run.close()
    orc.close()
