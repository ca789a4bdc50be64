"""Direct magnetFlux calls after iterations (the flux objects have their edge stores, so that
the lean form is open to them): components in either order, and one component named twice,
whose second advection starts from the first's result.  Against the oracle at <= 1e-12
relative L-inf (expected 0)."""
import pytest

import imogen_amd
from imogen_amd import iteration, problems

from .helpers import FLUID_FIELDS, MAG_FIELDS, compare, make_gpu, make_oracle

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("pair", [(0, 1), (1, 0), (0, 0), (1, 1)])
@pytest.mark.parametrize("bc", ["circ", "trans"])
@pytest.mark.parametrize("grid", [(33, 18, 1), (12, 16, 9), (300, 1, 1)])
def test_component_orders(grid, bc, pair):
    h = 1.0 / max(grid)
    ini = {"grid": grid, "dGrid": (h, h, h), "gamma": 5.0 / 3.0, "cfl": 0.3, "bcMode": bc,
           "bcInfinity": 20, "fluxLimiter": "vanleer", "minMass": 1e-5,
           "mode": {"fluid": True, "magnet": True}, "iterMax": 100, "timeMax": 1e9}
    st = problems.random_state(grid, seed=sum(grid), magnet=True)
    orc, run = make_oracle(ini, st), make_gpu(ini, st)
    mass, mom, ener, mag = run._arrays
    for _ in range(2):
        orc.iteration()
        iteration(run)
    for X in (1, 2, 3):
        if grid[X - 1] < 3:
            continue
        others = [i for i in (1, 2, 3) if i != X]
        I2 = [others[k] for k in pair]
        for _ in range(2):
            orc.magnet_flux(X, I2)
            imogen_amd.magnetFlux(run, mass, mom, mag, X, I2)
            compare(run, orc, FLUID_FIELDS + MAG_FIELDS, 1e-12)
    orc.iteration()
    iteration(run)
    compare(run, orc, FLUID_FIELDS + MAG_FIELDS, 1e-12)
    run.close()
    orc.close()
