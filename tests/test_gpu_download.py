"""Fields of all sizes come back whole: below, at and past the staged copy's threshold, chunk
and ring (download.cpp), FP64 and FP32, from two threads at once."""
import threading

import numpy as np
import pytest

import imogen_amd
from imogen_amd import problems

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("prec", ["fp64", "fp32"])
@pytest.mark.parametrize("grid", [(5, 7, 1), (181, 181, 1), (256, 255, 1), (257, 256, 1),
                                  (1024, 577, 1), (131, 127, 71)])
def test_round_trip(grid, prec):
    st = problems.random_state(grid, seed=sum(grid), magnet=False)
    ini = {"grid": grid, "dGrid": (0.1, 0.1, 0.1), "gamma": 1.4, "cfl": 0.4,
           "bcMode": {"x": "circ", "y": "circ", "z": "circ"}, "bcInfinity": 20,
           "fluxLimiter": "vanleer", "minMass": 1e-5, "mode": {"fluid": True, "magnet": False},
           "iterMax": 10, "timeMax": 1.0}
    run = imogen_amd.initialize(ini, prec)
    imogen_amd.create_arrays(run, st)
    want = {"mass": st["mass"], "ener": st["ener"], "momx": st["mom"][0]}
    if prec == "fp32":
        want = {k: np.asarray(v).astype(np.float32).astype(np.float64) for k, v in want.items()}
    got = {}

    def fetch(k):
        got[k] = run.download(k)

    threads = [threading.Thread(target=fetch, args=(k,)) for k in want]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    for k, v in want.items():
        np.testing.assert_array_equal(got[k].reshape(-1), np.asarray(v).reshape(-1), err_msg=k)
    run.close()
