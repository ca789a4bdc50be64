"""A magnetic simulation whose second scratch field is past the serving budget runs on one (the
general magnetic sweep), with the result of the same run alone: <= 1e-12 relative L-inf."""
import ctypes

import pytest

from imogen_amd import _lib, problems
from imogen_amd.config import from_ini
from imogen_amd.imogen import make_imh_config
from imogen_amd.serve import DONE, Server

from .helpers import FLUID_FIELDS, MAG_FIELDS, make_gpu, rel_linf

pytestmark = pytest.mark.gpu


def estimate(ini, precision):
    b = ctypes.c_size_t()
    _lib.check(_lib.lib().imh_memory_estimate(
        ctypes.byref(make_imh_config(from_ini(ini), precision)), ctypes.byref(b)))
    return b.value


@pytest.mark.parametrize("second", [False, True])
def test_budget_of_one_scratch_field(second):
    """Alone under the budget, and as the second of two that fit only so."""
    ini, st = problems.orszag_tang(48)
    ini = dict(ini, iterMax=10)
    full = estimate(ini, _lib.FP64)
    least = full - 48 * 48 * 8
    srv = Server("fp64", hbm_budget=full + least if second else least, max_active=4)
    ids = [srv.submit(ini, st) for _ in range(2 if second else 1)]
    running, queued = srv.step(2)
    assert (running, queued) == (len(ids), 0)
    assert srv.stats()["used_bytes"] == (full + least if second else least)
    for _ in range(20):
        if srv.step(4) == (0, 0):
            break
    run = make_gpu(ini, st)
    run.run_iterations(100)
    for rid in ids:
        assert srv.status(rid)[0] == DONE
        for f in FLUID_FIELDS + MAG_FIELDS:
            assert rel_linf(srv.download(rid, f), run.download(f)) <= 1e-12, f
        srv.release(rid)
    # the contexts go back to the pool and serve the next requests, each with its scratch
    again = [srv.submit(ini, st) for _ in ids]
    for _ in range(20):
        if srv.step(4) == (0, 0):
            break
    for rid in again:
        assert srv.status(rid)[0] == DONE
        assert rel_linf(srv.download(rid, "mass"), run.download("mass")) <= 1e-12
        srv.release(rid)
    assert srv.stats()["used_bytes"] == 0
    srv.close()
    run.close()
