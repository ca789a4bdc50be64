"""Device memory of a context (imh_memory_estimate): two scratch fields for the magnetic sweeps
where the lean form can run, else one (no GPU call is made)."""
import ctypes

import pytest

from imogen_amd import _lib, config
from imogen_amd.imogen import make_imh_config


def estimate(grid, bc, magnet, precision=_lib.FP64):
    rc = config.RunConfig(grid=grid, dgrid=(1, 1, 1), bc=[[bc[0]] * 3, [bc[1]] * 3],
                          magnet_active=magnet)
    b = ctypes.c_size_t()
    _lib.check(_lib.lib().imh_memory_estimate(ctypes.byref(make_imh_config(rc, precision)),
                                              ctypes.byref(b)))
    return b.value


@pytest.mark.parametrize("precision,esz", [(_lib.FP64, 8), (_lib.FP32_BULK, 4)])
@pytest.mark.parametrize("grid,bc,fields", [
    ((40, 30, 24), ("circ", "circ"), 2), ((256, 1, 1), ("const", "flip"), 2),
    ((7, 40, 1), ("circ", "circ"), 2),
    # fade ends, ends of which one is circular, pencils below eight cells: the general form
    ((40, 30, 24), ("fade", "fade"), 1), ((40, 30, 24), ("circ", "const"), 1),
    ((7, 6, 5), ("circ", "circ"), 1)])
def test_scratch_fields(grid, bc, fields, precision, esz):
    n = grid[0] * grid[1] * grid[2]
    more = estimate(grid, bc, True, precision) - estimate(grid, bc, False, precision)
    assert more == fields * n * esz


def test_small_contexts_hold_no_tile_maxima():
    """A simulation of one CFL tile (4096 cells) keeps no maxima of tiles."""
    base = estimate((16, 16, 16), ("circ", "circ"), False) - 4096 * 8 * 11
    assert estimate((8, 8, 8), ("circ", "circ"), False) - 512 * 8 * 11 == base
    assert estimate((256, 256, 1), ("circ", "circ"), False) - 65536 * 8 * 11 == base + 3 * 64 * 8
