"""The tile autotuner tries every tile that its rule names (on the CPU, with an ensemble that
records the tiles in place of one that runs them)."""
import pytest

from imogen_amd import autotune, problems


class Recorder:
    tiles = []

    def __init__(self, sims, precision):
        self.fused = True  # 1-D MHD simulations: one launch, no fluid sweeps

    def set_fused_1d(self, enable):
        self.fused = bool(enable)

    def step(self, n):
        pass

    def set_fluid_tile(self, i, X, bs, k, px):
        if i == 0:
            self.tiles.append((X, (bs, k, px)))

    def profile_step(self, n):
        return {"fluid": (0.0, 0.0, 0) if self.fused else (1.0, 0.0, 1)}

    def close(self):
        pass


@pytest.mark.parametrize("precision", ["fp64", "fp32"])
@pytest.mark.parametrize("n", [64, 128, 256, 512])
def test_every_candidate_is_timed(monkeypatch, precision, n):
    monkeypatch.setattr(autotune, "Ensemble", Recorder)
    monkeypatch.setattr(Recorder, "tiles", [])
    ini, st = problems.kelvin_helmholtz(4)
    ini = problems.resize(ini, (n, n, 1))
    autotune.tune([(ini, st)], precision)
    for X in (1, 2):
        want = autotune.candidates(n, 8 if precision == "fp64" else 4, X == 2, n)
        assert [t for x, t in Recorder.tiles if x == X] == want
    assert (2, (0, 0, 0)) in Recorder.tiles  # the column march along y


def test_candidates_take_the_lean_sweep():
    """No more pencils per tile than the lean sweep holds (LEAN_PXMAX)."""
    for esz in (4, 8):
        for n in (8, 16, 64, 200, 4096):
            assert all(px <= 16 for bs, k, px in autotune.candidates(n, esz, True, 1 << 20))


def test_one_dimensional_sweeps_are_timed(monkeypatch):
    """1-D MHD simulations run in one launch per iteration, without the sweep that the tile is
    for; the tuner times that sweep."""
    monkeypatch.setattr(autotune, "Ensemble", Recorder)
    table = autotune.tune([problems.mhd_riemann(300, seed=1)], "fp32")
    assert table and all(us > 0 for _, _, _, us in table.values())
