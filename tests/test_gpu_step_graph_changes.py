"""Step graphs past the team kernels' sizes, and parameters and variants changed
between calls of different lengths: each call gives the eager steps' results
bit for bit, before and after the handle's graphs of two and four steps are
built, with reads and eager work in between."""
import numpy as np
import pytest

import cudasphnew_amd as S
from cudasphnew_amd import Field
from tests.helpers import lattice_positions

pytestmark = pytest.mark.gpu

FIELDS = (Field.POSITION, Field.VELOCITY, Field.DENSITY, Field.SORTED_IDS)


def _pair(n, masks):
    m = int(np.ceil(n ** (1.0 / 3.0)))
    pos = lattice_positions((m, m, m), 0.01, (0.08, 0.08, 0.08))[:n].astype(np.float32)
    sc = S.make_scene("dam16k").with_positions(pos)
    sims = [S.ParticleSimulation(sc).Init() for _ in range(2)]
    for sim in sims:
        sim.set_tuning(hit_masks=masks)
    sims[1].use_graph(True)
    return sims


def _same(sims, what):
    for f in FIELDS:
        a, b = (sim.read(f) for sim in sims)
        assert np.array_equal(a, b), (what, f)


@pytest.mark.parametrize("masks", [0, 1])
@pytest.mark.parametrize("n", [1000, 16384, 30011])
def test_parameters_change_between_calls(n, masks):
    sims = _pair(n, masks)
    for round_, gravity in enumerate((9.81, 4.0, 12.0, 0.0)):
        for sim in sims:
            p = sim.get_params()
            p.gravity = gravity
            sim.set_params(p)
        for steps in (1, 2, 4, 7) if round_ < 3 else (4, 4, 4, 7, 2, 4, 1):
            for sim in sims:
                sim.Advance(steps)
            _same(sims, (round_, steps))


@pytest.mark.parametrize("masks", [0, 1])
def test_variants_and_two_scale_between_calls(masks):
    sims = _pair(30011, masks)
    for sim in sims:
        sim.Advance(14)
    _same(sims, "settled")
    for change in (dict(density_lanes=4, force_lanes=8), dict(hit_masks=masks), "two-scale", "two-scale"):
        for sim in sims:
            if change == "two-scale":
                sim.AdvanceTwoScale(1)
            else:
                sim.set_tuning(**change)
        for steps in (4, 7, 4):
            for sim in sims:
                sim.Advance(steps)
        _same(sims, change)
