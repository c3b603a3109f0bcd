"""Step graphs of one, two and four steps: calls of every remainder replay them
between eager work and give the eager steps' results bit for bit, also with an
autotune interval that cuts the calls."""
import numpy as np
import pytest

import cudasphnew_amd as S
from cudasphnew_amd import Field

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("masks", [0, 1])
@pytest.mark.parametrize("n", [1000, 16384])
def test_calls_of_every_remainder(n, masks):
    base = S.make_scene("dam16k")
    sc = base.with_positions(base.positions[:n].copy())
    eager, graph = S.ParticleSimulation(sc).Init(), S.ParticleSimulation(sc).Init()
    for sim in (eager, graph):
        sim.set_tuning(hit_masks=masks)
    graph.use_graph(True)
    for steps in (1, 2, 3, 4, 7, 1, 9, 6):
        eager.Advance(steps)
        graph.Advance(steps)
        for f in (Field.POSITION, Field.VELOCITY, Field.DENSITY, Field.SORTED_IDS):
            assert np.array_equal(graph.read(f), eager.read(f)), (steps, f)


def test_autotune_interval_is_kept():
    sc = S.make_scene("dam16k")
    sim, one = S.ParticleSimulation(sc).Init(), S.ParticleSimulation(sc).Init()
    for s in (sim, one):
        s.use_graph(True)
        s.set_autotune_interval(3)
    sim.Advance(11)
    for _ in range(11):
        one.Advance(1)
    sim.sync()
    one.sync()
    # the variants differ in summation order only
    assert np.allclose(sim.read(Field.DENSITY), one.read(Field.DENSITY), rtol=1e-5)
