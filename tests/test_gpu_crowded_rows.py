"""Default variants of one scene compressed until rows hold more than 128
candidates: the masks pair with the one-lane loops' sums (csrc/kernels.hip,
PLAIN) gives what the loops give the same scene in a batch, bit for bit, and
takes no longer than they do (about 1.3 times as long when it tested the
candidates of such particles one by one; 0.8 to 1.0 times since)."""
import numpy as np
import pytest

import cudasphnew_amd as S
from cudasphnew_amd import Field
from tests.helpers import lattice_positions

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("crowd", [4.0, 10.0])
def test_long_rows_like_the_loops(crowd):
    base = S.make_scene("dam16k")
    rng = np.random.default_rng(int(crowd))
    n, sp = 120000, 0.01 * crowd ** (-1.0 / 3.0)
    pos = lattice_positions((50, 48, 50), sp, (0.08, 0.08, 0.08)) + rng.uniform(-0.1 * sp, 0.1 * sp, (n, 3))
    sc = base.with_positions(pos.astype(np.float32))
    sc.params.time_step = 1e-7      # the block stays as compressed as it is
    tiny = base.with_positions(base.positions[:64].copy())
    alone, loops = S.ParticleSimulation(sc).Init(), S.Batch([sc, tiny])
    for sim in (alone, loops):
        sim.time_steps(3)
    start, end = alone.read(Field.CELL_START), alone.read(Field.CELL_END)
    count = np.where(start >= 0, end - start, 0)
    assert (count[:-2] + count[1:-1] + count[2:]).max() > 128
    t_alone, t_loops = (min(sim.time_steps(6) for _ in range(6)) for sim in (alone, loops))
    for f in (Field.POSITION, Field.VELOCITY, Field.DENSITY, Field.ACCEL, Field.SORTED_IDS):
        assert np.array_equal(alone.read(f), loops.read(0, f)), f
    assert t_alone < 1.12 * t_loops, (t_alone, t_loops)
