"""The default variants of one scene past the team kernels' sizes run as the
masks pair with the one-lane loops' sums (csrc/kernels.hip, PLAIN): bit for bit
what the loops give the same scene in a batch.

Sizes at the line (28,672 particles run in teams) and a ragged one; blocks at
rest density, 2.2 and 12 times (rows of more than 32 and more than 128
candidates), with coincident particles, touching the walls."""
import numpy as np
import pytest

import cudasphnew_amd as S
from cudasphnew_amd import Field
from tests.helpers import lattice_positions

pytestmark = pytest.mark.gpu

FIELDS = (Field.POSITION, Field.VELOCITY, Field.DENSITY, Field.ACCEL, Field.SORTED_IDS)


@pytest.mark.parametrize("n,crowd", [(28672, 1.0), (28673, 1.0), (45001, 2.2), (45000, 12.0)])
def test_alone_equals_batch(n, crowd):
    base = S.make_scene("dam16k")
    rng = np.random.default_rng(n)
    m = int(np.ceil(n ** (1.0 / 3.0)))
    sp = 0.01 * crowd ** (-1.0 / 3.0)
    pos = lattice_positions((m, m, m), sp, (0.004, 0.004, 0.03))[:n] + rng.uniform(-0.1 * sp, 0.1 * sp, (n, 3))
    pos = pos[rng.permutation(n)].astype(np.float32)
    pos[n // 2] = pos[n // 3]
    sc = base.with_positions(pos, (0.5 * rng.standard_normal((n, 3))).astype(np.float32))
    big = base.with_positions(lattice_positions((40, 40, 40), 0.01, (0.08, 0.08, 0.08)).astype(np.float32))
    alone, batch = S.ParticleSimulation(sc).Init(), S.Batch([big, sc])
    for step in range(2):
        alone.Advance(1)
        batch.step(1)
        for f in FIELDS:
            assert np.array_equal(alone.read(f), batch.read(1, f)), (step, f)
