"""The sixteen-lanes-per-particle kernels of small particle sets
(csrc/team.hip) against the one-thread kernels they stand in for: the same
scene alone (teams) and in a batch too large for teams gives the same
positions, velocities, densities and accelerations bit for bit.

Sizes at the edges of a team's workgroup (16 particles); blocks at rest
density (rows of up to 32 candidates, the fast path), at 2.2 times (longer
rows) and 12 times (more than 288 candidates within reach: the list is summed
in parts), touching the walls so that penalty, viscosity and collision act."""
import numpy as np
import pytest

import cudasphnew_amd as S
from cudasphnew_amd import Field
from tests.helpers import lattice_positions

pytestmark = pytest.mark.gpu

FIELDS = (Field.POSITION, Field.VELOCITY, Field.DENSITY, Field.ACCEL, Field.SORTED_IDS)


@pytest.fixture(scope="module")
def scenes():
    base = S.make_scene("dam16k")
    big = base.with_positions(lattice_positions((40, 40, 40), 0.01, (0.08, 0.08, 0.08)).astype(np.float32))
    return base, big


def _block(base, n, crowd):
    rng = np.random.default_rng(n)
    m = int(np.ceil(n ** (1.0 / 3.0)))
    sp = 0.01 * crowd ** (-1.0 / 3.0)
    pos = lattice_positions((m, m, m), sp, (0.004, 0.004, 0.03))[:n] + rng.uniform(-0.1 * sp, 0.1 * sp, (n, 3))
    vel = 0.5 * rng.standard_normal((n, 3))
    order = rng.permutation(n)
    return base.with_positions(pos[order].astype(np.float32), vel[order].astype(np.float32))


@pytest.mark.parametrize("masks", [0, 1])
@pytest.mark.parametrize("n,crowd", [(1, 1.0), (15, 1.0), (17, 1.0), (700, 1.0), (6000, 1.0), (700, 2.2), (6000, 2.2),
                                     (3000, 12.0)])
def test_small_set_alone_equals_large_batch(scenes, n, crowd, masks):
    base, big = scenes
    small = _block(base, n, crowd)
    alone, batch = S.ParticleSimulation(small).Init(), S.Batch([big, small])
    if masks:
        alone.set_tuning(hit_masks=1, hit_list=48)
        batch.set_tuning(hit_masks=1, hit_list=48)
    for step in range(2):
        alone.Advance(1)
        batch.step(1)
        for f in FIELDS:
            assert np.array_equal(alone.read(f), batch.read(1, f)), (step, f)
