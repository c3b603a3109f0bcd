"""A field read that is refused (the sub-particle capacity was exceeded)
reports it and leaves the caller's array as it was, over one chunk of the
transfer and over several."""
import numpy as np
import pytest

import cudasphnew_amd as S
from cudasphnew_amd import Field
from tests.helpers import lattice_positions

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("m", [20, 40])   # 96 KB and 768 KB of positions
def test_refused_read_writes_nothing(m):
    base = S.make_scene("dam16k")
    sc = base.with_positions(lattice_positions((m, m, m), 0.008, (0.08, 0.08, 0.08)).astype(np.float32))
    for a in range(3):
        sc.params.split_lo[a], sc.params.split_hi[a] = 0.0, 0.6      # every parent splits
    sc.params.max_sub_particles = 64
    sim = S.ParticleSimulation(sc).Init()
    sim.AdvanceTwoScale(1)
    for f, shape in ((Field.POSITION, (sc.n, 3)), (Field.DENSITY, (sc.n,))):
        out = np.full(shape, -7.0, np.float32)
        st = S.lib.sph_read_field(sim._h, int(f), out.ctypes.data, out.nbytes)
        assert st == S.Status.CAPACITY_EXCEEDED
        assert (out == -7.0).all(), f
