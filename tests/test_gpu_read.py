"""Field reads at the edges of the chunks in which they cross to the host
(512 KiB through four pinned slots): one chunk, one byte range more, one more
than the four slots.  The positions of a handle that has not stepped are its
inputs; after a step in a shuffled id order they are those of the same set
in another handle with the ids in order, and the pressure is k (rho - rho0)
of the density, all bit for bit."""
import numpy as np
import pytest

import cudasphnew_amd as S
from cudasphnew_amd import Field
from tests.helpers import lattice_positions

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [1, 43690, 43691, 174763])
def test_reads_across_chunks(n):
    base = S.make_scene("dam16k")
    rng = np.random.default_rng(n)
    m = int(np.ceil(n ** (1.0 / 3.0)))
    pos = lattice_positions((m, m, m), 0.5 / m, (0.07, 0.07, 0.07))[:n]
    pos = (pos + rng.uniform(-1e-4, 1e-4, pos.shape)).astype(np.float32)
    order = rng.permutation(n)
    a = S.ParticleSimulation(base.with_positions(pos)).Init()
    assert np.array_equal(a.positions(), pos)
    b = S.ParticleSimulation(base.with_positions(pos[order])).Init()
    for sim in (a, b):
        p = sim.get_params()
        p.gas_stiffness = 0.0     # no pressure or viscosity: sums over neighbours in
        p.dynamic_viscosity = 0.0   # another order leave the motion as it is
        p.tension_coefficient = 0.0
        sim.set_params(p)
        sim.Advance(1)
    for f in (Field.POSITION, Field.VELOCITY, Field.ACCEL):
        assert np.array_equal(b.read(f), a.read(f)[order]), f
    rho, p = b.read(Field.DENSITY), b.get_params()
    q = b.get_params()
    q.gas_stiffness = 3.0
    b.set_params(q)
    assert np.array_equal(b.read(Field.PRESSURE), np.float32(3.0) * (rho - np.float32(p.rest_density)))
    with pytest.raises(S.SphError):
        S.simulation.check(S.lib.sph_read_field(b._h, int(Field.DENSITY), rho.ctypes.data, rho.nbytes - 4), b._h)
