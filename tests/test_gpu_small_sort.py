"""The one-workgroup cell sort of small particle sets (csrc/small_sort.hip),
all exact: keys, ids and cell ranges against the oracle's sort on the first
step and after a step, and the step without a handle against sph_step.

Sizes around the workgroup (1,024 threads of four particles each) and its
upper line (4,097: the counting sort); grids with an odd number of cells, at
the most cells the kernel holds (48,128) and above; crowded cells."""
import ctypes as C

import numpy as np
import pytest

import cudasphnew_amd as S
from cudasphnew_amd import Field
from tests.helpers import lattice_positions
from tests.test_gpu_parity import _check_sort
from tests.test_zz_no_alloc import DevBuf, _handle, _hip, _noalloc

pytestmark = pytest.mark.gpu

SIZES = [(1, 1.0), (63, 1.0), (1023, 1.0), (1025, 1.0), (4095, 1.0), (4096, 1.0), (4097, 1.0), (3000, 30.0)]
GRIDS = [None, (35, 33, 31), (47, 32, 32), (33, 27, 55)]   # 46,656, 35,805, 48,128 and 49,005 cells


def _scene(n, crowd, grid=None):
    base = S.make_scene("dam16k")
    if grid:
        for a in range(3):
            base.params.grid_dim[a] = grid[a]
    rng = np.random.default_rng(n)
    m = int(np.ceil(n ** (1.0 / 3.0)))
    sp = 0.01 * crowd ** (-1.0 / 3.0)
    pos = lattice_positions((m, m, m), sp, (0.02, 0.02, 0.02))[:n] + rng.uniform(-0.1 * sp, 0.1 * sp, (n, 3))
    return base.with_positions(pos[rng.permutation(n)].astype(np.float32))


@pytest.mark.parametrize("grid", GRIDS)
@pytest.mark.parametrize("n,crowd", SIZES)
def test_sort_of_a_small_set(n, crowd, grid):
    sc = _scene(n, crowd, grid)
    sim = S.ParticleSimulation(sc).Init()
    pos = sc.positions
    for _ in range(2):
        sim.Advance(1)
        _check_sort(sc.params, pos, sim)
        pos = sim.positions()
    sim.close()


@pytest.mark.parametrize("steps", [1, 3])
@pytest.mark.parametrize("n,crowd", SIZES)
def test_step_without_a_handle(n, crowd, steps):
    hip, stream = _hip(), C.c_void_p()
    assert hip.hipStreamCreate(C.byref(stream)) == 0
    flags = DevBuf(hip, np.ones(1, np.uint32))
    sc = _scene(n, crowd)
    pos, vel = _noalloc(sc, steps, hip, stream, flags)
    x, v, rho = _handle(sc, steps)
    assert np.array_equal(pos[:, :3], x) and np.array_equal(vel[:, :3], v)
    assert np.array_equal(pos[:, 3], rho) and np.array_equal(vel[:, 3], rho)
    assert int(flags.get(np.zeros(1, np.uint32))[0]) == 0
    flags.free()
    hip.hipStreamDestroy(stream)


def test_a_particle_outside_the_domain_is_flagged():
    hip, stream = _hip(), C.c_void_p()
    assert hip.hipStreamCreate(C.byref(stream)) == 0
    flags = DevBuf(hip, np.zeros(1, np.uint32))
    sc = _scene(700, 1.0)
    far = sc.positions.copy()
    far[333] = (-5.0, 0.1, 0.1)
    _noalloc(sc.with_positions(far), 1, hip, stream, flags)
    assert int(flags.get(np.zeros(1, np.uint32))[0]) != 0
    flags.free()
    hip.hipStreamDestroy(stream)
