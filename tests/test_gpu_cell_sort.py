"""The counting sort's block totals (csrc/cell_sort.hip) on a key space wider
than the window of blocks a workgroup adds up in LDS (1,024 of 4,096 cells):
keys, ids and cell ranges equal the oracle's, from shuffled particles (of
the wider grid some outside the window) and from the sorted ones of the next step."""
import numpy as np
import pytest

import cudasphnew_amd as S
from tests.test_gpu_parity import _check_sort

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("grid,n", [((200, 200, 40), 101001), ((170, 160, 160), 280000)])   # 391, 1,063 blocks
def test_wide_key_space(grid, n):
    base = S.make_scene("dam16k")
    p = base.params
    for a in range(3):
        p.grid_dim[a] = grid[a]
    rng = np.random.default_rng(n)
    lo = np.array([p.grid_origin[a] for a in range(3)])
    ext = np.array([grid[a] * p.grid_spacing for a in range(3)])
    sc = base.with_positions((lo + ext * rng.uniform(0.01, 0.99, (n, 3))).astype(np.float32))
    sim = S.ParticleSimulation(sc).Init()
    pos = sc.positions
    for _ in range(2):
        sim.Advance(1)
        _check_sort(sc.params, pos, sim)
        pos = sim.positions()
    sim.close()
