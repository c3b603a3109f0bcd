"""The hit-mask variants and the 128-thread loops on sets past the team kernels'
sizes (28,672 particles with masks, 40,960 in a batch without), where each hit
list and block size is a kernel of its own: squeezed blocks with rows of more
than 32 candidates, and of more than 128, against the FP64 oracle."""
import os

import numpy as np
import pytest

import cudasphnew_amd as S
from cudasphnew_amd import Field
from oracle import oracle as O

pytestmark = pytest.mark.gpu

THREADS = min(16, os.cpu_count() or 1)


def _block(nx, ny, nz, squeeze):
    base = S.make_scene("dam16k")
    rng = np.random.default_rng(11)
    sp = 0.01 / squeeze
    g = np.stack(np.meshgrid(np.arange(nx), np.arange(ny), np.arange(nz), indexing="ij"), -1).reshape(-1, 3)
    pos = 0.1 + g * sp + 0.05 * sp * rng.standard_normal(g.shape)
    return base.with_positions(rng.permutation(pos).astype(np.float32))


def _longest_row(read):
    start, end = read(Field.CELL_START), read(Field.CELL_END)
    c = np.where(start >= 0, end - start, 0)
    return int((c[:-2] + c[1:-1] + c[2:]).max())


def _check(read, orc, squeeze):
    longest = _longest_row(read)
    assert longest > (128 if squeeze > 1.7 else 32), longest
    assert np.max(np.abs(read(Field.DENSITY) / orc.read(Field.DENSITY) - 1)) <= 1e-5
    a, ao = read(Field.ACCEL), orc.read(Field.ACCEL)
    scale = np.maximum(np.linalg.norm(ao, axis=1), 9.81)[:, None]
    # particles at the surface-tension threshold may fall on either side of it
    off = (np.abs(a - ao) / scale).max(1) > 1e-4
    assert off.mean() <= 1e-3, off.sum()
    assert np.max(np.abs(read(Field.POSITION) - orc.read(Field.POSITION))) <= 1e-6


@pytest.fixture(scope="module")
def squeezed():
    out = {}
    for squeeze in (1.3, 1.9):
        sc = _block(32, 30, 32, squeeze)
        orc = O.OracleSim(sc, real=0, threads=THREADS)
        orc.step(1)
        out[squeeze] = (sc, orc)
    return out


@pytest.mark.parametrize("squeeze", [1.3, 1.9])
@pytest.mark.parametrize("block", [128, 256])
@pytest.mark.parametrize("hit_list", [32, 40, 48, 64])
def test_hit_lists_and_blocks(squeezed, squeeze, block, hit_list):
    sc, orc = squeezed[squeeze]
    assert sc.n > 28672
    sim = S.ParticleSimulation(sc).Init()
    sim.set_tuning(hit_masks=1, hit_list=hit_list, block=block)
    sim.Advance(1)
    _check(sim.read, orc, squeeze)


@pytest.mark.parametrize("squeeze", [1.3, 1.9])
def test_loops_of_both_block_sizes(squeeze):
    sc, tiny = _block(35, 34, 35, squeeze), _block(4, 4, 4, 1.0)
    assert sc.n > 40960
    orc = O.OracleSim(sc, real=0, threads=THREADS)
    orc.step(1)
    out = []
    for block in (256, 128):
        b = S.Batch([sc, tiny])
        b.set_tuning(block=block)
        b.step(1)
        _check(lambda f: b.read(0, f), orc, squeeze)
        out.append([b.read(0, f) for f in (Field.POSITION, Field.VELOCITY, Field.DENSITY, Field.ACCEL)])
    for x, y in zip(*out):
        assert np.array_equal(x, y)
