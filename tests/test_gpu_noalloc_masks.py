"""The step without a handle on sets past the team kernels' sizes, where the
masks pair stands in for the one-lane kernels (csrc/kernels.hip, PLAIN): bit
for bit sph_step's default variants.

Sizes at the line (28,672 particles run in teams), a ragged one and the
largest; blocks at rest density, 2.2, 4 and 12 times (rows of more than 32 and
more than 128 candidates), with coincident particles.  A set with a non-finite
velocity beside a coincident particle leaves its neighbours what the team
kernels leave them."""
import ctypes as C

import numpy as np
import pytest

import cudasphnew_amd as S
from tests.helpers import lattice_positions
from tests.test_zz_no_alloc import DevBuf, _device_boundary, _handle, _hip, _noalloc
from cudasphnew_amd import _native as N

pytestmark = pytest.mark.gpu


def _block(n, crowd, origin=(0.02, 0.02, 0.02)):
    rng = np.random.default_rng(n)
    m = int(np.ceil(n ** (1.0 / 3.0)))
    sp = 0.01 * crowd ** (-1.0 / 3.0)
    pos = lattice_positions((m, m, m), sp, origin)[:n] + rng.uniform(-0.1 * sp, 0.1 * sp, (n, 3))
    pos = pos[rng.permutation(n)].astype(np.float32)
    pos[n // 2] = pos[n // 3]
    return pos


@pytest.fixture
def hip_stream():
    hip, stream = _hip(), C.c_void_p()
    assert hip.hipStreamCreate(C.byref(stream)) == 0
    yield hip, stream
    hip.hipStreamDestroy(stream)


@pytest.mark.parametrize("n,crowd,steps", [(28672, 1.0, 1), (28673, 1.0, 2), (45001, 2.2, 2), (45000, 12.0, 2),
                                           (100003, 1.0, 1), (262144, 4.0, 3)])
def test_large_set_equals_handle(hip_stream, n, crowd, steps):
    hip, stream = hip_stream
    sc = S.make_scene("dam16k").with_positions(_block(n, crowd))
    pos, vel = _noalloc(sc, steps, hip, stream)
    x, v, rho = _handle(sc, steps)
    assert np.array_equal(pos[:, 3], rho)
    assert np.array_equal(pos[:, :3], x) and np.array_equal(vel[:, :3], v)


def test_non_finite_velocity_spreads_no_further(hip_stream):
    hip, stream = hip_stream
    small = _block(700, 1.0)
    both = np.concatenate([small, _block(30000, 1.0, (0.02, 0.02, 0.3))])
    out = []
    for p in (small, both):
        sc = S.make_scene("dam16k").with_positions(p)
        b, keep = _device_boundary(sc, hip)
        p4, v4 = np.zeros((len(p), 4), np.float32), np.zeros((len(p), 4), np.float32)
        p4[:, :3] = p
        v4[350, 0], v4[20, 1] = np.inf, np.nan
        pos, vel = DevBuf(hip, p4), DevBuf(hip, v4)
        assert N.lib.sph_step_noalloc(C.byref(sc.params), C.byref(b), len(p), pos.ptr, vel.ptr, 1, None, stream) == 0
        assert hip.hipStreamSynchronize(stream) == 0
        out.append((pos.get(p4)[:700], vel.get(v4)[:700]))
        for x in (pos, vel, *keep):
            x.free()
    assert np.isfinite(out[0][1]).all(1).sum() > 500
    for a, b in zip(*out):
        assert np.array_equal(a, b, equal_nan=True)
