"""The memory that field reads take and what they do without it, on the CPU on
a fake runtime (fake_hip.cpp)."""
import pytest

from tests import fake_hip


@pytest.fixture(scope="module")
def fake(tmp_path_factory):
    return fake_hip.build(tmp_path_factory.mktemp("fake_hip"))


def test_small_reads_take_one_pinned_slot(fake):
    fake_hip.run(fake, """
        base = S.make_scene("dam16k")
        def sim_of(n):
            x = np.random.default_rng(n).uniform(0.1, 0.5, (n, 3)).astype(np.float32)
            return S.ParticleSimulation(base.with_positions(x)).Init(), x
        sim, x = sim_of(43690)                      # 512 KiB - 8
        events = count("event")
        assert np.array_equal(sim.positions(), x)
        sim.read(Field.DENSITY)
        assert count("pinned bytes") < (1 << 19) + 4096 and count("event") == events
        big, y = sim_of(43691)
        big.read(Field.DENSITY)                     # one slot, then all of them
        assert np.array_equal(big.positions(), y)
        big.read(Field.DENSITY)
        assert count("pinned bytes") < 5 * (1 << 19) + 8192
        sim.close(), big.close()
        assert count("pinned bytes") == 0
    """)
