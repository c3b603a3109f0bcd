"""The neighbour masks that stand in for the one-lane loops of a larger scene
are memory of the handles that read them only.  On the CPU, on a fake runtime
(fake_hip.cpp)."""
import pytest

from tests import fake_hip

_SIM = """
        N, MASKS = 50000, 180 * 50000
        x = np.random.default_rng(0).uniform(0.1, 0.5, (N, 3)).astype(np.float32)
        scene = S.make_scene("dam16k").with_positions(x)
        plain = lambda: launches("k_force_masksILi48ELi256ELb1ELb1EE")
        loops = lambda: launches("k_forceILi256ELb1EE")
        def held():
            assert abs(count("bytes") - base - (sim.GetSizeMemoryGPU() - size)) < 64
            return round((count("bytes") - base) / MASKS, 3)
"""


@pytest.fixture(scope="module")
def fake(tmp_path_factory):
    return fake_hip.build(tmp_path_factory.mktemp("fake_hip"))


def test_masks_follow_the_variants(fake):
    fake_hip.run(fake, _SIM + """
        sim = S.ParticleSimulation(scene).Init()
        base, size = count("bytes") - MASKS, sim.GetSizeMemoryGPU() - MASKS
        sim.use_graph(True)
        sim.Advance(3)
        assert plain() > 0 and held() == 1
        sim.set_tuning(density_lanes=4, force_lanes=8)      # variants that never read them
        assert held() == 0
        sim.Advance(3)
        assert launches("k_force_coop") > 0 and held() == 0
        sim.set_tuning()
        n = plain()
        sim.Advance(3)
        assert plain() > n and held() == 1 and loops() == 0
        sim.set_tuning(hit_masks=1)
        sim.set_tuning(density_lanes=4)                     # asked for: kept, as ever
        assert held() == 1
        sim.close()
        assert count("bytes") == 0 and count("bad free") == 0
    """)


def test_two_scale_handles_hold_none(fake):
    fake_hip.run(fake, _SIM + """
        sim = S.ParticleSimulation(scene).Init()
        total = sim.GetSizeMemoryGPU()
        sim.AdvanceTwoScale(1)
        two = sim.GetSizeMemoryGPU()
        sim.AdvanceTwoScale(3)
        assert sim.GetSizeMemoryGPU() == two and plain() == 0
        sim.Advance(1)                                      # a plain step takes them again
        assert sim.GetSizeMemoryGPU() == two + MASKS and plain() == 1
        sim.AdvanceTwoScale(1)
        sim.Advance(1)
        assert sim.GetSizeMemoryGPU() == two + MASKS and plain() == 2
        sim.close()
        assert count("bytes") == 0
        # the two-scale buffers alone, from a handle that reads no masks
        sim = S.ParticleSimulation(scene).Init()
        sim.set_tuning(density_lanes=2)
        a = sim.GetSizeMemoryGPU()
        assert a == total - MASKS
        sim.AdvanceTwoScale(1)
        assert sim.GetSizeMemoryGPU() - a == two - a
    """)


@pytest.mark.parametrize("how", ["fake.fake_free_bytes(MASKS * 7)", "fake.fake_fail(b'hipMalloc', 0)"])
def test_without_memory_for_them_the_loops_run(fake, how):
    fake_hip.run(fake, _SIM + f"""
        sim = S.ParticleSimulation(scene).Init()
        sim.set_tuning(density_lanes=4)
        {how}
        sim.set_tuning()
        sim.Advance(2)
        assert loops() == 2 and plain() == 0
        fake.fake_free_bytes(1 << 38)
        fake.fake_work(b"hipMalloc")
        sim.set_tuning()
        sim.Advance(1)
        assert loops() == 2 and plain() == 1
    """)
