"""What a handle or network creates after its creation is created on its own
device, whatever the calling thread's current device is, and the thread's
current device is left as it was.  On the CPU, on a fake runtime of two
devices (fake_hip.cpp)."""
import pytest

from tests import fake_hip


@pytest.fixture(scope="module")
def fake(tmp_path_factory):
    return fake_hip.build(tmp_path_factory.mktemp("fake_hip"))


@pytest.mark.parametrize("n", [1000, 50000])
def test_reads_from_a_thread_on_another_device(fake, n):
    fake_hip.run(fake, f"""
        import threading
        base = S.make_scene("dam16k")
        x = np.random.default_rng(0).uniform(0.1, 0.5, ({n}, 3)).astype(np.float32)
        fake.fake_set_device(1)
        sim = S.ParticleSimulation(base.with_positions(x)).Init()
        b = S.Batch([base.with_positions(x), base])
        before = count("bytes@0")
        def reader():
            assert fake.fake_get_device() == 0
            for _ in range(2):
                assert np.array_equal(sim.positions(), x)
                assert np.array_equal(b.read(0, Field.POSITION), x)
                sim.read(Field.PRESSURE)
            assert fake.fake_get_device() == 0
            done.append(1)
        done = []
        t = threading.Thread(target=reader)
        t.start(); t.join()
        assert done
        assert count("bytes@0") == before, "a read took memory of another device"
        assert fake.fake_wrong_device() == 0
    """)


def test_everything_created_later_is_on_the_handles_device(fake):
    fake_hip.run(fake, """
        fake.fake_set_device(1)
        sim = S.ParticleSimulation(S.make_scene("dam16k")).Init()
        net = S.NeuralSDF([0.0] * 3, [1.0] * 3, seed=1, out_scale=0.5)
        fake.fake_set_device(0)
        before = count("bytes@0")
        sim.enable_timing(True)
        sim.Advance(1)
        sim.set_tuning(hit_masks=1)
        sim.map()
        sim.extract_surface()
        sim.AdvanceTwoScale(1)
        sim.time_steps(1)
        p = np.zeros((100003, 3), np.float32)
        net.eval(p)
        net.set_samples(np.zeros((128, 4), np.float32))
        net.train(2, 64)
        assert count("bytes@0") == before
        assert fake.fake_wrong_device() == 0 and fake.fake_get_device() == 0
    """)
