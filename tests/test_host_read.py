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


@pytest.mark.parametrize("call", ["hipMalloc", "hipHostMalloc"])
@pytest.mark.parametrize("n", [1000, 100000])
def test_reads_without_memory_for_staging(fake, call, n):
    fake_hip.run(fake, f"""
        base = S.make_scene("dam16k")
        rng = np.random.default_rng(1)
        x = rng.uniform(0.1, 0.5, ({n}, 3)).astype(np.float32)
        v = rng.standard_normal(({n}, 3)).astype(np.float32)
        sim = S.ParticleSimulation(base.with_positions(x, v)).Init()
        fake.fake_fail(b"{call}", 0)
        # the densities of a handle that has not stepped are the 0 it was made with
        rho0 = np.float32(sim.get_params().rest_density)
        k = np.float32(sim.get_params().gas_stiffness)
        assert np.array_equal(sim.positions(), x)
        if "{call}" == "hipMalloc":
            assert np.array_equal(sim.read(Field.VELOCITY), v)
            assert not sim.read(Field.DENSITY).any()
            assert (sim.read(Field.PRESSURE) == k * (np.float32(0.0) - rho0)).all()
        fake.fake_work(b"{call}")
        assert np.array_equal(sim.positions(), x)
        assert np.array_equal(sim.read(Field.VELOCITY), v)
    """)


def test_evaluation_without_pinned_memory(fake):
    fake_hip.run(fake, """
        net = S.NeuralSDF([0.0] * 3, [1.0] * 3, seed=1, out_scale=0.5)
        fake.fake_fail(b"hipHostMalloc", 0)
        net.eval(np.zeros((100003, 3), np.float32))
        assert count("kernel k_mlp_eval") == 1
    """)
