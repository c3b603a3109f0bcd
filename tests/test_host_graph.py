"""Step graphs: one capture of one step when a handle's graphs start and after
each change of what its step launches; longer ones once it has settled, or for
a call that is long itself.  On the CPU, on a fake runtime (fake_hip.cpp)."""
import pytest

from tests import fake_hip

_SIM = """
        x = np.random.default_rng(0).uniform(0.1, 0.5, (2000, 3)).astype(np.float32)
        sim = S.ParticleSimulation(S.make_scene("dam16k").with_positions(x)).Init()
        sim.use_graph(True)
        def advance(n):
            a = count("capture"), count("replay"), count("captured"), sim.GetNumTimesSteps()
            sim.Advance(n)
            assert sim.GetNumTimesSteps() - a[3] == n
            return count("capture") - a[0], count("replay") - a[1], count("captured") - a[2]
"""


@pytest.fixture(scope="module")
def fake(tmp_path_factory):
    return fake_hip.build(tmp_path_factory.mktemp("fake_hip"))


def test_first_calls_capture_one_step_once(fake):
    fake_hip.run(fake, _SIM + """
        sim.enable_timing(False)
        k0 = count("kernels"); sim.Advance(1); per_step = count("kernels") - k0 - 1   # without the first keys
        assert advance(3) == (1, 3, per_step)
        assert advance(4) == (0, 4, 0)
        assert advance(4)[0] <= 1
        for _ in range(3):
            advance(4)
        assert advance(4) == (0, 1, 0)          # settled: one graph of four steps
        assert advance(7)[1] == 3 and advance(7) == (0, 3, 0)
    """)


def test_a_long_call_builds_the_longest_at_once(fake):
    fake_hip.run(fake, _SIM + """
        sim.Advance(1)
        assert advance(18)[:2] == (2, 6)        # four of four steps, two of one
        assert advance(16) == (0, 4, 0)
    """)


def test_changes_between_frames_capture_one_step_each(fake):
    fake_hip.run(fake, _SIM + """
        advance(4)
        for _ in range(12):
            sim.set_params(sim.get_params())
            assert advance(4)[:2] == (1, 4)
    """)


@pytest.mark.parametrize("interval", [16, 17, 18, 19])
def test_no_graph_runs_over_a_retuning(fake, interval):
    fake_hip.run(fake, _SIM + f"""
        sim.set_autotune_interval({interval})
        sim.Advance({interval} + 1)                          # retuned before the last of them
        for _ in range(4):
            assert sim.GetNumTimesSteps() % {interval} == 1
            sim.set_tuning(density_lanes=2, force_lanes=16)  # not what the fake's equal times pick
            sim.Advance({interval} - 3)                      # settled, two steps before the next one
            sim.Advance(1)
            assert sim.get_tuning()["hit_masks"] == 0
            sim.Advance(2)                                   # the step before it, and the retuned one
            assert sim.get_tuning()["hit_masks"] == 1
            sim.Advance({interval} - sim.GetNumTimesSteps() % {interval} + 1)
            sim.set_tuning(density_lanes=2, force_lanes=16)
            sim.Advance({interval} - 6)
            sim.Advance(10)                                  # one call over the next one
            assert sim.get_tuning()["hit_masks"] == 1
            sim.Advance({interval} - sim.GetNumTimesSteps() % {interval} + 1)
    """)
