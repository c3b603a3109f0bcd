"""The autotuner times the kernels that a step under its choice would run, and
each of them once.  On the CPU, on a fake runtime that records launches
(fake_hip.cpp)."""
import pytest

from tests import fake_hip

PLAIN_FORCE = "k_force_masksILi48ELi256ELb1ELb1EE"      # the masks pair with the loops' sums
_SIM = """
        x = np.random.default_rng(0).uniform(0.1, 0.5, ({n}, 3)).astype(np.float32)
        sim = S.ParticleSimulation(S.make_scene("dam16k").with_positions(x)).Init()
"""


@pytest.fixture(scope="module")
def fake(tmp_path_factory):
    return fake_hip.build(tmp_path_factory.mktemp("fake_hip"))


@pytest.mark.parametrize("n", [28673, 50000])
def test_one_lane_is_timed_as_the_pair_a_step_runs(fake, n):
    fake_hip.run(fake, _SIM.format(n=n) + f"""
        sim.Advance(1)
        assert launches("{PLAIN_FORCE}") == 1
        sim.autotune(2)
        assert launches("{PLAIN_FORCE}") >= 1 + 3
        assert launches("k_forceILi128E") == 0          # no step of this scene would
    """)


def test_sets_that_run_in_teams_have_one_form_of_each_pass(fake):
    fake_hip.run(fake, _SIM.format(n=2000) + """
        sim.set_tuning(hit_masks=1, hit_list=64, block=128)
        sim.Advance(1)
        b = [launches("k_force_teamILb%dELb1E" % m) for m in (0, 1)]
        t = sim.autotune(2)
        a = [launches("k_force_teamILb%dELb1E" % m) for m in (0, 1)]
        # a warm-up and two repetitions each, and the choice run once more
        assert [a[0] - b[0], a[1] - b[1]] in ([4, 3], [3, 4]), (a, b)
        assert (t["hit_list"], t["block"]) == (64, 128)
    """)


def test_a_two_scale_state_is_timed_with_the_kernels_of_its_step(fake):
    fake_hip.run(fake, _SIM.format(n=20000) + """
        sim.set_tuning(hit_masks=1)
        sim.AdvanceTwoScale(1)
        assert launches("k_density_masks") == 1 and launches("k_density_team") == 0
        sim.autotune(2)
        assert launches("k_density_teamILb1E") == 0 and launches("k_force_teamILb1E") == 0
        assert launches("k_force_masksILi32ELi128E") == 3
    """)


def test_batches_keep_the_loops(fake):
    fake_hip.run(fake, """
        base = S.make_scene("dam16k")
        x = np.random.default_rng(0).uniform(0.1, 0.5, (45000, 3)).astype(np.float32)
        b = S.Batch([base.with_positions(x), base])
        b.step(1)
        b.autotune(2)
        assert launches("k_forceILi128ELb0E") >= 3 and launches("ELi256ELb1ELb1EE") == 0
    """)


@pytest.mark.parametrize("masks", [0, 1])
@pytest.mark.parametrize("n", [2000, 28673, 41000])
def test_bench_names_the_kernels_that_ran(fake, n, masks):
    fake_hip.run(fake, _SIM.format(n=n) + f"""
        import bench
        sim.set_tuning(hit_masks={masks}, hit_list=40, block=128)
        sim.Advance(1)
        for stage in ("density", "force"):
            name, args = bench.kernel_name(stage, sim.get_tuning(), {n})[:-1].split("<")
            args = args.replace("plain", "true").split(",")
            mangled = name + "I" + "".join(dict(true="Lb1E", false="Lb0E").get(a, "Li" + a + "E") for a in args)
            assert launches(mangled) == 1, mangled
    """)
