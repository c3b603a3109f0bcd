"""A two-scale step that cannot have its buffers refuses, again on the next
call, launches nothing with what it could get, and runs once there is memory.
On the CPU, on a fake runtime (fake_hip.cpp)."""
import pytest

from tests import fake_hip


@pytest.fixture(scope="module")
def fake(tmp_path_factory):
    return fake_hip.build(tmp_path_factory.mktemp("fake_hip"))


@pytest.mark.parametrize("after", [0, 5, 20])
def test_no_step_on_missing_buffers(fake, after):
    fake_hip.run(fake, f"""
        sim = S.ParticleSimulation(S.make_scene("dam16k")).Init()
        held = count("bytes")
        for _ in range(2):
            fake.fake_fail(b"hipMalloc", {after})
            try:
                sim.AdvanceTwoScale(1)
                raise SystemExit("no error")
            except S.SphError as e:
                assert e.status == S.Status.OUT_OF_MEMORY
            assert launches("k_ts_") == 0 and count("bytes") == held
        fake.fake_work(b"hipMalloc")
        sim.Advance(1)
        sim.AdvanceTwoScale(1)
        assert launches("k_ts_") > 0
    """)
