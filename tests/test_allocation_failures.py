"""What the GPU library does when memory runs out half-way, on the CPU (the
runtime of tests/cpp/hip_stand_in.cpp): no later call works with a piece that
is not there, and everything is given back."""
import pytest

import stand_in


@pytest.fixture(scope="module")
def runtime(tmp_path_factory):
    return stand_in.build(tmp_path_factory.mktemp("hip"))


@pytest.mark.parametrize("what,count", [("hipStreamCreateWithFlags", 1), ("hipEventCreateWithFlags", 3),
                                        ("hipHostMalloc", 1)])
def test_frames_after_a_failed_first_use(runtime, what, count):
    """Whichever piece of the frame copies could not be made, that call and the
    next one with the same trouble are refused, and the one after it works."""
    stand_in.run(runtime, f"""
doc = pa.settings("lptl", "stream", inner_h=64, inner_v=32, time_steps=1)
for nth in range(1, {count} + 1):
    lat = pa.Lattice.from_settings(doc)
    log()
    for _ in range(2):
        fail({what!r}, nth)
        raises(lambda: lat.run_frames(10, 2))
        assert not [k for k in log() if "k_copy_frame" in k]
        nth = 1
    fail({what!r}, 0)
    lat.run_frames(10, 2)
    assert len([k for k in log() if "k_copy_frame" in k]) == 5
    lat.close()
    assert live()[:2] == [0, 0] and live()[2] == 0, live()
""")
