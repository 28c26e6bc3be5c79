"""The pinned staging of results, on the CPU (the runtime of
tests/cpp/hip_stand_in.cpp): as large as the largest read so far needs, kept
from one object to the next, and done without where it cannot be had."""
import pytest

import stand_in


@pytest.fixture(scope="module")
def runtime(tmp_path_factory):
    return stand_in.build(tmp_path_factory.mktemp("hip"))


def test_staging_grows_and_stays(runtime):
    stand_in.run(runtime, """
MIB = 1 << 20
def read(h, v):
    with pa.Lattice.from_settings(pa.settings("lptl", "stream", inner_h=h, inner_v=v, time_steps=1)) as lat:
        lat.run(3)
        lat.macros()
    return live()
assert read(64, 32) == [0, MIB, 1]        # 64 KiB: one slot, one event
assert read(64, 32) == [0, MIB, 1]
assert read(300, 200) == [0, 2 * MIB, 2]  # 1.9 MB
assert read(1100, 1000) == [0, 16 * MIB, 16]
assert read(64, 32) == [0, 16 * MIB, 16]
""")


@pytest.mark.parametrize("what,nth", [("hipHostMalloc", 1), ("hipEventCreateWithFlags", 1),
                                      ("hipEventCreateWithFlags", 2)])
def test_reads_without_staging(runtime, what, nth):
    stand_in.run(runtime, f"""
with pa.Lattice.from_settings(pa.settings("lptl", "stream", inner_h=300, inner_v=200, time_steps=1)) as lat:
    lat.run(3)
    before = live()
    fail({what!r}, {nth})
    first = np.stack(lat.macros())
    assert live() == before, (before, live())
    fail({what!r}, 0)
    np.testing.assert_array_equal(first, np.stack(lat.macros()))
    assert live()[1] == 2 << 20
""")
