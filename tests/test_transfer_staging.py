"""The pinned staging of results, on the CPU (the runtime of
tests/cpp/hip_stand_in.cpp): kept from one object to the next, and done without
where it cannot be had."""
import pytest

import stand_in


@pytest.fixture(scope="module")
def runtime(tmp_path_factory):
    return stand_in.build(tmp_path_factory.mktemp("hip"))


def test_staging_stays(runtime):
    stand_in.run(runtime, """
def read(h, v):
    with pa.Lattice.from_settings(pa.settings("lptl", "stream", inner_h=h, inner_v=v, time_steps=1)) as lat:
        lat.run(3)
        before = live()
        lat.macros()
        return [b - a for a, b in zip(before, live())]
assert live() == [0, 0, 0]
assert read(300, 200) == [0, 16 << 20, 16]
assert live() == [0, 16 << 20, 16]
assert read(64, 32) == read(1100, 1000) == [0, 0, 0]
""")


@pytest.mark.parametrize("what,nth", [("hipHostMalloc", 1), ("hipEventCreateWithFlags", 1),
                                      ("hipEventCreateWithFlags", 9)])
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
    assert live()[1] == 16 << 20
""")
