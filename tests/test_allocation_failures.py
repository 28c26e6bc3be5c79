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


def test_a_second_result_array_only_for_several_frames(runtime):
    """Two result arrays alternate so that steps need not wait for a copy: a
    run without a frame, or with one, takes no second one."""
    stand_in.run(runtime, """
doc = pa.settings("lptl", "stream", inner_h=64, inner_v=32, time_steps=1)
with pa.Lattice.from_settings(doc) as lat:
    before = live()[0]
    lat.run_frames(10, 0)
    lat.run_frames(9, 100)
    lat.run_frames(2, 10)
    assert live()[0] == before
    lat.run_frames(20, 10)
    assert live()[0] == before + 4 * 64 * 32 * 8
    assert lat.frame()[0] == 39
assert live() == [0, 0, 0], live()
# where it cannot be had, frames share one array
with pa.Lattice.from_settings(doc) as lat:
    before = live()[0]
    log()
    fail("hipMalloc", 1)
    lat.run_frames(20, 5)
    assert live()[0] == before and len([k for k in log() if "k_copy_frame" in k]) == 4
""")


IN_PLACE = """
def kernels(algorithm, layout, h, v, storage="f64", limit=None, nth=0, group=1024):
    memory(288 << 30)
    if limit:
        memory(limit)
    fail("hipMalloc", nth)
    doc = pa.settings(algorithm, layout, inner_h=h, inner_v=v, work_group_size=group, storage=storage, time_steps=1)
    with pa.Lattice.from_settings(doc) as lat:
        fail("hipMalloc", 0)
        log()
        lat.run(6)
        return sorted({k.split("k_")[1].split("<")[0] for k in log() if "k_step" in k or "k_tile_s" in k or "k_march" in k})
"""


def test_one_lattice_schemes_stay_in_place_without_memory(runtime):
    """npol and nsol take a second, unexpanded lattice where it is at most 1/64
    of the device's memory and can be had; otherwise the in-place kernel of
    their layout, storage and size."""
    stand_in.run(runtime, IN_PLACE + """
size = 9 * (256 + 2 + 127) * (64 + 2) * 8  # as plan_compact counts it
assert kernels("npol", "stream", 256, 64) == ["tile_steps"]
assert kernels("npol", "stream", 256, 64, limit=64 * size) == ["tile_steps"]
assert kernels("npol", "stream", 256, 64, limit=64 * size - 1) == ["step_npol"]
assert kernels("nsol", "bundle", 256, 64, limit=64 * size - 1) == ["step_nsol"]
for nth in range(1, 9):  # any allocation of the second context
    assert kernels("npol", "stream", 256, 64, nth=nth) == ["step_npol"], nth
fail("hipMemGetInfo", 1)
assert kernels("npol", "stream", 256, 64) == ["step_npol"]
# in place, by size, layout and storage
G = 1 << 30
assert kernels("npol", "stream", 2048, 512, limit=G) == ["step_tile_sweep"]
assert kernels("nsol", "bundle", 2048, 512, "f32", limit=G) == ["step_tile_sweep"]
assert kernels("npol", "collision", 2048, 512, limit=G) == ["step_tile_staged"]
assert kernels("nsol", "collision", 2048, 512, "f32", limit=G) == ["step_tile_staged"]
assert kernels("npol", "collision", 512, 128, limit=G // 8) == ["step_npol"]
assert kernels("npol", "collision", 2048, 512, "f16-shifted", limit=G) == ["step_tile_sweep"]
memory(288 << 30)
assert live()[0] == 0 and live()[2] == 0, live()
""")


@pytest.mark.parametrize("storage", ["f64", "f16-shifted"])
def test_buffer_nodes_without_memory(runtime, storage):
    """Where the expanded lattice cannot be had, setting populations or a state
    succeeds and the buffer nodes stay at rest."""
    stand_in.run(runtime, f"""
doc = pa.settings("npol", "stream", inner_h=65, inner_v=40, storage={storage!r}, time_steps=1)
with pa.Lattice.from_settings(doc) as lat:
    values, state = lat.populations(), lat.state()
    for nth in (1, 2, 3):  # its lattice, its column reference (16-bit) and its staging
        for call in (lambda: lat.set_populations(values), lambda: lat.set_state(state), lat.state, lat.populations):
            lat.init()
            fail("hipMalloc", nth)
            call()
            fail("hipMalloc", 0)
        lat.init()
        if nth > 1:
            assert live() == before, (before, live())
        before = live()
    lat.set_populations(values)
    assert live()[0] > before[0]
    extra = live()[0] - before[0]
    assert extra >= 9 * lat.N * {8 if storage == "f64" else 2}
assert live()[0] == 0, live()
""")
