"""How the steps of a run are put into launches, on the CPU (the runtime of
tests/cpp/hip_stand_in.cpp, which records the kernels): by marching waves, in
LDS regions or one by one, by element size, extents and layout."""
import pytest

import stand_in


@pytest.fixture(scope="module")
def runtime(tmp_path_factory):
    return stand_in.build(tmp_path_factory.mktemp("hip"))


CODE = """
def kernel(storage, layout, h, v):
    doc = pa.settings("lptl", layout, inner_h=h, inner_v=v, storage=storage, time_steps=1)
    with pa.Lattice(pa.desc_from_settings(doc)) as lat:
        lat.set_phase(np.zeros(lat.N, dtype=np.int8))
        lat.init()
        log()
        lat.run(12)
        steps = [k for k in log() if "k_step" in k or "k_march" in k or "k_tile" in k]
    if "k_march" in steps[0]:
        assert len(steps) == 3, steps
        return "march"
    if "k_tile" in steps[0]:
        return "x".join(steps[0].split("<")[1].split(">")[0].replace(" ", "").split(",")[2:4]) + f" {len(steps)}"
    assert len(steps) == 12, steps
    return "one"
"""

# inner extents, storage, layout: shape and number of launches for 12 steps
CASES = [
    # by size
    ((64, 32), "f64", "stream", "16x16 3"), ((256, 64), "f16-shifted", "bundle", "16x16 3"),
    ((512, 128), "f64", "collision", "32x32 2"), ((640, 380), "f64", "stream", "32x32 3"),
    ((1024, 256), "f32", "stream", "32x32 3"), ((1000, 600), "f64", "stream", "32x16 3"),
    ((1000, 600), "f32", "bundle", "32x16 4"), ((1999, 501), "bf16-shifted", "bundle", "32x16 4"),
    ((1999, 749), "f64", "stream", "32x16 3"), ((1999, 752), "f64", "stream", "march"),
    ((2499, 1000), "f32", "stream", "32x16 4"), ((2501, 1000), "f32", "stream", "march"),
    ((3499, 1000), "f16-shifted", "collision", "32x16 4"), ((3601, 1000), "f16-shifted", "collision", "march"),
    ((8192, 2048), "f16-shifted", "stream", "march"), ((8192, 2048), "bf16-shifted", "bundle", "march"),
    # the lattices that the tests of several steps per launch march and tile
    ((2240, 700), "f64", "stream", "march"), ((3001, 503), "f64", "bundle", "march"),
    ((85, 17700), "f64", "collision", "march"), ((2241, 1360), "f32", "stream", "march"),
    ((3001, 1171), "f16-shifted", "stream", "march"), ((2688, 1310), "bf16-shifted", "stream", "march"),
    ((2464, 1100), "f32", "stream", "march"), ((3001, 901), "f32", "collision", "march"),
    ((150, 18000), "f32", "bundle", "march"), ((235, 15400), "f16-shifted", "collision", "32x32 3"),
    ((190, 19000), "bf16-shifted", "bundle", "march"), ((4481, 801), "f16-shifted", "stream", "march"),
    # narrow: what of the waves' columns is used
    ((64, 30000), "f64", "stream", "march"), ((24, 65000), "f64", "stream", "32x16 3"),
    ((64, 60000), "f32", "bundle", "march"), ((48, 60000), "f32", "bundle", "32x16 4"),
    ((58, 65000), "f16-shifted", "stream", "32x32 3"), ((58, 65000), "bf16-shifted", "collision", "32x32 3"),
    ((80, 65000), "f16-shifted", "bundle", "32x16 4"), ((113, 30000), "f16-shifted", "bundle", "32x32 3"),
    ((226, 60000), "f16-shifted", "stream", "one"), ((226, 60000), "f16-shifted", "bundle", "32x32 3"),
    ((450, 30000), "bf16-shifted", "stream", "one"), ((450, 30000), "f16-shifted", "bundle", "march"),
    ((280, 60000), "f16-shifted", "stream", "march"),
    # thin
    ((65000, 3), "f64", "stream", "one"), ((65000, 3), "f64", "bundle", "32x16 3"),
    ((65000, 8), "f32", "stream", "32x16 3"), ((40000, 11), "f16-shifted", "collision", "32x16 4"),
    ((65000, 13), "f16-shifted", "stream", "one"), ((65000, 26), "f16-shifted", "bundle", "32x16 3"),
    ((8000, 4), "f64", "stream", "16x16 3"),
]


def test_launches_by_extents(runtime):
    stand_in.run(runtime, CODE + f"""
wrong = []
for (h, v), storage, layout, expect in {CASES!r}:
    got = kernel(storage, layout, h, v)
    if got != expect:
        wrong.append((h, v, storage, layout, expect, got))
assert not wrong, wrong
""")


def test_two_steps_take_smaller_regions(runtime):
    stand_in.run(runtime, """
with pa.Lattice.from_settings(pa.settings("nptl", "collision", inner_h=1024, inner_v=256, time_steps=1)) as lat:
    for steps, shape in ((2, "32, 16"), (3, "32, 32"), (7, "32, 32"), (2, "32, 16")):
        log()
        lat.run(steps)
        launches = [k for k in log() if "k_tile_steps" in k]
        assert launches and all(shape in k for k in launches), (steps, launches)
""")


@pytest.mark.parametrize("count,h,v,storage,expect", [
    (976, 64, 64, "f16-shifted", "k_batch_tiles"), (40, 700, 150, "f16-shifted", "k_batch_march"),
    (61, 256, 256, "bf16-shifted", "k_batch_tiles"), (40, 500, 150, "f32", "k_batch_march"),
    (12000, 16, 16, "f32", "k_batch_tiles"), (500, 64, 64, "f64", "k_batch_march")])
def test_launches_of_a_batch(runtime, count, h, v, storage, expect):
    stand_in.run(runtime, f"""
docs = [pa.settings("lptl", "stream", inner_h={h}, inner_v={v}, time_steps=1)] * {count}
with pa.Batch(docs, storage={storage!r}) as b:
    log()
    b.run(12, "persistent")
    steps = [k for k in log() if "k_batch" in k]
    assert steps and all({expect!r} in k for k in steps), steps
""")


def test_two_steps_of_a_batch(runtime):
    stand_in.run(runtime, """
docs = [pa.settings("lptl", "stream", inner_h=30, inner_v=30, time_steps=1)] * 300
for storage, steps, launches in (("f64", 2, ["k_batch_step"] * 2), ("f64", 3, ["k_batch_tiles"]),
                                 ("f32", 2, ["k_batch_tiles"]), ("f64", 7, ["k_batch_tiles"] * 2)):
    with pa.Batch(docs, storage=storage) as b:
        log()
        b.run(steps, "persistent")
        names = [k for k in log() if "k_batch" in k]
        assert len(names) == len(launches) and all(n in k for n, k in zip(launches, names)), (storage, steps, names)
""")
