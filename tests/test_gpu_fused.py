"""Several time steps in one launch against the same steps one at a time
(lbm_run(1) launches the one-step kernels): the same fields, reductions and
outlet history, bit for bit, in every layout and storage, on extents that
leave remainders in every direction of the launch."""
import numpy as np
import pytest

import portlbm_amd as pa

pytestmark = pytest.mark.gpu

STORAGES = [("f64", "nearest"), ("f32", "nearest"), ("f16-shifted", "nearest"), ("f16-shifted", "stochastic"),
            ("bf16-shifted", "nearest"), ("bf16-shifted", "stochastic")]


def document(algorithm, layout, storage, rounding, h, v, scenario, group=256, tau=0.7):
    ext = {"seed": 11, "porosity": 0.7, "radiusMin": 2.0, "radiusMax": 6.0, "obstacleMargin": 4} \
        if scenario == "porous-circles" else {}
    return pa.settings(algorithm, layout, inner_h=h, inner_v=v, scenario=scenario, work_group_size=group, tau=tau,
                       rho_in=1.02, storage=storage, rounding=rounding, time_steps=1, **ext)


def same(a, b):
    return all(np.array_equal(x, y, equal_nan=True) for x, y in zip(a, b))


def check(doc, steps, frame_interval=0):
    phase = pa.build_phase(doc)
    with pa.Lattice(pa.desc_from_settings(doc), phase) as one, pa.Lattice(pa.desc_from_settings(doc), phase) as many:
        for _ in range(steps):
            one.run(1)
        many.run(steps, frame_interval)
        assert one.iteration() == many.iteration() == steps
        assert same(one.macros(), many.macros())
        assert one.reduce() == many.reduce()
        # the outlet history and the lattice carry on alike, both ways
        one.run(5)
        for _ in range(5):
            many.run(1)
        assert same(one.macros(), many.macros())


# Inner extents.  Marching waves own strips of 56, 112 or 224 columns (FP64,
# FP32, 16-bit): whole strips, ragged ones, one strip and a half.
MARCHED = {"f64": [(2240, 700), (3001, 503), (85, 17700)], "f32": [(2240, 901), (1999, 1013), (2241, 1360)],
           "f16-shifted": [(3001, 1171)], "bf16-shifted": [(2688, 1310)]}
# Small lattices: less than a region, each shape's whole and ragged numbers of them.
TILED = [(4, 9), (30, 12), (61, 37), (256, 64), (257, 131), (500, 250), (1031, 301), (1030, 800), (700, 260)]


@pytest.mark.parametrize("storage,rounding", STORAGES)
@pytest.mark.parametrize("layout", ["collision", "stream", "bundle"])
def test_marched_steps_equal_single_steps(layout, storage, rounding):
    for k, (h, v) in enumerate(MARCHED[storage]):
        scenario = ["porous-circles", "walls", "circle"][k]
        check(document("nptl" if k != 1 else "lptl", layout, storage, rounding, h, v, scenario), 23)


@pytest.mark.parametrize("storage,rounding", STORAGES)
@pytest.mark.parametrize("layout", ["collision", "stream", "bundle"])
def test_tiled_steps_equal_single_steps(layout, storage, rounding):
    for k, (h, v) in enumerate(TILED):
        scenario = ["Hagen-Poiseuille", "walls", "porous", "porous-circles"][k % 4]
        check(document("lptl" if k % 2 else "nptl", layout, storage, rounding, h, v, scenario, 64 if h < 64 else 256),
              29 + k)


@pytest.mark.parametrize("size", [(2011, 801), (1031, 301), (300, 100)])
@pytest.mark.parametrize("steps", [1, 2, 3, 4, 5, 6, 7, 8])
def test_every_remainder(steps, size):
    check(document("nptl", "stream", "f64", "nearest", *size, "porous-circles"), steps)


@pytest.mark.parametrize("size", [(2011, 801), (300, 100)])
@pytest.mark.parametrize("interval", [1, 3, 10])
def test_frames_end_a_launch(interval, size):
    doc = document("lptl", "collision", "f64", "nearest", *size, "porous-circles")
    check(doc, 21, interval)
    phase = pa.build_phase(doc)
    with pa.Lattice(pa.desc_from_settings(doc), phase) as a, pa.Lattice(pa.desc_from_settings(doc), phase) as b:
        a.run_frames(21, interval)
        last, fields = a.frame()
        assert last == 21 // interval * interval - 1
        b.run(last + 1)
        assert same(fields, b.macros())


@pytest.mark.parametrize("size", [(3001, 1171), (300, 100)])
def test_reference_change_between_launches(size):
    """16-bit storage changes its column reference at step 128."""
    check(document("nptl", "stream", "f16-shifted", "nearest", *size, "porous-circles"), 134)


@pytest.mark.parametrize("size", [(2011, 801), (300, 100)])
def test_state_after_fused_steps(size):
    """A state taken after an odd number of launches continues elsewhere."""
    doc = document("nptl", "bundle", "f64", "nearest", *size, "porous-circles")
    phase = pa.build_phase(doc)
    with pa.Lattice(pa.desc_from_settings(doc), phase) as a, pa.Lattice(pa.desc_from_settings(doc), phase) as b:
        a.run(12)
        state = a.state()
        b.set_state(state)
        assert np.array_equal(b.state(), state)
        a.run(9)
        for _ in range(9):
            b.run(1)
        assert same(a.macros(), b.macros())


@pytest.mark.parametrize("size", [(2011, 801), (300, 100)])
@pytest.mark.parametrize("storage", ["f64", "f32"])
def test_diverging_flow_keeps_its_infinities(storage, size):
    """Populations that are not finite take the full sums, as the one-step kernels do."""
    doc = document("nptl", "stream", storage, "nearest", *size, "porous-circles", tau=0.503)
    phase = pa.build_phase(doc)
    with pa.Lattice(pa.desc_from_settings(doc), phase) as one, pa.Lattice(pa.desc_from_settings(doc), phase) as many:
        f = one.populations()
        f[::7919] = np.inf
        f[::15838] = 1e300 if storage == "f64" else 1e30
        for lattice in (one, many):
            lattice.set_populations(f)
        for _ in range(8):
            one.run(1)
        many.run(8)
        assert not np.all(np.isfinite(one.populations()))
        assert same(one.macros(), many.macros())


@pytest.mark.parametrize("size", [(3001, 1171), (300, 100)])
@pytest.mark.parametrize("storage", ["f16-shifted", "bf16-shifted"])
def test_stochastic_rounding_keeps_infinities(storage, size):
    """The random bits carry into neither an infinity nor a NaN: they stand
    where rounding to nearest leaves them."""
    fields = []
    for rounding in ("nearest", "stochastic"):
        doc = document("nptl", "stream", storage, rounding, *size, "walls")
        with pa.Lattice(pa.desc_from_settings(doc), pa.build_phase(doc)) as lattice:
            f = lattice.populations()
            f[::7919], f[1::15838], f[2::31676] = np.inf, -np.inf, np.nan
            lattice.set_populations(f)
            lattice.run(3)
            fields.append(lattice.populations())
    assert not np.all(np.isfinite(fields[0]))
    for kind in (np.isnan, np.isposinf, np.isneginf):
        np.testing.assert_array_equal(kind(fields[0]), kind(fields[1]))


@pytest.mark.parametrize("storage", ["f64", "f32", "f16-shifted", "bf16-shifted"])
@pytest.mark.parametrize("count", [1, 3, 40, 130])
def test_batched_domains(count, storage):
    """Persistent and graph runs, several steps per launch, against one launch
    per domain and step: few domains (LDS tiles) to many (marching waves)."""
    rng = np.random.default_rng(count)
    docs = []
    for _ in range(count):
        h, v = (int(rng.integers(a, b)) for a, b in ((4, 700 if count > 3 else 90), (4, 300 if count > 3 else 60)))
        docs.append(pa.settings("lptl", "stream", inner_h=h, inner_v=v, scenario="porous-circles", time_steps=1,
                                tau=float(rng.uniform(0.6, 0.9)), rho_in=float(rng.uniform(1.005, 1.03)),
                                storage=storage, seed=int(rng.integers(1, 1 << 40)), porosity=0.8, radiusMin=2.0,
                                radiusMax=5.0, obstacleMargin=2))
    with pa.Batch(docs, storage=storage) as one, pa.Batch(docs, storage=storage) as many:
        for steps, mode in ((9, "persistent"), (14, "graph"), (14, "graph"), (1, "graph"), (5, "persistent")):
            one.run(steps, "per-domain")
            many.run(steps, mode)
        one.residuals()
        many.residuals()
        one.run(7, "per-domain")
        many.run(7, "graph")
        assert np.array_equal(one.residuals(), many.residuals(), equal_nan=True)
        for d in range(count):
            assert same(one.macros(d), many.macros(d))
