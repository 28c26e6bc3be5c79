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


# inner extents: a whole number of strips and ragged ones (a strip is 56, 112
# or 224 columns in FP64, FP32 and 16-bit storage)
SIZES = {"f64": [(1120, 300), (3001, 103), (57, 5400)], "f32": [(2240, 560), (1999, 613)],
         "f16-shifted": [(3001, 2003)], "bf16-shifted": [(3001, 2003)]}


@pytest.mark.parametrize("storage,rounding", STORAGES)
@pytest.mark.parametrize("layout", ["collision", "stream", "bundle"])
def test_fused_steps_equal_single_steps(layout, storage, rounding):
    for k, (h, v) in enumerate(SIZES[storage]):
        scenario = ["porous-circles", "walls", "circle"][k]
        check(document("nptl" if k != 1 else "lptl", layout, storage, rounding, h, v, scenario), 23)


@pytest.mark.parametrize("steps", [1, 2, 3, 4, 5, 6, 7, 8])
def test_every_remainder(steps):
    check(document("nptl", "stream", "f64", "nearest", 1031, 301, "porous-circles"), steps)


@pytest.mark.parametrize("interval", [1, 3, 10])
def test_frames_end_a_launch(interval):
    doc = document("lptl", "collision", "f64", "nearest", 1031, 301, "porous-circles")
    check(doc, 21, interval)
    phase = pa.build_phase(doc)
    with pa.Lattice(pa.desc_from_settings(doc), phase) as a, pa.Lattice(pa.desc_from_settings(doc), phase) as b:
        a.run_frames(21, interval)
        last, fields = a.frame()
        assert last == 21 // interval * interval - 1
        b.run(last + 1)
        assert same(fields, b.macros())


def test_reference_change_between_launches():
    """16-bit storage changes its column reference at step 128."""
    check(document("nptl", "stream", "f16-shifted", "nearest", 3001, 2003, "porous-circles"), 134)


def test_state_after_fused_steps():
    """A state taken after an odd number of launches continues elsewhere."""
    doc = document("nptl", "bundle", "f64", "nearest", 1031, 301, "porous-circles")
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


def test_diverging_flow_keeps_its_infinities():
    """Populations that are not finite take the full sums, as the one-step kernels do."""
    doc = document("nptl", "stream", "f64", "nearest", 1031, 301, "porous-circles", tau=0.503)
    phase = pa.build_phase(doc)
    with pa.Lattice(pa.desc_from_settings(doc), phase) as one, pa.Lattice(pa.desc_from_settings(doc), phase) as many:
        f = one.populations()
        f[::7919] = np.inf
        f[::15838] = 1e300
        for lattice in (one, many):
            lattice.set_populations(f)
        for _ in range(8):
            one.run(1)
        many.run(8)
        assert not np.all(np.isfinite(one.populations()))
        assert same(one.macros(), many.macros())
