"""npol and nsol under the automatic tile kernel, which works on the unexpanded
lattice where a second one is cheap, against their in-place block kernels: the
same fields, node tables, populations and states, bit for bit, on whole and
ragged tile grids and where a buffer column meets the outlet."""
import numpy as np
import pytest

import portlbm_amd as pa

pytestmark = pytest.mark.gpu

# inner extents and work-group: 16 x 16 (npol) / 14 x 15 (nsol) tiles and others
SHAPES = [(64, 32, 256), (65, 40, 256), (57, 31, 256), (131, 77, 64), (31, 30, 1024), (900, 700, 1024)]
STORAGES = ["f64", "f32", "f16-shifted", "bf16-shifted"]


def document(algorithm, layout, storage, h, v, group, tile_kernel, scenario="porous-circles"):
    return pa.settings(algorithm, layout, inner_h=h, inner_v=v, scenario=scenario, work_group_size=group, tau=0.7,
                       rho_in=1.02, time_steps=1, storage=storage, tileKernel=tile_kernel, seed=5, porosity=0.8,
                       radiusMin=2.0, radiusMax=4.0, obstacleMargin=4)


def fluid_slots(phase, layout, N):
    n = np.nonzero(phase == 0)[0].astype(np.int64)
    d = np.arange(9)[:, None]
    if layout == "collision":
        return (9 * n + d).ravel()
    return (N * d + n).ravel() if layout == "stream" else (3 * (d // 3) * N + d % 3 + 3 * n).ravel()


def lattices(algorithm, layout, storage, shape):
    auto = document(algorithm, layout, storage, *shape, "auto")
    phase = pa.build_phase(auto)
    block = pa.desc_from_settings(document(algorithm, layout, storage, *shape, "block"))
    return pa.Lattice(pa.desc_from_settings(auto), phase), pa.Lattice(block, phase), phase


@pytest.mark.parametrize("storage", STORAGES)
@pytest.mark.parametrize("layout", ["collision", "stream", "bundle"])
@pytest.mark.parametrize("algorithm", ["npol", "nsol"])
def test_fields_tables_and_populations(algorithm, layout, storage):
    for k, shape in enumerate(SHAPES):
        if k == 5 and layout != "stream":
            continue
        a, b, phase = lattices(algorithm, layout, storage, shape)
        with a, b:
            slots = fluid_slots(phase, layout, a.N)
            np.testing.assert_array_equal(a.phase(), phase)
            np.testing.assert_array_equal(a.node_codes(), b.node_codes())
            a.run(33)
            b.run(33)
            for x, y in zip(a.macros(), b.macros()):
                np.testing.assert_array_equal(x, y)
            np.testing.assert_array_equal(a.populations()[slots], b.populations()[slots])
            ra, rb = a.reduce(), b.reduce()
            assert ra["fluid"] == rb["fluid"] and abs(ra["mass"] / rb["mass"] - 1) < 1e-12


@pytest.mark.parametrize("layout,storage", [("collision", "f64"), ("stream", "f32"), ("bundle", "f16-shifted")])
@pytest.mark.parametrize("algorithm", ["npol", "nsol"])
def test_states_and_populations_move_between_them(algorithm, layout, storage):
    a, b, phase = lattices(algorithm, layout, storage, (65, 40, 256))
    with a, b:
        slots = fluid_slots(phase, layout, a.N)
        b.run(21)
        a.set_state(b.state())
        for lattice in (a, b):
            lattice.run(10)
        np.testing.assert_array_equal(a.populations()[slots], b.populations()[slots])
        state = a.state()
        assert state.size == b.state().size
        b.set_state(state)
        assert b.iteration() == a.iteration() == 31
        for lattice in (a, b):
            lattice.run(7)
        for x, y in zip(a.macros(), b.macros()):
            np.testing.assert_array_equal(x, y)
        b.set_populations(a.populations())
        a.set_populations(a.populations())
        rho, jx, jy = (np.linspace(s, s + 0.01, a.D) for s in (1.0, 0.0, -0.01))
        for lattice in (a, b):
            lattice.run(9)
            lattice.run_split(2)
            lattice.run_frames(20, 6)
        for x, y in zip(a.macros() + a.frame()[1], b.macros() + b.frame()[1]):
            np.testing.assert_array_equal(x, y)
        for lattice in (a, b):
            lattice.set_equilibrium_field(rho, jx, jy)
            lattice.run(3)
        for x, y in zip(a.macros(), b.macros()):
            np.testing.assert_array_equal(x, y)


def test_calls_out_of_order_are_refused():
    desc = pa.desc_from_settings(document("npol", "stream", "f64", 64, 32, 256, "auto"))
    with pa.Lattice(desc) as lattice:
        np.testing.assert_array_equal(lattice.phase(), np.full(lattice.N, -1, dtype=np.int8))
        with pytest.raises(pa.LbmError, match="lbm_set_phase"):
            lattice.init()
        for call in (lambda: lattice.run(1), lattice.reduce, lattice.state, lattice.node_codes,
                     lambda: lattice.set_populations(np.zeros(9 * lattice.N)), lambda: lattice.run_split(1),
                     lambda: lattice.run_frames(1, 1)):
            with pytest.raises(pa.LbmError, match="lbm_init_populations"):
                call()
        with pytest.raises(pa.LbmError, match="node_count"):
            lattice.set_phase(np.zeros(lattice.N - 1, dtype=np.int8))
