"""Flows that leave the range of their numbers, several steps per launch
against the same steps one at a time: the populations of every fluid node
themselves, bit for bit (the results pass a clamp that makes NaN and infinities
alike; solid nodes' populations are never read and left in either state)."""
import numpy as np
import pytest

import portlbm_amd as pa

pytestmark = pytest.mark.gpu

CASES = [("f64", (2011, 801)), ("f32", (2401, 1201)), ("f64", (300, 100)), ("f32", (300, 100)),
         ("f64", (200, 60)), ("f32", (700, 300))]  # marched, then the LDS regions


def document(layout, storage, size, tau, nan_protection):
    return pa.settings("lptl", layout, inner_h=size[0], inner_v=size[1], scenario="walls", work_group_size=256,
                       tau=tau, rho_in=1.02, time_steps=1, storage=storage, nanProtection=nan_protection)


def slots(layout, d, n, N):
    return 9 * n + d if layout == "collision" else (N * d + n if layout == "stream" else 3 * (d // 3) * N + d % 3 + 3 * n)


def both(doc, edit):
    phase = pa.build_phase(doc)
    one, many = (pa.Lattice(pa.desc_from_settings(doc), phase) for _ in range(2))
    f = one.populations()
    edit(f)
    one.set_populations(f)
    many.set_populations(f)
    layout, N = doc["algorithmic"]["dataLayout"], phase.size
    fluid = np.nonzero(phase == 0)[0].astype(np.int64)
    return one, many, slots(layout, np.arange(9)[:, None], fluid, N).ravel()


def check(one, many, fluid):
    np.testing.assert_array_equal(one.populations()[fluid], many.populations()[fluid])
    for a, b in zip(one.macros(), many.macros()):
        np.testing.assert_array_equal(a, b)


@pytest.mark.parametrize("nan_protection", [True, False])
@pytest.mark.parametrize("storage,size", CASES)
@pytest.mark.parametrize("layout", ["collision", "stream", "bundle"])
def test_momentum_overflows_while_the_density_does_not(layout, storage, size, nan_protection):
    """At tau 0.4 a relaxation stretches a population by -1.5.  The first step
    pulls f3 = f5 = -s a, f1 = f7 = s a: density and momentum 0.  s changes its
    sign along the diagonals so that the second step pulls f3 = f7 = -f1 = -f5,
    1.5 a each: density 0, momentum 3 a, past the largest number."""
    H, V = size[0] + 2, size[1] + 2
    a = {"f64": 0.38 * np.finfo(np.float64).max, "f32": 0.38 * float(np.finfo(np.float32).max)}[storage]

    def edit(f):
        y, x = np.mgrid[1:V - 1, 1:H - 1]
        n = (y * H + x).ravel()
        s = lambda k: np.where(k % 4 < 2, a, -a).ravel()
        f[:] = 0.0
        f[slots(layout, 1, n, H * V)] = s(x + y - 1)
        f[slots(layout, 3, n, H * V)] = -s(x + y - 1)
        f[slots(layout, 5, n, H * V)] = -s(x + y + 1)
        f[slots(layout, 7, n, H * V)] = s(x + y + 1)

    one, many, fluid = both(document(layout, storage, size, 0.4, nan_protection), edit)
    with one, many:
        for _ in range(2):
            one.run(1)
        many.run(2)
        if not nan_protection:
            rho, jx = one.macros()[:2]
            assert np.count_nonzero(np.isfinite(rho) & np.isinf(jx)) > 0.9 * size[0] * size[1] * 0.9
        check(one, many, fluid)
        for _ in range(3):
            one.run(1)
        many.run(3)
        check(one, many, fluid)


@pytest.mark.parametrize("nan_protection", [True, False])
@pytest.mark.parametrize("steps", [1, 2, 3, 4, 5, 8])
@pytest.mark.parametrize("storage,size", CASES[:4])
@pytest.mark.parametrize("layout", ["collision", "stream", "bundle"])
def test_infinities_spread_alike(layout, storage, size, steps, nan_protection):
    def edit(f):
        f[::7919] = np.inf
        f[3::15838] = -np.inf
        f[5::31676] = np.nan
        f[::15838] = 1e300 if storage == "f64" else 1e30

    one, many, fluid = both(document(layout, storage, size, 0.503, nan_protection), edit)
    with one, many:
        for _ in range(steps):
            one.run(1)
        many.run(steps)
        check(one, many, fluid)
