"""Results reach pageable host arrays through pinned slots of 1 MiB: sizes
around a slot, around the ring of 16 of them and above one thread's share, and
from several threads at once, against the results inside a saved state (which
a plain copy fetches)."""
import threading

import numpy as np
import pytest

import portlbm_amd as pa

pytestmark = pytest.mark.gpu

# 4 arrays of h x v doubles: 1 KiB, one slot less a row, one slot, one more, 6 MiB, the ring, several rings
SIZES = [(8, 4), (256, 127), (256, 128), (257, 128), (512, 384), (1024, 512), (1031, 1203)]


def lattice(h, v):
    doc = pa.settings("lptl", "stream", inner_h=h, inner_v=v, scenario="Hagen-Poiseuille", rho_in=1.01, time_steps=1)
    return pa.Lattice.from_settings(doc)


def saved(lat):
    return lat.state()[-32 * lat.D:].view(np.float64).reshape(4, lat.D)


@pytest.mark.parametrize("h,v", SIZES)
def test_results_of_every_size(h, v):
    with lattice(h, v) as lat:
        lat.run(12)
        for _ in range(2):  # fresh pages, then the ring in use before
            np.testing.assert_array_equal(np.stack(lat.macros()), saved(lat))


def test_several_threads_at_once():
    lats = [lattice(400 + 100 * k, 300) for k in range(4)]
    expect, bad = [], []
    for lat in lats:
        lat.run(10)
        expect.append(saved(lat))

    def read(k):
        for _ in range(20):
            if not np.array_equal(np.stack(lats[k].macros()), expect[k]):
                bad.append(k)

    threads = [threading.Thread(target=read, args=(k,)) for k in range(4)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    for lat in lats:
        lat.close()
    assert not bad
    with lattice(64, 32) as again:  # the staging was given back with the last lattice
        again.run(3)
        np.testing.assert_array_equal(np.stack(again.macros()), saved(again))
