"""The persistent launch of one step under every tile width: the same fields
as launches of several steps, whose partition does not depend on them."""
import numpy as np
import pytest

import portlbm_amd as pa

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("storage", ["f64", "f32", "f16-shifted", "bf16-shifted"])
@pytest.mark.parametrize("widths", [[64, 64, 64, 64], [128, 64, 256, 128], [256, 256, 256, 64]])
def test_single_steps_under_other_tile_widths(widths, storage):
    docs = [pa.settings("lptl", "stream", inner_h=h, inner_v=v, scenario="porous-circles", time_steps=1, tau=0.7,
                        rho_in=1.02, storage=storage, seed=h, porosity=0.8, radiusMin=2.0, radiusMax=4.0,
                        obstacleMargin=2) for h, v in ((30, 20), (128, 33), (129, 40), (257, 64), (513, 70), (700, 31))]
    with pa.Batch(docs, storage=storage) as one, pa.Batch(docs, storage=storage) as many:
        one.set_tiles(widths)
        for _ in range(13):
            one.run(1, "persistent")
        many.run(13, "persistent")
        np.testing.assert_allclose(one.residuals(), many.residuals(), rtol=1e-12)
        for d in range(len(docs)):
            for a, b in zip(one.macros(d), many.macros(d)):
                np.testing.assert_array_equal(a, b)
