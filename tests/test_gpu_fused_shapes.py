"""Several steps per launch against single steps, bit for bit: marching waves
in FP32 and 16-bit storage on whole, ragged and single strips (the sizes march,
tests/test_fusion_plan.py), and lattices and batches whose launches are chosen
for being narrow or thin."""
import numpy as np
import pytest

import portlbm_amd as pa
from test_gpu_fused import STORAGES, check, document, same

pytestmark = pytest.mark.gpu

# strips of 112 (FP32) and 224 (16-bit) columns: 22 and 20 whole ones and a column, ragged ones, one and a part
MARCHED = {"f32": [(2464, 1100), (3001, 901), (150, 18000)], "f16-shifted": [(4481, 801), (190, 19000)],
           "bf16-shifted": [(4481, 801), (190, 19000)]}


@pytest.mark.parametrize("storage,rounding", STORAGES[1:])
@pytest.mark.parametrize("layout", ["collision", "stream", "bundle"])
def test_marched_steps(layout, storage, rounding):
    for k, (h, v) in enumerate(MARCHED[storage]):
        check(document("lptl" if k else "nptl", layout, storage, rounding, h, v, ["porous-circles", "walls", "circle"][k]),
              23)


@pytest.mark.parametrize("size", [(58, 65000), (24, 65000), (113, 30000), (280, 20000), (65000, 26), (65000, 13),
                                  (40000, 11), (65000, 8), (30000, 5), (65000, 3)])
@pytest.mark.parametrize("storage", ["f64", "f32", "f16-shifted"])
@pytest.mark.parametrize("layout", ["collision", "stream", "bundle"])
def test_narrow_and_thin_lattices(layout, storage, size):
    check(document("lptl", layout, storage, "nearest", *size, "walls"), 13)


@pytest.mark.parametrize("count,h,v,storage", [(976, 64, 64, "f16-shifted"), (130, 256, 120, "bf16-shifted"),
                                               (12000, 16, 16, "f32"), (9000, 13, 15, "f64")])
def test_batches_of_small_domains(count, h, v, storage):
    """Domains of every extent up to (h, v); all compared in total, some node by node."""
    docs = [pa.settings("lptl", "stream", inner_h=h - k % 5, inner_v=v - k % 3, scenario="walls", time_steps=1,
                        tau=0.6 + 0.001 * (k % 200), rho_in=1.01, storage=storage) for k in range(count)]
    with pa.Batch(docs, storage=storage) as one, pa.Batch(docs, storage=storage) as many:
        for _ in range(13):
            one.run(1, "persistent")
        many.run(13, "persistent")
        assert np.array_equal(one.residuals(), many.residuals(), equal_nan=True)
        for d in [*range(0, count, max(1, count // 40)), count - 1]:
            assert same(one.macros(d), many.macros(d))
