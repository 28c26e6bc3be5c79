"""Runs of two steps, which take regions of their own, against single steps:
sizes of the 32 x 32 plan, whole and ragged regions of 30 x 14 owned nodes."""
import pytest

from test_gpu_fused import STORAGES, check, document

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("storage,rounding", STORAGES)
@pytest.mark.parametrize("layout", ["collision", "stream", "bundle"])
@pytest.mark.parametrize("size", [(1024, 256), (600, 140), (601, 141), (629, 155), (300, 127)])
def test_pairs_of_steps(size, layout, storage, rounding):
    check(document("lptl", layout, storage, rounding, *size, "porous-circles"), 2)
