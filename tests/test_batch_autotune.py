"""The autotuner's trials on the CPU (the runtime of tests/cpp/hip_stand_in.cpp,
which records the kernels): they launch the kernel whose tiles they choose."""
import pytest

import stand_in


@pytest.fixture(scope="module")
def runtime(tmp_path_factory):
    return stand_in.build(tmp_path_factory.mktemp("hip"))


@pytest.mark.parametrize("count", [4, 60])
def test_trials_launch_the_single_step_kernel(runtime, count):
    stand_in.run(runtime, f"""
docs = [pa.settings("lptl", "stream", inner_h=h, inner_v=300, time_steps=1) for h in (100, 200, 400, 600)] * ({count} // 4)
with pa.Batch(docs) as b:
    log()
    b.autotune(20)
    steps = [k for k in log() if any(n in k for n in ("k_batch_step", "k_batch_march", "k_batch_tiles"))]
    assert len(steps) == 4 * 3 * 22 and all("k_batch_step" in k for k in steps), set(steps)
    b.run(20, "persistent")
    fused = [k for k in log() if "k_batch" in k]
    assert fused and not any("k_batch_step" in k for k in fused), fused
""")
