"""Fused heat sweeps of lines in more than 8 partitions (257 to 512 cells), whose
reduced rows are read by the lanes of partition 0, against the materialized
ones, bit for bit: 16-line tiles in x, the partitions of y and z beside them."""
import numpy as np
import pytest

from filtered_tdma_amd.heat import SolveTheta

pytestmark = pytest.mark.gpu

pytest.importorskip("torch")


@pytest.mark.parametrize("shape", [(257, 19, 21), (289, 33, 12), (400, 20, 34), (512, 17, 9),
                                   (500, 7, 300), (20, 512, 18), (18, 23, 480)])
def test_long_lines_fused_equal_materialized(shape):
    print(f"[gpu-case] heat long lines {shape}", flush=True)
    sims = [SolveTheta(*shape, backend="pascal", dt=2e-4) for _ in range(2)]
    try:
        sims[1].set_fused(False)
        for steps in (1, 3):
            for sim in sims:
                sim.run(steps, use_graph=True)
            np.testing.assert_array_equal(sims[0].field(), sims[1].field())
        assert sims[0].last_plan().count("fused") == 3, sims[0].last_plan()
        assert sims[1].last_plan().count("materialized") == 3, sims[1].last_plan()
    finally:
        for sim in sims:
            sim.close()
