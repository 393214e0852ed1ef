"""The filtered kind's fused sweeps (k_adi_filt1, k_filt_correct) against the
materialized ones, bit for bit, at the edges of their shapes: how a wave
holds the factor table (64, 32 and 16 systems per workgroup), partitions of
the fewest and the most rows, and on both sides of the tile count from which
J has a launch of its own."""
import numpy as np
import pytest

from filtered_tdma_amd.heat import SolveTheta

pytestmark = pytest.mark.gpu

pytest.importorskip("torch")


@pytest.mark.parametrize("shape,parts", [
    ((128, 128, 40), (1, 1, 4)),   # 64 systems, 16-row lanes
    ((130, 129, 100), (1, 1, 2)),  # 64 systems, a ragged last tile, 64-row lanes
    ((181, 181, 31), (1, 1, 2)),   # 512 tiles: J found by the correction
    ((183, 180, 31), (1, 1, 2)),   # 515 tiles: J's own launch
    ((91, 95, 9), (1, 1, 3)),      # partitions of 3 rows, 32 systems
    ((33, 31, 128), (1, 1, 2)),    # 64 rows in every lane, 16 systems
    ((40, 192, 30), (1, 3, 1)),    # y, 64 rows in every lane
    ((150, 37, 120), (1, 4, 8)),   # y and z
])
def test_filtered_fused_sweeps_equal_materialized(shape, parts):
    print(f"[gpu-case] heat filtered {shape} parts={parts}", flush=True)
    sims = [SolveTheta(*shape, parts=parts, backend="filtered", dt=2e-4) for _ in range(2)]
    try:
        sims[1].set_fused(False)
        for steps in (1, 3):
            for sim in sims:
                sim.run(steps, use_graph=True)
            np.testing.assert_array_equal(sims[0].field(), sims[1].field())
        assert "filtered_fused" in sims[0].last_plan()
    finally:
        for sim in sims:
            sim.close()
