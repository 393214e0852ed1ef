"""Many steps in one call (graphs of several steps whose x sweeps leave the
next step's Dirichlet ghosts) against the same steps one by one, ghosts
included, bit for bit; called again on the captured graphs."""
import numpy as np
import pytest

from filtered_tdma_amd.heat import SolveTheta

pytestmark = pytest.mark.gpu

pytest.importorskip("torch")


@pytest.mark.parametrize("kind,shape,parts,periodic", [
    ("pascal", (48, 33, 40), (1, 1, 1), (0, 0, 0)),
    ("pascal", (130, 20, 35), (1, 1, 2), (0, 0, 0)),  # x lines in partitions, odd y and z
    ("filtered", (40, 40, 32), (1, 1, 4), (0, 0, 0)),
    ("filtered_v2", (33, 3, 24), (2, 1, 2), (0, 0, 0)),  # x materialized: ghosts by launch
    ("pascal", (40, 32, 36), (1, 1, 1), (0, 1, 0)),      # periodic y: ghosts by launch
    ("pascal", (3, 3, 3), (1, 1, 1), (0, 0, 0)),
])
def test_steps_in_one_call_equal_steps_one_by_one(kind, shape, parts, periodic):
    print(f"[gpu-case] heat graph {kind} {shape} parts={parts} periodic={periodic}", flush=True)
    sims = [SolveTheta(*shape, parts=parts, backend=kind, dt=2e-4, periodic=periodic)
            for _ in range(2)]
    try:
        for steps in (42, 9, 20, 1):
            sims[0].run(steps, use_graph=True)
            for _ in range(steps):
                sims[1].run(1, use_graph=False)
            np.testing.assert_array_equal(sims[0].field(), sims[1].field())
    finally:
        for sim in sims:
            sim.close()
