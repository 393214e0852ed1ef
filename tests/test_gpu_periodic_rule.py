"""Periodic batches of 257 to 448 rows on both sides of the line from which
whole-line ones take 64-row lanes; bit for bit the oracle's periodic PaScaL of
the partitions that the path names."""
import sys

import numpy as np
import pytest

import oracle as O
from filtered_tdma_amd import Kind, TdmaBackendGPU, cases

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")


@pytest.mark.parametrize("n_sys,n_row,M", [
    (24576, 257, 64), (24592, 448, 64), (24560, 257, 32), (24577, 300, 32), (24576, 256, 32),
])
def test_periodic_rule(n_sys, n_row, M):
    print(f"[gpu-case] periodic rule n_sys={n_sys} n_row={n_row}", flush=True)
    sys.stdout.flush()
    A, B, C, D = cases.general_batch(n_sys, n_row, seed=n_row)
    be = TdmaBackendGPU(Kind.PASCAL, n_sys, n_row, 1)
    try:
        t = [torch.from_numpy(x).cuda() for x in (A, B, C, D)]
        be.solve_cyclic(*t)
        x, path = t[3].cpu().numpy(), be.last_path()
    finally:
        be.close()
    assert path.startswith(f"pascal_fused M={M} "), path
    np.testing.assert_array_equal(x, O.pascal(A, B, C, D, int(path.split("Q=")[1].split()[0]),
                                              sem=O.SEM_GPU, cyclic=True))
