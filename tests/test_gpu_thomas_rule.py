"""Real batches of one partition of 33 to 64 rows: plain Thomas or 16-row
partitions, on both sides of the rule's lines; bit for bit the oracle's solve
that the path names."""
import sys

import numpy as np
import pytest

import oracle as O
from filtered_tdma_amd import Kind, TdmaBackendGPU, cases

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")


@pytest.mark.parametrize("n_sys,n_row,thomas", [
    (49152, 64, True), (49136, 64, False), (49152, 48, False),
    (57344, 33, True), (57328, 48, False), (65536, 64, True), (65537, 64, False),
    (65552, 64, False), (98304, 49, True), (98288, 64, False), (98304, 48, False),
    (114688, 48, True), (114672, 48, False), (131071, 64, False), (131072, 64, True),
])
def test_thomas_rule(n_sys, n_row, thomas):
    print(f"[gpu-case] thomas rule n_sys={n_sys} n_row={n_row}", flush=True)
    sys.stdout.flush()
    A, B, C, D = cases.general_batch(n_sys, n_row, seed=n_row)
    be = TdmaBackendGPU(Kind.PASCAL, n_sys, n_row, 1)
    try:
        t = [torch.from_numpy(x).cuda() for x in (A, B, C, D)]
        be.solve(*t)
        x, path = t[3].cpu().numpy(), be.last_path()
    finally:
        be.close()
    assert path.startswith("thomas_fused" if thomas else "pascal_fused M=16"), path
    ref = (O.thomas(A, B, C, D, sem=O.SEM_GPU) if thomas else
           O.pascal(A, B, C, D, int(path.split("Q=")[1].split()[0]), sem=O.SEM_GPU))
    np.testing.assert_array_equal(x, ref)
