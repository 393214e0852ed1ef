"""Column-0 bounds with a row's own ratio in every row, the largest in a
partition's first row (which J leaves out), second or last: J and x bit for
bit the oracle's, for partitions up to 64 rows and longer ones."""
import sys

import numpy as np
import pytest

import oracle as O
from filtered_tdma_amd import TdmaBackendGPU

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")


@pytest.mark.parametrize("kind,version", [("filtered", 1), ("filtered_v2", 2)])
@pytest.mark.parametrize("n_row,P", [(9, 3), (255, 4), (256, 4), (257, 4), (512, 8), (700, 2),
                                     (2600, 2)])
@pytest.mark.parametrize("where", [0, 1, -1])
def test_bounds(n_row, P, where, kind, version):
    n_sys = 35
    print(f"[gpu-case] set_rho {kind} n_row={n_row} P={P} where={where}", flush=True)
    sys.stdout.flush()
    rng = np.random.default_rng(n_row + P)
    r = rng.uniform(0.1, 0.3, n_row)
    r[[x[where] for x in np.array_split(np.arange(n_row), P)]] = 1.5
    A = np.tile(-r[:, None], (1, n_sys))
    C = np.tile(-0.9 * r[:, None], (1, n_sys))
    B = 1 - A - C
    D = rng.uniform(-1, 1, (n_row, n_sys))
    be = TdmaBackendGPU(kind, n_sys, n_row, P)
    try:
        be.set_eps(1e-5)
        t = [torch.from_numpy(x.copy()).cuda() for x in (A, B, C, D)]
        be.set_rho_device(*t[:3])
        be.solve(*t)
        x, J = t[3].cpu().numpy(), be.last_J()
    finally:
        be.close()
    ref, Jref = O.filtered(A, B, C, D, P, version, 1e-5, eps_direct=True, sem=O.SEM_GPU,
                           rho="auto", return_J=True)
    assert list(J) == list(Jref)
    np.testing.assert_array_equal(x, ref)
