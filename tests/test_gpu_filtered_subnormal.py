"""Filtered v1 where the scale from which a tile tells its own J is subnormal
(a column-0 bound near 1e-6 over 60 rows) and the boundary values are near
1e303, on both sides of J = m - 1: x and J bit for bit the oracle's, on the
streamed and the fused kernel."""
import sys

import numpy as np
import pytest

import oracle as O
from filtered_tdma_amd import TdmaBackendGPU

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")

# J of these is m - 1 from boundary values of about 2.65e303 on; the scale itself
# rounds to the smallest subnormal, which puts it at 1.55e303
RHO, EPS = 3.2443508865633046e-06, 7.686052368823148e-21


@pytest.mark.parametrize("n_sys", [64, 33])
@pytest.mark.parametrize("v", [1e300, 1.4e303, 1.6e303, 1.83e303, 2.5e303, 1e306])
def test_subnormal_scale(n_sys, v):
    n_row, P = 480, 8
    print(f"[gpu-case] v1 subnormal scale n_sys={n_sys} v={v}", flush=True)
    sys.stdout.flush()
    rng = np.random.default_rng(n_sys)
    A = np.full((n_row, n_sys), -RHO)
    B = np.ones((n_row, n_sys))
    D = v * rng.uniform(0.97, 1.0, (n_row, n_sys))
    ref, J = O.filtered(A, B, A, D, P, 1, EPS, eps_direct=True, sem=O.SEM_GPU, rho="auto",
                        return_J=True)
    be = TdmaBackendGPU("filtered", n_sys, n_row, P)
    try:
        be.set_eps(EPS)
        t = [torch.from_numpy(x.copy()).cuda() for x in (A, B, A, D)]
        be.set_rho_device(*t[:3])
        be.solve(*t)
        x, Jg, path = t[3].cpu().numpy(), be.last_J(), be.last_path()
    finally:
        be.close()
    assert path.startswith("filtered_v1_stream" if n_sys % 32 == 0 else "filtered_v1_fused"), path
    assert list(Jg) == list(J)
    np.testing.assert_array_equal(x, ref)
