"""Profiling the pressure step's wall-normal solver times the solve that the step
runs: same path, same result, a device time after each step and 0 without."""
import ctypes

import numpy as np
import pytest

from filtered_tdma_amd import _lib
from filtered_tdma_amd.poisson import ChannelPoisson

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")


@pytest.mark.parametrize("nz,P,modes", [(64, 1, True), (513, 1, False), (64, 4, False)])
def test_profiled_solver_keeps_the_path(nz, P, modes):
    print(f"[gpu-case] poisson profiled nz={nz} P={P}", flush=True)
    nx, ny = 16, 6
    rhs = torch.from_numpy(np.random.default_rng(nz).standard_normal((nz, ny, nx))).cuda()
    ps = ChannelPoisson(nx, ny, nz, 6.0, 3.0, 2.0, 1.0, "pascal", P)
    try:
        solver = ctypes.c_void_p(_lib.load().ftd_poisson_solver(ps._h))
        got = []
        for on in (0, 1, 0):
            _lib.check(_lib.load().ftd_set_profiling(solver, on))
            got.append(torch.empty_like(rhs))
            ps.solve_rhs(rhs, got[-1])
            assert ps.solver_path().startswith("pascal_modes") == modes, ps.solver_path()
            assert (_lib.load().ftd_last_gpu_ms(solver) > 0.0) == bool(on)
    finally:
        ps.close()
    for g in got[1:]:
        np.testing.assert_array_equal(g.cpu().numpy(), got[0].cpu().numpy())
