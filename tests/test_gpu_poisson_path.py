"""Asking which path the pressure step's wall-normal solve took makes nothing:
the FFT plans of the solve on arrays are made when its handle is asked for."""
import pytest

from filtered_tdma_amd import _lib
from filtered_tdma_amd.poisson import ChannelPoisson

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")


def free():
    torch.cuda.synchronize()
    return torch.cuda.mem_get_info()[0]


def test_path_makes_no_plans():
    nx, ny, nz = 262, 131, 64  # 132 modes in lines of 136; a prime factor, so that plans take memory
    print(f"[gpu-case] poisson path nx={nx} ny={ny} nz={nz}", flush=True)
    ps = ChannelPoisson(nx, ny, nz, 6.0, 3.0, 2.0, 1.0)
    try:
        rhs = torch.ones((nz, ny, nx), dtype=torch.float64, device="cuda")
        dp = torch.empty_like(rhs)
        ps.solve_rhs(rhs, dp)
        before = free()
        assert ps.solver_path().startswith("pascal_modes")
        assert free() == before
        assert _lib.load().ftd_poisson_solver(ps._h)
        assert free() < before  # (so the measure does see plans)
    finally:
        ps.close()
