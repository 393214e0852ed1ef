"""The pressure step's own wall-normal solve (one caller partition: coefficients
formed in the kernel, padded spectra) against the oracle, at the edges of its
partitions and of the padding, and against the solve on arrays that a tuned
handle takes. Tolerances as in test_gpu_poisson.py: the FFTs differ."""
import ctypes
import sys

import numpy as np
import pytest

import poisson_oracle as PO
from filtered_tdma_amd import _lib
from filtered_tdma_amd.poisson import ChannelPoisson

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")

# nx, ny, nz: one and two partitions, counts that split unevenly, a mode count
# that is no multiple of a workgroup's, padded lines (41 modes in 48), 17 and 32
# partitions, and one row more than the kernel holds
CASES = [(16, 6, 16), (16, 6, 17), (20, 7, 33), (80, 5, 47), (80, 9, 64), (16, 5, 257),
         (18, 3, 512), (16, 3, 513)]


@pytest.mark.parametrize("kind", ["pascal", "filtered_v2"])
@pytest.mark.parametrize("nx,ny,nz", CASES)
def test_modes_match_oracle_and_array_solve(nx, ny, nz, kind):
    print(f"[gpu-case] poisson modes nx={nx} ny={ny} nz={nz} kind={kind}", flush=True)
    sys.stdout.flush()
    rhs = np.random.default_rng(nx + ny + nz).standard_normal((nz, ny, nx))
    ref = PO.Channel(nx, ny, nz, 2 * np.pi, np.pi, 2.0, 1.0).solve_rhs(rhs)
    scale = np.max(np.abs(ref))
    ps = ChannelPoisson(nx, ny, nz, 2 * np.pi, np.pi, 2.0, 1.0, kind)
    try:
        t_rhs = torch.from_numpy(rhs).cuda()
        own, arrays, again = (torch.empty_like(t_rhs) for _ in range(3))
        ps.solve_rhs(t_rhs, own)
        assert ps.solver_path().startswith("pascal_modes") == (17 <= nz <= 512), ps.solver_path()
        solver = _lib.load().ftd_poisson_solver(ps._h)
        _lib.check(_lib.load().ftd_set_tuning(ctypes.c_void_p(solver), -2, 0, 0, 0))
        ps.solve_rhs(t_rhs, arrays)
        assert not ps.solver_path().startswith("pascal_modes")
        _lib.check(_lib.load().ftd_set_tuning(ctypes.c_void_p(solver), 0, 0, 0, 0))
        ps.solve_rhs(t_rhs, again)
    finally:
        ps.close()
    own, arrays, again = (t.cpu().numpy() for t in (own, arrays, again))
    assert np.max(np.abs(own - ref)) <= 1e-11 * scale
    assert np.max(np.abs(own - arrays)) <= 1e-11 * scale
    np.testing.assert_array_equal(own, again)
