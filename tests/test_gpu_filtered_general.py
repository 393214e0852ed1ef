"""The general filtered kernels (partitions longer than a lane holds, or
forced): rows are read in blocks of 8 and corrected in blocks of 8, one wave
per 64 systems. Partitions at the edges of a block, systems at the edges of a
wave, J at both ends and inside; bit for bit the oracle's Filtered."""
import sys

import numpy as np
import pytest

import oracle as O
from filtered_tdma_amd import Kind, TdmaBackendGPU, cases

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")


@pytest.mark.parametrize("kind", [Kind.FILTERED, Kind.FILTERED_V2])
@pytest.mark.parametrize("n_sys,n_row,P,forced", [
    (1, 6, 2, True), (63, 9, 3, True), (64, 21, 2, True), (65, 38, 4, True),   # m = 3 .. 11
    (129, 33, 2, True), (64, 50, 2, True),        # m = 17 / 16, 25
    (65, 131, 2, False), (257, 260, 4, False), (7, 1029, 8, False),
])
def test_general_block_and_wave_edges(n_sys, n_row, P, forced, kind):
    version = 1 if kind == Kind.FILTERED else 2
    A, B, C, D, _ = cases.toeplitz_batch(n_sys, n_row, 0.05, 0.5, seed=n_sys)
    for cyclic in (False, True):
        # J = 0, interior, and m - 1
        for scale, eps in ((1e-14, 1e-6), (1.0, 1e-4), (1.0, 1e-300)):
            print(f"[gpu-case] filtered_general v{version} n_sys={n_sys} n_row={n_row} P={P} "
                  f"cyclic={cyclic} scale={scale} eps={eps}", flush=True)
            sys.stdout.flush()
            Ds = D * scale
            be = TdmaBackendGPU(kind, n_sys, n_row, P)
            try:
                if forced:
                    be.set_tuning(-1, 0, 0, 0)
                be.set_eps(eps)
                t = [torch.from_numpy(v.copy()).cuda() for v in (A, B, C, Ds)]
                be.set_rho_device(*t[:3])
                (be.solve_cyclic if cyclic else be.solve)(*t)
                torch.cuda.synchronize()
                x, J, path = t[3].cpu().numpy(), be.last_J(), be.last_path()
            finally:
                be.close()
            assert "general" in path, path
            ref, Jref = O.filtered(A, B, C, Ds, P, version, eps, eps_direct=True, sem=O.SEM_GPU,
                                   cyclic=cyclic, rho="auto", return_J=True)
            assert list(J) == list(Jref)
            np.testing.assert_array_equal(x, ref)
