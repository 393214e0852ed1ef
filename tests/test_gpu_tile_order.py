"""Fused exact and filtered solves whose tiles are whole 128-byte lines (which
run round the XCDs as they come) and those beside them that are not, with tile
counts off the XCDs' number: bit for bit the oracle's."""
import sys

import numpy as np
import pytest

import oracle as O
from filtered_tdma_amd import TdmaBackendGPU, cases

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")


def note(msg):
    print(f"[gpu-case] {msg}", flush=True)
    sys.stdout.flush()


def path_Q(path):
    return int(path.split("Q=")[1].split()[0])


# systems on and off the lines, whole tiles and a last one of 16 or 1
N_SYS = [64 * 9, 64 * 8 + 16, 64 * 8 + 1, 16]


@pytest.mark.parametrize("n_sys", N_SYS)
@pytest.mark.parametrize("tuning", [None, (32, 512, 16, 0), (32, 512, 64, 0), (32, 256, 8, 0)])
def test_exact(n_sys, tuning):
    n_row = 96
    A, B, C, D = cases.general_batch(n_sys, n_row, seed=n_sys)
    note(f"tile order exact n_sys={n_sys} tuning={tuning}")
    be = TdmaBackendGPU("pascal", n_sys, n_row, 1)
    try:
        if tuning:
            be.set_tuning(*tuning)
        t = [torch.from_numpy(x.copy()).cuda() for x in (A, B, C, D)]
        be.solve(*t)
        x, path = t[3].cpu().numpy(), be.last_path()
        Z = torch.from_numpy(D - 2j * D[::-1]).cuda()
        be.solve_complex(*t[:3], Z)
        z, zpath = Z.cpu().numpy(), be.last_path()
        f = [v.float() for v in t[:3]]
        t[3].copy_(torch.from_numpy(D))
        be.solve_f32c(*f, t[3])
        x32, path32 = t[3].cpu().numpy(), be.last_path()
    finally:
        be.close()
    np.testing.assert_array_equal(x, O.pascal(A, B, C, D, path_Q(path), sem=O.SEM_GPU))
    np.testing.assert_array_equal(z.real, O.pascal(A, B, C, D, path_Q(zpath), sem=O.SEM_GPU))
    np.testing.assert_array_equal(z.imag, O.pascal(A, B, C, -2 * D[::-1], path_Q(zpath),
                                                   sem=O.SEM_GPU))
    w = [v.cpu().numpy().astype(np.float64) for v in f]
    np.testing.assert_array_equal(x32, O.pascal(*w, D, path_Q(path32), sem=O.SEM_GPU))


@pytest.mark.parametrize("kind,version", [("filtered", 1), ("filtered_v2", 2)])
@pytest.mark.parametrize("n_sys", N_SYS)
@pytest.mark.parametrize("r", [0.3, 8.0])  # J inside, and every row
def test_filtered(n_sys, kind, version, r):
    n_row, P, eps = 150, 5, 1e-6
    A = np.full((n_row, n_sys), -r)
    B = np.full((n_row, n_sys), 1 + 2 * r)
    D = np.random.default_rng(n_sys).uniform(-1, 1, (n_row, n_sys))
    note(f"tile order {kind} n_sys={n_sys} r={r}")
    be = TdmaBackendGPU(kind, n_sys, n_row, P, eps)
    try:
        t = [torch.from_numpy(x.copy()).cuda() for x in (A, B, A, D)]
        be.set_rho_device(*t[:3])
        be.solve(*t)
        x, path = t[3].cpu().numpy(), be.last_path()
        Z = torch.from_numpy(D + 1j * D[::-1]).cuda()
        be.solve_complex(*t[:3], Z)
        z = Z.cpu().numpy()
    finally:
        be.close()
    assert f"v{version}_fused M=32" in path, path
    np.testing.assert_array_equal(x, O.filtered(A, B, A, D, P, version, eps, rho="auto"))
    np.testing.assert_array_equal(z.real, O.filtered(A, B, A, D, P, version, eps, rho="auto"))
    np.testing.assert_array_equal(z.imag, O.filtered(A, B, A, D[::-1].copy(), P, version, eps,
                                                     rho="auto"))
