"""Filtered v1, tiles that take the full correction in the first pass: bitwise
against the oracle where all tiles, some of them or none ask for every row by
their own boundary maxima, on the streamed and the fused kernels, plain,
cyclic and with complex right-hand sides."""
import sys

import numpy as np
import pytest

import oracle as O
from filtered_tdma_amd import TdmaBackendGPU

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")

EPS = 1e-6
# n_sys, n_row, P: streamed (32 and 64 rows, all three partition counts),
# fused with ragged tiles, uneven partitions, one partition per wave
SIZES = [(256, 512, 8), (96, 250, 4), (128, 512, 16), (33, 100, 4), (65, 509, 8), (70, 41, 5)]
# the ratio of column 0 (which bounds J) and the scale from tile to tile: every
# tile full, none full, and a fall over many decades in which the first tiles
# are and the last are not
DATA = [(8.0, 1.0), (0.3, 1.0), (6.0, 1e-3), (2.0, 1e-6)]


def make(n_sys, n_row, r, fall, seed):
    rng = np.random.default_rng(seed)
    rr = np.full(n_sys, r)
    A = np.tile(-rr, (n_row, 1))
    B = np.tile(1 + 2 * rr, (n_row, 1))
    D = rng.uniform(-1.0, 1.0, (n_row, n_sys)) * fall ** (np.arange(n_sys) // 32)
    return A, B, A.copy(), D


@pytest.mark.parametrize("r,fall", DATA)
@pytest.mark.parametrize("n_sys,n_row,P", SIZES)
@pytest.mark.parametrize("cyclic", [False, True])
def test_first_pass_bits(n_sys, n_row, P, r, fall, cyclic):
    print(f"[gpu-case] v1 first pass {n_sys}x{n_row} P={P} r={r} fall={fall} cyclic={cyclic}",
          flush=True)
    sys.stdout.flush()
    A, B, C, D = make(n_sys, n_row, r, fall, n_sys + n_row)
    ref, J = O.filtered(A, B, C, D, P, 1, EPS, rho="auto", cyclic=cyclic, return_J=True)
    be = TdmaBackendGPU("filtered", n_sys, n_row, P, EPS)
    t = [torch.from_numpy(x).cuda() for x in (A, B, C, D)]
    be.set_rho_device(*t[:3])
    (be.solve_cyclic if cyclic else be.solve)(*t)
    path = be.last_path()
    assert path.startswith("filtered_v1_stream" if n_sys % 32 == 0 else "filtered_v1_fused"), path
    np.testing.assert_array_equal(t[3].cpu().numpy(), ref)
    np.testing.assert_array_equal(be.last_J(), J)


@pytest.mark.parametrize("r,fall", DATA)
def test_first_pass_complex(r, fall):
    n_sys, n_row, P = 40, 96, 4
    print(f"[gpu-case] v1 first pass complex r={r} fall={fall}", flush=True)
    A, B, C, D = make(n_sys, n_row, r, fall, 5)
    E = make(n_sys, n_row, r, fall, 6)[3] * 1e-5  # the parts keep their own J
    be = TdmaBackendGPU("filtered", n_sys, n_row, P, EPS)
    t = [torch.from_numpy(x).cuda() for x in (A, B, C)]
    be.set_rho_device(*t)
    Z = torch.from_numpy(D + 1j * E).cuda()
    be.solve_complex(*t, Z)
    z = Z.cpu().numpy()
    np.testing.assert_array_equal(z.real, O.filtered(A, B, C, D, P, 1, EPS, rho="auto"))
    np.testing.assert_array_equal(z.imag, O.filtered(A, B, C, E, P, 1, EPS, rho="auto"))
