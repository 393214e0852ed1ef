"""Filtered v1 on the streamed kernel where a workgroup takes several turns: the
second pass leaves out the (tile, partition pair)s that the first has stored.
Stored and remaining ones mixed at random, remaining ones alone, and more than
64 turns a workgroup (the list of turns is filled again), its first 64 all
stored in some; bit for bit the oracle's."""
import sys

import numpy as np
import pytest

import oracle as O
from filtered_tdma_amd import TdmaBackendGPU

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")

R = 0.3  # a = c = -R, b = 1 + 2 R
LIMIT = 1e-3


def eps_of(m):
    """The eps for which a boundary maximum of LIMIT or more asks for J = m - 1."""
    rho = R / (1 + 2 * R)
    q = rho / ((1 + np.sqrt(1 - 4 * rho * rho)) * 0.5)
    return LIMIT * q * (2 + q) / ((1 - q) * (1 - 2 * rho)) * q ** (m - 2)


def solve(n_sys, n_row, P, high):
    """high [tiles, P]: where D is of order 1, else of order 1e-9."""
    rng = np.random.default_rng(n_sys)
    m = n_row // P
    D = rng.uniform(0.5, 1.0, (n_row, n_sys))
    D *= np.repeat(np.repeat(np.where(high, 1.0, 1e-9).T, m, axis=0), 32, axis=1)
    A = np.full((n_row, n_sys), -R)
    B = np.full((n_row, n_sys), 1 + 2 * R)
    be = TdmaBackendGPU("filtered", n_sys, n_row, P)
    try:
        be.set_eps(eps_of(m))
        t = [torch.from_numpy(x).cuda() for x in (A, B, A, D)]
        be.set_rho_device(*t[:3])
        be.solve(*t)
        x, J, path = t[3].cpu().numpy(), be.last_J(), be.last_path()
    finally:
        be.close()
    assert path.startswith("filtered_v1_stream"), path
    ref, Jref = O.filtered(A, B, A, D, P, 1, eps_of(m), eps_direct=True, sem=O.SEM_GPU, rho="auto",
                           return_J=True)
    assert list(J) == list(Jref)
    np.testing.assert_array_equal(x, ref)
    # which (tile, partition pair)s the first pass could store
    ends = np.maximum(np.abs(ref[0::m]), np.abs(ref[m - 1::m]))  # [P, n_sys]
    full = ends.reshape(P, -1, 32).max(axis=2) >= LIMIT
    return full.reshape(P // 2, 2, -1).all(axis=1)


# 64-row lanes, one and two workgroups per CU, and 32-row ones
@pytest.mark.parametrize("n_sys,n_row,P", [(40000, 40 * 8, 8), (50016, 36 * 4, 4), (40000, 24, 8),
                                           (36000, 48, 16)])
@pytest.mark.parametrize("share", [0.0, 0.05, 0.3])
def test_mixed_turns(n_sys, n_row, P, share):
    print(f"[gpu-case] v1 turns {n_sys}x{n_row} P={P} share={share}", flush=True)
    sys.stdout.flush()
    high = np.random.default_rng(P).uniform(size=(n_sys // 32, P)) < share
    stored = solve(n_sys, n_row, P, high)
    assert stored.any() == (share > 0) and not stored.all()


def test_more_than_64_turns():
    n_sys, n_row, P = 33000 * 32, 24, 8
    print(f"[gpu-case] v1 turns {n_sys}x{n_row} P={P}", flush=True)
    sys.stdout.flush()
    rng = np.random.default_rng(7)
    high = rng.uniform(size=(33000, P)) < 0.2
    first = np.arange(33000) % 512 < 100  # workgroups of a grid of 512
    high[first] = True
    high[:100] = False  # and the one turn left to each of them
    stored = solve(n_sys, n_row, P, high)
    assert stored[:, 512:][:, first[512:]].all() and not stored[:, :100].any()
