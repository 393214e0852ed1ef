"""A heat field of more lines than one grid of the packing kernel holds (2^25
lines of 128 threads are 2^32): the initial field, ghosts included, against the
formula at lines from both ends, the middle and beside that count."""
import numpy as np
import pytest

from filtered_tdma_amd.heat import SolveTheta

pytestmark = pytest.mark.gpu

pytest.importorskip("torch")


def test_initial_field_of_many_lines():
    nx, n = 3, 5792  # 5794 * 5794 lines of 5 values, 1.3 GB
    assert (n + 2) ** 2 > 1 << 25
    print(f"[gpu-case] heat field {nx}x{n}x{n}", flush=True)
    sim = SolveTheta(nx, n, n, backend="pascal", dt=1e-4)
    try:
        f = sim.field()
    finally:
        sim.close()
    c = [-1 + 1 / m + (np.arange(m + 2) - 1) * (2 / m) for m in (nx, n)]
    s, k = [np.sin(np.pi * x) for x in c], [np.cos(np.pi * x) for x in c]
    last = (1 << 25) // (n + 2)  # the plane of line 2^25
    for z in (1, 2, n // 2, last - 1, last, last + 1, n):
        want = (s[1][z] * s[1][1:-1, None] * s[0][None, 1:-1]
                + k[1][z] * k[1][1:-1, None] * k[0][None, 1:-1])
        np.testing.assert_allclose(f[z, 1:-1, 1:-1], want, rtol=0, atol=1e-14)
        # the Dirichlet ghosts of the x walls: 2 u_wall - u
        wall = -k[1][z] * k[1][1:-1]
        np.testing.assert_allclose(f[z, 1:-1, 0], 2 * wall - f[z, 1:-1, 1], rtol=0, atol=1e-14)
        np.testing.assert_allclose(f[z, 1:-1, -1], 2 * wall - f[z, 1:-1, -2], rtol=0, atol=1e-14)
