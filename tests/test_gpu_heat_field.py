"""ftd_heat_field to pageable memory (through the pinned ring from 16 MiB on)
against the same field copied by the runtime into pinned memory, on both
sides of that size and with whole and partial last pieces."""
import ctypes

import numpy as np
import pytest

from filtered_tdma_amd import _lib
from filtered_tdma_amd.heat import SolveTheta

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")


@pytest.mark.parametrize("nx,ny,nz", [
    (126, 126, 126),  # 16 MiB: the smallest field of the ring, whole pieces
    (125, 126, 126),  # just below
    (127, 126, 126),  # a partial last piece
    (254, 62, 142),   # 18 MiB: three rounds of the six threads
    (301, 97, 203),   # odd sizes, a ragged number of pieces
])
def test_heat_field_to_pageable_equals_pinned(nx, ny, nz):
    print(f"[gpu-case] heat field {nx}x{ny}x{nz}", flush=True)
    sim = SolveTheta(nx, ny, nz, backend="pascal", dt=1e-4)
    try:
        for _ in range(2):  # the second call with the ring in place
            sim.run(1)
            got = sim.field()
            pinned = torch.empty(sim.shape, dtype=torch.float64, pin_memory=True)
            _lib.check_heat(_lib.load().ftd_heat_field(sim._h, ctypes.c_void_p(pinned.data_ptr())))
            np.testing.assert_array_equal(got, pinned.numpy())
    finally:
        sim.close()
