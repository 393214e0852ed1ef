"""The field of a handle read by a thread whose current device is another one
(new threads start on device 0), below and above the pinned ring's size."""
import threading

import numpy as np
import pytest

from filtered_tdma_amd.heat import SolveTheta

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")


@pytest.mark.skipif(torch.cuda.device_count() < 2, reason="needs two GPUs")
@pytest.mark.parametrize("shape", [(40, 33, 36), (160, 130, 120)])
def test_field_read_on_another_current_device(shape):
    print(f"[gpu-case] heat field from another device {shape}", flush=True)
    with torch.cuda.device(1):
        sim = SolveTheta(*shape, backend="pascal", dt=2e-4)
        try:
            sim.run(1)
            got = []

            def read():
                torch.cuda.set_device(0)
                got.append(sim.field())
                got.append(torch.cuda.current_device())

            t = threading.Thread(target=read)
            t.start()
            t.join()
            assert got[1] == 0
            np.testing.assert_array_equal(got[0], sim.field())
        finally:
            sim.close()
