"""One handle's field read by several threads at once, and by one while another
steps: every field read is one of the run's, whole, on both sides of the size
from which it goes through the pinned ring."""
import threading

import numpy as np
import pytest

from filtered_tdma_amd.heat import SolveTheta

pytestmark = pytest.mark.gpu

pytest.importorskip("torch")


@pytest.mark.parametrize("shape", [(40, 33, 36), (160, 130, 120)])
def test_field_from_several_threads(shape):
    print(f"[gpu-case] heat field threads {shape}", flush=True)
    sim = SolveTheta(*shape, backend="pascal", dt=2e-4)
    try:
        sim.run(1)
        want = sim.field()
        got = [None] * 4

        def read(k):
            for _ in range(5):
                got[k] = sim.field()
                if not np.array_equal(got[k], want):
                    return

        threads = [threading.Thread(target=read, args=(k,)) for k in range(4)]
        for t in threads:
            t.start()
        for t in threads:
            t.join()
        for f in got:
            np.testing.assert_array_equal(f, want)
    finally:
        sim.close()


@pytest.mark.parametrize("shape", [(40, 33, 36), (160, 130, 120)])
def test_field_beside_steps(shape):
    print(f"[gpu-case] heat field beside steps {shape}", flush=True)
    calls, steps = 8, 3
    sims = [SolveTheta(*shape, backend="pascal", dt=2e-4) for _ in range(2)]
    try:
        fields = [sims[1].field()]
        for _ in range(calls):
            sims[1].run(steps, use_graph=True)
            fields.append(sims[1].field())
        done = threading.Event()

        def step():
            for _ in range(calls):
                sims[0].run(steps, use_graph=True)
            done.set()

        t = threading.Thread(target=step)
        t.start()
        got = []
        while not done.is_set() and len(got) < 100:
            got.append(sims[0].field())
        t.join()
        got.append(sims[0].field())
        for f in got:
            assert any(np.array_equal(f, g) for g in fields)
        np.testing.assert_array_equal(got[-1], fields[-1])
    finally:
        for sim in sims:
            sim.close()
