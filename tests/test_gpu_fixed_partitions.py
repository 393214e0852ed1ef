"""With rows per lane and threads given, the exact solve's partitions depend on
n_row alone: a system has the same bits in batches of any size. (Left to the
engine they depend on n_sys too.) And the general kernels keep plain Thomas."""
import sys

import numpy as np
import pytest

import oracle as O
from filtered_tdma_amd import Kind, TdmaBackendGPU, cases

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")


def solve(arrays, n, tuning):
    n_row = arrays[0].shape[0]
    be = TdmaBackendGPU(Kind.PASCAL, n, n_row, 1)
    try:
        be.set_tuning(*tuning)
        t = [torch.from_numpy(np.ascontiguousarray(x[:, :n])).cuda() for x in arrays]
        be.solve(*t)
        return t[3].cpu().numpy(), be.last_path()
    finally:
        be.close()


@pytest.mark.parametrize("n_row", [48, 64, 200, 480, 700, 1024])
def test_tuned_partitions_do_not_depend_on_the_batch(n_row):
    sizes = [1, 100, 8193, 70000 if n_row <= 200 else 10016]
    arrays = cases.general_batch(sizes[-1], n_row, seed=n_row)[:4]
    first, paths = None, set()
    for n in sizes:
        print(f"[gpu-case] fixed partitions n_sys={n} n_row={n_row}", flush=True)
        sys.stdout.flush()
        x, path = solve(arrays, n, (32, 512, 0, 0))
        paths.add(path)
        first = x[:, :1] if first is None else first
        np.testing.assert_array_equal(x[:, :1], first)
        if n >= 100:
            np.testing.assert_array_equal(x[:, :100], O.pascal(
                *[np.ascontiguousarray(v[:, :100]) for v in arrays],
                int(path.split("Q=")[1].split()[0]), sem=O.SEM_GPU))
    assert len(paths) == 1, paths


@pytest.mark.parametrize("n_row", [48, 700, 1500])
def test_general_kernels_keep_thomas(n_row):
    print(f"[gpu-case] thomas kept n_row={n_row}", flush=True)
    arrays = cases.general_batch(33, n_row, seed=n_row)[:4]
    # a zero on the diagonal that the whole system's elimination carries
    arrays[1][n_row // 2, 5] = 0.0
    x, path = solve(arrays, 33, (-1, 0, 0, 0))
    assert path == "thomas_general", path
    ref = O.thomas(*arrays, sem=O.SEM_GPU)
    assert np.isfinite(ref).all()
    np.testing.assert_array_equal(x, ref)
