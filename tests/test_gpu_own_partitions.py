"""Exact solves over partitions the engine chooses (one caller partition, or
more rows in one than a lane holds): every kernel and tile shape the choice
has, at the sizes where it changes, with rows on and off the 128-byte lines
and last tiles of one system. Bit for bit the oracle's PaScaL of the
partition count the path names, and within 1e-13 of serial Thomas."""
import sys

import numpy as np
import pytest

import oracle as O
from filtered_tdma_amd import Kind, TdmaBackendGPU, cases

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")


def note(msg):
    print(f"[gpu-case] {msg}", flush=True)
    sys.stdout.flush()


def path_Q(path):
    return int(path.split("Q=")[1].split()[0])


def solve(A, B, C, D, P=1, cyclic=False, tuning=None, shift=0):
    """x, path and the coefficients after the solve; shift: elements by which
    the arrays start off their allocation."""
    n_row, n_sys = D.shape

    def place(x):
        flat = torch.empty(x.size + shift, dtype=torch.float64, device="cuda")
        flat[shift:].copy_(torch.from_numpy(np.ascontiguousarray(x).reshape(-1)))
        return flat[shift:].view(n_row, n_sys)

    be = TdmaBackendGPU(Kind.PASCAL, n_sys, n_row, P)
    try:
        if tuning is not None:
            be.set_tuning(*tuning)
        t = [place(x) for x in (A, B, C, D)]
        (be.solve_cyclic if cyclic else be.solve)(*t)
        torch.cuda.synchronize()
        return t[3].cpu().numpy(), be.last_path(), [v.cpu().numpy() for v in t[:3]]
    finally:
        be.close()


def check(n_sys, n_row, P=1, cyclic=False, shift=0):
    A, B, C, D = cases.general_batch(n_sys, n_row, seed=n_sys + n_row)
    x, path, after = solve(A, B, C, D, P, cyclic, shift=shift)
    note(f"own partitions n_sys={n_sys} n_row={n_row} P={P} cyclic={cyclic} shift={shift}: {path}")
    ref = O.pascal(A, B, C, D, path_Q(path), sem=O.SEM_GPU, cyclic=cyclic)
    np.testing.assert_array_equal(x, ref, err_msg=path)
    for v, w in zip(after, (A, B, C)):
        np.testing.assert_array_equal(v, w, err_msg=path)
    th = O.thomas(A, B, C, D, sem=O.SEM_GPU, cyclic=cyclic)
    assert np.max(np.max(np.abs(x - th), 0) / np.max(np.abs(th), 0)) <= 1e-13, path
    return A, B, C, D, x, path


@pytest.mark.parametrize("cyclic", [False, True])
@pytest.mark.parametrize("n_sys,n_row", [
    (1, 65), (4096, 80), (4097, 256),      # 16-row lanes, 16- and 32-system tiles
    (8193, 100), (16385, 130),             # 64-system tiles; 32 off the lines
    (16400, 150), (16400, 256),            # 5 partitions (32) and 8 (64) on the lines
    (8208, 300), (8209, 300), (40, 448),   # above 256 rows: 32 on the lines, else 16
    (64, 449), (8224, 512), (65, 512),     # 8 streamed partitions, and off whole tiles
])
def test_own_partitions_bitwise(n_sys, n_row, cyclic):
    check(n_sys, n_row, cyclic=cyclic)


@pytest.mark.parametrize("n_sys,n_row", [(1, 33), (1000, 48), (16385, 64)])
def test_short_rows_of_a_small_batch(n_sys, n_row):
    """33 to 64 rows below 131072 systems: 16-row partitions; the periodic
    solve stays Sherman-Morrison Thomas."""
    path = check(n_sys, n_row)[5]
    assert path.startswith("pascal_fused M=16"), path
    A, B, C, D = cases.general_batch(n_sys, n_row, seed=2)
    x, path, _ = solve(A, B, C, D, cyclic=True)
    assert path.startswith("thomas_cyclic"), path
    np.testing.assert_array_equal(x, O.thomas(A, B, C, D, sem=O.SEM_GPU, cyclic=True))


@pytest.mark.parametrize("cyclic", [False, True])
@pytest.mark.parametrize("n_sys,n_row", [
    (8192, 513), (8193, 1024),             # 16 systems per tile, last tile of 1
    (2, 1025), (9, 1025), (2051, 1500), (24, 2048),   # 8 per tile
    (3, 2049), (5, 3000), (1030, 4095), (4, 4096),    # 4 per tile
])
def test_long_systems_bitwise(n_sys, n_row, cyclic):
    A, B, C, D, x, path = check(n_sys, n_row, cyclic=cyclic)
    assert path.startswith("pascal_stream"), path
    # the same partitions without the streamed kernels
    xf, pathf, _ = solve(A, B, C, D, cyclic=cyclic, tuning=(-2, 0, 0, 0))
    assert pathf.startswith("pascal_fused") and path_Q(pathf) == path_Q(path), pathf
    np.testing.assert_array_equal(xf, x)


@pytest.mark.parametrize("n_sys,n_row,P", [(100, 1500, 2), (33, 1030, 8), (5000, 200, 2)])
def test_caller_partitions_longer_than_a_lane(n_sys, n_row, P):
    check(n_sys, n_row, P=P)


@pytest.mark.parametrize("n_sys,n_row", [(2048, 100), (512, 300), (33, 1100), (2048, 2100)])
def test_own_partitions_at_element_alignment(n_sys, n_row):
    check(n_sys, n_row, shift=1)


@pytest.mark.parametrize("cyclic", [False, True])
@pytest.mark.parametrize("n_sys,n_row", [(131072, 33), (33, 32), (5, 3)])
def test_thomas_where_it_stays(n_sys, n_row, cyclic):
    A, B, C, D = cases.general_batch(n_sys, n_row, seed=9)
    note(f"thomas n_sys={n_sys} n_row={n_row} cyclic={cyclic}")
    x, path, _ = solve(A, B, C, D, cyclic=cyclic)
    assert path.startswith("thomas"), path
    np.testing.assert_array_equal(x, O.thomas(A, B, C, D, sem=O.SEM_GPU, cyclic=cyclic))


@pytest.mark.parametrize("d32", [False, True])
@pytest.mark.parametrize("n_sys,n_row", [(100, 40), (2048, 100), (16400, 256), (16416, 256),
                                         (8200, 300), (9000, 600)])
def test_f32_storage_own_partitions(n_sys, n_row, d32):
    A, B, C, D, _ = cases.toeplitz_batch(n_sys, n_row, 5.0, 500.0, seed=4)
    f = [v.astype(np.float32) for v in (A, B, C)]
    D32 = D.astype(np.float32) if d32 else D
    note(f"f32 own partitions n_sys={n_sys} n_row={n_row} d32={d32}")
    be = TdmaBackendGPU(Kind.PASCAL, n_sys, n_row, 1)
    try:
        t = [torch.from_numpy(v).cuda() for v in f]
        tD = torch.from_numpy(D32.copy()).cuda()
        X = torch.empty((n_row, n_sys), dtype=torch.float64, device="cuda") if d32 else tD
        if d32:
            be.solve_f32(*t, tD, X)
        else:
            be.solve_f32c(*t, X)
        torch.cuda.synchronize()
        x, path = X.cpu().numpy(), be.last_path()
    finally:
        be.close()
    w = [v.astype(np.float64) for v in f] + [D32.astype(np.float64)]
    np.testing.assert_array_equal(x, O.pascal(*w, path_Q(path), sem=O.SEM_GPU), err_msg=path)


def test_beyond_the_long_system_kernel():
    """Above 4096 rows, and a single system above 512 rows in a batch the
    other shapes do not hold: the lane-per-system Thomas, as before."""
    for n_sys, n_row in ((3, 4097), (1, 1025)):
        A, B, C, D = cases.general_batch(n_sys, n_row, seed=3)
        note(f"general n_sys={n_sys} n_row={n_row}")
        x, path, _ = solve(A, B, C, D)
        assert path == "thomas_general", path
        np.testing.assert_array_equal(x, O.thomas(A, B, C, D, sem=O.SEM_GPU))
