"""The partition stage on rows in ascending degree order, whose entries are computed by their number: edges of the
pass that finds the runs (four rows per thread, workgroups that take several tiles), runs that are missing, and
fewer entries wanted than there are."""
import ctypes as C

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def entries(gpu, indptr, capacity):
    out, n = np.full((capacity + 1, 4), -7, np.int32), C.c_int64(0)
    gpu._lib.check(gpu.lib().accel_partition_gpu(gpu._lib.ptr(indptr, C.c_int32), indptr.size - 1,
                                                 gpu._lib.ptr(out, C.c_int32), capacity, C.byref(n)))
    return out, n.value


@pytest.mark.parametrize("rows", [1, 3, 4, 5, 63, 64, 255, 256, 257, 1023, 1024, 1025, 1_048_575, 1_048_576, 1_048_577, 1_300_001])
@pytest.mark.parametrize("kind", ["mixed", "one degree", "zero", "long"])
def test_edges_and_missing_runs(gpu, rows, kind):
    rng = np.random.default_rng(rows)
    if kind == "long":
        rows = min(rows, 2000)                             # (row pointers are int32)
    deg = {"mixed": lambda: np.sort(rng.choice([0, 1, 2, 33, 192, 383, 384, 385, 1000], rows, p=[.1, .4, .4, .04, .02, .01, .01, .01, .01])),
           "one degree": lambda: np.full(rows, 12), "zero": lambda: np.zeros(rows, np.int64),
           "long": lambda: np.sort(rng.integers(385, 5000, rows))}[kind]()
    indptr = np.concatenate([[0], np.cumsum(deg)]).astype(np.int32)
    want = gpu.block_level_partition.partition(indptr, backend="host").reshape(-1, 4)
    got, n = entries(gpu, indptr, len(want) + 3)
    assert n == len(want)
    assert np.array_equal(got[:n], want) and (got[n:] == -7).all()


@pytest.mark.parametrize("share", [0.0, 0.3, 0.9, 0.97, 1.0])
def test_fewer_entries_than_there_are(gpu, share):
    deg = np.sort(np.concatenate([np.random.default_rng(1).integers(0, 384, 5000), [385, 400, 384 * 3, 7000] * 10]))
    indptr = np.concatenate([[0], np.cumsum(deg)]).astype(np.int32)
    want = gpu.block_level_partition.partition(indptr, backend="host").reshape(-1, 4)
    capacity = int(len(want) * share)
    got, n = entries(gpu, indptr, capacity)
    assert n == len(want)
    assert np.array_equal(got[:capacity], want[:capacity]) and (got[capacity:] == -7).all()


def test_bad_row_pointers_are_refused(gpu):
    out, n = np.zeros((10, 4), np.int32), C.c_int64(0)
    for bad in ([1, 2, 3], [0, 3, 2]):
        indptr = np.asarray(bad, np.int32)
        rc = gpu.lib().accel_partition_gpu(gpu._lib.ptr(indptr, C.c_int32), indptr.size - 1, gpu._lib.ptr(out, C.c_int32), 10, C.byref(n))
        assert rc == gpu._lib.ERR_CSR
