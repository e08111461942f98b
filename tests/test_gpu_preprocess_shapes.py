"""The preprocessing at the sizes where its kernels change: the last share of rows, tiles of
many runs, the ranking of long rows by comparison and by radix sort, chunks of wide rows, and
a launch plan that does not fit the room it is first given."""
import numpy as np
import pytest

from oracle import spmm_oracle as so
from test_gpu_preprocess import check_plan, check_preprocess

pytestmark = pytest.mark.gpu


def graph(gpu, deg, n_cols, seed=0):
    """Columns are a run of consecutive ones from a random start, wrapped: distinct within a row."""
    rng = np.random.default_rng(seed)
    deg = np.asarray(deg, dtype=np.int64)
    indptr = np.concatenate([[0], np.cumsum(deg)])
    k = np.arange(indptr[-1]) - np.repeat(indptr[:-1], deg)
    cols = (np.repeat(rng.integers(0, n_cols, deg.size), deg) + k) % n_cols
    values = rng.uniform(-1, 1, cols.size).astype(np.float32)
    return gpu.synthetic.Graph("shapes", indptr.astype(np.int32), cols.astype(np.int32), values, deg.size, n_cols)


def degrees(kind):
    rng = np.random.default_rng(5)
    if kind == "every degree":
        return rng.permutation(np.arange(386))                    # each once: every tile holds many runs
    if kind == "one row past a share":
        return np.full(64 * 4096 + 1, 1)                          # 64-row shares no longer reach
    if kind == "wide rows":
        return rng.permutation([1023, 1024, 1025, 4095, 4096, 4097, 8192, 8193, 20000, 3, 0, 192, 193, 384, 385])
    if kind == "8192 long rows":
        return rng.permutation(np.concatenate([np.full(8192, 385) + np.arange(8192) % 3, np.full(50, 2)]))
    if kind == "8193 long rows":
        return rng.permutation(np.concatenate([np.full(8193, 385) + np.arange(8193) % 3, [70000, 0, 5]]))
    raise ValueError(kind)


@pytest.mark.parametrize("kind", ["every degree", "one row past a share", "wide rows", "8192 long rows",
                                  "8193 long rows"])
def test_sizes_where_the_kernels_change(gpu, kind):
    g = graph(gpu, degrees(kind), 70_001)
    op = check_preprocess(gpu, g, plan_team=1, plan_unit=384)
    if g.n_rows < 1000:
        check_plan(op, g.n_cols)
    N = 4
    X = np.random.default_rng(1).uniform(-1, 1, (g.n_cols, N)).astype(np.float32)
    Y = op.matmul(X)
    assert so.check(Y, g.indptr, g.indices, g.values, X) <= so.TOL
    v = np.random.default_rng(2).uniform(-1, 1, g.nnz).astype(np.float32)      # the position map's kernels
    op.update_values(v)
    assert so.check(op.matmul(X), g.indptr, g.indices, v, X) <= so.TOL
    op.close()


def test_a_plan_that_does_not_fit_its_first_room(gpu):
    """Single light rows first, full units last: level in cost, the first queues hold six times
    their share of the units."""
    deg = np.concatenate([np.full(12 * 8000, 1), np.full(8000, 384)])
    g = graph(gpu, deg, 5000)
    op = gpu.AccelSpMM(g.indptr, g.indices, g.values, g.n_cols).preprocess(plan_team=1, plan_unit=384, plan_split=384)
    live = op.plan()[:, 3] != 0
    assert op.info.n_plan_units > 2 * live.sum()
    X = np.random.default_rng(3).uniform(-1, 1, (g.n_cols, 8)).astype(np.float32)
    assert so.check(op.matmul(X), g.indptr, g.indices, g.values, X) <= so.TOL
    op.close()


def test_memory_is_kept_for_the_next_handle_and_given_back(gpu):
    """A second handle of about the same size takes no new device memory, with and without streams in
    between; what is kept is freed on demand."""
    import ctypes as C
    hip = C.CDLL("libamdhip64.so.7")

    def free_bytes():
        assert hip.hipDeviceSynchronize() == 0
        free, total = C.c_size_t(), C.c_size_t()
        assert hip.hipMemGetInfo(C.byref(free), C.byref(total)) == 0
        return free.value

    def use(g):
        op = gpu.AccelSpMM(g.indptr, g.indices, g.values, g.n_cols).preprocess()
        op.run(dX, dY, 8)
        op.close()

    g1, g2 = graph(gpu, np.full(120_000, 40), 60_000), graph(gpu, np.full(118_000, 40), 60_000, seed=1)
    dX, dY = gpu.DeviceBuffer(60_000 * 8 * 4), gpu.DeviceBuffer(120_000 * 8 * 4)
    dX.fill_u32(0x3F800000)
    use(g1)
    before = free_bytes()
    use(g2)
    assert before - free_bytes() < 4 << 20
    gpu._lib.check(gpu.lib().accel_release_memory())
    assert free_bytes() - before > 50 << 20            # the CSR and its sorted copy: 77 MB
    use(g2)                                            # and it can be taken again
    assert so.check(dY.to_numpy(np.float32, (120_000, 8))[:118_000], g2.indptr, g2.indices, g2.values,
                    np.ones((60_000, 8), np.float32)) <= so.TOL
    dX.close()
    dY.close()


@pytest.mark.parametrize("rows", [524_287, 524_288, 4_194_303, 4_300_000])
def test_partition_stage_at_the_transfers_pieces(gpu, rows):
    """Row pointers that end at a piece of the transfer buffer (2 MiB), at the buffer itself
    (16 MiB) and beyond; the metadata of the last is longer than the buffer too."""
    deg = np.sort(np.random.default_rng(rows).integers(0, 40, rows))
    deg[-3:] = (400, 5000, 384 * 7)
    deg.sort()
    indptr = np.concatenate([[0], np.cumsum(deg)]).astype(np.int32)
    got = gpu.block_level_partition.partition(indptr, backend="gpu")
    assert np.array_equal(got, gpu.block_level_partition.partition(indptr, backend="host"))
