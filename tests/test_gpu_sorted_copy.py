"""The sorted copy at the sizes where its kernels change: rows of one chunk, placed by four wavefronts that share their rounds
evenly, next to rows of several; more than 1,024 chunks, placed by smaller workgroups; tiles of whole rows that hold one
degree, a few, or very many.  Whole numbers, compared exactly with the oracle; products within its tolerance."""
import numpy as np
import pytest

from oracle import spmm_oracle as so
from test_gpu_preprocess import check_plan, check_preprocess
from test_gpu_preprocess_shapes import graph

pytestmark = pytest.mark.gpu


def check(gpu, deg, cols, groups=0, **options):
    g = graph(gpu, deg, cols)
    op = check_preprocess(gpu, g, plan_team=1, plan_groups=groups, **options)
    check_plan(op, g.n_cols)
    X = np.random.default_rng(2).uniform(-1, 1, (g.n_cols, 4)).astype(np.float32)
    assert so.check(op.matmul(X), g.indptr, g.indices, g.values, X) <= so.TOL
    v = np.random.default_rng(3).uniform(-1, 1, g.nnz).astype(np.float32)
    op.update_values(v)                                  # the same kernels, with positions instead of values
    assert so.check(op.matmul(X), g.indptr, g.indices, v, X) <= so.TOL
    op.close()


@pytest.mark.parametrize("groups", [0, 8, 16, 32, 64])
def test_rows_of_one_chunk(gpu, groups):
    edges = [64 * k + e for k in (16, 17, 20, 32, 48, 63, 64) for e in (-1, 0, 1)]
    small = [193, 255, 256, 257, 383, 384, 385, 640, 641, 1023, 1024, 0, 1, 5]
    check(gpu, np.random.default_rng(5).permutation(edges + small), 50_021, groups, plan_unit=384)


def test_many_chunks(gpu):
    rng = np.random.default_rng(6)
    check(gpu, rng.permutation(np.concatenate([4097 + 4 * rng.integers(0, 1200, 520), rng.integers(1, 1500, 300)])), 60_013,
          plan_unit=384)


@pytest.mark.parametrize("kind", ["ones", "one run", "two runs", "every degree", "few", "empty rows"])
@pytest.mark.parametrize("rows", [1, 300, 2047, 2049, 5000])
def test_tiles_of_whole_rows(gpu, kind, rows):
    rng = np.random.default_rng(rows)
    deg = {"ones": np.ones(rows, int), "one run": np.full(rows, 13), "two runs": np.where(np.arange(rows) % 2, 1, 191),
           "every degree": np.arange(rows) % 193, "few": rng.integers(1, 4, rows), "empty rows": rng.integers(0, 2, rows) * 7}[kind]
    deg[rng.integers(0, rows)] = 9                       # (at least one row that makes the order another)
    check(gpu, deg, 10_007, plan_unit=192)


@pytest.mark.parametrize("n", [15, 16, 17, 4096, 4097, 8191, 8192, 8193])
def test_number_of_long_rows(gpu, n):
    """Long rows compared with each other, sixteen to a workgroup and against 2,048 at a time, up to 8,192 of them."""
    rng = np.random.default_rng(n)
    deg = np.concatenate([385 + rng.integers(0, 3, n), rng.integers(0, 20, 300)])
    deg[:5] = (1024, 1025, 4097, 9000, 1025)
    check(gpu, rng.permutation(deg), 30_011, plan_unit=384)


@pytest.mark.parametrize("n", [64 * 2048, 64 * 2048 + 1])
def test_tiles_of_the_long_rows_sort(gpu, n):
    """Up to 64 tiles of 2,048 long rows the sort's second kernel adds up the counts of all tiles itself."""
    rng = np.random.default_rng(n)
    deg = rng.permutation(np.concatenate([385 + rng.integers(0, 9, n - 2), [1025, 70_000], rng.integers(0, 3, 100)]))
    indptr = np.concatenate([[0], np.cumsum(deg)]).astype(np.int32)
    op = gpu.AccelSpMM(indptr, np.zeros(indptr[-1], np.int32), np.ones(indptr[-1], np.float32), 4).preprocess()
    assert op.info.n_long_rows == n
    order = np.argsort(deg, kind="stable")
    assert np.array_equal(op.perm(), order)
    Y = op.matmul(np.ones((4, 4), np.float32))
    assert np.array_equal(Y, np.repeat(deg[:, None], 4, 1))           # whole numbers below 2^24: exact
    op.close()


@pytest.mark.parametrize("rows, degrees", [(70_000, (3, 30)), (9_000, (1, 193)), (4_000_000, (1, 2)), (300_000, (60, 64))])
def test_bands_of_tiles(gpu, rows, degrees):
    """8 to 256 bands of tiles, runs of one tile and of hundreds: every non-zero of the whole rows is copied once."""
    rng = np.random.default_rng(rows)
    deg = rng.integers(*degrees, rows)
    deg[rng.integers(0, rows, 3)] = (5, 9, 11)
    g = graph(gpu, deg, 20_011, seed=rows)
    op = gpu.AccelSpMM(g.indptr, g.indices, g.values, g.n_cols).preprocess()
    order = np.argsort(deg, kind="stable")
    start = np.concatenate([[0], np.cumsum(deg[order])])
    source = np.arange(g.nnz) - np.repeat(start[:-1] - g.indptr[order], deg[order])
    ip, ix, v = op.sorted_csr()
    assert np.array_equal(ip, start) and np.array_equal(ix, g.indices[source]) and np.array_equal(v, g.values[source])
    op.close()
