"""Rows of more than 384 non-zeros at the sizes where their kernels change: 64 to a workgroup, all of them in LDS up
to 2,048, equal degrees (ranked by row), wide rows of one to many chunks next to the counting of the split rows, rows in
order and not, and the partition stage by itself."""
import numpy as np
import pytest

from oracle import spmm_oracle as so
from test_gpu_preprocess import check_plan, check_preprocess
from test_gpu_preprocess_shapes import graph

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("order", ["any", "sorted"])
@pytest.mark.parametrize("n", [1, 63, 64, 65, 1000, 2047, 2048, 2049])
def test_number_of_long_rows(gpu, n, order):
    rng = np.random.default_rng(n)
    deg = np.concatenate([385 + rng.integers(0, 4, n), rng.integers(0, 30, 500)])
    deg[:min(n, 5)] = (1024, 1025, 4097, 9000, 1025)[:min(n, 5)]
    deg = np.sort(deg) if order == "sorted" else rng.permutation(deg)
    g = graph(gpu, deg, 30_011, seed=n)
    op = check_preprocess(gpu, g, plan_team=1, plan_unit=384)
    check_plan(op, g.n_cols)
    X = np.random.default_rng(1).uniform(-1, 1, (g.n_cols, 4)).astype(np.float32)
    assert so.check(op.matmul(X), g.indptr, g.indices, g.values, X) <= so.TOL
    op.close()
    if order == "sorted":
        got = gpu.block_level_partition.partition(g.indptr, backend="gpu")
        assert np.array_equal(got, gpu.block_level_partition.partition(g.indptr, backend="host"))


@pytest.mark.parametrize("groups", [0, 8, 64])
def test_chunks_of_wide_rows(gpu, groups):
    """1 to 18 chunks (more than the sixteen wavefronts that add up their counts), and split rows with none."""
    deg = np.random.default_rng(7).permutation(
        [1025, 4096, 4097, 2 * 4096, 2 * 4096 + 1, 16 * 4096, 16 * 4096 + 1, 17 * 4096 + 5, 193, 200, 384, 385, 1024, 7, 0])
    g = graph(gpu, deg, 100_003)
    op = check_preprocess(gpu, g, plan_team=1, plan_unit=384, plan_groups=groups)
    check_plan(op, g.n_cols)
    X = np.random.default_rng(2).uniform(-1, 1, (g.n_cols, 8)).astype(np.float32)
    assert so.check(op.matmul(X), g.indptr, g.indices, g.values, X) <= so.TOL
    v = np.random.default_rng(3).uniform(-1, 1, g.nnz).astype(np.float32)
    op.update_values(v)
    assert so.check(op.matmul(X), g.indptr, g.indices, v, X) <= so.TOL
    op.close()
