"""Units of every size: rows of each degree up to the longest that a unit holds whole, with one and with several column
vectors, lane groups and units per workgroup."""
import numpy as np
import pytest

from test_gpu_preprocess_shapes import graph

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("team", [1, 2])
@pytest.mark.parametrize("N", [3, 6, 16, 33, 64, 256, 300])
def test_every_degree(gpu, team, N):
    rng = np.random.default_rng(N)
    deg = rng.permutation(np.concatenate([np.arange(1, 386), np.full(25, 1), np.full(23, 2), np.full(13, 5), np.full(12, 31)]))
    g = graph(gpu, deg, 3_001, seed=N)
    op = gpu.AccelSpMM(g.indptr, g.indices, g.values, g.n_cols).preprocess(plan_team=team, plan_split=384, plan_unit=384)
    X = rng.uniform(-1, 1, (g.n_cols, N)).astype(np.float32)
    Y = op.matmul(X)
    op.close()
    want = np.zeros((g.n_rows, N))
    rows = np.repeat(np.arange(g.n_rows), np.diff(g.indptr))
    np.add.at(want, rows, g.values.astype(np.float64)[:, None] * X[g.indices].astype(np.float64))
    assert np.abs(Y - want).max() <= 1e-5 * np.abs(want).max()
