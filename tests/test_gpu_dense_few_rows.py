"""The dense product on few rows, where the column tiles of a block of rows are workgroups of their own and narrower ones:
row counts around blocks of 128 and the lines of the rule, column counts around tiles, both ways to take values apart."""
import numpy as np
import pytest

from oracle import spmm_oracle as so
from test_gpu_dense_two_parts import product

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("rows", [1, 31, 129, 2000, 8192, 8193, 16385, 32769])
@pytest.mark.parametrize("N", [33, 64, 65, 96, 127, 128, 129, 200, 256, 300])
def test_rows_and_columns_around_the_lines(gpu, rows, N):
    rng = np.random.default_rng(rows + N)
    for K, pad in ((16, 0), (17, 3), (65, 1)):
        X = rng.standard_normal((rows, K + pad), dtype=np.float32)
        W = rng.standard_normal((K, N)).astype(np.float32)
        Z = product(gpu, X, W, ldx=K + pad if pad else 0, ldz=N + pad if pad else 0)
        X = X[:, :K]
        assert so.check_dense(Z, X, W) <= (K + 1) * 2.0 ** -24      # K sums, each rounded to 24 bits, and the products left out
        want = X.astype(np.float64) @ W.astype(np.float64)
        # roundings that go either way: sqrt(K) / 2 of them, and half a bit for a K as short as 16
        assert np.linalg.norm(Z - want) <= 2.0 ** -24 * (np.sqrt(K) / 2 + 0.5) * np.linalg.norm(want)


@pytest.mark.parametrize("K,rows,N", [(64, 32_768, 512), (250, 20_000, 256), (250, 30_001, 193), (700, 11_000, 130), (602, 10_000, 256)])
@pytest.mark.parametrize("what", ["ordinary", "far apart"])
def test_two_parts_with_tiles_apart(gpu, K, rows, N, what):
    """1e9 multiplications and more, and at most 512 tiles of 128 x 128; far apart: goes on in three parts."""
    assert rows * K * N >= 1e9 and -(-rows // 128) * -(-N // 128) <= 1024
    rng = np.random.default_rng(K)
    X = rng.standard_normal((rows, K), dtype=np.float32)
    if what == "far apart":
        X *= np.exp2(rng.integers(-50, 50, X.shape)).astype(np.float32)
    W = rng.standard_normal((K, N)).astype(np.float32)
    Z = product(gpu, X, W)
    pick = np.unique(np.concatenate([np.arange(150), np.arange(rows - 150, rows), rng.integers(0, rows, 1500)]))
    want = X[pick].astype(np.float64) @ W.astype(np.float64)
    scale = np.abs(X[pick]).astype(np.float64) @ np.abs(W).astype(np.float64)
    assert (np.abs(Z[pick] - want) <= (K + 1) * 2.0 ** -24 * scale).all()
    if what == "ordinary":
        assert so.check_dense(Z[pick], X[pick], W) <= 2 * 2.0 ** -23 + 2.0 ** -24


@pytest.mark.parametrize("K,rows,N", [(17, 66_000, 129), (40, 70_001, 200), (64, 70_000, 300), (100, 130_945, 515), (33, 200_000, 257)])
@pytest.mark.parametrize("what", ["ordinary", "far apart"])
def test_more_blocks_of_rows_than_are_under_way(gpu, K, rows, N, what):
    """Workgroups that keep their column tile and go from block to block (512 or 768 of them: more than 65,536 rows)."""
    rng = np.random.default_rng(K)
    X = rng.standard_normal((rows, K), dtype=np.float32)
    if what == "far apart":
        X *= np.exp2(rng.integers(-50, 50, X.shape)).astype(np.float32)
    W = rng.standard_normal((K, N)).astype(np.float32)
    Z = product(gpu, X, W)
    pick = np.unique(np.concatenate([np.arange(0, rows, 128), np.arange(127, rows, 128), np.arange(rows - 300, rows)]))
    want = X[pick].astype(np.float64) @ W.astype(np.float64)
    scale = np.abs(X[pick]).astype(np.float64) @ np.abs(W).astype(np.float64)
    assert (np.abs(Z[pick] - want) <= (K + 1) * 2.0 ** -24 * scale).all()
