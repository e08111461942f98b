"""Runs that copy X to rows on whole cache lines first give the packed run's result (accel_run_static never copies),
whatever the column count, the stride and the alignment of X; the GCN layer lays its own buffer out so."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

ROWS, COLS, NNZ = 100_003, 200_003, 8_000_000


@pytest.fixture(scope="module")
def graph(gpu):
    """Random columns, 80 non-zeros per row on average, some rows long enough to be split, some empty."""
    rng = np.random.default_rng(7)
    weight = rng.pareto(2.0, ROWS) + 0.2
    weight[rng.integers(0, ROWS, 50)] = 0
    deg = np.minimum(rng.poisson(weight * (NNZ / weight.sum())), 9_000)
    indptr = np.zeros(ROWS + 1, np.int32)
    np.cumsum(deg, out=indptr[1:])
    idx = rng.integers(0, COLS, indptr[-1]).astype(np.int32)
    val = rng.standard_normal(indptr[-1]).astype(np.float32)
    op = gpu.AccelSpMM(indptr, idx, val, COLS).preprocess()
    yield indptr, idx, val, op
    op.close()


def expected(graph, X, rows):
    indptr, idx, val, _ = graph
    return np.stack([val[a:b].astype(np.float64) @ X[idx[a:b]].astype(np.float64) for a, b in
                     zip(indptr[rows], indptr[rows + 1])])


@pytest.mark.parametrize("N,ld,shift", [(16, 16, 3), (17, 17, 0), (25, 25, 1), (50, 50, 0), (56, 56, 0), (59, 61, 4),
                                        (95, 95, 0), (127, 127, 2), (127, 130, 0)])
def test_padded_run_is_the_packed_one(gpu, graph, N, ld, shift):
    op = graph[3]
    rng = np.random.default_rng(N)
    X = rng.standard_normal((COLS, N)).astype(np.float32)
    flat = np.full(shift + COLS * ld, np.nan, np.float32)
    flat[shift:].reshape(COLS, ld)[:, :N] = X
    dX = gpu.DeviceBuffer.from_numpy(flat)
    dP = gpu.DeviceBuffer.from_numpy(X)
    dY, dS = gpu.DeviceBuffer(ROWS * ld * 4), gpu.DeviceBuffer(ROWS * N * 4)
    dY.fill_u32(0x7FC00000)
    dS.fill_u32(0x7FC00000)
    try:
        op.run_strided(dX.address + 4 * shift, dY, N, ld)
        op.run_static(dP, dS, N)
        op.synchronize()
        Y = dY.to_numpy(np.float32, (ROWS, ld))
        S = dS.to_numpy(np.float32, (ROWS, N))
    finally:
        for b in (dX, dP, dY, dS):
            b.close()
    assert np.isnan(Y[:, N:]).all()
    if N > 96:                                         # two column panels: the sums are grouped otherwise
        assert np.abs(Y[:, :N] - S).max() <= 2e-5 * np.abs(S).max()
    else:
        assert np.array_equal(Y[:, :N].view(np.int32), S.view(np.int32))
    rows = np.concatenate([np.arange(0, ROWS, 997), [ROWS - 1, int(np.argmax(np.diff(graph[0])))]])
    want = expected(graph, X, rows)
    assert np.abs(Y[rows, :N] - want).max() <= 2e-5 * np.abs(want).max()


def test_layer_on_padded_rows(gpu, graph):
    op = graph[3]
    K, N = 24, 25
    assert op.row_stride(N) == 32 and op.row_stride(64) == 64
    rng = np.random.default_rng(3)
    X = rng.standard_normal((COLS, K)).astype(np.float32)
    W = rng.standard_normal((K, N)).astype(np.float32)
    b = rng.standard_normal(N).astype(np.float32)
    layer = gpu.GcnLayer(op, W, b, relu=True)
    Y = layer.forward_numpy(X)
    layer.close()
    rows = np.arange(0, ROWS, 499)
    want = np.maximum(expected(graph, (X.astype(np.float64) @ W), rows) + b, 0)
    assert np.abs(Y[rows] - want).max() <= 2e-5 * np.abs(want).max()
