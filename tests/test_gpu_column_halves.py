"""Launches in which every other die computes the other half of the columns: widths of two and of several panels, a
last panel that is not full, rows of Y on whole lines or not, rows without non-zeros, split rows added up in the
launch and by a second kernel, bias and ReLU."""
import numpy as np
import pytest

from test_gpu_preprocess_shapes import graph

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module", params=[1, 2], ids=["reduced in the launch", "reduced behind it"])
def product(gpu, request):
    rng = np.random.default_rng(11)
    deg = rng.permutation(np.concatenate([np.zeros(700, int), rng.integers(1, 40, 2000), np.arange(180, 420), [3000, 9000]]))
    g = graph(gpu, deg, 10_007, seed=2)
    op = gpu.AccelSpMM(g.indptr, g.indices, g.values, g.n_cols).preprocess(plan_team=1, plan_reduce=request.param)
    yield g, op
    op.close()


@pytest.mark.parametrize("N,ld", [(64, 64), (97, 128), (128, 128), (127, 128), (192, 192), (227, 256), (256, 260), (320, 320)])
@pytest.mark.parametrize("epilogue", [False, True])
def test_column_halves(gpu, product, N, ld, epilogue):
    g, op = product
    rng = np.random.default_rng(N)
    X = np.full((g.n_cols, ld), np.nan, np.float32)
    X[:, :N] = rng.uniform(-1, 1, (g.n_cols, N))
    bias = rng.uniform(-1, 1, N).astype(np.float32)
    dX, dY, dB = gpu.DeviceBuffer.from_numpy(X), gpu.DeviceBuffer(g.n_rows * ld * 4), gpu.DeviceBuffer.from_numpy(bias)
    dY.fill_u32(0x7FC00000)
    try:
        for _ in range(2):                             # the second run finds the counters of the first
            op.run_ex(dX, dY, N, ld=ld, bias=dB if epilogue else None, relu=epilogue)
        op.synchronize()
        Y = dY.to_numpy(np.float32, (g.n_rows, ld))
    finally:
        for b in (dX, dY, dB):
            b.close()
    assert np.isnan(Y[:, N:]).all()
    rows = np.repeat(np.arange(g.n_rows), np.diff(g.indptr))
    want = np.zeros((g.n_rows, N))
    np.add.at(want, rows, g.values.astype(np.float64)[:, None] * X[g.indices, :N].astype(np.float64))
    if epilogue:
        want = np.maximum(want + bias, 0)
    assert np.abs(Y[:, :N] - want).max() <= 1e-5 * np.abs(want).max()
