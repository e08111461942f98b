"""Runs that copy X to rows on whole cache lines first give the packed run's result (accel_run_static never copies),
whatever the column count, the stride and the alignment of X; the GCN layer lays its own buffer out so."""
import ctypes as C

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
    assert np.array_equal(Y[:, :N].view(np.int32), S.view(np.int32))
    rows = np.concatenate([np.arange(0, ROWS, 997), [ROWS - 1, int(np.argmax(np.diff(graph[0])))]])
    want = expected(graph, X, rows)
    assert np.abs(Y[rows, :N] - want).max() <= 2e-5 * np.abs(want).max()


@pytest.mark.parametrize("N,shift", [(25, 0), (97, 0), (97, 3), (100, 0), (100, 1), (112, 2), (127, 0), (127, 2), (128, 0),
                                     (128, 1), (191, 0), (225, 1), (256, 3)])
def test_same_bits_where_nothing_can_be_copied(gpu, graph, N, shift):
    """Packed rows: a run that may copy X, accel_run_static and a captured run, on the same operands."""
    op = graph[3]
    hip = C.CDLL("libamdhip64.so.7")
    X = np.random.default_rng(N).standard_normal(shift + COLS * N).astype(np.float32)
    dX, dY = gpu.DeviceBuffer.from_numpy(X), gpu.DeviceBuffer(ROWS * N * 4)
    address = dX.address + 4 * shift
    stream, graph_, exe = C.c_void_p(), C.c_void_p(), C.c_void_p()
    assert hip.hipStreamCreate(C.byref(stream)) == 0

    def bits(run):
        dY.fill_u32(0x7FC00000)
        run()
        assert hip.hipDeviceSynchronize() == 0
        return dY.to_numpy(np.uint32, (ROWS, N))

    try:
        eager = bits(lambda: op.run(address, dY, N))
        assert np.isfinite(eager.view(np.float32)).all()
        if op.info.n_plan_pieces * N * 4 <= gpu._lib.STATIC_SCRATCH_BYTES:
            assert np.array_equal(bits(lambda: op.run_static(address, dY, N)), eager)
        assert hip.hipStreamBeginCapture(stream, 0) == 0
        op.run(address, dY, N, stream=stream.value)
        assert hip.hipStreamEndCapture(stream, C.byref(graph_)) == 0
        assert hip.hipGraphInstantiate(C.byref(exe), graph_, None, None, 0) == 0
        for _ in range(2):
            assert np.array_equal(bits(lambda: hip.hipGraphLaunch(exe, stream)), eager)
        assert hip.hipGraphExecDestroy(exe) == 0 and hip.hipGraphDestroy(graph_) == 0
    finally:
        assert hip.hipStreamDestroy(stream) == 0
        dX.close()
        dY.close()


def test_main_time_is_the_gather_kernels_alone(gpu, graph):
    """What a run that copies X first takes beyond its gather kernel holds the copy (204 MB, 12 us at twice the
    memory's rate), next to the same run on rows that are on whole lines already."""
    op, N = graph[3], 127
    dX, dY = gpu.DeviceBuffer.from_numpy(np.ones((COLS, 128), np.float32)), gpu.DeviceBuffer(ROWS * 128 * 4)
    beyond = [np.median(np.subtract(*op.time_ex(dX, dY, N, ld=ld, warmup=4, iters=20))) for ld in (127, 128)]
    dX.close()
    dY.close()
    assert beyond[0] - beyond[1] >= 0.012, beyond


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
