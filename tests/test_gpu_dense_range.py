"""The dense product where its three-part bf16 arithmetic could go wrong: magnitudes from the
smallest to the largest, infinities and NaN, values that need all 24 bits, K around the halves and
steps of the walk, and the shapes that take W apart beforehand, on two streams and in a graph."""
import ctypes as C

import numpy as np
import pytest

from oracle import spmm_oracle as so

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("K", [15, 16, 17, 31, 32, 33, 47, 48, 63, 65, 95, 602])
@pytest.mark.parametrize("N", [5, 33, 100])
def test_k_around_halves_and_steps(gpu, K, N):
    rng = np.random.default_rng(K * 7 + N)
    X = rng.standard_normal((259, K)).astype(np.float32)
    W = rng.standard_normal((K, N)).astype(np.float32)
    assert so.check_dense(gpu.dense_xw_numpy(X, W), X, W) <= 3e-7       # what fp32 arithmetic gives


@pytest.mark.parametrize("exponent", [-120, -100, -60, 60, 100])
def test_magnitudes(gpu, exponent):
    """Scaling X by a power of two scales the result by it exactly."""
    rng = np.random.default_rng(abs(exponent))
    X = rng.uniform(0.5, 1, (200, 64)).astype(np.float32) * np.where(rng.random((200, 64)) < 0.5, -1, 1).astype(np.float32)
    W = rng.standard_normal((64, 40)).astype(np.float32)
    Z = gpu.dense_xw_numpy(np.ldexp(X, exponent).astype(np.float32), W)
    want = np.ldexp(gpu.dense_xw_numpy(X, W).astype(np.float64), exponent)
    err = np.abs(Z - want) / np.ldexp(np.abs(X).astype(np.float64) @ np.abs(W), exponent)
    assert err.max() <= 3e-7


@pytest.mark.parametrize("where", ["X", "W"])
@pytest.mark.parametrize("value", [np.inf, -np.inf, np.nan, 3.4e38, 1.8e38])
def test_values_the_matrix_path_does_not_take(gpu, where, value):
    rng = np.random.default_rng(9)
    X = rng.uniform(0.1, 1, (300, 50)).astype(np.float32)
    W = np.exp2(rng.integers(-3, 3, (50, 70))).astype(np.float32) * np.float32(0.25)     # bf16 values: one part
    (X if where == "X" else W)[37, 20] = value
    if where == "X":
        X[38, 3] = -3.3e38
    Z = gpu.dense_xw_numpy(X, W)
    with np.errstate(all="ignore"):
        want = (X.astype(np.float64) @ W.astype(np.float64))
    special = ~np.isfinite(want) | (np.abs(want) > np.finfo(np.float32).max)
    assert np.array_equal(np.isnan(Z), np.isnan(want))
    assert np.array_equal(np.sign(Z[special & ~np.isnan(want)]), np.sign(want[special & ~np.isnan(want)]))
    assert np.isinf(Z[special & ~np.isnan(want)]).all()
    ok = ~special
    assert np.max(np.abs(Z[ok] - want[ok]) / (np.abs(X).astype(np.float64) @ np.abs(W))[ok]) <= 1e-6


def test_all_24_bits_survive(gpu):
    """Columns of X picked by a unit weight come back bit for bit, whatever their bits."""
    rng = np.random.default_rng(2)
    bits = rng.integers(0, 1 << 23, (500, 33)).astype(np.uint32) | (rng.integers(90, 160, (500, 33)).astype(np.uint32) << 23)
    X = bits.view(np.float32)
    for N in (20, 64, 128):
        W = np.zeros((33, N), np.float32)
        W[np.arange(min(N, 33)), np.arange(min(N, 33))] = 1
        Z = gpu.dense_xw_numpy(X, W)
        assert np.array_equal(Z[:, :min(N, 33)].view(np.uint32), X[:, :min(N, 33)].view(np.uint32))


def test_prepared_weights_on_two_streams(gpu):
    """Products large enough to take W apart beforehand, with different weights, queued in turn on the
    null stream and on another: each gets its own weights."""
    hip = C.CDLL("libamdhip64.so.7")
    rows, K, N = 300_000, 300, 128                       # 1.15e10 multiplications
    rng = np.random.default_rng(4)
    X = rng.uniform(-1, 1, (rows, K)).astype(np.float32)
    Ws = [rng.standard_normal((K, N)).astype(np.float32) for _ in range(4)]
    dX = gpu.DeviceBuffer.from_numpy(X)
    dW = [gpu.DeviceBuffer.from_numpy(w) for w in Ws]
    dZ = [gpu.DeviceBuffer(rows * N * 4) for _ in Ws]
    stream = C.c_void_p()
    assert hip.hipStreamCreateWithFlags(C.byref(stream), 1) == 0          # does not wait for the null stream
    for rep in range(3):
        for i, z in enumerate(dZ):
            gpu.dense_xw(dX, dW[i], z, rows, K, N, stream=stream.value if i % 2 else None)
    assert hip.hipStreamSynchronize(stream) == 0
    gpu._lib.check(gpu.lib().accel_stream_sync(None))
    pick = rng.integers(0, rows, 2000)
    for i, z in enumerate(dZ):
        Z = z.to_numpy(np.float32, (rows, N))
        assert so.check_dense(Z[pick], X[pick], Ws[i]) <= 3e-7
        z.close(); dW[i].close()
    dX.close()
    assert hip.hipStreamDestroy(stream) == 0


@pytest.mark.parametrize("where", ["X", "W", "both"])
@pytest.mark.parametrize("K,N", [(9, 40), (33, 20), (100, 50), (160, 128), (67, 130)])
def test_small_magnitudes_among_ordinary_values(gpu, where, K, N):
    """Values below 2^-100 (denormals among them) next to ordinary ones, in a few places or everywhere, also where
    whole rows hold nothing else: every element as exact as fp32 sums are."""
    rng = np.random.default_rng(K + N)
    rows = 300
    X = rng.standard_normal((rows, K)).astype(np.float32)
    W = rng.standard_normal((K, N)).astype(np.float32)
    if where != "W":
        X[rng.random(X.shape) < 0.02] = 3e-38
        X[40:80] *= np.float32(2.0 ** -110)
        X[81, K // 2] = 1e-42
    if where != "X":
        W[K // 3] *= np.float32(2.0 ** -104)
        W[:, N // 2] *= np.float32(2.0 ** -101) if where == "W" else np.float32(1)
    Z = gpu.dense_xw_numpy(X, W)
    want = X.astype(np.float64) @ W.astype(np.float64)
    scale = np.abs(X).astype(np.float64) @ np.abs(W).astype(np.float64)
    # K additions, each rounded to 24 bits or to a multiple of the smallest number
    assert (np.abs(Z - want) <= (K + 1) * (2.0 ** -24 * scale + 2.0 ** -149)).all()


@pytest.mark.parametrize("value", [2.0 ** 78, 2.0 ** 80, 2.0 ** 103])
def test_large_magnitudes_among_ordinary_values(gpu, value):
    """Where an operand or a sum leaves the range of the scaled values, the tile is computed again."""
    rng = np.random.default_rng(3)
    X = rng.standard_normal((200, 70)).astype(np.float32)
    W = rng.standard_normal((70, 100)).astype(np.float32)
    X[100, 60] = value
    W[4, 99] = -value
    Z = gpu.dense_xw_numpy(X, W)
    assert so.check_dense(Z, X, W) <= 71 * 2.0 ** -24


@pytest.mark.parametrize("where,value,limit", [("W", 1e-38, 2), ("X", 1e-38, 2), ("X", np.inf, 8)])
def test_speed_does_not_hang_on_single_values(gpu, where, value, limit):
    """Small values cost nothing; an infinity makes its tile be computed again, by fp32 instructions (in every
    tile that is some three times the time)."""
    hip = C.CDLL("libamdhip64.so.7")
    rows, K, N = 60_000, 256, 128
    rng = np.random.default_rng(1)
    X = rng.uniform(-1, 1, (rows, K)).astype(np.float32)
    W = rng.standard_normal((K, N)).astype(np.float32)

    def milliseconds():
        dX, dW, dZ = gpu.DeviceBuffer.from_numpy(X), gpu.DeviceBuffer.from_numpy(W), gpu.DeviceBuffer(rows * N * 4)
        ev = [C.c_void_p() for _ in range(2)]
        for e in ev:
            assert hip.hipEventCreate(C.byref(e)) == 0
        for _ in range(3):
            gpu.dense_xw(dX, dW, dZ, rows, K, N)
        assert hip.hipEventRecord(ev[0], None) == 0
        for _ in range(5):
            gpu.dense_xw(dX, dW, dZ, rows, K, N)
        assert hip.hipEventRecord(ev[1], None) == 0 and hip.hipEventSynchronize(ev[1]) == 0
        t = C.c_float()
        assert hip.hipEventElapsedTime(C.byref(t), *ev) == 0
        for e in ev:
            assert hip.hipEventDestroy(e) == 0
        for b in (dX, dW, dZ):
            b.close()
        return t.value / 5

    plain = milliseconds()
    (W if where == "W" else X)[K // 2, 5] = value
    if where == "X":
        X[rng.integers(0, rows, 200), rng.integers(0, K, 200)] = value
    assert milliseconds() <= limit * plain


@pytest.mark.parametrize("rows,N", [(1, 1), (31, 33), (300, 20), (1000, 100), (129, 300)])
def test_one_product_per_sum_is_rounded_once(gpu, rows, N):
    """K = 1: every element is one fp32 product, correctly rounded."""
    rng = np.random.default_rng(rows + N)
    X = rng.standard_normal((rows, 1)).astype(np.float32)
    W = rng.standard_normal((1, N)).astype(np.float32)
    assert np.array_equal(gpu.dense_xw_numpy(X, W).view(np.uint32), (X * W).view(np.uint32))


@pytest.mark.parametrize("K", [2, 3, 7, 8, 14, 15])
@pytest.mark.parametrize("N", [5, 33, 100, 260])
def test_short_k(gpu, K, N):
    """Below half a step of the walk: sums of K rounded additions, infinities where they belong, and in rows that
    are further apart than K nothing between them is read."""
    rng = np.random.default_rng(K + N)
    X = rng.standard_normal((1000, K)).astype(np.float32)
    W = rng.standard_normal((K, N)).astype(np.float32)
    assert so.check_dense(gpu.dense_xw_numpy(X, W), X, W) <= (K + 1) * 2.0 ** -24
    ld = K + 3
    wide = np.full((1000, ld), np.nan, np.float32)
    wide[:, :K] = X
    wide[70, K - 1] = np.inf
    W[0, 3] = np.inf
    dX, dW, dZ = gpu.DeviceBuffer.from_numpy(wide), gpu.DeviceBuffer.from_numpy(W), gpu.DeviceBuffer(1000 * (N + 5) * 4)
    dZ.fill_u32(0x7FC00000)
    gpu.dense_xw(dX, dW, dZ, 1000, K, N, ldx=ld, ldz=N + 5)
    gpu._lib.check(gpu.lib().accel_stream_sync(None))
    Z = dZ.to_numpy(np.float32, (1000, N + 5))
    for b in (dX, dW, dZ):
        b.close()
    X[70, K - 1] = np.inf
    with np.errstate(all="ignore"):
        want = X.astype(np.float64) @ W.astype(np.float64)
    assert np.isnan(Z[:, N:]).all()
    assert np.array_equal(np.isfinite(Z[:, :N]), np.isfinite(want))
    assert np.array_equal(np.isnan(Z[:, :N]), np.isnan(want))
