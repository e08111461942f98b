"""The dense product by two fp16 values per fp32 value (K >= 64, 1e9 multiplications and more for N > 64, 4e9 for
N = 33..64): edges of steps and tiles, strides, and magnitudes that its short range does not take."""
import numpy as np
import pytest

from oracle import spmm_oracle as so

pytestmark = pytest.mark.gpu


def rows_for(K, N):
    return int((1e9 if N > 64 else 4e9) / (K * N)) + 1


def product(gpu, X, W, ldx=0, ldz=0):
    rows, K = X.shape[0], W.shape[0]
    N = W.shape[1]
    dX, dW = gpu.DeviceBuffer.from_numpy(X), gpu.DeviceBuffer.from_numpy(W)
    dZ = gpu.DeviceBuffer((rows + 1) * (ldz or N) * 4)
    dZ.fill_u32(0x7FC00000)
    gpu.dense_xw(dX, dW, dZ, rows, K, N, ldx=ldx, ldz=ldz)
    gpu._lib.check(gpu.lib().accel_stream_sync(None))
    Z = dZ.to_numpy(np.float32, (rows + 1, ldz or N))
    for b in (dX, dW, dZ):
        b.close()
    assert np.isnan(Z[rows]).all() and np.isnan(Z[:, N:]).all()      # nothing written behind the rows and columns
    return Z[:rows, :N]


def picked(rng, rows):
    return np.unique(np.concatenate([np.arange(200), np.arange(rows - 200, rows), rng.integers(0, rows, 3000)]))


@pytest.mark.parametrize("K,N,more,pad", [(64, 128, 0, 0), (65, 65, 1, 3), (79, 100, 31, 0), (80, 127, 127, 5), (95, 130, 2, 0),
                                          (96, 256, 33, 0), (127, 193, 64, 1), (602, 128, 5, 0), (64, 64, 0, 0), (67, 33, 97, 2)])
def test_edges_of_steps_and_tiles(gpu, K, N, more, pad):
    rng = np.random.default_rng(K + N)
    rows = rows_for(K, N) + more
    X = rng.standard_normal((rows, K + pad), dtype=np.float32)
    W = rng.standard_normal((K, N)).astype(np.float32)
    Z = product(gpu, X, W, ldx=K + pad if pad else 0, ldz=N + pad if pad else 0)
    X = X[:, :K]
    pick = picked(rng, rows)
    # two operands to 2^-23, the product of what is below 2^-11 in both, and sums of 32 products rounded K / 32 times
    assert so.check_dense(Z[pick], X[pick], W) <= 2 * 2.0 ** -23 + 2.0 ** -24
    # and no further off than sums in fp32 (K roundings at random: sqrt(K) / 2 of 2^-24 of the result)
    want = X[pick].astype(np.float64) @ W.astype(np.float64)
    assert np.linalg.norm(Z[pick] - want) <= 2.0 ** -24 * (np.sqrt(K) / 2) * np.linalg.norm(want)


@pytest.mark.parametrize("case", ["few small", "rows", "row ends", "everywhere", "W entry", "W column", "growing columns", "sparse",
                                  "large"])
def test_magnitudes_far_apart(gpu, case):
    """Tiles whose magnitudes do not fit are computed another way: every element as exact as fp32 sums are."""
    rng = np.random.default_rng(5)
    K, N = 100, 128
    rows = rows_for(K, N) + 77
    X = rng.standard_normal((rows, K), dtype=np.float32)
    W = rng.standard_normal((K, N)).astype(np.float32)
    if case == "few small":
        X[::997, 3] = 3e-38
        X[5, 7] = 1e-42
    elif case == "rows":
        X[64:640] *= np.float32(2.0 ** -110)
    elif case == "row ends":
        X[:, -1] *= np.float32(2.0 ** -40)
    elif case == "everywhere":
        X *= np.exp2(rng.integers(-60, 60, X.shape)).astype(np.float32)
    elif case == "W entry":
        W[K // 2, 5] = 1e-38
    elif case == "W column":
        W[:, N // 2] *= np.float32(2.0 ** -101)
    elif case == "growing columns":
        X *= np.exp2(np.arange(K) // 8).astype(np.float32)
    elif case == "sparse":
        X *= rng.random(X.shape) < 0.02
        X[:, :40] = 0
        X[100:300] = 0
    elif case == "large":
        X[1000, 60] = 2.0 ** 103
        X[7, 0] = 2.0 ** 80
    Z = product(gpu, X, W)
    pick = picked(rng, rows)
    want = X[pick].astype(np.float64) @ W.astype(np.float64)
    scale = np.abs(X[pick]).astype(np.float64) @ np.abs(W).astype(np.float64)
    assert (np.abs(Z[pick] - want) <= (K + 1) * (2.0 ** -24 * scale + 2.0 ** -149)).all()


@pytest.mark.parametrize("where,value", [("X", np.inf), ("X", np.nan), ("X", -3.4e38), ("W", -np.inf), ("W", np.nan), ("W", 3.4e38)])
def test_infinities_and_nan(gpu, where, value):
    rng = np.random.default_rng(9)
    K, N = 70, 100
    rows = rows_for(K, N)
    X = rng.uniform(0.1, 1, (rows, K)).astype(np.float32)
    W = rng.uniform(1, 2, (K, N)).astype(np.float32)
    if where == "X":
        X[[37, 5000, rows - 1], [20, 69, 0]] = value
    else:
        W[37, 20] = value
    Z = product(gpu, X, W)
    pick = np.concatenate([np.arange(400), np.arange(4990, 5010), np.arange(rows - 100, rows)])
    with np.errstate(all="ignore"):
        want = X[pick].astype(np.float64) @ W.astype(np.float64)
        fits = np.abs(want) <= np.finfo(np.float32).max
        assert np.array_equal(np.isnan(Z[pick]), np.isnan(want))
        assert np.array_equal(np.isinf(Z[pick]), ~fits & ~np.isnan(want))
        assert np.array_equal(np.signbit(Z[pick])[~np.isnan(want)], np.signbit(want)[~np.isnan(want)])
    assert np.max(np.abs(Z[pick][fits] - want[fits]) / np.abs(want[fits])) <= (K + 1) * 2.0 ** -24
