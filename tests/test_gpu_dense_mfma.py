"""The many-token fp32 product (one MFMA product per output element, the adds
in column order) against the oracle's sequential loop, bit for bit: token and
row remainders of its four tile shapes, column remainders of its chunks, the
few-token sizes where it takes over from the chain kernel, and special values.
"""
import numpy as np
import pytest

import oracle as O

pytestmark = pytest.mark.gpu


def bits(a):
    return np.ascontiguousarray(a, dtype=np.float32).view(np.uint32)


def f32_dev(moehip, A, W):
    M, K = A.shape
    N = W.shape[0]
    dA, dW = moehip.DeviceBuffer.from_array(A), moehip.DeviceBuffer.from_array(W)
    dC = moehip.DeviceBuffer(M * N * 4)
    moehip.check(moehip.lib().moe_matmul_f32_dev(dA.ptr, dW.ptr, dC.ptr, M, N, K), "f32")
    return dC.download((M, N), np.float32)


# (M, N, K): one chunk and less, chunk tails of 4..60 columns, one row, rows
# and tokens one past a tile; the 32 x 64, 64 x 64 and 64 x 80 tiles with
# partial last tiles (many blocks, few columns); 5-16 tokens on both sides of
# the chain kernel's rule (its third, second and only block a CU: 6, 9 and 10
# tokens; one row past a round of its blocks); more 32-row, then 64-row tiles
# than a grid holds
SHAPES = [(17, 1, 4), (17, 31, 32), (32, 32, 60), (33, 33, 64), (31, 79, 68), (65, 81, 100),
          (48, 130, 2044), (500, 2050, 36), (505, 5100, 68), (1000, 8150, 36), (9, 1025, 2048),
          (16, 1100, 68), (5, 8001, 132), (5, 7999, 132), (8, 4999, 64), (8, 5001, 64),
          (9, 2048, 2048), (9, 2049, 2048), (10, 1024, 4100), (10, 1025, 4100), (6, 3072, 516), (6, 3073, 516),
          (7, 257, 8192), (16, 64, 8192), (12, 1030, 8192),
          (2097185, 3, 4), (4194305, 3, 4)]


@pytest.mark.parametrize("M,N,K", SHAPES)
def test_dense_mfma_shapes(moehip, M, N, K):
    print("dense case", M, N, K, flush=True)
    A = O.normal(M * K, 31 + M + K, 0.0, 1.0).reshape(M, K)
    W = O.normal(N * K, 37 + N, 0.0, 0.05).reshape(N, K)
    np.testing.assert_array_equal(bits(f32_dev(moehip, A, W)), bits(O.matmul_f32(A, W)))


def test_dense_mfma_special_values(moehip):
    """Products in and below the denormal range, overflow to infinity, signed
    zeros and infinities as the sequential loop gives them; NaN where it has
    NaN (the payload of a NaN is not compared)."""
    M, N, K = 40, 50, 132
    A = O.normal(M * K, 5, 0.0, 1.0).reshape(M, K)
    W = O.normal(N * K, 6, 0.0, 1.0).reshape(N, K)
    A[0] *= np.float32(1e-30)
    W[:10] *= np.float32(1e-12)       # row 0: sums of denormal and vanishing products
    A[1] *= np.float32(1e30)
    W[10:14] *= np.float32(1e9)       # row 1: products past the largest float
    A[2] = np.where(np.arange(K) % 2, np.float32(0.0), np.float32(-0.0))
    A[3, 100] = np.inf
    A[4, 131] = np.nan
    W[20, 7] = -np.inf
    with np.errstate(all="ignore"):
        want = O.matmul_f32(A, W)
    got = f32_dev(moehip, A, W)
    nan = np.isnan(want)
    assert nan.any() and np.isinf(want).any()
    assert (np.abs(want[0, :10]) < 1.2e-38).all() and (want[0, :10] != 0).any()
    np.testing.assert_array_equal(np.isnan(got), nan)
    np.testing.assert_array_equal(bits(got)[~nan], bits(want)[~nan])
