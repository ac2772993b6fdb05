"""The fp32 product on rows of any length and 4-byte alignment against the
oracle's sequential loop, bit for bit: lengths under, at and past a chunk of
its four tile shapes, few short rows (a thread an output), every remainder of four columns, one row and one token,
and aligned lengths read from unaligned addresses."""
import numpy as np
import pytest

import oracle as O

pytestmark = pytest.mark.gpu


def bits(a):
    return np.ascontiguousarray(a, dtype=np.float32).view(np.uint32)


# (M, N, K, floats past a 16-byte boundary of A, of W)
SHAPES = [(1, 1, 1, 0, 0), (1, 70, 3, 0, 0), (4, 33, 63, 0, 0), (1, 1000, 65, 0, 0), (7, 31, 129, 1, 3),
          (33, 40, 1030, 0, 0), (20, 33, 64, 1, 0), (2, 50, 128, 0, 2), (500, 2050, 31, 0, 0), (505, 5100, 33, 0, 1),
          (1000, 8150, 35, 0, 0), (1000, 8150, 32, 3, 3),
          (2097185, 2, 5, 0, 0), (4, 33, 7, 0, 0), (300, 2048, 5, 0, 0), (300, 2800, 5, 0, 0), (64, 2000, 9, 0, 0),
          (20, 300, 15, 1, 1), (20, 300, 17, 0, 0), (5, 1000, 23, 0, 0), (5, 1000, 25, 0, 0), (9, 50, 8, 1, 0)]


@pytest.mark.parametrize("M,N,K,oa,ow", SHAPES)
def test_dense_any_rows(moehip, M, N, K, oa, ow):
    print("dense any case", M, N, K, oa, ow, flush=True)
    A = O.normal(M * K, 31 + M + K, 0.0, 1.0).reshape(M, K)
    W = O.normal(N * K, 37 + N, 0.0, 0.05).reshape(N, K)
    A[0, K - 1] = np.float32(3e38)      # a column past its row's end would show
    W[0, 0] = np.float32(-1e-38)
    dA, dW = moehip.DeviceBuffer(A.nbytes + 4 * oa), moehip.DeviceBuffer(W.nbytes + 4 * ow)
    dA.upload(A, 4 * oa)
    dW.upload(W, 4 * ow)
    dC = moehip.DeviceBuffer(M * N * 4)
    moehip.check(moehip.lib().moe_matmul_f32_dev(dA.ptr + 4 * oa, dW.ptr + 4 * ow, dC.ptr, M, N, K), "f32")
    with np.errstate(all="ignore"):
        want = O.matmul_f32(A, W)
    np.testing.assert_array_equal(bits(dC.download((M, N), np.float32)), bits(want))
