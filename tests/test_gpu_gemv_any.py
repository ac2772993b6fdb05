"""The untiled-shape GEMV kernel (unaligned 16-byte row chunks, activations
quantized per block) against the oracle, bit for bit."""
import ctypes

import numpy as np
import pytest

import oracle as O

pytestmark = pytest.mark.gpu


def bits(a):
    return np.ascontiguousarray(a, dtype=np.float32).view(np.uint32)


# (dtype, N, K): rows of exactly one chunk, one byte more, whole chunks, a
# last chunk that repeats 15 bytes; 31 / 32 / 33 chunks (16 lanes a row below
# 32, a wave from 32), 64 and 65 chunks (one and two per lane); 2048 rows and
# more with several tokens, 4096 with one (16 lanes a row for longer rows too),
# 4096 rows and more with 70 tokens (four rows a lane); the largest K of each
# token count (8 x 8192, 4 x 16384, 1 x 65536) and one past
SHAPES = [(2, 5, 16), (2, 7, 17), (2, 9, 48), (2, 33, 31), (2, 20, 496), (2, 20, 511), (2, 17, 513),
          (2, 130, 1023), (2, 130, 1030), (2, 4099, 66), (2, 9, 8191), (2, 9, 8193), (2, 6, 16385),
          (2, 3, 65535), (2, 3, 65537), (2, 2060, 1030), (2, 4100, 1023),
          (3, 5, 32), (3, 7, 34), (3, 33, 62), (3, 20, 992), (3, 17, 1026), (3, 130, 2050),
          (3, 4097, 70), (3, 9, 8190), (3, 9, 8194), (3, 6, 16386), (3, 3, 65534), (3, 2051, 1090)]


def variant(dtype, M, N, K):
    """The kernel these shapes are meant to reach."""
    nc = -(-(K if dtype == 2 else K // 2) // 16)
    if K > 65536:
        return "generic"
    mt = next(m for m in (1, 4, 8) if M <= m or m == 8)
    while mt > 1 and mt * K > 65536:
        mt = 4 if mt == 8 else 1
    rows = N * -(-M // mt)
    if mt > 1 and N >= 4096 and rows >= 32768:
        return "any_l16r4"
    many = rows >= max(2048, 12 * nc) if mt > 1 else rows >= max(4096, 20 * nc)
    return "any_l16" if nc < 32 or many else "any_l64"


def test_variants_reached():
    reached = {variant(d, M, N, K) for d, N, K in SHAPES for M in (1, 5, 70)}
    assert reached == {"any_l16", "any_l16r4", "any_l64", "generic"}
    assert any(variant(d, M, N, K) == "any_l16" and K > 1024 for d, N, K in SHAPES for M in (1, 5))


@pytest.mark.parametrize("dtype,N,K", SHAPES)
@pytest.mark.parametrize("M,scale", [(1, 1.0), (4, 0.05), (5, 30.0), (9, 1.0), (2, 1e5), (9, 1e5), (1, 1e9), (70, 300.0)])
def test_gemv_any_shapes(moehip, dtype, N, K, M, scale):
    print("gemv any case", dtype, N, K, M, scale, flush=True)
    assert moehip.gemv_variant(dtype, M, N, K) == variant(dtype, M, N, K)
    seed = dtype * 100000 + N * 31 + K * 7 + M
    A = O.normal(M * K, seed, 0.0, scale).reshape(M, K)
    rb = K if dtype == 2 else K // 2
    q = (O.uniform_u32(N * rb, seed + 1) & 0xFF).astype(np.uint8)
    q = (q.view(np.int8) if dtype == 2 else q).reshape(N, rb)
    s = O.normal(N, seed + 2, 0.0, 0.01)
    want = (O.gemv_q8 if dtype == 2 else O.gemv_q4)(A, q, s, N, K)
    L = moehip.lib()
    # the weights from an odd address, with bytes of another value around them
    raw = np.full(rb * N + 65, 0x5A, np.uint8)
    raw[33:33 + rb * N] = q.reshape(-1).view(np.uint8)
    dA, dq, ds = (moehip.DeviceBuffer.from_array(v) for v in (A, raw, s))
    dC = moehip.DeviceBuffer(M * N * 4)
    f = L.moe_matmul_q8_dev if dtype == 2 else L.moe_matmul_q4_dev
    moehip.check(f(dA.ptr, dq.ptr + 33, ds.ptr, dC.ptr, M, N, K), "gemv")
    np.testing.assert_array_equal(bits(dC.download((M, N), np.float32)), bits(want))


# (dtype, jobs, M, N, K): rows a multiple of 16 bytes without a tiled
# geometry; blocks of one row unit and, past 2048 units, of several with a
# partial last one; 16 lanes and (7 rows) a wave a row; tokens past a block's
@pytest.mark.parametrize("dtype,nj,M,N,K", [(2, 3, 1, 7, 1040), (2, 5, 4, 100, 96), (3, 5, 9, 100, 96),
                                            (2, 300, 1, 200, 112), (3, 40, 5, 1000, 96), (2, 2, 2, 9000, 80),
                                            (3, 9, 3, 4100, 160), (2, 1, 1, 40000, 48)])
@pytest.mark.parametrize("scale", [1.0, 1e5])
def test_gemv_any_batched(moehip, dtype, nj, M, N, K, scale):
    print("gemv any batched", dtype, nj, M, N, K, scale, flush=True)
    assert moehip.gemv_variant(dtype, M, N, K).startswith("any")
    rb = K if dtype == 2 else K // 2
    q = (O.uniform_u32(nj * N * rb, 11 + K) & 0xFF).astype(np.uint8)
    q = (q.view(np.int8) if dtype == 2 else q).reshape(nj, N, rb)
    s = O.normal(nj * N, 12, 0.0, 0.01).reshape(nj, N)
    A = O.normal(nj * M * K, 13 + M, 0.0, scale).reshape(nj, M, K)
    dq, ds, dA = (moehip.DeviceBuffer.from_array(v) for v in (q, s, A))
    dC = moehip.DeviceBuffer(nj * M * N * 4)
    jobs = (moehip.QJob * nj)(*[moehip.QJob(dq.ptr + j * N * rb, ds.ptr + j * N * 4, dA.ptr + j * M * K * 4,
                                            dC.ptr + j * M * N * 4) for j in range(nj)])
    dj = moehip.DeviceBuffer(ctypes.sizeof(jobs))
    L = moehip.lib()
    moehip.check(L.moe_memcpy_h2d(dj.ptr, ctypes.addressof(jobs), ctypes.sizeof(jobs)))
    moehip.check(L.moe_matmul_q_batched_dev(dtype, dj.ptr, nj, M, N, K), "batched")
    got = dC.download((nj, M, N), np.float32)
    f = O.gemv_q8 if dtype == 2 else O.gemv_q4
    for j in range(nj):
        np.testing.assert_array_equal(bits(got[j]), bits(f(A[j], q[j], s[j], N, K)), err_msg=f"job {j}")
