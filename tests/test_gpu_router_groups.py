"""Layers of 17-32 tokens on the per-pair kernels: the router's chain kernel
in two groups of 16 tokens (up to 256 experts), the general product past that,
against the oracle, bit for bit; with and without the norm in front, and from
rows that are not 16-byte aligned."""
import numpy as np
import pytest

import oracle as O

pytestmark = pytest.mark.gpu


def bits(a):
    return np.ascontiguousarray(a, dtype=np.float32).view(np.uint32)


@pytest.mark.parametrize("dtype,T,E,bias", [(2, 17, 128, False), (3, 17, 16, True), (3, 31, 60, False),
                                            (2, 32, 256, True), (3, 18, 257, False), (3, 33, 32, False)])
def test_router_token_groups(moehip, dtype, T, E, bias):
    print("router groups case", dtype, T, E, bias, flush=True)
    D, dff = 256, 128
    seed = 9700 + T + E
    ex = O.make_experts(dtype, E, D, dff, seed)
    rw = O.normal(E * D, seed + 10, 0.0, 0.05).reshape(E, D)
    rb = O.normal(E, seed + 11, 0.0, 0.05) if bias else None
    rms = O.normal(D, seed + 13, 1.0, 0.1)
    x = O.normal(T * D, seed + 12, 0.0, 1.0).reshape(T, D)
    x[T - 1] *= np.float32(30.0)     # the last token needs more limbs than the others
    layer = moehip.MoeLayer.from_arrays(dtype, rw, rb, ex.gq, ex.gs, ex.uq, ex.us, ex.dq, ex.ds, rms2_w=rms)
    layer.set_grouped_min_tokens(1000)   # the per-pair kernels at every T
    want, widx, wp, _ = O.moe_block(x, x, rw, rb, ex)
    for _ in range(2):
        got, idx, p = layer.forward(x, x)
        np.testing.assert_array_equal(idx, widx)
        np.testing.assert_array_equal(bits(p), bits(wp))
        np.testing.assert_array_equal(bits(got), bits(want))
    # a fresh layer call with the rows 4 bytes past a 16-byte boundary
    buf = moehip.DeviceBuffer(x.nbytes + 4)
    buf.upload(x, 4)
    out = moehip.DeviceBuffer(x.nbytes)
    layer.forward_dev(buf.ptr + 4, None, T, out.ptr)
    want0, _, _, _ = O.moe_block(x, None, rw, rb, ex)
    np.testing.assert_array_equal(bits(out.download((T, D), np.float32)), bits(want0))
    # norm in front
    xn = O.rmsnorm(x, rms, 1e-6)
    wantn, _, _, _ = O.moe_block(xn, x, rw, rb, ex)
    np.testing.assert_array_equal(bits(layer.block_forward(x, 1e-6)), bits(wantn))
