"""The expert-major Q8 kernels' two-limb passes against the oracle, bit for
bit, at the edges of their pair tiles: 8 experts with top-8, so that every
expert takes every token."""
import numpy as np
import pytest

import oracle as O

pytestmark = pytest.mark.gpu


def bits(a):
    return np.ascontiguousarray(a, dtype=np.float32).view(np.uint32)


# tokens = pairs per expert: one tile of 32 and less, just past it, the 256-pair
# shape with 64 and 65 pairs, a full two-limb pass of 128 and one more, a split
# task; x scales for 1-, 2- and 4-limb activations
# (2 limbs: one pass; 4: two passes); d_ff = 192: a partial gate/up tile and
# three down stages; d_ff = 128: fewer stages than the ring holds
@pytest.mark.parametrize("scale", [0.3, 1.0, 400.0])
@pytest.mark.parametrize("T,dff", [(1, 128), (24, 192), (33, 192), (64, 128), (65, 192), (128, 192),
                                   (129, 192), (257, 128)])
def test_expert_limb_passes(moehip, T, dff, scale):
    E, D, dtype = 8, 384, 2
    print("expert limbs case", T, dff, scale, flush=True)
    seed = 9300 + T
    ex = O.make_experts(dtype, E, D, dff, seed)
    rw = O.normal(E * D, seed + 10, 0.0, 0.02).reshape(E, D)
    xn = O.normal(T * D, seed + 12, 0.0, scale).reshape(T, D)
    want, widx, wp, _ = O.moe_block(xn, xn, rw, None, ex)
    layer = moehip.MoeLayer.from_arrays(dtype, rw, None, ex.gq, ex.gs, ex.uq, ex.us, ex.dq, ex.ds)
    layer.set_grouped_min_tokens(1)
    got, idx, p = layer.forward(xn, xn)
    np.testing.assert_array_equal(idx, widx)
    np.testing.assert_array_equal(bits(p), bits(wp))
    np.testing.assert_array_equal(bits(got), bits(want))


# E experts, T tokens, pairs of one expert: its full tiles, one pair more and
# several tasks where the mean over the experts takes the 32-pair shape (T = 192
# of 64 experts: 24), the 64-pair shape (300: 37) and the 256-pair shape (500:
# 62); the counts that end a tile of any shape occur under each mean
SKEWED = [(192, n) for n in (32, 33, 64, 65, 128, 129, 192)] + [(300, n) for n in (32, 33, 64, 65, 128, 129, 257)] + [
    (500, n) for n in (65, 129, 256, 257)]


@pytest.mark.parametrize("scale", [1.0, 400.0])
@pytest.mark.parametrize("T,pairs", SKEWED)
def test_expert_limb_passes_skewed(moehip, T, pairs, scale):
    E, D, dff, dtype, hot = 64, 256, 192, 2, 37
    print("expert limbs skewed case", T, pairs, scale, flush=True)
    seed = 9700 + T + pairs
    ex = O.make_experts(dtype, E, D, dff, seed)
    # column 0 marks the tokens of the hot expert, whose router row sees nothing else
    rw = O.normal(E * D, seed + 10, 0.0, 0.02 / scale).reshape(E, D)
    rw[:, 0] = 0.0
    rw[hot] = 0.0
    rw[hot, 0] = 10.0 / scale
    xn = O.normal(T * D, seed + 12, 0.0, scale).reshape(T, D)
    xn[:, 0] = np.where((np.arange(T) * 7919) % T < pairs, 3.0 * scale, -3.0 * scale)
    want, widx, wp, _ = O.moe_block(xn, xn, rw, None, ex)
    assert (widx == hot).sum() == pairs
    layer = moehip.MoeLayer.from_arrays(dtype, rw, None, ex.gq, ex.gs, ex.uq, ex.us, ex.dq, ex.ds)
    layer.set_grouped_min_tokens(1)
    got, idx, p = layer.forward(xn, xn)
    np.testing.assert_array_equal(idx, widx)
    np.testing.assert_array_equal(bits(p), bits(wp))
    np.testing.assert_array_equal(bits(got), bits(want))
