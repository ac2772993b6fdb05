"""The many-row attention kernels (32-row tiles, MFMA products) against the
oracle, bit for bit, through whole small models: head widths of part of one,
one, two and several 64-column stages, row counts around the tiles, key counts
around the 32-key tiles and 128-key blocks, chunks that start at odd
positions, cache lengths that are no multiple of 4, head counts that 8 does not
divide."""
import numpy as np
import pytest

import oracle as O

pytestmark = pytest.mark.gpu


def bits(a):
    return np.ascontiguousarray(a, dtype=np.float32).view(np.uint32)


# (head_dim, query heads, KV heads, cache length, prompt chunks)
CASES = [(128, 8, 2, 131, (5, 16, 32, 17, 33, 28)), (64, 6, 2, 70, (31, 33, 6)), (32, 5, 1, 67, (32, 35)),
         (96, 16, 16, 200, (129, 65, 5)), (68, 3, 3, 65, (64,)), (256, 8, 1, 150, (15, 128)),
         (512, 2, 1, 49, (33, 16)), (4, 8, 8, 300, (257, 6, 37)),
         # 4095 and 4224 head rows, on both sides of the head kernel's rule
         (64, 15, 15, 92, (91,)), (512, 16, 16, 90, (88,))]


@pytest.mark.parametrize("hd,nq,nkv,max_seq,chunks", CASES)
def test_attention_tiles(moehip, hd, nq, nkv, max_seq, chunks):
    print("attention tiles case", hd, nq, nkv, max_seq, chunks, flush=True)
    tm = O.TinyModel(seed=61 + hd, D=128, L=2, hd=hd, nq=nq, nkv=nkv, dff=128, E=8, V=90, dtype=3)
    m = moehip.model_from_tiny(tm, max_seq=max_seq)
    cache = tm.new_cache(max_seq)
    pos = 0
    for T in chunks:
        ids = (O.uniform_u32(T, 17 * pos + hd) % tm.V).astype(np.int32)
        want = tm.forward_kv(ids, pos, cache)
        got, _ = m.forward(ids)
        np.testing.assert_array_equal(bits(got), bits(want), err_msg=f"{T} rows at position {pos}")
        pos += T
