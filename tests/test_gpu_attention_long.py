"""GPU parity of causal attention at real context lengths
(test_model_trace.c:399-425: the score, softmax and weighted-V loops over
every cached position), through the whole-model C ABI.

The model tests in test_gpu_model.py stay inside one 64-key block.  These
run the kernels' multi-block paths at the 30B-A3B model's head geometry
(head_dim 128, 32 query heads, 4 KV heads) with small D and L:

* a 320-token prompt in one chunk: the query-tiled score kernel over five
  64-key blocks, the query-tiled softmax / V kernel with its V rows staged
  128 positions at a time (three stages);
* 70 single-token decode steps across two more key-block boundaries (320,
  384), each step's logits checked;
* a second prompt chunk at position 390 (query tiles at pos0 > 0);
* the one-row kernels with two to four rows, past several chunks of V;
* 2060 cached positions (decode's scores no longer fit in registers,
  several 1024-position V chunks) and 4650, where four score rows no longer fit
  a softmax block's LDS share (two a block), with 4 / 1 query heads so that the
  CPU oracle stays fast; narrow heads to the longest cache, 16384 positions
  (one row a block from 8961 on).

Bar: bit-exact against oracle/model_oracle.c's KV-cached forward, itself
pinned to the compiled reference's model_forward_f32 (tests/golden/
ref_model.json, tests/test_oracle_model.py).
"""
import numpy as np
import pytest

import oracle as O

pytestmark = pytest.mark.gpu


def bits(a):
    return np.ascontiguousarray(a, dtype=np.float32).view(np.uint32)


def _check(got, want, what):
    np.testing.assert_array_equal(bits(got), bits(want), err_msg=what)


GEOM = dict(D=256, L=2, hd=128, nq=32, nkv=4, dff=128, E=16, V=300, dtype=3)


def test_long_prompt_decode_and_second_chunk(moehip):
    """The 30B-A3B model's heads: 320-token prompt, 70 decode steps, a 70-token
    chunk at position 390, then forward_full of the whole sequence."""
    print("attention long: prompt 320 / decode 70 / chunk 70", flush=True)
    tm = O.TinyModel(seed=41, **GEOM)
    max_seq = 512
    m = moehip.model_from_tiny(tm, max_seq=max_seq)
    cache = tm.new_cache(max_seq)
    ids = (O.uniform_u32(320, 141) % tm.V).astype(np.int32)
    want = tm.forward_kv(ids, 0, cache)
    got, nxt = m.forward(ids)
    _check(got, want, "prompt 320")
    assert nxt == O.greedy(want)
    seq = ids.tolist()
    for step in range(70):
        seq.append(nxt)
        want = tm.forward_kv([nxt], len(seq) - 1, cache)
        got, nxt = m.forward([nxt])
        _check(got, want, f"decode step {step} (position {len(seq) - 1})")
        assert nxt == O.greedy(want)
    chunk = (O.uniform_u32(70, 142) % tm.V).astype(np.int32)
    want = tm.forward_kv(chunk, len(seq), cache)
    got, nxt = m.forward(chunk)
    _check(got, want, "chunk at 390")
    seq += chunk.tolist()
    assert m.position == len(seq) == 460
    _check(m.forward_full(seq), got, "forward_full of 460 tokens")
    m.close()


def test_long_rowwise_kernels(moehip):
    """The one-row score and softmax / V kernels with two to four rows at
    positions 296-318 (the block-parallel exact sum of each row's exponentials,
    three 128-position pieces of V), then decode steps."""
    print("attention long: two to four rows at 296", flush=True)
    tm = O.TinyModel(seed=43, **GEOM)
    m = moehip.model_from_tiny(tm, max_seq=400)
    cache = tm.new_cache(400)
    ids = (O.uniform_u32(296, 143) % tm.V).astype(np.int32)
    want = tm.forward_kv(ids, 0, cache)
    got, nxt = m.forward(ids)
    _check(got, want, "prompt 296")
    pos = 296
    for T in (4, 3, 2, 4, 4, 3, 2):
        chunk = (O.uniform_u32(T, 144 + pos) % tm.V).astype(np.int32)
        want = tm.forward_kv(chunk, pos, cache)
        got, nxt = m.forward(chunk)
        _check(got, want, f"{T} rows at {pos}")
        pos += T
    for step in range(12):
        want = tm.forward_kv([nxt], pos, cache)
        got, nxt = m.forward([nxt])
        _check(got, want, f"rowwise decode step {step}")
        pos += 1
    m.close()


def test_context_2060(moehip):
    """2060-token prompt, then decode past 2048 cached positions (the
    decode softmax reads its scores from memory instead of registers; its V
    sums run over three 1024-position chunks)."""
    print("attention long: prompt 2040 / decode to 2060", flush=True)
    tm = O.TinyModel(D=128, L=1, hd=128, nq=4, nkv=1, dff=128, E=16, V=300, dtype=3, seed=44)
    max_seq = 2100
    m = moehip.model_from_tiny(tm, max_seq=max_seq)
    cache = tm.new_cache(max_seq)
    ids = (O.uniform_u32(2040, 145) % tm.V).astype(np.int32)
    want = tm.forward_kv(ids, 0, cache)
    got, nxt = m.forward(ids)
    _check(got, want, "prompt 2040")
    pos = 2040
    for step in range(20):
        want = tm.forward_kv([nxt], pos, cache)
        got, nxt = m.forward([nxt])
        _check(got, want, f"decode at position {pos}")
        pos += 1
    m.close()


def test_context_past_tile_lds(moehip):
    """A 4600-token prompt and a 50-token chunk behind it: past 4352 scores a
    softmax block holds two rows instead of four; then decode steps."""
    print("attention long: prompt 4600 / chunk 50 / decode", flush=True)
    tm = O.TinyModel(D=128, L=1, hd=128, nq=1, nkv=1, dff=128, E=16, V=300, dtype=3, seed=45)
    max_seq = 4700
    m = moehip.model_from_tiny(tm, max_seq=max_seq)
    cache = tm.new_cache(max_seq)
    ids = (O.uniform_u32(4600, 146) % tm.V).astype(np.int32)
    want = tm.forward_kv(ids, 0, cache)
    got, nxt = m.forward(ids)
    _check(got, want, "prompt 4600")
    chunk = (O.uniform_u32(50, 147) % tm.V).astype(np.int32)
    want = tm.forward_kv(chunk, 4600, cache)
    got, nxt = m.forward(chunk)
    _check(got, want, "chunk at 4600")
    pos = 4650
    for step in range(4):
        want = tm.forward_kv([nxt], pos, cache)
        got, nxt = m.forward([nxt])
        _check(got, want, f"decode at position {pos}")
        pos += 1
    m.close()


def test_context_to_the_longest_cache(moehip):
    """A 9200-token prompt, chunks of 7 and 40 rows behind it (a softmax row of
    more than 8960 scores: one row a block), a prompt to 16340 and chunks that
    end at the longest cache, 16384 positions."""
    print("attention long: 16384 positions", flush=True)
    tm = O.TinyModel(D=64, L=1, hd=8, nq=1, nkv=1, dff=32, E=8, top_k=2, V=60, dtype=3, seed=46)
    m = moehip.model_from_tiny(tm, max_seq=16384)
    cache = tm.new_cache(16384)
    pos = 0
    for T in (9200, 7, 40, 7093, 39, 5):
        ids = (O.uniform_u32(T, 150 + T) % tm.V).astype(np.int32)
        want = tm.forward_kv(ids, pos, cache)
        got, _ = m.forward(ids)
        _check(got, want, f"{T} rows at {pos}")
        pos += T
    assert pos == 16384 == m.position
    m.close()
