"""The drop-in matmul_adaptive on weights it has seen before: the product
starts on the cached device copy while the host bytes are checked, so a weight
changed in place must still give the new weights' result, bit for bit."""
import os
import shutil
import subprocess
import sys
import threading

import numpy as np
import pytest

import oracle as O

pytestmark = pytest.mark.gpu


def bits(a):
    return np.ascontiguousarray(a, dtype=np.float32).view(np.uint32)


def want_of(dtype, A, w, s, N, K):
    if dtype == 0:
        return O.matmul_f32(A, w)
    return (O.gemv_q8 if dtype == 2 else O.gemv_q4)(A, w, s, N, K)


# (dtype, M, N, K): C stored straight into pinned memory, C just past 64 KB
# (copied), C past 1 MB and A past 1 MB (no pinned staging); weight bytes a
# multiple of the digest's 128-byte block and not
CASES = [(2, 1, 768, 2048), (3, 2, 70, 98), (0, 3, 33, 68), (2, 3, 6000, 64), (3, 40, 8000, 64),
         (0, 300, 20, 1000), (2, 1, 1, 130)]


@pytest.mark.parametrize("dtype,M,N,K", CASES)
def test_dropin_weights_changed_in_place(moehip, dtype, M, N, K):
    print("drop-in case", dtype, M, N, K, flush=True)
    A = O.normal(M * K, 5, 0.0, 1.0).reshape(M, K)
    if dtype == 0:
        w, s = O.normal(N * K, 6, 0.0, 0.05).reshape(N, K), None
    else:
        w, s = (O.quant_q8 if dtype == 2 else O.quant_q4)(O.normal(N * K, 6, 0.0, 0.02).reshape(N, K))

    def call():
        if dtype == 0:
            return moehip.matmul_adaptive(A, w, None, N, K)
        return moehip.matmul_adaptive(A, None, {"q": w, "s": s, "dtype": dtype}, N, K)

    for _ in range(2):
        np.testing.assert_array_equal(bits(call()), bits(want_of(dtype, A, w, s, N, K)))
    raw = w.reshape(-1).view(np.uint8)
    for at in (0, raw.size // 2, raw.size - 1):
        raw[at] ^= 0x11     # (an fp32 weight keeps its exponent: bits of the mantissa or of its low byte)
        for _ in range(2):
            np.testing.assert_array_equal(bits(call()), bits(want_of(dtype, A, w, s, N, K)))
    if s is not None:
        s[N - 1] *= np.float32(1.5)
        np.testing.assert_array_equal(bits(call()), bits(want_of(dtype, A, w, s, N, K)))
    # trusted addresses keep the last upload; verified again, the change is seen
    L = moehip.lib()
    old = want_of(dtype, A, w, s, N, K)
    moehip.check(L.moe_weight_cache_mode(1))
    raw[3] ^= 0x11
    try:
        np.testing.assert_array_equal(bits(call()), bits(old))
    finally:
        moehip.check(L.moe_weight_cache_mode(0))
    np.testing.assert_array_equal(bits(call()), bits(want_of(dtype, A, w, s, N, K)))
    moehip.check(L.moe_weight_cache_clear())
    np.testing.assert_array_equal(bits(call()), bits(want_of(dtype, A, w, s, N, K)))


def test_dropin_calls_from_several_threads(moehip):
    """Calls on different operands from three host threads (C within 64 KB, C
    past it, operands past the pinned staging) while a fourth clears the
    weight cache: every result is its own call's."""
    print("drop-in threads", flush=True)
    work = []
    for i, (dtype, M, N, K) in enumerate([(2, 1, 768, 2048), (3, 8, 4000, 256), (2, 130, 2100, 96)]):
        A = O.normal(M * K, 31 + i, 0.0, 1.0).reshape(M, K)
        w, s = (O.quant_q8 if dtype == 2 else O.quant_q4)(O.normal(N * K, 41 + i, 0.0, 0.02).reshape(N, K))
        work.append((A, {"q": w, "s": s, "dtype": dtype}, N, K, want_of(dtype, A, w, s, N, K)))
    wrong, left = [], [len(work)]
    done = threading.Event()

    def caller(i):
        A, w, N, K, want = work[i]
        try:
            for it in range(40):
                if not np.array_equal(bits(moehip.matmul_adaptive(A, None, w, N, K)), bits(want)):
                    wrong.append((i, it))
        finally:
            left[0] -= 1
            if not left[0]:
                done.set()

    threads = [threading.Thread(target=caller, args=(i,)) for i in range(len(work))]
    for t in threads:
        t.start()
    while not done.wait(0.01):
        moehip.check(moehip.lib().moe_weight_cache_clear())
    for t in threads:
        t.join()
    assert not wrong, wrong


CHILD = """
import ctypes, sys
ctypes.CDLL(sys.argv[1], mode=ctypes.RTLD_GLOBAL)   # its hipHostMalloc comes first
import numpy as np
import moehip, oracle as O
assert not any(m.startswith("torch") for m in sys.modules)
for dtype, M, N, K in ((2, 1, 768, 2048), (3, 8, 4000, 256)):
    A = O.normal(M * K, 51, 0.0, 1.0).reshape(M, K)
    w, s = (O.quant_q8 if dtype == 2 else O.quant_q4)(O.normal(N * K, 52, 0.0, 0.02).reshape(N, K))
    for _ in range(3):
        want = (O.gemv_q8 if dtype == 2 else O.gemv_q4)(A, w, s, N, K)
        got = moehip.matmul_adaptive(A, None, {"q": w, "s": s, "dtype": dtype}, N, K)
        assert np.array_equal(got.view(np.uint32), want.view(np.uint32))
        w.reshape(-1).view(np.uint8)[5] ^= 0x11
assert ctypes.c_int.in_dll(ctypes.CDLL(sys.argv[1]), "refused").value > 0
print("child ok")
"""


@pytest.mark.skipif(shutil.which("gcc") is None, reason="needs gcc for the refusing allocator")
def test_dropin_without_pinned_memory(moehip, tmp_path):
    """A host that refuses pinned memory: the drop-in takes its waiting copies,
    as it did before it had a pinned staging."""
    print("drop-in without pinned memory", flush=True)
    src, so = tmp_path / "refuse.c", tmp_path / "refuse.so"
    src.write_text("#include <stddef.h>\nint refused;\n"
                   "int hipHostMalloc(void** p, size_t n, unsigned f) { (void)p; (void)n; (void)f; ++refused; return 2; }\n")
    subprocess.run(["gcc", "-shared", "-fPIC", "-o", str(so), str(src)], check=True)
    root = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
    env = dict(os.environ, PYTHONPATH=os.pathsep.join([os.path.join(root, "moe.cc_amd"), os.path.join(root, "oracle")]))
    r = subprocess.run([sys.executable, "-c", CHILD, str(so)], env=env, capture_output=True, text=True, timeout=100)
    assert r.returncode == 0 and "child ok" in r.stdout, r.stdout + r.stderr
