"""The work whose speed is watched on an MI355X, as calls of the public entry points.

Sizes are those of the repository's configurations, tests and benchmark: Qwen3-30B-A3B
(d_model 2048, d_ff 768, 128 experts, top-8, 32 / 4 heads of 128, vocabulary 151,936), its
expert matrices [768 x 2048] and [2048 x 768], and generic ones around them.  Weights are
N(0, 0.02^2) quantized per row with the exporter's rule, activations N(0, 1), as a
normalised hidden state is.  A case is a dict of plain values; `kind` names its entry point:

  dropin   matmul_adaptive on host arrays: the gate, up and down projection of one expert
  gemv     moe_matmul_q8_dev / moe_matmul_q4_dev, one product on device arrays
  pool     moe_act_pack_dev + moe_matmul_q_prepacked_dev, many products in one launch
  moe      moe_layer_forward or (norm) moe_block_forward, on `layers` layers one after another
  dense    moe_matmul_f32_dev, the fp32 products of attention and head
  model    moe_model_forward: a prompt, then greedy steps fed from device memory

Every result is defined bit for bit (integer dots, and fp32 sums in one stated order, each
operation rounded once), so the tolerance is "exact" throughout.
"""
import ctypes
import math
import os
import sys

import numpy as np
import torch  # loaded before the library, so that both use one HIP runtime

sys.path.insert(0, os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "moe.cc_amd"))
import moehip as M  # noqa: E402

LEVELS = {2: 127, 3: 7}  # 2 = Q8, 3 = Q4
SHAPE = {"D": 2048, "dff": 768, "E": 128, "k": 8}  # the MoE block of Qwen3-30B-A3B
VOCAB = 151936


def listed():
    return [
        # the drop-in in an unmodified host program: three calls for one routed expert
        {"name": "dropin_q8_expert", "kind": "dropin", "dtype": 2, "M": 1, "D": 2048, "dff": 768},
        # the smallest device call: one expert's down projection for one token
        {"name": "gemv_q4_down", "kind": "gemv", "dtype": 3, "M": 1, "N": 2048, "K": 768},
        # odd sizes that no tiled geometry fits
        {"name": "gemv_q8_ragged", "kind": "gemv", "dtype": 2, "M": 7, "N": 1000, "K": 1030},
        # the benchmark's pool: 1 GiB of distinct Q4 matrices at batch 1
        {"name": "pool_q4_down", "kind": "pool", "dtype": 3, "jobs": 1366, "N": 2048, "K": 768},
        # decode, one sequence: six consecutive MoE blocks
        {"name": "moe_q8_t1", "kind": "moe", "dtype": 2, "T": 1, "norm": False, "layers": 6, **SHAPE},
        # decode, a batch of sequences
        {"name": "moe_q8_t16", "kind": "moe", "dtype": 2, "T": 16, "norm": False, "layers": 6, **SHAPE},
        # a few tokens, with the norm in front (speculative steps, small ragged batches)
        {"name": "block_q4_t5", "kind": "moe", "dtype": 3, "T": 5, "norm": True, "layers": 6, **SHAPE},
        # a short ragged prompt, Q8
        {"name": "moe_q8_t300", "kind": "moe", "dtype": 2, "T": 300, "norm": False, "layers": 1, **SHAPE},
        # the largest prompt chunk, Q4
        {"name": "moe_q4_t2048", "kind": "moe", "dtype": 3, "T": 2048, "norm": False, "layers": 1, **SHAPE},
        # the joint Q/K/V projection of a 512-token prompt
        {"name": "dense_qkv_m512", "kind": "dense", "M": 512, "N": 5120, "K": 2048},
        # the whole model: a 512-token prompt
        {"name": "model_prefill", "kind": "model", "dtype": 3, "L": 48, "V": VOCAB, "untied": True, "prompt": 512, "new": 0},
        # the whole model: a short chat turn, prompt and greedy steps
        {"name": "model_chat", "kind": "model", "dtype": 3, "L": 48, "V": VOCAB, "untied": True, "prompt": 100, "new": 24},
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["dropin", "gemv", "pool", "moe", "moe", "moe", "moe", "dense", "dense", "model", "model"])
    dtype = rng.choice([2, 3])
    if kind == "dropin":
        return {"kind": kind, "dtype": dtype, "M": rng.randint(1, 8), "D": 64 * rng.randint(8, 64), "dff": 64 * rng.randint(4, 32)}
    if kind == "gemv":
        N, K = _log(rng, 64, 8192), _log(rng, 64, 8192)
        if rng.random() < 0.5:
            K = max(64, K // 128 * 128)
        return {"kind": kind, "dtype": dtype, "M": _log(rng, 1, 64), "N": N, "K": K if dtype == 2 else K + K % 2}
    if kind == "pool":
        N, K = rng.choice([(768, 2048), (2048, 768), (1024, 2048), (2048, 1024)])
        return {"kind": kind, "dtype": dtype, "jobs": _log(rng, 24, 1366 if dtype == 3 else 683), "N": N, "K": K}
    if kind == "moe":
        c = dict(SHAPE) if rng.random() < 0.6 else {"D": rng.choice([1024, 1536, 2048]), "dff": rng.choice([512, 768, 1024]),
                                                    "E": rng.choice([32, 60, 64, 128]), "k": rng.choice([4, 8])}
        T = _log(rng, 1, 2048)
        return {"kind": kind, "dtype": dtype, "T": T, "norm": rng.random() < 0.4, "layers": 6 if T < 32 else 1, **c}
    if kind == "dense":
        N, K = _log(rng, 64, 8192), _log(rng, 64, 4096)
        if rng.random() < 0.7:
            K = max(64, K // 64 * 64)
        return {"kind": kind, "M": _log(rng, 1, 1024), "N": N, "K": K}
    return {"kind": kind, "dtype": dtype, "L": rng.randint(1, 4), "V": rng.choice([8192, VOCAB]), "untied": rng.random() < 0.5,
            "prompt": _log(rng, 1, 700), "new": rng.randint(0, 12)}


def _gen(seed):
    return torch.Generator(device="cuda").manual_seed(int(seed) & 0x7FFFFFFF)


def _normal(gen, shape, std=1.0):
    return torch.randn(shape, generator=gen, device="cuda", dtype=torch.float32) * std


def _quantized(gen, dtype, rows, K):
    """(bytes [rows, K or K / 2], scales [rows]) of N(0, 0.02^2) rows."""
    q = torch.empty((rows, K if dtype == 2 else K // 2), device="cuda", dtype=torch.int8 if dtype == 2 else torch.uint8)
    s = torch.empty(rows, device="cuda", dtype=torch.float32)
    step = max(1, (64 << 20) // K)
    for r in range(0, rows, step):
        w = _normal(gen, (min(step, rows - r), K), 0.02)
        sc = w.abs().amax(1).clamp_min(1e-8) / LEVELS[dtype]
        v = torch.round(w / sc[:, None])
        if dtype == 2:
            q[r:r + step] = v.to(torch.int8)
        else:
            u = v.clamp(-8, 7).to(torch.int32) + 8
            q[r:r + step] = (u[:, 0::2] | (u[:, 1::2] << 4)).to(torch.uint8)
        s[r:r + step] = sc
    return q, s


def _moe_weights(gen, case):
    D, dff, E = case["D"], case["dff"], case["E"]
    w = {"router": _normal(gen, (E, D), 0.02), "rms2": 1.0 + _normal(gen, (D,), 0.1)}
    for name, rows, K in (("g", dff, D), ("u", dff, D), ("d", D, dff)):
        w[name] = _quantized(gen, case["dtype"], E * rows, K)
    return w


def _moe_input(gen, case):
    """(normalised rows, residual rows) of T tokens"""
    x = _normal(gen, (case["T"], case["D"]))
    return x / x.pow(2).mean(1, keepdim=True).add(1e-6).sqrt(), x


def prepare(case, seed):
    kind, gen = case["kind"], _gen(seed)
    state = {"case": case}
    if kind == "dropin":
        D, dff = case["D"], case["dff"]
        state["w"] = []
        for rows, K in ((dff, D), (dff, D), (D, dff)):
            q, s = _quantized(gen, case["dtype"], rows, K)
            state["w"].append(({"q": q.cpu().numpy(), "s": s.cpu().numpy(), "dtype": case["dtype"]}, rows, K))
        state["x"] = _normal(gen, (case["M"], D)).cpu().numpy()
        state["h"] = _normal(gen, (case["M"], dff)).cpu().numpy()
    elif kind == "gemv":
        state["w"] = _quantized(gen, case["dtype"], case["N"], case["K"])
        state["x"] = _normal(gen, (case["M"], case["K"]))
        state["y"] = torch.empty((case["M"], case["N"]), device="cuda")
    elif kind == "pool":
        n, N, K = case["jobs"], case["N"], case["K"]
        q, s = _quantized(gen, case["dtype"], n * N, K)
        x, y = _normal(gen, (1, K)), torch.empty((n, N), device="cuda")
        i = np.arange(n, dtype=np.int64)
        jobs = np.stack([q.data_ptr() + i * N * q.shape[1], s.data_ptr() + i * N * 4, np.full(n, x.data_ptr()), y.data_ptr() + i * N * 4], 1)
        state.update(w=(q, s), x=x, y=y, jobs=torch.from_numpy(jobs).cuda(),
                     tabs=torch.empty(M.lib().moe_act_table_bytes(K), device="cuda", dtype=torch.uint8))
    elif kind == "moe":
        state["calls"] = []
        for _ in range(case["layers"]):
            w = _moe_weights(gen, case)
            h = ctypes.c_void_p()
            torch.cuda.synchronize()
            M.check(M.lib().moe_layer_create_raw(
                case["dtype"], case["D"], case["dff"], case["E"], case["k"], w["router"].data_ptr(), None, w["rms2"].data_ptr(),
                *(t.data_ptr() for n in "gud" for t in w[n]), 1, ctypes.byref(h)), "moe_layer_create_raw")
            del w
            layer = M.MoeLayer(h.value, case["dtype"], case["D"], case["dff"], case["E"], case["k"])
            xn, x = _moe_input(gen, case)
            out = {"out": torch.empty_like(x)}
            if not case["norm"]:
                out["expert"] = torch.empty((case["T"], case["k"]), device="cuda", dtype=torch.int32)
                out["gate"] = torch.empty((case["T"], case["k"]), device="cuda")
            state["calls"].append((layer, xn, x, out))
    elif kind == "dense":
        state["w"] = _normal(gen, (case["N"], case["K"]), 0.02)
        state["x"] = _normal(gen, (case["M"], case["K"]))
        state["y"] = torch.empty((case["M"], case["N"]), device="cuda")
    elif kind == "model":
        cfg = M.qwen_config(2048, case["L"], 128, 32, 4, 768, 128, 8, case["V"])
        state["model"] = M.Model.synthetic(cfg, case["dtype"], case["untied"], int(seed) + 1, 0.02, 2048)
        state["ids"] = torch.randint(0, case["V"], (case["prompt"],), generator=gen, device="cuda", dtype=torch.int32)
        state["logits"] = torch.empty((case["new"] + 1, case["V"]), device="cuda")
        state["next"] = torch.empty(case["new"] + 1, device="cuda", dtype=torch.int32)
    torch.cuda.synchronize()  # the library works on a stream of its own
    return state


def run(state):
    case, L = state["case"], M.lib()
    kind = case["kind"]
    if kind == "dropin":
        (g, n, k), (u, _, _), (d, nd, kd) = state["w"]
        return [M.matmul_adaptive(state["x"], None, g, n, k), M.matmul_adaptive(state["x"], None, u, n, k),
                M.matmul_adaptive(state["h"], None, d, nd, kd)]
    if kind == "gemv":
        f = L.moe_matmul_q8_dev if case["dtype"] == 2 else L.moe_matmul_q4_dev
        q, s = state["w"]
        M.check(f(state["x"].data_ptr(), q.data_ptr(), s.data_ptr(), state["y"].data_ptr(), case["M"], case["N"], case["K"]), "gemv")
        return state["y"]
    if kind == "pool":
        M.check(L.moe_act_pack_dev(case["dtype"], state["x"].data_ptr(), 1, case["K"], state["tabs"].data_ptr()), "pack")
        M.check(L.moe_matmul_q_prepacked_dev(case["dtype"], state["jobs"].data_ptr(), case["jobs"], 1, case["N"], case["K"],
                                             state["tabs"].data_ptr()), "pool")
        return state["y"]
    if kind == "moe":
        for layer, xn, x, out in state["calls"]:
            if case["norm"]:
                M.check(L.moe_block_forward(layer.h, x.data_ptr(), case["T"], out["out"].data_ptr(), 1e-6), "moe_block_forward")
            else:
                layer.forward_dev(xn.data_ptr(), x.data_ptr(), case["T"], out["out"].data_ptr(), out["expert"].data_ptr(), out["gate"].data_ptr())
        return [c[3] for c in state["calls"]]
    if kind == "dense":
        M.check(L.moe_matmul_f32_dev(state["x"].data_ptr(), state["w"].data_ptr(), state["y"].data_ptr(), case["M"], case["N"], case["K"]), "dense")
        return state["y"]
    m, logits, nxt = state["model"], state["logits"], state["next"]
    m.reset()
    M.check(L.moe_model_forward(m.h, state["ids"].data_ptr(), case["prompt"], 1, logits.data_ptr(), nxt.data_ptr()), "prompt")
    for i in range(1, case["new"] + 1):
        M.check(L.moe_model_forward(m.h, nxt.data_ptr() + 4 * (i - 1), 1, 1, logits.data_ptr() + 4 * case["V"] * i, nxt.data_ptr() + 4 * i), "step")
    return {"logits": logits, "next": nxt}


def _row_bytes(dtype, K):
    return K if dtype == 2 else K // 2


def _qbytes(dtype, N, K):
    return N * (_row_bytes(dtype, K) + 4)


def _moe_work(dtype, T, D, dff, E, k):
    """Router, the experts that T tokens reach on average, rows in and out."""
    used = E * (1 - (1 - k / E) ** T)
    expert = 2 * _qbytes(dtype, dff, D) + _qbytes(dtype, D, dff)
    return 4 * E * D + used * expert + 8 * T * D, 2 * T * (E * D + k * 3 * D * dff)


def work(case):
    kind = case["kind"]
    if kind == "dropin":
        D, dff, rows = case["D"], case["dff"], case["M"]
        b = 2 * _qbytes(case["dtype"], dff, D) + _qbytes(case["dtype"], D, dff) + 4 * rows * 3 * (D + dff)
        return {"bytes": b, "flops": 2 * rows * 3 * D * dff}
    if kind in ("gemv", "pool"):
        n, rows, N, K = case.get("jobs", 1), case.get("M", 1), case["N"], case["K"]
        return {"bytes": n * (_qbytes(case["dtype"], N, K) + 4 * rows * N) + 4 * rows * K, "flops": 2 * n * rows * N * K}
    if kind == "moe":
        b, f = _moe_work(case["dtype"], case["T"], case["D"], case["dff"], case["E"], case["k"])
        return {"bytes": case["layers"] * b, "flops": case["layers"] * f}
    if kind == "dense":
        rows, N, K = case["M"], case["N"], case["K"]
        return {"bytes": 4 * (rows * N + N * K + rows * K), "flops": 2 * rows * N * K}
    # the model: each call reads the dense weights, its experts, the head and the cache so far
    D, L, hd, nq, nkv = 2048, case["L"], 128, 32, 4
    proj = (nq + 2 * nkv) * hd * D + nq * hd * D
    b = f = 0
    ctx = 0
    for T in [case["prompt"]] + [1] * case["new"]:
        mb, mf = _moe_work(case["dtype"], T, D, SHAPE["dff"], SHAPE["E"], SHAPE["k"])
        seen = T * ctx + T * (T + 1) // 2  # (token, position) pairs
        ctx += T
        b += L * (mb + 4 * proj + 8 * nkv * hd * ctx) + 4 * case["V"] * (D + 1)
        f += L * (mf + 2 * T * proj + 4 * nq * hd * seen) + 2 * case["V"] * D
    return {"bytes": b, "flops": f}


def tolerance(case):
    return "exact"


def _acts(x, dtype):
    return torch.trunc(x * LEVELS[dtype])


def _ints(q, dtype):
    if dtype == 2:
        return q.double()
    q = q.int()
    return torch.stack([(q & 15) - 8, (q >> 4) - 8], -1).flatten(-2).double()


def _product(x, q, s, dtype):
    """x [M, K] in 64 bits times the quantized rows"""
    return (_acts(x, dtype) @ _ints(q, dtype).T) / LEVELS[dtype] * s.double()


def exact(case, seed):
    kind, gen = case["kind"], _gen(seed)
    if kind == "dropin":
        D, dff, dt = case["D"], case["dff"], case["dtype"]
        ws = [_quantized(gen, dt, rows, K) for rows, K in ((dff, D), (dff, D), (D, dff))]
        x, h = _normal(gen, (case["M"], D)), _normal(gen, (case["M"], dff))
        return [_product(a.double(), *w, dt).cpu().numpy() for a, w in zip((x, x, h), ws)]
    if kind == "gemv":
        w = _quantized(gen, case["dtype"], case["N"], case["K"])
        return _product(_normal(gen, (case["M"], case["K"])).double(), *w, case["dtype"])
    if kind == "pool":
        n, N, K = case["jobs"], case["N"], case["K"]
        q, s = _quantized(gen, case["dtype"], n * N, K)
        x = _normal(gen, (1, K)).double()
        return torch.cat([_product(x, q[r:r + 64 * N], s[r:r + 64 * N], case["dtype"])[0] for r in range(0, n * N, 64 * N)]).reshape(n, N)
    if kind == "moe":
        return [_exact_moe(gen, case) for _ in range(case["layers"])]
    if kind == "dense":
        w = _normal(gen, (case["N"], case["K"]), 0.02)
        return _normal(gen, (case["M"], case["K"])).double() @ w.double().T
    return None  # the synthetic model's weights are made inside the library


def _exact_moe(gen, case):
    dt, D, dff, E, k = case["dtype"], case["D"], case["dff"], case["E"], case["k"]
    w = _moe_weights(gen, case)
    xn, x = _moe_input(gen, case)
    xn, x = xn.double(), x.double()
    if case["norm"]:
        xn = x / x.pow(2).mean(1, keepdim=True).add(1e-6).sqrt() * w["rms2"].double()
    top, idx = (xn @ w["router"].double().T).topk(k, dim=1)
    p = (top - top[:, :1]).exp()
    p = p / (p.sum(1, keepdim=True) + 1e-9)
    out = x.clone()
    for e in range(E):
        t, j = (idx == e).nonzero(as_tuple=True)
        if not t.numel():
            continue
        m = {n: (w[n][0][e * r:(e + 1) * r], w[n][1][e * r:(e + 1) * r]) for n, r in (("g", dff), ("u", dff), ("d", D))}
        g, u = _product(xn[t], *m["g"], dt), _product(xn[t], *m["u"], dt)
        out.index_add_(0, t, p[t, j][:, None] * _product(g / (1 + (-g).exp()) * u, *m["d"], dt))
    return {"out": out} if case["norm"] else {"out": out, "expert": None, "gate": p}
