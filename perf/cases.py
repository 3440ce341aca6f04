"""What this library is timed on: eviction layer-calls, scoring calls, a
chunked prefill and decode steps, each through the entry point that a program
calls.

A case is a dict of plain values; ``op`` names the entry point:

* ``update``    one layer's prefill eviction, ``DropKVCache.update`` on a fresh
                cache, with Q/K/V as a decoder layer has them (projections
                ``[B, L, H, D]`` seen as ``[B, H, L, D]``), or with K/V
                contiguous per head where ``per_head`` is set;
* ``plan``      the same work through a kept ``EvictPlan`` on contiguous K/V,
                which also returns the scores;
* ``scores``    ``dropkv_scores_triton`` alone;
* ``deployed``  ``ops.scores`` with the rounding of the deployed PyTorch path
                (p and y in the input type), which also takes float32 inputs
                and head dimensions that are no power of two;
* ``chunked``   ``prefill_chunked`` over one layer of a preallocated cache;
* ``decode``    ``ops.decode_attention`` on a preallocated cache, once per
                layer of one decode step;
* ``graph``     the same step captured as a HIP graph and replayed, as
                ``CompressedDecoder`` does.
"""

import math

import torch

from dropkv_amd import DropKVCache, dropkv_scores_triton, ops, prefill_chunked

_DTYPES = {"bf16": torch.bfloat16, "fp16": torch.float16, "fp32": torch.float32}
_BYTES = {"bf16": 2, "fp16": 2, "fp32": 4}


def listed():
    return [
        # The smallest call: a short prompt on a small model (the head shape
        # of the plumbing configuration).  Launches and host work are all of it.
        dict(name="update_short_prompt", op="update", B=1, Hq=8, Hkv=2, D=64, Lq=512, Lk=512, dtype="bf16", window=8,
             kernel=11, ratio=0.1, keys="normal"),
        # One layer of the Qwen2-0.5B architecture at its 16K prompt.
        dict(name="update_qwen_16k", op="update", B=1, Hq=14, Hkv=2, D=64, Lq=16384, Lk=16384, dtype="bf16", window=8,
             kernel=11, ratio=0.1, keys="normal"),
        # One layer of Llama-3.1-8B at a 32K prompt: the headline configuration.
        dict(name="update_llama_32k", op="update", B=1, Hq=32, Hkv=8, D=128, Lq=32768, Lk=32768, dtype="bf16", window=8,
             kernel=11, ratio=0.1, keys="lognormal"),
        # A batch of medium prompts of an odd length, in float16.
        dict(name="update_batch_7001", op="update", B=3, Hq=32, Hkv=8, D=128, Lq=7001, Lk=7001, dtype="fp16", window=16,
             kernel=7, ratio=0.2, keys="lognormal"),
        # The long-context configuration (the last chunk of four prompts of
        # 128K): eight query heads per KV head, a wide window, heavy-tailed keys.
        dict(name="update_gqa8_128k", op="update", B=4, Hq=64, Hkv=8, D=128, Lq=4096, Lk=131072, dtype="bf16", window=32,
             kernel=11, ratio=0.05, keys="student"),
        # The headline configuration on a plan that a serving loop keeps.
        dict(name="plan_llama_32k", op="plan", B=1, Hq=32, Hkv=8, D=128, Lq=32768, Lk=32768, dtype="bf16", window=8,
             kernel=11, ratio=0.1, keys="lognormal"),
        # Scores alone at a head dimension of 256.
        dict(name="scores_d256_8k", op="scores", B=1, Hq=8, Hkv=4, D=256, Lq=8192, Lk=8192, dtype="bf16", window=8,
             p_round=True, keys="normal"),
        # float32 inputs, which the deployed path scores.
        dict(name="deployed_fp32_8k", op="deployed", B=1, Hq=14, Hkv=2, D=64, Lq=8192, Lk=8192, dtype="fp32", window=8,
             keys="normal"),
        # A head dimension that is no power of two, one query head per KV
        # head, an odd length.
        dict(name="deployed_d96_4099", op="deployed", B=1, Hq=16, Hkv=16, D=96, Lq=4099, Lk=4099, dtype="fp16",
             window=8, keys="normal"),
        # A chunked prefill: the cache grows chunk by chunk and is evicted
        # once at the end.
        dict(name="chunked_llama_32k", op="chunked", B=1, Hq=32, Hkv=8, D=128, Lk=32768, chunk=4096, dtype="bf16",
             window=8, kernel=11, ratio=0.1, keys="normal", strategy="last_chunk"),
        # A decode step on the compressed 16K cache, as the decoder replays it.
        dict(name="graph_qwen_24_layers", op="graph", layers=24, B=1, Hq=14, Hkv=2, D=64, rows=1638, room=320,
             dtype="bf16"),
        # A batch decoding over longer caches.
        dict(name="decode_llama_batch", op="decode", layers=1, B=8, Hq=32, Hkv=8, D=128, rows=8003, room=509,
             dtype="bf16"),
    ]


def _log(rng, lo, hi):
    """A whole number spread over the logarithm of [lo, hi], odd as often as even."""
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


# (Hq, Hkv, D) of the matrix-core head dimensions.
_HEADS = ((8, 2, 64), (14, 2, 64), (32, 8, 128), (28, 4, 128), (8, 8, 128), (16, 8, 64), (64, 8, 128), (12, 4, 32))
# Keys of all heads and sequences together: a call's K and V stay under 0.6 GB.
_MOST_KV = 1 << 29


def draw(rng):
    op = rng.choice(("update", "update", "update", "plan", "scores", "deployed", "chunked", "decode", "graph"))
    Hq, Hkv, D = rng.choice(_HEADS)
    dtype = rng.choice(("bf16", "bf16", "fp16"))
    if op in ("decode", "graph"):
        Hq, Hkv, D = rng.choice([h for h in _HEADS if h[2] >= 64])
        layers = 1 if op == "decode" else rng.choice((4, 16, 24))
        B, rows = rng.choice((1, 1, 2, 8)), _log(rng, 100, 12000)
        while layers * B * Hkv * rows * D * 4 > _MOST_KV // 2:
            rows //= 2
        return dict(op=op, layers=layers, B=B, Hq=Hq, Hkv=Hkv, D=D, rows=rows, room=rng.randrange(1, 600), dtype=dtype)
    keys = rng.choice(("normal", "lognormal", "student"))
    window = rng.choice((4, 8, 8, 16, 32))
    if op == "deployed":
        dtype = rng.choice(("fp32", "fp32", "fp16", "bf16"))
        Hq, Hkv, D = rng.choice(((14, 2, 64), (8, 2, 64), (8, 4, 128), (12, 4, 32)) if dtype == "fp32" else
                                ((16, 16, 96), (8, 2, 80), (8, 4, 256)))
        L = _log(rng, 300, 9000)
        return dict(op=op, B=1, Hq=Hq, Hkv=Hkv, D=D, Lq=L, Lk=L, dtype=dtype, window=min(window, 16), keys="normal")
    B = rng.choice((1, 1, 1, 2, 3))
    Lk = _log(rng, 400, 65536)
    if op == "scores" and rng.random() < 0.4:
        Hq, Hkv, D = rng.choice(((8, 4, 256), (16, 8, 256), (8, 1, 256)))
        B, Lk, window = 1, _log(rng, 400, 9000), min(window, 16)
    while B * Hkv * Lk * D * 4 > _MOST_KV:
        Lk = Lk // 2 + 1
    Lq = Lk if rng.random() < 0.7 else max(window, min(Lk, 4096))
    case = dict(op=op, B=B, Hq=Hq, Hkv=Hkv, D=D, Lk=Lk, dtype=dtype, window=window, keys=keys)
    if op == "scores":
        return dict(case, Lq=Lq, p_round=rng.random() < 0.7)
    case.update(kernel=rng.choice((5, 7, 11, 21, 63)), ratio=rng.choice((0.05, 0.1, 0.2, 0.5)))
    if op == "chunked":
        return dict(case, chunk=rng.choice((1024, 4096, 4096)) + rng.choice((0, 0, 37)),
                    strategy=rng.choice(("last_chunk", "last_chunk", "every_chunk")))
    return dict(case, Lq=Lq, per_head=rng.random() < 0.3) if op == "update" else dict(case, Lq=Lq)


def _normal(g, dtype, *shape):
    return torch.randn(*shape, generator=g, device="cuda", dtype=torch.float32).to(dtype)


def _keys(g, case, dtype, B, L, H, D):
    """Keys [B, L, H, D]: normal; with an outlier scale per channel, as trained
    models have; or heavy-tailed (Student-t with three degrees of freedom)."""
    z = torch.randn(B, L, H, D, generator=g, device="cuda", dtype=torch.float32)
    if case["keys"] == "lognormal":
        z *= torch.exp(torch.randn(B, 1, H, D, generator=g, device="cuda", dtype=torch.float32))
    elif case["keys"] == "student":
        chi = torch.zeros_like(z)
        for _ in range(3):
            chi += torch.randn(B, L, H, D, generator=g, device="cuda", dtype=torch.float32).square_()
        z /= (chi / 3).sqrt_()
    return z.to(dtype)


def _qkv(case, seed):
    """Q, K, V as [B, H, L, D] views of [B, L, H, D] projections."""
    g = torch.Generator(device="cuda").manual_seed(seed)
    dtype = _DTYPES[case["dtype"]]
    B, Hq, Hkv, D, Lk = (case[k] for k in ("B", "Hq", "Hkv", "D", "Lk"))
    k = _keys(g, case, dtype, B, Lk, Hkv, D)
    v = _normal(g, dtype, B, Lk, Hkv, D)
    q = _normal(g, dtype, B, case.get("Lq", Lk), Hq, D)
    return q.transpose(1, 2), k.transpose(1, 2), v.transpose(1, 2)


class _OneLayer:
    """Stands for a model of one layer: each call hands the cache the
    projections of its tokens."""

    def __init__(self, q, k, v):
        self.q, self.k, self.v = q, k, v

    def __call__(self, input_ids, past_key_values, use_cache):
        s = past_key_values.get_seq_length()
        e = s + input_ids.shape[1]
        past_key_values.update(self.q[:, :, s:e], self.k[:, :, s:e], self.v[:, :, s:e], 0)


def _decode_state(case, seed):
    g = torch.Generator(device="cuda").manual_seed(seed)
    dtype = _DTYPES[case["dtype"]]
    B, Hq, Hkv, D, n = (case[k] for k in ("B", "Hq", "Hkv", "D", "rows"))
    C = (n + case["room"] + 63) // 64 * 64
    s = {"scale": D ** -0.5, "layers": []}
    for _ in range(case["layers"]):
        kb, vb = (torch.zeros(B, Hkv, C, D, dtype=dtype, device="cuda") for _ in range(2))
        kb[:, :, :n] = _normal(g, dtype, B, Hkv, n, D)
        vb[:, :, :n] = _normal(g, dtype, B, Hkv, n, D)
        q = _normal(g, dtype, B, 1, Hq, D).transpose(1, 2)
        kn = _normal(g, dtype, B, 1, Hkv, D).transpose(1, 2)
        vn = _normal(g, dtype, B, 1, Hkv, D).transpose(1, 2)
        out = torch.empty(B, 1, Hq, D, dtype=dtype, device="cuda")
        s["layers"].append((q, kn, vn, kb, vb, out))
    s["n"] = torch.full((1,), n, dtype=torch.int32, device="cuda")
    s["ws"] = ops.decode_workspace(B, Hq, Hkv, D, C, "cuda")
    return s


def _decode_step(s):
    for q, kn, vn, kb, vb, out in s["layers"]:
        ops.decode_attention(q, kn, vn, kb, vb, s["n"], s["scale"], out, s["ws"])
    return {"out": [lay[5] for lay in s["layers"]], "k": s["layers"][-1][3], "v": s["layers"][-1][4]}


def prepare(case, seed):
    op = case["op"]
    if op in ("decode", "graph"):
        s = _decode_state(case, seed)
        if op == "graph":
            side = torch.cuda.Stream()
            side.wait_stream(torch.cuda.current_stream())
            with torch.cuda.stream(side):
                _decode_step(s)
            torch.cuda.current_stream().wait_stream(side)
            s["graph"] = torch.cuda.CUDAGraph()
            with torch.cuda.graph(s["graph"]):
                s["result"] = _decode_step(s)
        return dict(s, case=case)
    q, k, v = _qkv(case, seed)
    s = {"case": case}
    if op == "chunked":
        s["model"] = _OneLayer(q, k, v)
        s["ids"] = torch.zeros(case["B"], case["Lk"], dtype=torch.int64, device="cuda")
        return s
    if op in ("plan", "scores", "deployed") or case.get("per_head"):
        k, v = k.contiguous(), v.contiguous()
    if op == "plan":
        keep = max(int(case["ratio"] * case["Lk"]), case["window"], 1)
        s["plan"] = ops.EvictPlan(q, k, case["window"], case["kernel"], keep, keep_scores=True)
    return dict(s, q=q, k=k, v=v)


def run(state):
    case = state["case"]
    op = case["op"]
    if op == "graph":
        state["graph"].replay()
        return state["result"]
    if op == "decode":
        return _decode_step(state)
    if op == "scores":
        return dropkv_scores_triton(state["q"], state["k"], state["v"], case["window"],
                                    match_pytorch_precision=case["p_round"])
    if op == "deployed":
        return ops.scores(state["q"], state["k"], state["v"], case["window"], y_round=True)
    if op == "plan":
        plan = state["plan"]
        idx, k, v = plan(state["q"], state["k"], state["v"])
        return {"scores": plan.scores, "idx": idx, "k": k, "v": v}
    if op == "chunked":
        cache = DropKVCache(case["ratio"], case["window"], case["kernel"], capacity=case["Lk"] + 64)
        prefill_chunked(state["model"], state["ids"], cache, chunk_size=case["chunk"], evict_strategy=case["strategy"])
        return {"k": cache.key_cache[0], "v": cache.value_cache[0]}
    cache = DropKVCache(case["ratio"], case["window"], case["kernel"])
    cache.update(state["q"], state["k"], state["v"], 0)
    return {"k": cache.key_cache[0], "v": cache.value_cache[0]}


def work(case):
    """K and V read once and what is kept written once; the products Q K^T,
    P V and Y V^T of the scores, or the two of an attention step."""
    B, Hq, Hkv, D, eb = case["B"], case["Hq"], case["Hkv"], case["D"], _BYTES[case["dtype"]]
    if case["op"] in ("decode", "graph"):
        n = case["rows"] + 1
        return {"bytes": case["layers"] * B * (2 * Hkv * n + 2 * Hq) * D * eb,
                "flops": case["layers"] * 4 * B * Hq * n * D}
    L, W = case["Lk"], case["window"]
    size = 2 * B * Hkv * L * D * eb + B * Hq * W * D * eb
    flops = 6 * B * Hq * W * L * D
    if case["op"] in ("scores", "deployed"):
        return {"bytes": size + 4 * B * Hkv * L, "flops": flops}
    keep = max(int(case["ratio"] * L), W, 1)
    size += 2 * B * Hkv * keep * D * eb
    if case["op"] == "plan":
        size += B * Hkv * (4 * L + 8 * keep)
    if case["op"] == "chunked":
        size += 2 * B * Hkv * L * D * eb  # every chunk is stored
        chunks = -(-L // case["chunk"])
        if case["strategy"] == "every_chunk":
            flops = flops * (0.5 + 0.05 * chunks)  # kept rows are scored again with each later chunk
    return {"bytes": size, "flops": flops}


def tolerance(case):
    """About four times what the scores of two summation orders (other key
    splits), and the scores and the 64-bit ones, were seen to differ by.  The
    largest differences come from a p that rounds the other way to 16 bits, and
    with heavy-tailed keys from p close to 1.  Kept rows are copies: the
    selection was the same in every order that was tried."""
    op = case["op"]
    if op in ("update", "chunked"):
        return "exact"
    if op in ("decode", "graph"):
        return {"rel": 4e-3 if case["dtype"] == "bf16" else 6e-4, "max": 0.04}
    if case["dtype"] == "fp32":
        return {"rel": 6e-6, "max": 3e-5}
    heavy = case["keys"] == "student"
    if not case.get("p_round", True):
        return {"rel": 6e-6, "max": 3e-5} if case["keys"] == "normal" else {"rel": 1e-3 if heavy else 2e-4, "max": 5e-3}
    return {"rel": 1.2e-2, "max": 0.16} if heavy else {"rel": 8e-4, "max": 0.05}


def _round(x, dtype):
    return x.to(dtype).double()


def exact(case, seed):
    op = case["op"]
    if op in ("decode", "graph"):
        s = _decode_state(case, seed)
        n, g = case["rows"], case["Hq"] // case["Hkv"]
        outs = []
        for q, kn, vn, kb, vb, _ in s["layers"]:
            per_b = []
            for b in range(case["B"]):
                k = torch.cat([kb[b, :, :n], kn[b]], dim=1).double()
                v = torch.cat([vb[b, :, :n], vn[b]], dim=1).double()
                heads = []
                for h in range(case["Hq"]):
                    p = torch.softmax((q[b, h].double() @ k[h // g].t()) * s["scale"], dim=-1)
                    heads.append(p @ v[h // g])
                per_b.append(torch.stack(heads, dim=1))
            outs.append(torch.stack(per_b))
        return {"out": outs, "k": None, "v": None}
    if op in ("update", "chunked"):
        return None  # rows of K and V, copied
    q, k, v = _qkv(case, seed)
    dtype = q.dtype
    B, Hq, Hkv, D, L, W = (case[x] for x in ("B", "Hq", "Hkv", "D", "Lk", "window"))
    g = Hq // Hkv
    p_round, y_round = case.get("p_round", True), op == "deployed"
    bound = torch.arange(L - W, L, device="cuda").repeat(g)
    seen = torch.arange(L, device="cuda")[None, :] <= bound[:, None]
    out = torch.empty(B, Hkv, L, dtype=torch.float64, device="cuda")
    for b in range(B):
        for h in range(Hkv):
            qt = q[b, h * g:(h + 1) * g, -W:].reshape(g * W, D).double()
            kd, vd = k[b, h].double(), v[b, h].double()
            logits = (qt @ kd.t()) / math.sqrt(D)
            p = torch.softmax(logits.masked_fill(~seen, -math.inf), dim=-1)
            if p_round and dtype != torch.float32:
                p = _round(p, dtype)
            y = p @ vd
            if y_round and dtype != torch.float32:
                y = _round(y, dtype)
            d2 = vd.square().sum(-1)[None, :] - 2 * (y @ vd.t()) + y.square().sum(-1)[:, None]
            out[b, h] = ((p / (1 - p + 1e-6)).square() * d2.clamp_min_(0)).sum(0) / g
    if op == "plan":
        return {"scores": out, "idx": None, "k": None, "v": None}
    return out
