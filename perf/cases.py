"""The work that programs have this package do: cases with their inputs, one pass of each through the public entry
points (the torch operators `torch.ops.ckopt.*` and the package's functions), the work each pass cannot do without, and
its result in 64 bits.

A case is a dict of plain values; "op" names the entry point:
  softmax      torch.ops.ckopt.softmax            rows of logits, or attention scores with a causal mask
  rmsnorm      torch.ops.ckopt.rmsnorm            hidden states, or every head's query and key vectors, with a weight
  rmsnorm_add  torch.ops.ckopt.rmsnorm_add        the residual add in front of a decoder layer's norm
  rope         rope() / torch.ops.ckopt.rope      rotation on the fly from inverse frequencies, or from a cos/sin cache
  rope_kv      rope_kv()                          rotation and the write of keys and values into a paged cache
  topk         torch.ops.ckopt.topk               a sampler's candidates from logits, or a router's experts
  topk_sample  torch.ops.ckopt.topk_and_sample    the candidates and a draw from them

listed() is the fixed set, draw(rng) gives more of the same ranges. Every input is drawn on the GPU from the seed.
"""

import importlib
import math

import torch

_PACKAGE = "cuda-kernels-optimized-for-rtx5090_amd"
_DTYPES = {"fp32": torch.float32, "bf16": torch.bfloat16, "fp16": torch.float16}
_BYTES = {"fp32": 4, "bf16": 2, "fp16": 2}
_THETA = 10000.0
_EPS = 1e-6
_MOST = 1 << 26  # elements of the largest case's activations (16384 x 4096)


def listed():
    return [
        # fp32 attention or classifier rows of a model's hidden length, many rows: the bandwidth-bound softmax
        {"name": "softmax_rows", "op": "softmax", "dtype": "fp32", "rows": 4096, "cols": 4096, "masked": False},
        # attention scores while a sequence grows by a token at a time: 32 heads x 256 queries over a length that is no
        # multiple of anything, with the causal mask's -inf in place
        {"name": "softmax_attention", "op": "softmax", "dtype": "bf16", "rows": 8192, "cols": 3001, "masked": True},
        # probabilities over a vocabulary for a small decode batch: few, long rows
        {"name": "softmax_vocab", "op": "softmax", "dtype": "fp32", "rows": 16, "cols": 128256, "masked": False},
        # a decoder layer's norm over a prefill of 4 x 4096 tokens: the largest case
        {"name": "rmsnorm_prefill", "op": "rmsnorm", "dtype": "bf16", "rows": 16384, "cols": 4096},
        # the norm of each query and key head (head size 128) of a 4096-token prefill with 32 + 8 heads
        {"name": "rmsnorm_heads", "op": "rmsnorm", "dtype": "bf16", "rows": 163840, "cols": 128},
        # the residual add and norm of one decode step of 48 sequences: launch-bound
        {"name": "rmsnorm_add_decode", "op": "rmsnorm_add", "dtype": "fp16", "rows": 48, "cols": 5120},
        # RoPE of a prefill of 4 x 4096 tokens, grouped-query heads, on the fly
        {"name": "rope_prefill", "op": "rope", "dtype": "bf16", "batch": 4, "seq": 4096, "q_heads": 32, "kv_heads": 8,
         "head_dim": 128, "cache": "none"},
        # one decode step of 64 sequences: RoPE and the write into a paged KV cache, launch-bound
        {"name": "rope_kv_decode", "op": "rope_kv", "dtype": "bf16", "batch": 64, "seq": 1, "q_heads": 32,
         "kv_heads": 8, "head_dim": 128, "slots": 8192},
        # the sampler of a serving step: top 50 of a large vocabulary and a draw, for 128 sequences
        {"name": "topk_sample", "op": "topk_sample", "dtype": "fp32", "rows": 128, "cols": 128256, "k": 50},
        # a sampler's candidates from bf16 logits over a vocabulary of odd size
        {"name": "topk_ragged", "op": "topk", "dtype": "bf16", "rows": 64, "cols": 49999, "k": 50},
        # a wide candidate list (reranking, beams, truncated distributions kept for distillation)
        {"name": "topk_wide", "op": "topk", "dtype": "fp32", "rows": 128, "cols": 128256, "k": 1024},
        # a mixture-of-experts router: 8 of 128 experts for each token of a prefill
        {"name": "topk_router", "op": "topk", "dtype": "fp32", "rows": 16384, "cols": 128, "k": 8},
    ]


def _log(rng, low, high):
    """An integer from low to high, spread over the logarithm."""
    return min(high, max(low, int(round(math.exp(rng.uniform(math.log(low), math.log(high)))))))


def _length(rng, low, high):
    """A row length: any integer half of the time, else a multiple of 8 or of 256."""
    n, unit = _log(rng, low, high), rng.choice([1, 1, 8, 256])
    return min(high, max(low, n // unit * unit)) if n >= unit else n


def draw(rng):
    kind = rng.choice(["softmax", "attention", "rmsnorm", "heads", "rmsnorm_add", "rope", "rope_kv", "topk", "topk",
                       "topk_sample", "router"])
    if kind in ("softmax", "attention"):
        dtype = rng.choice(["fp32", "bf16"])
        cols = _length(rng, 512, 262144) if kind == "softmax" else _log(rng, 128, 16384)
        most = min(65536, (_MOST // 4) * 4 // _BYTES[dtype] // cols)
        return {"op": "softmax", "dtype": dtype, "rows": _log(rng, 1, most), "cols": cols,
                "masked": kind == "attention"}
    if kind in ("rmsnorm", "rmsnorm_add"):
        cols = _log(rng, 512, 16384) // 8 * 8 if rng.random() < 0.75 else _log(rng, 500, 9000)
        most = _MOST // cols if kind == "rmsnorm" else _MOST // 2 // cols
        return {"op": kind, "dtype": rng.choice(["bf16", "fp16"]), "rows": _log(rng, 1, most), "cols": cols}
    if kind == "heads":
        cols = rng.choice([64, 80, 96, 128, 192, 256])
        return {"op": "rmsnorm", "dtype": rng.choice(["bf16", "fp16"]), "rows": _log(rng, 64, _MOST // 2 // cols),
                "cols": cols}
    if kind in ("rope", "rope_kv"):
        kv_heads = rng.choice([1, 2, 4, 8])
        q_heads = kv_heads * rng.choice([1, 3, 4, 7, 8])
        head_dim = rng.choice([64, 80, 96, 128, 128, 256])
        tokens = _log(rng, 1, _MOST // 2 // ((q_heads + 2 * kv_heads) * head_dim))
        batch = min(tokens, _log(rng, 1, 64))
        case = {"op": kind, "dtype": rng.choice(["bf16", "fp16"]), "batch": batch, "seq": min(16384, tokens // batch),
                "q_heads": q_heads, "kv_heads": kv_heads, "head_dim": head_dim}
        if kind == "rope":
            case["cache"] = rng.choice(["none", "fp32", "bf16"])
        else:
            case["slots"] = max(1024, case["batch"] * case["seq"] * 5 // 4)
        return case
    dtype = rng.choice(["fp32", "bf16"])
    if kind == "router":
        cols = _log(rng, 16, 512)
        return {"op": "topk", "dtype": dtype, "rows": _log(rng, 1, 32768), "cols": cols, "k": rng.randint(1, min(16, cols))}
    cols = _length(rng, 16000, 262144)
    rows = _log(rng, 1, min(512, _MOST // 4 // cols))
    k = _log(rng, 1, 1024) if kind == "topk" else _log(rng, 2, 100)
    return {"op": kind, "dtype": dtype, "rows": rows, "cols": cols, "k": k}


def _generator(seed):
    return torch.Generator(device="cuda").manual_seed(int(seed))


def _normal(g, shape, dtype, scale=1.0):
    return (torch.randn(shape, generator=g, device="cuda", dtype=torch.float32) * scale).to(dtype)


def _softmax_input(case, g):
    rows, cols = case["rows"], case["cols"]
    x = _normal(g, (rows, cols), torch.float32, 3.0)
    if case["masked"]:
        # causal: the last queries of a sequence of `cols` keys; query i of a head sees all but the keys after it
        queries = min(256, rows, cols)
        seen = cols - queries + 1 + torch.arange(rows, device="cuda") % queries
        x.masked_fill_(torch.arange(cols, device="cuda")[None, :] >= seen[:, None], float("-inf"))
    return x.to(_DTYPES[case["dtype"]])


def _positions(case, g):
    """Prefills start somewhere in a sequence; a decode step's sequences are each at a place of their own."""
    batch, seq = case["batch"], case["seq"]
    start = torch.randint(0, 8192, (batch, 1), generator=g, device="cuda")
    return (start + torch.arange(seq, device="cuda")[None, :]).contiguous()


def _inv_freq(head_dim):
    return 1.0 / (_THETA ** (torch.arange(0, head_dim, 2, dtype=torch.int64).float() / head_dim))


def _inputs(case, seed):
    g, dtype, op = _generator(seed), _DTYPES[case["dtype"]], case["op"]
    if op == "softmax":
        return {"x": _softmax_input(case, g)}
    if op in ("rmsnorm", "rmsnorm_add"):
        t = {"x": _normal(g, (case["rows"], case["cols"]), dtype)}
        t["weight"] = (torch.rand(case["cols"], generator=g, device="cuda") + 0.5).to(dtype)
        if op == "rmsnorm_add":
            t["residual"] = _normal(g, (case["rows"], case["cols"]), dtype)
        return t
    if op in ("rope", "rope_kv"):
        batch, seq, d = case["batch"], case["seq"], case["head_dim"]
        t = {"q": _normal(g, (batch, seq, case["q_heads"], d), dtype),
             "k": _normal(g, (batch, seq, case["kv_heads"], d), dtype),
             "position_ids": _positions(case, g), "inv_freq": _inv_freq(d).cuda()}
        if op == "rope" and case["cache"] != "none":
            freqs = torch.outer(torch.arange(8192 + seq, dtype=torch.float32, device="cuda"), t["inv_freq"])
            emb = torch.cat((freqs, freqs), dim=-1)
            t["cos"], t["sin"] = emb.cos().to(_DTYPES[case["cache"]]), emb.sin().to(_DTYPES[case["cache"]])
        if op == "rope_kv":
            tokens, slots = batch * seq, case["slots"]
            t["v"] = _normal(g, (batch, seq, case["kv_heads"], d), dtype)
            mapping = torch.randperm(slots, generator=g, device="cuda")[:tokens].view(batch, seq)
            if seq > 8:  # a padded prefill: the last tokens of the first sequence are not written
                mapping[0, -3:] = -1
            t["slot_mapping"] = mapping.contiguous()
            t["k_cache"] = _normal(g, (slots, case["kv_heads"], d), dtype)
            t["v_cache"] = _normal(g, (slots, case["kv_heads"], d), dtype)
        return t
    t = {"x": _normal(g, (case["rows"], case["cols"]), torch.float32, 2.0).to(dtype)}
    if op == "topk_sample":
        t["uniforms"] = torch.rand(case["rows"], generator=g, device="cuda")
    return t


def prepare(case, seed):
    package = importlib.import_module(_PACKAGE)
    state = _inputs(case, seed)
    state["case"], state["package"], state["ops"] = dict(case), package, package.ops()
    return state


def run(state):
    case, ops, package = state["case"], state["ops"], state["package"]
    op = case["op"]
    if op == "softmax":
        return ops.softmax(state["x"])
    if op == "rmsnorm":
        return ops.rmsnorm(state["x"], state["weight"], _EPS)
    if op == "rmsnorm_add":
        return ops.rmsnorm_add(state["x"], state["residual"], state["weight"], _EPS)
    if op == "rope":
        if case["cache"] == "none":
            return package.rope(state["q"], state["k"], state["position_ids"], inv_freq=state["inv_freq"])
        return ops.rope(state["q"], state["k"], state["cos"], state["sin"], state["position_ids"])
    if op == "rope_kv":
        q = package.rope_kv(state["q"], state["k"], state["v"], state["position_ids"], state["inv_freq"],
                            state["k_cache"], state["v_cache"], state["slot_mapping"])
        return q, state["k_cache"], state["v_cache"]
    if op == "topk":
        return ops.topk(state["x"], case["k"])
    return ops.topk_and_sample(state["x"], case["k"], state["uniforms"], 0.8, 0.9)


def work(case):
    op, size = case["op"], _BYTES[case["dtype"]]
    if op in ("softmax", "rmsnorm", "rmsnorm_add"):
        n = case["rows"] * case["cols"]
        if op == "softmax":
            return {"bytes": 2 * n * size, "flops": 4 * n}
        streams = 2 if op == "rmsnorm" else 4
        return {"bytes": streams * n * size + case["cols"] * size, "flops": (4 if op == "rmsnorm" else 5) * n}
    if op in ("rope", "rope_kv"):
        tokens, d = case["batch"] * case["seq"], case["head_dim"]
        q, kv = tokens * case["q_heads"] * d, tokens * case["kv_heads"] * d
        n = 2 * (q + kv) * size + tokens * 8
        if op == "rope_kv":
            n += 2 * kv * size + tokens * 8
        elif case["cache"] != "none":
            n += 2 * min(8192 + case["seq"], tokens) * d * _BYTES[case["cache"]]
        return {"bytes": n, "flops": 3 * (q + kv)}
    n = case["rows"] * case["cols"] * size + case["rows"] * case["k"] * (size + 8)
    return {"bytes": n + (case["rows"] * 12 if op == "topk_sample" else 0), "flops": case["rows"] * case["cols"]}


def tolerance(case):
    """fp32 softmax: sums and exponentials in 32 bits. The 16-bit outputs: their own rounding (2^-9 for bf16, 2^-12 for
    fp16, about 0.6 of it in the 2-norm), for RMSNorm also that of the row's factor and of the product before the
    weight. Top-k and the draw from it are whole values and copies of inputs."""
    op = case["op"]
    if op == "softmax":
        return {"rel": 1e-6} if case["dtype"] == "fp32" else {"rel": 7e-3}
    if op in ("topk", "topk_sample"):
        return "exact"
    bf16 = case["dtype"] == "bf16"
    if op in ("rmsnorm", "rmsnorm_add"):
        return {"rel": 1.2e-2} if bf16 else {"rel": 1.5e-3}
    return {"rel": 7e-3 if bf16 else 1e-3}


def _rotate64(x, cos, sin):
    a, b = x.double().chunk(2, dim=-1)
    (c1, c2), (s1, s2) = cos.chunk(2, dim=-1), sin.chunk(2, dim=-1)
    return torch.cat((a * c1 - b * s1, b * c2 + a * s2), dim=-1)


def exact(case, seed):
    t, op = _inputs(case, seed), case["op"]
    if op == "softmax":
        return torch.softmax(t["x"].double(), dim=-1)
    if op == "rmsnorm":
        x = t["x"].double()
        return x * torch.rsqrt(x.square().mean(-1, keepdim=True) + _EPS) * t["weight"].double()
    if op == "rmsnorm_add":
        h = t["x"].double() + t["residual"].double()
        # the norm is of the sum as it is kept, in the tensors' own type
        n = h.to(_DTYPES[case["dtype"]]).double()
        return n * torch.rsqrt(n.square().mean(-1, keepdim=True) + _EPS) * t["weight"].double(), h
    if op in ("rope", "rope_kv"):
        if "cos" in t:
            cos, sin = (t[n].double()[t["position_ids"]].unsqueeze(2) for n in ("cos", "sin"))
        else:
            # the angle is the fp32 product of position and inverse frequency, as the cache's is
            angle = (t["position_ids"].float()[..., None] * t["inv_freq"]).double()
            angle = torch.cat((angle, angle), dim=-1).unsqueeze(2)
            cos, sin = angle.cos(), angle.sin()
        q, k = _rotate64(t["q"], cos, sin), _rotate64(t["k"], cos, sin)
        if op == "rope":
            return q, k
        slots = t["slot_mapping"].view(-1)
        kept = slots >= 0
        k_cache, v_cache = t["k_cache"].double(), t["v_cache"].double()
        k_cache[slots[kept]] = k.flatten(0, 1)[kept]
        v_cache[slots[kept]] = t["v"].double().flatten(0, 1)[kept]
        return q, k_cache, v_cache
    # a stable descending sort: ties by the lower index
    values, indices = torch.sort(t["x"], dim=-1, descending=True, stable=True)
    out = values[:, : case["k"]].contiguous(), indices[:, : case["k"]].contiguous()
    return out if op == "topk" else (*out, None)
