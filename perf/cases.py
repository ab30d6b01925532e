"""The work a program gives this framework, as cases that can be timed and compared.

A program decodes with cached block steps (32 rows to refine a block, 8 for a sub-block), prefills a
prompt, scores continuations against a long prefix, refines many sequences' blocks at once, runs a short
sequence without a cache, takes the lm_head's logits or confidence, or keeps its own model and calls the
attention alone.  Sizes are the 1.5B configuration's and the benchmark's workloads (prefixes of 512, 2048
and 8192 rows, 16 sequences with prefixes in [128, 1024], blocks of 32 and sub-blocks of 8).  Steps run a
few decoder layers: a layer costs the same in a deeper model, and rounding does not travel as far.  A
prefill runs all 28, since what its last layer has to do is less than the others'.
"""

from __future__ import annotations

import math
import random

import torch

import __graft_entry__

__graft_entry__.load_package()

from fast_dllm_relax_amd.config import fast_dllm_v2_1p5b  # noqa: E402
from fast_dllm_relax_amd.params import TORCH_DTYPES, param_names, param_shapes  # noqa: E402
from fast_dllm_relax_amd.runtime import build_prefix_block_attention_bias  # noqa: E402
from fast_dllm_relax_amd.vm import HipVM  # noqa: E402

DEV = "cuda"
BLOCK = 32
VOCAB = 151936
SMALL_VOCAB = 4096  # layers alone: the embedding table and the head play no part in what is timed

# a case's fields: `layers` deep; `rows` of one call; `prefix` rows in the cache before it; `nseq`
# sequences whose prefixes are drawn from [lo, hi] with `lens`; `rp` a partial step's row in its block


def listed():
    return [
        # the attention callback of a program that keeps its own projections, once per layer and block step
        dict(name="callback_32_p2048", kind="callback", layers=4, rows=32, prefix=2048, dtype="bfloat16"),
        # the decode loop's most frequent call: 8 rows of a sub-block, a short conversation
        dict(name="partial_8_p512", kind="partial", layers=4, rows=8, prefix=512, rp=16, dtype="bfloat16"),
        # a block refinement step, a prompt of 2048: embedding, layers and logits with their confidence
        dict(name="call_32_p2048", kind="call", layers=8, rows=32, prefix=2048, dtype="bfloat16"),
        # a block step after a long prompt, which is not a whole number of blocks
        dict(name="step_32_p8175", kind="step", layers=4, rows=32, prefix=8175, dtype="bfloat16"),
        # scoring a continuation of 64 tokens (and the prompt's tail) against a long prefix, with its logits
        dict(name="score_83_p8192", kind="score", layers=4, rows=83, prefix=8192, dtype="bfloat16"),
        # many sequences' blocks refined together, and a sub-block of each
        dict(name="batch_16x32", kind="batch", layers=4, rows=32, nseq=16, lo=128, hi=1024, lens=3, dtype="float16"),
        dict(name="batch_16x8", kind="batch_partial", layers=4, rows=8, rp=8, nseq=16, lo=128, hi=1024, lens=3,
             dtype="float16"),
        # the confidence of those sub-blocks' rows: the lm_head without its logits
        dict(name="head_128", kind="head", rows=128, dtype="float16"),
        # a sequence without a cached prefix: an explicit bias and logits for every row
        dict(name="stateless_84", kind="stateless", layers=4, rows=84, dtype="bfloat16"),
        # prompts: an ordinary one of odd length, a long one, the longest
        dict(name="prefill_509", kind="prefill", layers=28, rows=509, dtype="bfloat16"),
        dict(name="prefill_2048", kind="prefill", layers=28, rows=2048, dtype="bfloat16"),
        dict(name="prefill_8192", kind="prefill", layers=28, rows=8192, dtype="bfloat16"),
    ]


def _log_size(rng, lo, hi):
    """A whole number of [lo, hi], spread over its logarithm."""
    return min(hi, int(math.exp(rng.uniform(math.log(lo), math.log(hi + 1)))))


def draw(rng: random.Random):
    kind = rng.choice(("callback", "partial", "step", "step", "call", "score", "batch", "batch_partial", "head", "stateless",
                       "prefill", "prefill"))
    dtype = rng.choice(("bfloat16", "bfloat16", "float16"))
    prefix = _log_size(rng, 64, 8192)
    if rng.random() < 0.5:
        prefix = prefix // BLOCK * BLOCK
    if kind == "callback":
        return dict(kind=kind, layers=4, rows=_log_size(rng, 4, 300), prefix=prefix, dtype=dtype)
    if kind == "partial":
        return dict(kind=kind, layers=4, rows=8, prefix=prefix, rp=rng.choice((0, 8, 16, 24)), dtype=dtype)
    if kind == "step":
        return dict(kind=kind, layers=4, rows=rng.choice((BLOCK, _log_size(rng, 1, 200))), prefix=prefix, dtype=dtype)
    if kind == "call":
        return dict(kind=kind, layers=4, rows=BLOCK, prefix=prefix, dtype=dtype)
    if kind == "score":
        return dict(kind=kind, layers=4, rows=_log_size(rng, BLOCK, 160), prefix=prefix, dtype=dtype)
    if kind in ("batch", "batch_partial"):
        lo = _log_size(rng, 64, 512)
        c = dict(kind=kind, layers=4, rows=BLOCK if kind == "batch" else BLOCK // 4, nseq=_log_size(rng, 2, 32), lo=lo,
                 hi=lo + _log_size(rng, 32, 1500), lens=rng.randrange(1 << 20), dtype=dtype)
        return c if kind == "batch" else dict(c, rp=rng.choice((0, 8, 16, 24)))
    if kind == "head":
        return dict(kind=kind, rows=_log_size(rng, 1, 512), dtype=dtype)
    if kind == "stateless":
        return dict(kind=kind, layers=4, rows=_log_size(rng, 8, 300), dtype=dtype)
    return dict(kind=kind, layers=28, rows=_log_size(rng, 48, 8192), dtype=dtype)


def _config(case):
    full = case["kind"] in ("call", "score", "head", "stateless")
    return fast_dllm_v2_1p5b(num_hidden_layers=case.get("layers", 1), vocab_size=VOCAB if full else SMALL_VOCAB)


def _generator(seed):
    g = torch.Generator(device=DEV)
    g.manual_seed(seed)
    return g


def _normal(g, shape, dtype, std=1.0):
    return (torch.empty(shape, dtype=torch.float32, device=DEV).normal_(0.0, 1.0, generator=g) * std).to(dtype)


def _params(cfg, g, td):
    """Weights N(0, 0.02), as the benchmark makes them, and norm weights near 1."""
    shapes = param_shapes(cfg)
    return [(1.0 + _normal(g, shapes[n], torch.float32, 0.1)).to(td) if n.endswith("norm.weight") else
            _normal(g, shapes[n], td, 0.02) for n in param_names(cfg)]


def _prefixes(case):
    """The sequences' prefixes, each a whole number of blocks, as the batched loop aligns them."""
    rng = random.Random(case["lens"])
    return [max(1, rng.randint(case["lo"], case["hi"]) // BLOCK) * BLOCK for _ in range(case["nseq"])]


def _inputs(case, seed):
    """The tensors of a case, from the seed alone: weights, token ids or rows, and the cache's earlier rows,
    whose values have the size the projections give them (N(0, 0.02) weights over unit-RMS rows)."""
    cfg, td, g = _config(case), TORCH_DTYPES[case["dtype"]], _generator(seed)
    kind, L, nkv, hd = case["kind"], case.get("layers", 1), cfg.num_key_value_heads, cfg.head_dim
    kv_std = 0.02 * math.sqrt(cfg.hidden_size)
    d = {}
    if kind != "callback":
        d["params"] = _params(cfg, g, td)
    if kind == "callback":
        P, R = case["prefix"], case["rows"]
        d["q"] = _normal(g, (L, 1, R, cfg.num_attention_heads, hd), td, kv_std)
        d["kr"] = _normal(g, (L, 1, R, nkv, hd), td, kv_std)
        d["vr"] = _normal(g, (L, 1, R, nkv, hd), td, kv_std)
        cap = -(-(P + R) // BLOCK) * BLOCK
        shape = (L, 1, cap, nkv, hd)
    elif kind == "head":
        d["hidden"] = _normal(g, (1, case["rows"], cfg.hidden_size), td)
        return cfg, d
    else:
        n = case["rows"] * case.get("nseq", 1)
        d["ids"] = torch.randint(0, cfg.vocab_size, (n,), dtype=torch.int32, device=DEV, generator=g)
        if kind == "stateless":
            return cfg, d
        if kind == "prefill":
            shape = (L, 1, -(-case["rows"] // BLOCK) * BLOCK, nkv, hd)
        elif kind in ("batch", "batch_partial"):
            shape = (L, case["nseq"], max(_prefixes(case)) + BLOCK, nkv, hd)
        else:
            shape = (L, 1, -(-(case["prefix"] + max(case["rows"], BLOCK)) // BLOCK) * BLOCK, nkv, hd)
    if kind == "prefill":
        d["k"], d["v"] = torch.zeros(shape, dtype=td, device=DEV), torch.zeros(shape, dtype=td, device=DEV)
    else:
        d["k"], d["v"] = _normal(g, shape, td, kv_std), _normal(g, shape, td, kv_std)
    return cfg, d


def prepare(case, seed):
    cfg, s = _inputs(case, seed)
    kind = case["kind"]
    if kind == "callback":
        # the callbacks need no weights; the model's own are elsewhere
        cfg = fast_dllm_v2_1p5b(num_hidden_layers=case["layers"], vocab_size=SMALL_VOCAB, intermediate_size=128)
        s["params"] = _params(cfg, _generator(seed), TORCH_DTYPES[case["dtype"]])
    vm = HipVM(cfg, s["params"], dtype=case["dtype"], max_rows=max(64, case["rows"] * case.get("nseq", 1)))
    s.update(case=case, vm=vm)
    if kind in ("step", "call", "score"):
        s["off"] = torch.tensor(case["prefix"], dtype=torch.int32, device=DEV)
    elif kind == "partial":
        s["off"] = torch.tensor(case["prefix"] + case["rp"], dtype=torch.int32, device=DEV)
        s["fn"] = vm[f"forward_block_partial_rp{case['rp']}"]
    elif kind in ("batch", "batch_partial"):
        s["lens"] = _prefixes(case)
        s["off"] = torch.tensor([p + case.get("rp", 0) for p in s["lens"]], dtype=torch.int32, device=DEV)
    elif kind == "stateless":
        prefix = (case["rows"] - 1) // BLOCK * BLOCK
        bias = build_prefix_block_attention_bias(prefix, case["rows"] - prefix, block_size=BLOCK)
        s["bias"] = torch.from_numpy(bias).to(DEV)
    return s


def run(s):
    case, vm = s["case"], s["vm"]
    kind = case["kind"]
    if kind == "callback":
        out = []
        for layer in range(case["layers"]):
            out.append(vm.attn_inplace(s["q"][layer], s["kr"][layer], s["vr"][layer], s["k"], s["v"], layer, case["prefix"],
                                       0, case["rows"])[2])
        return {"out": out, "k": s["k"], "v": s["v"]}
    if kind == "head":
        ids, maxp = vm.get_confidence(s["hidden"])
        return {"ids": ids, "maxp": maxp}
    x = vm.embed_unchecked(s["ids"])
    if kind == "prefill":
        vm.build_prefix_cache(x[None], None, s["k"], s["v"])
        return {"k": s["k"], "v": s["v"]}
    if kind == "stateless":
        hidden = vm.forward_hidden(x[None], s["bias"])
        return {"hidden": hidden, "logits": vm.get_logits(hidden)}
    if kind == "partial":
        hidden = s["fn"](x[None], s["k"], s["v"], s["off"], case["prefix"])
    elif kind == "batch":
        hidden = vm.forward_cached_batch(x.view(case["nseq"], case["rows"], -1), s["k"], s["v"], s["off"], s["lens"])
    elif kind == "batch_partial":
        hidden = vm.forward_block_partial_batch(case["rp"], x.view(case["nseq"], case["rows"], -1), s["k"], s["v"],
                                                s["off"], s["lens"])
    else:
        hidden = vm.forward_cached(x[None], s["k"], s["v"], s["off"], case["prefix"])
    out = {"hidden": hidden, "k": s["k"], "v": s["v"]}
    if kind == "call":
        # the logits and the probability of each row's choice (the choice is the logits' argmax)
        out["logits"] = torch.empty((1, case["rows"], vm.cfg.vocab_size), dtype=torch.float32, device=DEV)
        _, out["maxp"] = vm.get_confidence(hidden, logits=out["logits"])
    elif kind == "score":
        out["logits"] = vm.get_logits(hidden)
    return out


def _spans(case):
    """(first row's position, cache rows before the call's, rows attended) of each sequence of the call."""
    kind, rows = case["kind"], case["rows"]
    if kind in ("prefill", "stateless"):
        return [(0, 0, rows)]
    lens = _prefixes(case) if kind.startswith("batch") else [case["prefix"]]
    rp = case.get("rp", 0)
    return [(p + rp, p, p + BLOCK if "rp" in case else p + rows) for p in lens]


def work(case):
    cfg, kind, rows = _config(case), case["kind"], case["rows"]
    H, I, hd, nq, nkv = (cfg.hidden_size, cfg.intermediate_size, cfg.head_dim, cfg.num_attention_heads,
                         cfg.num_key_value_heads)
    lm = (2 * cfg.vocab_size * H, 2 * rows * cfg.vocab_size * H)  # the head's bytes and operations
    if kind == "head":
        return {"bytes": lm[0] + 2 * rows * H + 8 * rows, "flops": lm[1]}
    L, M = case["layers"], rows * case.get("nseq", 1)
    kv = 2 * nkv * hd * 2  # bytes of one row of K and V
    if kind == "callback":
        keys = case["prefix"] + rows
        return {"bytes": L * (kv * keys + kv * rows + 2 * 2 * rows * nq * hd), "flops": L * 4 * rows * keys * nq * hd}
    pairs = 0  # (query, key) pairs of one head
    for _, _, attended in _spans(case):
        if kind in ("prefill", "stateless"):
            pairs += sum(min(rows, (r // BLOCK + 1) * BLOCK) for r in range(rows))
        else:
            pairs += rows * attended
    lin = cfg.qkv_dim * H + H * nq * hd + 3 * H * I
    read = sum(a for _, _, a in _spans(case)) if kind not in ("prefill", "stateless") else 0
    w = {"bytes": L * (cfg.layer_bytes() + kv * read + (0 if kind == "stateless" else kv * M)) + 2 * M * H,
         "flops": L * (2 * M * lin + 4 * pairs * nq * hd)}
    if kind != "prefill":
        w["bytes"] += 2 * M * H
    if kind == "stateless":
        w["bytes"] += 4 * rows * rows
    if kind in ("call", "score", "stateless"):
        w["bytes"] += lm[0] + 4 * rows * cfg.vocab_size
        w["flops"] += lm[1]
    return w


def tolerance(case):
    """Every tensor between two operators is rounded to 8 (bfloat16) or 11 bits, so another order of the fp32
    sums moves the results by about as much as either is from exact().  Measured: 0.0022 of the attention's
    output, 0.0006 (float16) of the head's probabilities, and after the layers (the farthest output) 0.013
    at 4, 0.020 at 8 and, of a prefill's cache, 0.017 at 28 in bfloat16; 0.0019 at 4 and 0.0022 in float16."""
    bf16 = case["dtype"] == "bfloat16"
    if case["kind"] == "callback":
        return {"rel": 0.01 if bf16 else 0.0015}
    if case["kind"] == "head":
        return {"rel": 0.02 if bf16 else 0.003, "differ": 0.01}
    return {"rel": 0.03 if bf16 else 0.009}


def _rope64(x, pos, theta):
    """x [rows, heads, 128] rotated at the rows' positions (pairs d and d + 64)."""
    half = x.shape[-1] // 2
    inv = torch.exp(-math.log(theta) * torch.arange(half, dtype=torch.float64, device=x.device) / half)
    ang = pos.double()[:, None] * inv
    c, s = torch.cos(ang)[:, None], torch.sin(ang)[:, None]
    a, b = x[..., :half], x[..., half:]
    return torch.cat([a * c - b * s, b * c + a * s], dim=-1)


def _attend64(q, k, v, mask):
    """q [rows, nq, hd] over k / v [keys, nkv, hd]; mask [rows, keys]: True where a row does not see a key."""
    rows, nq, hd = q.shape
    grp = nq // k.shape[1]
    out = torch.empty_like(q)
    for h in range(nq):
        s = (q[:, h] @ k[:, h // grp].t().contiguous()) / math.sqrt(hd)
        if mask is not None:
            s.masked_fill_(mask, -math.inf)
        out[:, h] = torch.softmax(s, dim=-1) @ v[:, h // grp].contiguous()
    return out


def _norm64(x, w, eps):
    return x / torch.sqrt((x * x).mean(dim=-1, keepdim=True) + eps) * w.double()


def exact(case, seed):
    cfg, d = _inputs(case, seed)
    kind, rows = case["kind"], case["rows"]
    nq, nkv, hd, H = cfg.num_attention_heads, cfg.num_key_value_heads, cfg.head_dim, cfg.hidden_size
    if "k" in d:
        k64, v64 = d["k"].double(), d["v"].double()
    if kind == "callback":
        P, out = case["prefix"], []
        for layer in range(case["layers"]):
            k64[layer, 0, P:P + rows], v64[layer, 0, P:P + rows] = d["kr"][layer, 0].double(), d["vr"][layer, 0].double()
            out.append(_attend64(d["q"][layer, 0].double(), k64[layer, 0, :P + rows], v64[layer, 0, :P + rows], None)[None])
        return {"out": out, "k": k64, "v": v64}
    by = dict(zip(param_names(cfg), d["params"]))

    def head(hidden):
        """Logits of hidden [rows, H], a slice of the vocabulary at a time."""
        w = by["model.embed_tokens.weight"]
        return torch.cat([hidden @ w[i:i + 16384].double().t().contiguous() for i in range(0, cfg.vocab_size, 16384)], dim=1)

    def chosen(logits):
        return torch.softmax(logits, dim=-1).amax(dim=-1)[None]

    if kind == "head":
        return {"ids": None, "maxp": chosen(head(d["hidden"][0].double()))}
    spans = _spans(case)
    x = by["model.embed_tokens.weight"][d["ids"].long()].double()
    pos = torch.cat([p + torch.arange(rows, device=DEV) for p, _, _ in spans])
    mask = None
    if kind in ("prefill", "stateless"):
        blk = torch.arange(rows, device=DEV) // BLOCK
        mask = blk[:, None] < blk[None, :]
    for layer in range(case["layers"]):
        p = f"model.layers.{layer}."
        y = _norm64(x, by[p + "input_layernorm.weight"], cfg.rms_norm_eps)
        y = y @ by[p + "self_attn.qkv_proj.weight"].double().t().contiguous() + by[p + "self_attn.qkv_proj.bias"].double()
        y = y.view(-1, nq + 2 * nkv, hd)
        q, kn, vn = _rope64(y[:, :nq], pos, cfg.rope_theta), _rope64(y[:, nq:nq + nkv], pos, cfg.rope_theta), y[:, nq + nkv:]
        o = torch.empty_like(q)
        for b, (first, _, attended) in enumerate(spans):
            r = slice(b * rows, (b + 1) * rows)
            if kind == "stateless":
                o[r] = _attend64(q[r], kn[r], vn[r], mask)
                continue
            k64[layer, b, first:first + rows], v64[layer, b, first:first + rows] = kn[r], vn[r]
            o[r] = _attend64(q[r], k64[layer, b, :attended], v64[layer, b, :attended], mask)
        x = x + o.reshape(-1, nq * hd) @ by[p + "self_attn.o_proj.weight"].double().t().contiguous()
        y = _norm64(x, by[p + "post_attention_layernorm.weight"], cfg.rms_norm_eps)
        y = y @ by[p + "mlp.gate_up_proj.weight"].double().t().contiguous()
        gate, up = y[:, :cfg.intermediate_size], y[:, cfg.intermediate_size:]
        x = x + (gate * torch.sigmoid(gate) * up) @ by[p + "mlp.down_proj.weight"].double().t().contiguous()
    if kind == "prefill":
        return {"k": k64, "v": v64}
    x = _norm64(x, by["model.norm.weight"], cfg.rms_norm_eps)
    out = {"hidden": x.view(case.get("nseq", 1), rows, H)}
    if kind == "stateless":
        out["logits"] = head(x)[None]
        return out
    out.update(k=k64, v=v64)
    if kind in ("call", "score"):
        out["logits"] = head(x)[None]
    if kind == "call":
        out["maxp"] = chosen(out["logits"][0])
    return out
