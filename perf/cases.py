"""The workloads by which this framework's speed is judged: the calls that a program built on it makes, over their real ranges.

Each kind is one public entry point with the sizes, layouts, data types and options that it is used with: the linears of a decode
step and of a prompt, plain and ragged matrix products in every supported type, causal prefill, the ymodel2 example's transposed
cache, the MATH backend, the masked product, decode attention over ragged caches, and the Qwen3-0.6B shape as a whole model.
`listed` holds one case of each kind, `draw` gives more over the same ranges.
"""
from __future__ import annotations

import math

import torch

import ytensor_amd as yt
from ytensor_amd import ops
from ytensor_amd.qwen3 import Qwen3, Qwen3Config, weight_layout

DEV = "cuda"
DTYPES = {"bf16": torch.bfloat16, "fp16": torch.float16, "fp32": torch.float32}
SIZE = {"bf16": 2, "fp16": 2, "fp32": 4}
# (in, out) features of the projections of the Qwen3-0.6B shape: qkv, attention output, gate_up, down
PROJECTIONS = ((1024, 4096), (2048, 1024), (1024, 6144), (3072, 1024))


def listed() -> list[dict]:
    return [
        # One decode step's projection: a single activation row against a weight, where the launch and its latency are what counts.
        {"name": "linear_decode", "kind": "linear", "m": 1, "k": 1024, "n": 3072, "dtype": "bf16", "bias": False},
        # A prompt's down projection (512 tokens): a long sum into few columns, the product that leaves most of the chip idle.
        {"name": "linear_prompt", "kind": "linear", "m": 512, "k": 3072, "n": 1024, "dtype": "bf16", "bias": False},
        # The large square product.
        {"name": "matmul_large", "kind": "matmul", "batch": 0, "m": 4096, "n": 4096, "k": 4096, "dtype": "bf16"},
        # A product none of whose sizes is a multiple of anything: a user's own data matrix.
        {"name": "matmul_ragged", "kind": "matmul", "batch": 0, "m": 1021, "n": 1003, "k": 779, "dtype": "bf16"},
        # The reference's own type, at a round decimal size.
        {"name": "matmul_fp32", "kind": "matmul", "batch": 0, "m": 1000, "n": 1000, "k": 1000, "dtype": "fp32"},
        # Prefill attention of a 2048-token prompt, 16 query and 8 key/value heads.
        {"name": "attention_prompt", "kind": "attention", "b": 1, "hq": 16, "hkv": 8, "sq": 2048, "skv": 2048, "d": 128,
         "dtype": "bf16", "mask": "causal", "bias": False, "backend": "flash"},
        # The ymodel2 example's attention: fp32, the ring cache stored transposed, values shared by both key heads, a ring mask.
        {"name": "attention_transposed", "kind": "pega2", "b": 1, "hh": 4, "sq": 256, "skv": 1024, "d": 64},
        # The MATH backend on a prompt.
        {"name": "attention_math", "kind": "attention", "b": 1, "hq": 16, "hkv": 8, "sq": 1024, "skv": 1024, "d": 128,
         "dtype": "bf16", "mask": "causal", "bias": False, "backend": "math"},
        # The masked product under a causal mask.
        {"name": "masked_matmul", "kind": "masked", "m": 2048, "n": 2048, "k": 2048, "dtype": "bf16", "mask": "causal"},
        # One token for each of 16 sequences whose caches are filled to different lengths.
        {"name": "attention_decode", "kind": "decode", "b": 16, "hq": 16, "hkv": 8, "ctx": 4096, "d": 128, "dtype": "bf16"},
        # The whole model: a 512-token prompt up to its first token.
        {"name": "qwen3_prompt", "kind": "qwen3", "prompt": 512, "tokens": 1},
        # The whole model: a short question and its greedy answer, which is decode steps almost throughout.
        {"name": "qwen3_answer", "kind": "qwen3", "prompt": 24, "tokens": 24},
    ]


def _log(rng, lo: int, hi: int) -> int:
    return max(lo, min(hi, round(math.exp(rng.uniform(math.log(lo), math.log(hi + 1))))))


def draw(rng) -> dict:
    kind = rng.choice(("linear_decode", "linear_prompt", "matmul", "matmul_ragged", "attention", "attention", "pega2", "math",
                       "masked", "decode", "qwen3_prompt", "qwen3_answer"))
    half = rng.choice(("bf16", "bf16", "fp16"))
    any_type = rng.choice(("bf16", "fp16", "fp32"))
    if kind == "linear_decode":
        k, n = rng.choice(PROJECTIONS + ((_log(rng, 8, 512) * 8, _log(rng, 64, 8192)),))
        return {"kind": "linear", "m": rng.randint(1, 16), "k": k, "n": n, "dtype": half, "bias": rng.random() < 0.3}
    if kind == "linear_prompt":
        k, n = rng.choice(PROJECTIONS + ((_log(rng, 8, 512) * 8, _log(rng, 64, 8192)),))
        return {"kind": "linear", "m": _log(rng, 17, 2048), "k": k, "n": n, "dtype": half, "bias": rng.random() < 0.3}
    if kind == "matmul":  # round sizes, in batches too
        batch = rng.choice((0, 0, 4, 16))
        top = 64 if batch == 0 else 16
        return {"kind": "matmul", "batch": batch, "m": 64 * _log(rng, 1, top), "n": 64 * _log(rng, 1, top),
                "k": 64 * _log(rng, 1, top), "dtype": any_type}
    if kind == "matmul_ragged":
        return {"kind": "matmul", "batch": rng.choice((0, 0, 3)), "m": _log(rng, 30, 2500), "n": _log(rng, 30, 2500),
                "k": _log(rng, 30, 2500), "dtype": any_type}
    if kind == "attention":
        dtype = rng.choice(("bf16", "bf16", "fp16", "fp32"))
        s = _log(rng, 100, 8192 if dtype != "fp32" else 4096)
        return {"kind": "attention", "b": 1 if s > 2048 else rng.choice((1, 1, 2)), "hq": 16, "hkv": rng.choice((8, 8, 4, 16)),
                "sq": s, "skv": s if rng.random() < 0.7 else s + _log(rng, 16, 1024), "d": rng.choice((128, 128, 64)),
                "dtype": dtype, "mask": rng.choice(("causal", "causal", "none", "bytes")), "bias": False, "backend": "flash"}
    if kind == "pega2":
        skv = _log(rng, 64, 1024)
        return {"kind": "pega2", "b": rng.choice((1, 1, 2)), "hh": rng.choice((2, 4)), "sq": _log(rng, 2, min(256, skv)),
                "skv": skv, "d": rng.choice((64, 64, 128))}
    if kind == "math":
        s = _log(rng, 100, 1024)
        return {"kind": "attention", "b": 1, "hq": 16, "hkv": rng.choice((8, 16)), "sq": s, "skv": s, "d": rng.choice((64, 128)),
                "dtype": any_type, "mask": rng.choice(("causal", "none", "bytes")), "bias": rng.random() < 0.3, "backend": "math"}
    if kind == "masked":
        m, n, k = (rng.choice((1, 8)) * _log(rng, 30, 256) for _ in range(3))
        return {"kind": "masked", "m": m, "n": n, "k": k, "dtype": any_type, "mask": rng.choice(("causal", "bytes"))}
    if kind == "decode":
        b = _log(rng, 1, 32)
        return {"kind": "decode", "b": b, "hq": 16, "hkv": rng.choice((8, 8, 4)), "ctx": _log(rng, 128, 131072 // max(b, 8)),
                "d": rng.choice((128, 128, 64)), "dtype": half}
    if kind == "qwen3_prompt":
        return {"kind": "qwen3", "prompt": _log(rng, 17, 512), "tokens": 1}
    return {"kind": "qwen3", "prompt": _log(rng, 4, 64), "tokens": rng.randint(4, 24)}


# ---------------------------------------------------------------------------
# inputs
# ---------------------------------------------------------------------------

def _rand(gen, *shape, dtype="bf16", scale=1.0):
    x = torch.randn(*shape, device=DEV, generator=gen)
    return (x * scale if scale != 1.0 else x).to(DTYPES[dtype])


def _offdiagonal_mask(gen, m: int, n: int, what: str):
    """None, "causal", or that mask as bytes with one key in sixteen hidden besides (padding); each row sees its first key."""
    if what == "none":
        return None
    if what == "causal":
        return "causal"
    i, j = torch.arange(m, device=DEV)[:, None], torch.arange(n, device=DEV)[None, :]
    mask = (j <= i + max(n - m, 0)) & (torch.rand(n, device=DEV, generator=gen) > 1 / 16)[None, :]
    mask[:, 0] = True
    return mask


def _decode_lengths(case) -> list[int]:
    """Filled rows of each sequence's cache, from half of it to all of it."""
    b, ctx = case["b"], case["ctx"]
    return [ctx - (i * 2654435761 % 4096) * (ctx // 2) // 4096 for i in range(b)]


def _model_weights(cfg, gen):
    """Random weights of the Qwen3-0.6B shape that a 16-bit type holds exactly: matrices N(0, 0.02), norm weights about 1, and
    embedding rows (the tied head) of unit values, which make the greedy choice decisive as a trained model's is."""
    parts = []
    for name, shape in weight_layout(cfg):
        n = math.prod(shape)
        if name == "embed":
            w = torch.randn(n, device=DEV, generator=gen)
        elif "norm" in name:
            w = 1.0 + 0.1 * torch.randn(n, device=DEV, generator=gen)
        else:
            w = 0.02 * torch.randn(n, device=DEV, generator=gen)
        parts.append(w.bfloat16().float())
    return torch.cat(parts)


def _inputs(case, seed):
    """What both prepare and exact start from, made from the seed alone."""
    gen = torch.Generator(device=DEV)
    gen.manual_seed(int(seed))
    kind = case["kind"]
    if kind == "linear":
        x = _rand(gen, case["m"], case["k"], dtype=case["dtype"])
        w = _rand(gen, case["n"], case["k"], dtype=case["dtype"], scale=0.02)
        return {"x": x, "w": w, "b": _rand(gen, case["n"], dtype=case["dtype"]) if case["bias"] else None}
    if kind == "matmul":
        lead = (case["batch"],) if case["batch"] else ()
        return {"a": _rand(gen, *lead, case["m"], case["k"], dtype=case["dtype"]),
                "b": _rand(gen, *lead, case["k"], case["n"], dtype=case["dtype"], scale=0.02)}
    if kind == "attention":
        q = _rand(gen, case["b"], case["hq"], case["sq"], case["d"], dtype=case["dtype"])
        k = _rand(gen, case["b"], case["hkv"], case["skv"], case["d"], dtype=case["dtype"])
        v = _rand(gen, case["b"], case["hkv"], case["skv"], case["d"], dtype=case["dtype"])
        bias = _rand(gen, case["sq"], case["skv"], dtype="fp32") if case["bias"] else None
        return {"q": q, "k": k, "v": v, "mask": _offdiagonal_mask(gen, case["sq"], case["skv"], case["mask"]), "bias": bias}
    if kind == "pega2":
        b, hh, sq, skv, d = (case[x] for x in ("b", "hh", "sq", "skv", "d"))
        q = _rand(gen, b, 2, hh, sq, d, dtype="fp32")
        kv = _rand(gen, b, 2, d, skv, dtype="fp32").transpose(-1, -2)  # [b, 2, skv, d] seen through the transposed cache
        start = int(seed) % skv  # the ring's write position
        i, j = torch.arange(sq, device=DEV)[:, None], torch.arange(skv, device=DEV)[None, :]
        return {"q": q, "k": kv.unsqueeze(2).expand(b, 2, hh, skv, d),
                "v": kv[:, 1:2].expand(b, 2, skv, d).unsqueeze(2).expand(b, 2, hh, skv, d),
                "mask": (j - start) % skv <= skv - sq + i}
    if kind == "masked":
        return {"a": _rand(gen, case["m"], case["k"], dtype=case["dtype"]),
                "b": _rand(gen, case["k"], case["n"], dtype=case["dtype"], scale=0.02),
                "mask": _offdiagonal_mask(gen, case["m"], case["n"], case["mask"])}
    if kind == "decode":
        k = _rand(gen, case["b"], case["hkv"], case["ctx"], case["d"], dtype=case["dtype"])
        v = _rand(gen, case["b"], case["hkv"], case["ctx"], case["d"], dtype=case["dtype"])
        return {"q": _rand(gen, case["b"], case["hq"], case["d"], dtype=case["dtype"]), "k": k, "v": v,
                "len": torch.tensor(_decode_lengths(case), dtype=torch.int32, device=DEV)}
    cfg = Qwen3Config()
    prompt = torch.randint(0, cfg.vocab, (case["prompt"],), device=DEV, generator=gen)
    return {"cfg": cfg, "weights": _model_weights(cfg, gen), "prompt": prompt.cpu().numpy()}


def prepare(case, seed):
    s = _inputs(case, seed)
    s["case"] = case
    if case["kind"] == "decode":
        s["workspace"] = torch.empty(ops.decode_workspace_bytes(case["b"], case["hq"], case["ctx"], case["d"]),
                                     dtype=torch.uint8, device=DEV)
    if case["kind"] == "qwen3":
        s["model"] = Qwen3(s["cfg"], s.pop("weights"), max_prompt=512)
    return s


def run(state):
    case = state["case"]
    kind = case["kind"]
    if kind == "linear":
        return yt.linear(state["x"], state["w"], state["b"])
    if kind == "matmul":
        return yt.matmul(state["a"], state["b"])
    if kind == "attention":
        return yt.scaled_dot_product_attention(state["q"], state["k"], state["v"], mask=state["mask"], bias=state["bias"],
                                               backend=case["backend"])
    if kind == "pega2":
        return yt.scaled_dot_product_attention(state["q"], state["k"], state["v"], mask=state["mask"])
    if kind == "masked":
        return yt.masked_matmul(state["a"], state["b"], state["mask"])
    if kind == "decode":
        return yt.decode_attention(state["q"], state["k"], state["v"], kv_len=state["len"], workspace=state["workspace"])
    model = state["model"]
    tokens = model.generate(state["prompt"], case["tokens"])
    return {"tokens": tokens, "logits": model.logits}


# ---------------------------------------------------------------------------
# what a pass cannot do without, how far two correct ones may differ, and the result in 64 bits
# ---------------------------------------------------------------------------

def _visible(case) -> float:
    """Query-key pairs that a mask leaves visible (bytes hide one key in sixteen more)."""
    sq, skv = (case["sq"], case["skv"]) if "sq" in case else (case["m"], case["n"])
    if case.get("mask", "causal") == "none":
        return sq * skv
    off = skv - sq if "sq" in case or case["mask"] == "causal" else max(skv - sq, 0)
    full = sum(max(0, min(skv, i + off + 1)) for i in range(sq))
    return full * (15 / 16 if case.get("mask") == "bytes" else 1)


def work(case) -> dict:
    kind, es = case["kind"], SIZE[case.get("dtype", "fp32")]
    if kind == "linear":
        m, n, k = case["m"], case["n"], case["k"]
        return {"bytes": es * (m * k + n * k + m * n + (n if case["bias"] else 0)), "flops": 2 * m * n * k}
    if kind == "matmul":
        b, m, n, k = max(1, case["batch"]), case["m"], case["n"], case["k"]
        return {"bytes": es * b * (m * k + n * k + m * n), "flops": 2 * b * m * n * k}
    if kind == "attention":
        rows = case["b"] * case["d"] * (2 * case["hq"] * case["sq"] + 2 * case["hkv"] * case["skv"])
        extra = case["sq"] * case["skv"] * ((case["mask"] == "bytes") + 4 * case["bias"])
        return {"bytes": es * rows + extra, "flops": 4 * case["b"] * case["hq"] * case["d"] * _visible(case)}
    if kind == "pega2":
        rows = case["b"] * case["d"] * (2 * 2 * case["hh"] * case["sq"] + 2 * case["skv"])
        return {"bytes": 4 * rows + case["sq"] * case["skv"],
                "flops": 4 * case["b"] * 2 * case["hh"] * case["d"] * _visible(case)}
    if kind == "masked":
        m, n, k = case["m"], case["n"], case["k"]
        return {"bytes": es * (m * k + n * k + m * n) + (m * n if case["mask"] == "bytes" else 0), "flops": 2 * k * _visible(case)}
    if kind == "decode":
        rows = sum(_decode_lengths(case))
        return {"bytes": es * case["d"] * (2 * case["hkv"] * rows + 2 * case["b"] * case["hq"]),
                "flops": 4 * case["hq"] * case["d"] * rows}
    cfg = Qwen3Config()
    sizes = {name: math.prod(shape) for name, shape in weight_layout(cfg)}
    layers = sum(n for name, n in sizes.items() if name not in ("embed", "norm"))
    p, t = case["prompt"], case["tokens"]
    steps = t - 1
    weights = 2 * (layers + sizes["embed"])
    kv = 2 * 2 * cfg.layers * cfg.n_kv * cfg.head_dim
    pairs = p * (p + 1) / 2 + sum(p + i + 1 for i in range(steps))
    return {"bytes": (1 + steps) * weights + kv * (p + steps * p + steps * (steps + 1) / 2) + 4 * t * cfg.vocab,
            "flops": 2 * layers * (p + steps) + 2 * sizes["embed"] * t + 4 * cfg.layers * cfg.n_heads * cfg.head_dim * pairs}


def tolerance(case) -> dict:
    """About four times how far the results are from `exact`: 16-bit rounding of the result and, in attention, of the weights
    (measured 1.7e-3 to 2.5e-3 in bf16, an eighth of that in fp16), 32-bit sums (6e-7), and 28 layers of both (5e-3)."""
    if case["kind"] == "qwen3":  # 28 layers of 16-bit activations; the tokens are decisive and do not differ
        return {"rel": 2e-2, "max": 0.2, "differ": 0.0}
    dtype = case.get("dtype", "fp32")
    if dtype == "fp32":
        return {"rel": 5e-6, "max": 1e-4}
    return {"rel": 1e-2 if dtype == "bf16" else 2e-3, "max": 0.1 if dtype == "bf16" else 2e-2}


def _attention64(q, k, v, visible=None, bias=None):
    """softmax(q k^T / sqrt(d) + bias) v over the visible keys; [..., S, d] in float64, head by head."""
    out = torch.empty(*q.shape[:-1], v.shape[-1], dtype=torch.float64, device=q.device)
    for idx in torch.cartesian_prod(*[torch.arange(n) for n in q.shape[:-2]]).reshape(-1, q.dim() - 2).tolist():
        idx = tuple(idx)
        s = (q[idx].double() @ k[idx].double().T) / math.sqrt(q.shape[-1])
        if bias is not None:
            s += bias.double()
        if visible is not None:
            s.masked_fill_(~visible, -math.inf)
        s = torch.nan_to_num(torch.softmax(s, -1), nan=0.0)  # a row that sees no key is zero
        out[idx] = s @ v[idx].double()
    return out


def _visible_matrix(mask, m: int, n: int):
    if mask is None or isinstance(mask, torch.Tensor):
        return mask
    i, j = torch.arange(m, device=DEV)[:, None], torch.arange(n, device=DEV)[None, :]
    return j <= i + (n - m)


def _qwen3_64(case, s):
    """The decoder in float64 from the same weights: the tokens that it is given and takes greedily, and the last step's logits."""
    cfg, flat = s["cfg"], s["weights"]
    w, at = {}, 0
    for name, shape in weight_layout(cfg):
        n = math.prod(shape)
        w[name] = flat[at:at + n].reshape(shape)
        at += n
    hd, nh, nkv = cfg.head_dim, cfg.n_heads, cfg.n_kv
    freq = cfg.theta ** (-torch.arange(0, hd, 2, device=DEV, dtype=torch.float64) / hd)

    def norm(x, weight):
        return x / torch.sqrt((x * x).mean(-1, keepdim=True) + cfg.eps) * weight.double()

    def rope(x, pos):  # [h, S, hd]
        a = pos[:, None] * freq[None, :]
        c, sn = torch.cos(a).repeat(1, 2), torch.sin(a).repeat(1, 2)
        return x * c + torch.cat((-x[..., hd // 2:], x[..., :hd // 2]), -1) * sn

    def linear(x, weight):
        return x @ weight.double().T

    cache = [None] * cfg.layers
    ids = torch.as_tensor(s["prompt"], device=DEV)
    tokens, logits, seen = [], None, 0
    for _ in range(case["tokens"]):
        n = ids.numel()
        x = w["embed"][ids].double()
        pos = torch.arange(seen, seen + n, device=DEV, dtype=torch.float64)
        for i in range(cfg.layers):
            L = lambda part: w[f"{i}.{part}"]  # noqa: E731
            h = norm(x, L("norm1"))
            q = rope(norm(linear(h, L("q")).view(n, nh, hd).transpose(0, 1), L("q_norm")), pos)
            k = rope(norm(linear(h, L("k")).view(n, nkv, hd).transpose(0, 1), L("k_norm")), pos)
            v = linear(h, L("v")).view(n, nkv, hd).transpose(0, 1)
            if cache[i] is not None:
                k, v = torch.cat((cache[i][0], k), 1), torch.cat((cache[i][1], v), 1)
            cache[i] = (k, v)
            group = nh // nkv
            o = _attention64(q, k.repeat_interleave(group, 0), v.repeat_interleave(group, 0), _visible_matrix("causal", n, seen + n))
            x = x + linear(o.transpose(0, 1).reshape(n, nh * hd), L("o"))
            h = norm(x, L("norm2"))
            x = x + linear(torch.nn.functional.silu(linear(h, L("gate"))) * linear(h, L("up")), L("down"))
        logits = linear(norm(x[-1:], w["norm"]), w["embed"])
        ids = logits[0].argmax().reshape(1)
        tokens.append(int(ids))
        seen += n
    return {"tokens": torch.tensor(tokens, dtype=torch.int32).numpy(), "logits": logits}


def exact(case, seed):
    s = _inputs(case, seed)
    kind = case["kind"]
    if kind == "linear":
        y = s["x"].double() @ s["w"].double().T
        return y if s["b"] is None else y + s["b"].double()
    if kind == "matmul":
        return s["a"].double() @ s["b"].double()
    if kind == "attention":
        group = case["hq"] // case["hkv"]
        return _attention64(s["q"], s["k"].repeat_interleave(group, 1), s["v"].repeat_interleave(group, 1),
                            _visible_matrix(s["mask"], case["sq"], case["skv"]), s["bias"])
    if kind == "pega2":
        return _attention64(s["q"], s["k"], s["v"], s["mask"])
    if kind == "masked":
        return (s["a"].double() @ s["b"].double()).masked_fill(~_visible_matrix(s["mask"], case["m"], case["n"]), 0.0)
    if kind == "decode":
        group = case["hq"] // case["hkv"]
        visible = torch.arange(case["ctx"], device=DEV)[None, :] < s["len"][:, None]
        out = [_attention64(s["q"][i].unsqueeze(1), s["k"][i].repeat_interleave(group, 0), s["v"][i].repeat_interleave(group, 0),
                            visible[i][None]) for i in range(case["b"])]
        return torch.stack(out).squeeze(2)
    return _qwen3_64(case, s)
