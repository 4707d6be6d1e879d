"""The attention calls whose speed this package is judged by, from one decode
step to a long training batch, each through the public Python interface.

A case is a dict of plain values with a "path":

* "train":  forward and backward of flash_attn_func or of its packed forms
* "varlen": the same on a packed batch of sequences of mixed lengths
* "prompt": forward only, no gradients (prefill, scoring, evaluation)
* "cache":  flash_attn_with_kvcache: decode steps and prompt chunks on a
            contiguous, remapped or paged cache, with an append

Inputs are fp16 (the interface's type) and normal with unit variance, as
projections after a normalisation are.  Lengths of mixed batches follow from
the case alone (its "lengths" number), values from the seed.
"""

import math
import os
import random
import sys

import torch

sys.path.insert(0, os.path.join(os.getcwd(), "flash-attention-turing_amd"))
import flash_attention_interface as fai  # noqa: E402

PAGE = 256  # tokens of a cache page
THETA = 10000.0  # base of the rotary angles


def _train(name, batch, seqlen, heads, heads_k, dim, causal, packed):
    return {"name": name, "path": "train", "batch": batch, "seqlen_q": seqlen, "seqlen_k": seqlen, "heads": heads,
            "heads_k": heads_k, "dim": dim, "causal": causal, "packed": packed}


def _cache(name, batch, queries, heads, heads_k, dim, shortest, longest, layout, **more):
    """queries: query tokens a sequence; as many new tokens are appended, except where "append" says none.
    shortest, longest: tokens that are in the cache before the call."""
    case = {"name": name, "path": "cache", "batch": batch, "queries": queries, "append": True, "heads": heads,
            "heads_k": heads_k, "dim": dim, "shortest": shortest, "longest": longest, "layout": layout, "lengths": 3,
            "splits": 0, "window": -1, "rotary": False, "validate": False}
    case.update(more)
    return case


def listed():
    return [
        # One user's next token in a chat: one sequence, the drop-in call with its default host checks.
        _cache("decode_one", 1, 1, 32, 8, 128, 1500, 1500, "contiguous", validate=True),
        # A serving step: 64 sequences of 1k to 32k tokens in a paged cache, the host checks off.
        _cache("decode_batch", 64, 1, 32, 8, 128, 1024, 32768, "paged", splits=8),
        # Drafted tokens checked against long documents: 4 queries on 65k to 131k tokens of a remapped cache.
        _cache("decode_long", 4, 4, 16, 16, 64, 65536, 131068, "remapped", splits=16),
        # A serving step of a model with rotary positions and a sliding window, both done by the call.
        _cache("decode_rotary_window", 16, 1, 32, 8, 128, 512, 8192, "paged", window=4095, rotary=True),
        # A short prompt's only pass: scoring or the first answer of a chat.
        {"name": "prompt_short", "path": "prompt", "batch": 1, "seqlen_q": 509, "seqlen_k": 509, "heads": 32,
         "heads_k": 8, "dim": 128, "causal": True, "packed": "none"},
        # The next piece of two long prompts in a paged serving cache (chunked prefill).
        _cache("chunk_paged", 2, 512, 32, 8, 128, 4096, 12000, "paged"),
        # The same on a contiguous cache: a document that is read 1024 tokens at a time.
        _cache("chunk_contiguous", 1, 1024, 32, 8, 128, 15000, 15000, "contiguous"),
        # An encoder's training step on short, padded texts: packed projections, no mask.
        _train("train_short", 8, 509, 16, 16, 64, False, "qkv"),
        # The benchmark's headline step.
        _train("train_4k", 4, 4096, 16, 16, 128, True, "none"),
        # One long text on each GPU, grouped heads: the usual shape of long-context training.
        _train("train_long", 1, 8192, 32, 8, 128, True, "kv"),
        # A packed batch of documents of mixed lengths, grouped heads.
        {"name": "train_varlen", "path": "varlen", "batch": 16, "heads": 32, "heads_k": 8, "dim": 128, "shortest": 128,
         "longest": 4096, "causal": True, "lengths": 2},
        # Long sequences without a mask (images, audio, proteins): the largest call.
        _train("train_full", 4, 8192, 16, 16, 64, False, "none"),
    ]


HEADS = [(8, 8), (16, 16), (12, 4), (16, 4), (32, 8), (32, 4), (32, 2)]
MOST_FLOPS = 14 * 4 * 16 * 64 * 8192 ** 2  # the largest listed case's
MOST_TOKENS = 64 * 16384  # cache tokens x (kv heads x dim / 1024) of the largest listed decode step


def _log(rng, lo, hi):
    return min(hi, max(lo, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    path = rng.choice(["train", "train", "varlen", "prompt", "decode", "decode", "chunk"])
    heads, heads_k = rng.choice(HEADS)
    dim = rng.choice([64, 128, 128])
    causal = rng.random() < 0.7
    if path in ("train", "prompt"):
        seqlen = _log(rng, 100 if path == "train" else 16, 16384)
        case = {"path": path, "batch": _log(rng, 1, 16), "seqlen_q": seqlen, "seqlen_k": seqlen, "heads": heads,
                "heads_k": heads_k, "dim": dim, "causal": causal,
                "packed": rng.choice(["none", "none", "kv"] + (["qkv"] if heads == heads_k else []))}
        if case["packed"] != "qkv" and rng.random() < 0.25:  # cross attention, or a prompt behind a prefix
            case["seqlen_k"] = _log(rng, seqlen, 16384)
    elif path == "varlen":
        longest = _log(rng, 128, 8192)
        case = {"path": path, "batch": _log(rng, 3, 32), "heads": heads, "heads_k": heads_k, "dim": dim,
                "shortest": rng.randint(16, longest), "longest": longest, "causal": causal,
                "lengths": rng.randrange(1 << 20)}
    else:
        chunk = path == "chunk"
        longest = _log(rng, 256, 32768)
        case = _cache("", _log(rng, 1, 4 if chunk else 64), _log(rng, 32, 1024) if chunk else rng.choice([1, 1, 1, 2, 4]),
                      heads, heads_k, dim, rng.randint(longest // 4, longest), longest,
                      rng.choice(["contiguous", "remapped", "paged", "paged"]), lengths=rng.randrange(1 << 20),
                      window=rng.choice([-1, -1, -1, 1023, 4095]), validate=rng.random() < 0.5)
        case["append"] = chunk or rng.random() < 0.85
        case["rotary"] = case["append"] and rng.random() < 0.3
        del case["name"]
        while case["batch"] > 1 and case["batch"] * longest * heads_k * dim > MOST_TOKENS * 1024:
            case["batch"] -= 1
    while work(case)["flops"] > MOST_FLOPS:
        if case["batch"] > 1:
            case["batch"] -= 1
        else:
            case["seqlen_q"], case["seqlen_k"] = case["seqlen_q"] * 7 // 8, case["seqlen_k"] * 7 // 8
    return case


def _lengths(case):
    r = random.Random(case["lengths"])
    return [r.randint(case["shortest"], case["longest"]) for _ in range(case["batch"])]


def _pairs(sq, sk, causal, window=-1):
    """Visible (query, key) pairs; queries are the last sq of the sk positions."""
    if not causal and window < 0:
        return sq * sk
    n = 0
    for i in range(sq):
        p = i + sk - sq
        hi = min(sk - 1, p) if causal else sk - 1
        lo = max(0, p - window) if window >= 0 else 0
        n += max(0, hi - lo + 1)
    return n


def _capacity(case):
    top = case["longest"] + (case["queries"] if case["append"] else 0)
    return (top + PAGE - 1) // PAGE * PAGE


def work(case):
    h, hk, d = case["heads"], case["heads_k"], case["dim"]
    if case["path"] == "cache":
        sq, new = case["queries"], case["queries"] if case["append"] else 0
        pairs = keys = 0
        for n in _lengths(case):
            n += new
            pairs += _pairs(sq, n, True, case["window"])
            keys += min(n, case["window"] + sq) if case["window"] >= 0 else n
        b = case["batch"]
        # K and V of the visible keys; q, out and lse; the new keys and values read and written.
        byts = keys * hk * d * 4 + b * sq * h * (d * 4 + 4) + b * new * hk * d * 8
        return {"bytes": byts, "flops": 4 * h * d * pairs}
    if case["path"] == "varlen":
        lens = _lengths(case)
        pairs = sum(_pairs(n, n, case["causal"]) for n in lens)
        rows = cols = sum(lens)
    else:
        rows, cols = case["batch"] * case["seqlen_q"], case["batch"] * case["seqlen_k"]
        pairs = case["batch"] * _pairs(case["seqlen_q"], case["seqlen_k"], case["causal"])
    if case["path"] == "prompt":
        return {"bytes": 4 * d * (rows * h + cols * hk), "flops": 4 * h * d * pairs}
    # q, dout read, out, dq written; k, v read, dk, dv written.
    return {"bytes": 8 * d * (rows * h + cols * hk), "flops": 14 * h * d * pairs}


def tolerance(case):
    # About four times the largest error against 64 bits measured over the
    # listed and a dozen drawn cases: relative 3.2e-4 with gradients and 3.0e-4
    # without (outputs are rounded to fp16; the tiled kernels round the
    # probabilities too); single values 3.1e-2 (gradients and causal rows that
    # see few keys), 3.8e-3 (prompts) and 1.5e-3 (cache calls).
    if case["path"] == "cache":
        return {"rel": 1.2e-3, "max": 6e-3}
    if case["path"] == "prompt":
        return {"rel": 1.2e-3, "max": 3e-2}
    return {"rel": 1.3e-3, "max": 0.12}


def _randn(shape, gen):
    return torch.randn(shape, generator=gen, device="cuda", dtype=torch.float16)


def prepare(case, seed):
    g = torch.Generator(device="cuda").manual_seed(seed)
    h, hk, d = case["heads"], case["heads_k"], case["dim"]
    if case["path"] == "cache":
        return _prepare_cache(case, seed, g)
    state = {"case": case}
    if case["path"] == "varlen":
        lens = _lengths(case)
        cu = [0]
        for n in lens:
            cu.append(cu[-1] + n)
        state["cu"] = torch.tensor(cu, dtype=torch.int32, device="cuda")
        state["longest"] = max(lens)
        shapes = {"q": (cu[-1], h, d), "k": (cu[-1], hk, d), "v": (cu[-1], hk, d), "dout": (cu[-1], h, d)}
    else:
        b, sq, sk = case["batch"], case["seqlen_q"], case["seqlen_k"]
        shapes = {"q": (b, sq, h, d), "k": (b, sk, hk, d), "v": (b, sk, hk, d), "dout": (b, sq, h, d)}
        if case["packed"] == "qkv":
            shapes = {"qkv": (b, sq, 3, h, d), "dout": shapes["dout"]}
        elif case["packed"] == "kv":
            shapes = {"q": shapes["q"], "kv": (b, sk, 2, hk, d), "dout": shapes["dout"]}
        if case["path"] == "prompt":
            del shapes["dout"]
    for name, shape in shapes.items():
        state[name] = _randn(shape, g)
        if case["path"] != "prompt" and name != "dout":
            state[name].requires_grad_(True)
    return state


def _prepare_cache(case, seed, g):
    b, sq, h, hk, d = case["batch"], case["queries"], case["heads"], case["heads_k"], case["dim"]
    new = sq if case["append"] else 0
    lens, cap = _lengths(case), _capacity(case)
    state = {"case": case, "lens": lens, "q": _randn((b, sq, h, d), g), "k": None, "v": None, "table": None,
             "rows": None, "cos": None, "sin": None,
             "seqlens": torch.tensor(lens, dtype=torch.int32, device="cuda")}
    if new:
        state["k"], state["v"] = _randn((b, new, hk, d), g), _randn((b, new, hk, d), g)
    if case["layout"] == "paged":
        pages = [(n + new + PAGE - 1) // PAGE for n in lens]
        order = list(range(sum(pages)))
        random.Random(seed).shuffle(order)
        table, at = [], 0
        for n in pages:
            table.append(order[at : at + n] + [0] * (cap // PAGE - n))
            at += n
        state["table"] = torch.tensor(table, dtype=torch.int32, device="cuda")
        shape = (sum(pages), PAGE, hk, d)
    elif case["layout"] == "remapped":
        rows = random.Random(seed).sample(range(2 * b), b)
        state["rows"] = torch.tensor(rows, dtype=torch.int32, device="cuda")
        shape = (2 * b, cap, hk, d)
    else:
        shape = (b, cap, hk, d)
    state["k_cache"], state["v_cache"] = _randn(shape, g), _randn(shape, g)
    if case["rotary"]:
        freq = THETA ** (-torch.arange(0, d, 2, device="cuda", dtype=torch.float64) / d)
        angle = torch.arange(cap, device="cuda", dtype=torch.float64)[:, None] * freq[None]
        state["cos"], state["sin"] = angle.cos().half(), angle.sin().half()
    return state


def run(state):
    case = state["case"]
    if case["path"] == "cache":
        out, lse = fai.flash_attn_with_kvcache(
            state["q"], state["k_cache"], state["v_cache"], k=state["k"], v=state["v"], rotary_cos=state["cos"],
            rotary_sin=state["sin"], cache_seqlens=state["seqlens"], cache_batch_idx=state["rows"],
            block_table=state["table"], causal=True, window_size=(case["window"], -1), rotary_interleaved=False,
            num_splits=case["splits"], return_softmax_lse=True, validate=case["validate"])
        answer = {"out": out, "lse": lse}
        if case["append"]:
            answer["k_cache"], answer["v_cache"] = state["k_cache"], state["v_cache"]
        return answer
    if case["path"] == "prompt":
        with torch.no_grad():
            return {"out": _attend(state, case)}
    out = _attend(state, case)
    names = [n for n in ("q", "k", "v", "kv", "qkv") if n in state]
    grads = torch.autograd.grad(out, [state[n] for n in names], state["dout"])
    answer = {"d" + n: t for n, t in zip(names, grads)}
    answer["out"] = out
    return answer


def _attend(state, case):
    if case["path"] == "varlen":
        return fai.flash_attn_varlen_func(state["q"], state["k"], state["v"], state["cu"], state["cu"],
                                          state["longest"], state["longest"], causal=case["causal"])
    if case["packed"] == "qkv":
        return fai.flash_attn_qkvpacked_func(state["qkv"], causal=case["causal"])
    if case["packed"] == "kv":
        return fai.flash_attn_kvpacked_func(state["q"], state["kv"], causal=case["causal"])
    return fai.flash_attn_func(state["q"], state["k"], state["v"], causal=case["causal"])


# The same results in float64 by plain torch, one (sequence, query head) at a time.


def _scores(q, k, first, causal, window):
    """Softmax inputs of queries at key positions first, first + 1, ... (float64, [rows, keys])."""
    s = q @ k.t().contiguous() * q.shape[-1] ** -0.5
    if causal or window >= 0:
        p = torch.arange(first, first + q.shape[0], device=q.device)[:, None]
        j = torch.arange(k.shape[0], device=q.device)[None, :]
        hide = j > p if causal else torch.zeros_like(s, dtype=torch.bool)
        if window >= 0:
            hide = hide | (j < p - window)
        s = s.masked_fill(hide, -math.inf)
    return s


ROWS = 4096  # query rows worked on at a time


def _exact_head(q, k, v, dout, causal, window=-1):
    """out, lse and (with dout) dq, dk, dv of one head, float64 [rows, dim] operands."""
    out, lse = torch.empty_like(q), torch.empty_like(q[:, 0])
    dq, dk, dv = torch.empty_like(q), torch.zeros_like(k), torch.zeros_like(v)
    scale = q.shape[-1] ** -0.5
    for at in range(0, q.shape[0], ROWS):
        rows = slice(at, at + ROWS)
        s = _scores(q[rows], k, at + k.shape[0] - q.shape[0], causal, window)
        lse[rows] = torch.logsumexp(s, -1)
        p = torch.exp(s - lse[rows, None])
        out[rows] = p @ v
        if dout is not None:
            do = dout[rows]
            dv += p.t().contiguous() @ do
            ds = p * (do @ v.t().contiguous() - (do * out[rows]).sum(-1, keepdim=True))
            dq[rows] = ds @ k * scale
            dk += ds.t().contiguous() @ q[rows] * scale
    return out, lse, dq, dk, dv


def _exact_batch(q, k, v, dout, causal):
    """[rows, heads, dim] operands of one sequence: out, dq, dk, dv in float64."""
    group = q.shape[1] // k.shape[1]
    wide = [torch.empty(t.shape, dtype=torch.float64, device=t.device) for t in (q, q)]
    narrow = [torch.zeros(t.shape, dtype=torch.float64, device=t.device) for t in (k, v)]
    for h in range(q.shape[1]):
        one = [t[:, i].double().contiguous() for t, i in ((q, h), (k, h // group), (v, h // group))]
        do = None if dout is None else dout[:, h].double().contiguous()
        out, _, dq, dk, dv = _exact_head(*one, do, causal)
        wide[0][:, h], wide[1][:, h] = out, dq
        narrow[0][:, h // group] += dk
        narrow[1][:, h // group] += dv
    return wide[0], wide[1], narrow[0], narrow[1]


def _rotated(x, cos, sin, first, each):
    """x [tokens, heads, dim] turned to positions first, first + 1, ... (or all to first)."""
    at = first + torch.arange(x.shape[0], device=x.device) * (1 if each else 0)
    c, s = cos[at].double()[:, None], sin[at].double()[:, None]
    a, b = x.double().chunk(2, -1)
    return torch.cat([a * c - b * s, a * s + b * c], -1)


def _exact_cache(case, state):
    b, sq, h, hk, d = case["batch"], case["queries"], case["heads"], case["heads_k"], case["dim"]
    out = torch.empty((b, sq, h, d), dtype=torch.float64, device="cuda")
    lse = torch.empty((b, h, sq), dtype=torch.float64, device="cuda")
    for i, n in enumerate(state["lens"]):
        q, kn, vn = state["q"][i].double(), state["k"], state["v"]
        if state["table"] is not None:
            pages = state["table"][i, : (n + PAGE - 1) // PAGE].long()
            k, v = (state[c][pages].reshape(-1, hk, d)[:n] for c in ("k_cache", "v_cache"))
        else:
            row = i if state["rows"] is None else int(state["rows"][i])
            k, v = state["k_cache"][row, :n], state["v_cache"][row, :n]
        k, v = k.double(), v.double()
        if kn is not None:
            kn, vn = kn[i].double(), vn[i].double()
            if case["rotary"]:
                kn = _rotated(kn, state["cos"], state["sin"], n, True)
                q = _rotated(q, state["cos"], state["sin"], n, True)
            k, v = torch.cat([k, kn]), torch.cat([v, vn])
        for j in range(hk):
            kj, vj = k[:, j].contiguous(), v[:, j].contiguous()
            for head in range(j * (h // hk), (j + 1) * (h // hk)):
                out[i, :, head], lse[i, head] = _exact_head(q[:, head].contiguous(), kj, vj, None, True,
                                                            case["window"])[:2]
    return {"out": out, "lse": lse, "k_cache": None, "v_cache": None}


def exact(case, seed):
    state = prepare(case, seed)
    if case["path"] == "cache":
        answer = _exact_cache(case, state)
        return answer if case["append"] else {"out": answer["out"], "lse": answer["lse"]}
    with torch.no_grad():
        return _exact_dense(case, state)


def _exact_dense(case, state):
    if "qkv" in state:
        q, k, v = state["qkv"].unbind(2)
    elif "kv" in state:
        q, (k, v) = state["q"], state["kv"].unbind(2)
    else:
        q, k, v = state["q"], state["k"], state["v"]
    dout = state.get("dout")
    if case["path"] == "varlen":
        cu = state["cu"].tolist()
        parts = [_exact_batch(*(t[a:b] for t in (q, k, v, dout)), case["causal"]) for a, b in zip(cu, cu[1:])]
        out, dq, dk, dv = (torch.cat(t) for t in zip(*parts))
    else:
        parts = [_exact_batch(q[i], k[i], v[i], None if dout is None else dout[i], case["causal"])
                 for i in range(q.shape[0])]
        out, dq, dk, dv = (torch.stack(t) for t in zip(*parts))
    if case["path"] == "prompt":
        return {"out": out}
    if "qkv" in state:
        return {"out": out, "dqkv": torch.stack([dq, dk, dv], 2)}
    if "kv" in state:
        return {"out": out, "dq": dq, "dkv": torch.stack([dk, dv], 2)}
    return {"out": out, "dq": dq, "dk": dk, "dv": dv}
