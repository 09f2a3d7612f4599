"""The work this engine is measured on: traces of token ids through the step function.

A trace is what `python -m holon_amd replay` plays and what serving comes down to: prompts go in, cut into portions under
a step's budget, then every live request brings one token a step, and the logits at the places a sampler would draw from
come back. The tokens are given, so a pass does the same work whatever its logits are. One pass plays a whole trace:
requests are admitted at its start and gone at its end, so that the next pass finds the cache as this one did.

Cases differ in the architecture and its size (the configurations of `holon_amd.benchmark`), the dtype, how many requests
there are, their prompts' lengths, how many tokens they decode and whether they arrive together or one behind the other.
Between them prompts go from a few tokens to several portions, steps from one row to sixteen, and every mixer,
feed-forward and norm that the package has takes part in prompt and in decode steps.
"""
from __future__ import annotations

import hashlib
import math
import random

import numpy as np
import torch

from holon_amd import benchmark
from holon_amd.engine.loading import load_model
from holon_amd.engine.replay import Replayer

PORTION = 4096                    # the token budget of one step, the engine's default
ROUTED = ("dopirax", "falisun", "nevodra")                # experts in bfloat16 traces
# (model, size) -> layers, where fewer than the configuration has are taken: two correct evaluations of a deep bfloat16
# stack of random weights drift apart, the more so where a rounding turns a router's near tie round, and a comparison
# would say nothing. A layer costs what it costs in the whole stack.
LAYERS = {("qwen3", "2k"): 4, ("qwen3", "8b"): 4, ("falisun", "2k"): 2, ("falisun", "4k"): 2, ("sopepel", "2k"): 4}


# -- the cases ------------------------------------------------------------------------------------------------------
def _trace(name: str | None, model: str, size: str, requests: int, shortest: int, longest: int, decode: int, *,
           dtype: str = "bfloat16", arrive: str = "together", portion: int = PORTION) -> dict:
    case = {"model": model, "size": size, "dtype": dtype, "requests": requests, "shortest": shortest,
            "longest": longest, "decode": decode, "arrive": arrive, "portion": portion}
    return case if name is None else dict(case, name=name)


def listed() -> list[dict]:
    return [
        # one person asks about a document: a prompt of two portions, then one row a step
        _trace("document", "qwen3", "8b", 1, 6007, 6007, 64),
        # eight chats that came at once: ordinary prompts of unequal length in shared steps, then eight rows a step
        _trace("chats", "qwen3", "8b", 8, 500, 1400, 64),
        # requests that come one behind the other: portions of a prompt beside the rows that already decode
        _trace("arrivals", "qwen3", "4k", 12, 300, 1500, 24, arrive="in turn", portion=512),
        # the 32-bit path, as it serves to compare logits with: short prompts and a few tokens each
        _trace("yardstick", "qwen3", "2k", 3, 150, 400, 12, dtype="float32"),
        # the same of a design with a recurrence: one longer prompt
        _trace("comparison", "sopepel", "2k", 1, 700, 700, 8, dtype="float32"),
        # a prompt of half a step, and its first tokens
        _trace("summary", "tolurax", "2k", 1, 2048, 2048, 4),
        # the smallest call: one prompt of a few words, one answer
        _trace("few words", "relanex", "2k", 1, 37, 37, 0),
        # a few prompts of a thousand tokens and more at once, their next tokens
        _trace("pages", "relanex", "2k", 4, 700, 1500, 8),
        # a batch job that only scores prompts: full steps of ragged requests
        _trace("scoring", "nevodra", "4k", 5, 600, 1900, 0),
        # one stream behind a short question
        _trace("stream", "nevodra", "2k", 1, 50, 50, 64),
        # four streams that go on for a while
        _trace("streams", "dopirax", "2k", 4, 200, 700, 48),
        # a small server's ordinary load: prompts of a page, sixteen rows a step
        _trace("server", "falisun", "2k", 16, 100, 1100, 32),
    ]


def draw(rng: random.Random) -> dict:
    """A case of the same ranges that costs no more than the largest listed one."""
    def log(lo: int, hi: int) -> int:
        return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))
    while True:
        if rng.random() < 1 / 6:                          # 32-bit: what logits are compared on, short prompts
            dtype, model, size = "float32", rng.choice(("qwen3", "sopepel", "relanex", "tolurax")), "2k"
        else:
            dtype, model = "bfloat16", rng.choice(("qwen3", "qwen3", "qwen3", "tolurax", "relanex", *ROUTED))
            size = rng.choice(("2k", "4k", "8b") if model == "qwen3" else ("2k", "2k", "4k"))
        requests, longest = log(1, 16), log(32, 800 if dtype == "float32" else 6000)
        decode = rng.choice((0, log(1, 64), log(1, 64)))
        if dtype == "bfloat16" and model in ROUTED:       # (enough rows that one near tie of a router does not rule)
            decode = max(decode, -(-48 // requests))
        in_turn = requests > 1 and decode > 0 and rng.random() < 0.25
        case = _trace(None, model, size, requests, rng.randint(max(1, longest // 3), longest), longest, decode, dtype=dtype,
                      arrive="in turn" if in_turn else "together", portion=512 if in_turn else PORTION)
        if _weight(case) <= max(_weight(c) for c in listed()) and sum(_prompt_lens(case)) <= 10000:
            return case


def _weight(case: dict) -> float:
    w = work(case)
    return w["bytes"] / 4e12 + w["flops"] / (4e13 if case["dtype"] == "float32" else 6e14)


# -- a case's configuration and trace --------------------------------------------------------------------------------
def _config(case: dict) -> dict:
    if case["size"] == "8b":
        return dict(benchmark.QWEN3_8B, num_hidden_layers=LAYERS["qwen3", "8b"])
    z = dict(benchmark.DESIGN_SIZES[case["size"]])
    z["layers"] = LAYERS.get((case["model"], case["size"]), z["layers"])
    return benchmark.qwen3_config(z) if case["model"] == "qwen3" else benchmark.DESIGN_CONFIGS[case["model"]](z)


def _vocab(case: dict) -> int:
    cfg = _config(case)
    return cfg["vocab_size"] if case["model"] == "qwen3" else cfg["vocab"]


def _prompt_lens(case: dict) -> list[int]:
    """Lengths between the case's two, in no particular order, from the case alone (a seed changes the tokens, not the
    work)."""
    n, lo, hi = case["requests"], case["shortest"], case["longest"]
    if n == 1:
        return [hi]
    lens = [lo + round((hi - lo) * i / (n - 1)) for i in range(n)]
    random.Random(n * 7919 + lo).shuffle(lens)
    return lens


def _steps(case: dict) -> list[list[tuple[int, int, int, bool]]]:
    """The trace: per step its rows as (request, first token, tokens, whether the last one's logits are asked for)."""
    lens, more, portion = _prompt_lens(case), case["decode"], case["portion"]
    at, steps = [0] * len(lens), []
    while any(a < n + more for a, n in zip(at, lens)):
        rows, budget = [], portion
        prompts = [r for r, n in enumerate(lens) if at[r] < n]
        decoding = [r for r, n in enumerate(lens) if n <= at[r] < n + more]
        if case["arrive"] == "in turn" or not prompts:
            rows += [(r, at[r], 1, True) for r in decoding]
        for r in prompts:
            take = min(lens[r] - at[r], budget)
            if take:
                rows.append((r, at[r], take, at[r] + take == lens[r]))
            budget -= take
            if case["arrive"] == "in turn":
                break                                     # the next request comes in the next step
        for r, start, n, _ in rows:
            at[r] = start + n
        steps.append(rows)
    return steps


def _tokens(case: dict, seed: int) -> list[list[int]]:
    rng = np.random.default_rng(seed)
    return [rng.integers(0, _vocab(case), n + case["decode"]).tolist() for n in _prompt_lens(case)]


# -- what a user's program has, and one pass -------------------------------------------------------------------------
def prepare(case: dict, seed: int):
    lens, steps = _prompt_lens(case), _steps(case)
    page = 16
    loaded = load_model("random", device="cuda", dtype=case["dtype"], page_size=page, max_seqs=len(lens),
                        max_model_len=max(lens) + case["decode"] + page, max_step_tokens=case["portion"] + len(lens),
                        cache_tokens=sum(-(-(n + case["decode"]) // page) * page for n in lens) + page, graphs=True,
                        random_config=_config(case), seed=seed)
    tokens = _tokens(case, seed)
    trace = [[{"id": r, "tokens": tokens[r][start: start + n], "want": [n - 1] if want else []}
              for r, start, n, want in rows] for rows in steps]
    wanted = sum(want for rows in steps for *_, want in rows)
    logits = torch.empty((wanted, _vocab(case)), dtype=torch.float32, device="cuda")
    return {"replayer": Replayer(loaded), "trace": trace, "logits": logits, "requests": list(range(len(lens)))}


def run(state) -> torch.Tensor:
    """Plays the trace -> the logits asked for, in the trace's order. (A step's logits are kept, as a caller that reads
    them later has to: a replayed step leaves them in a buffer of its own.)"""
    replayer, logits, at = state["replayer"], state["logits"], 0
    last = len(state["trace"]) - 1
    for i, entries in enumerate(state["trace"]):
        out = replayer.step(entries, state["requests"] if i == last else ())
        if out is not None:
            logits[at: at + out.shape[0]].copy_(out)
            at += out.shape[0]
    return logits


# -- what a pass cannot do without -----------------------------------------------------------------------------------
def _layers(case: dict) -> list[dict]:
    """Per layer: `always` and `expert` weights (values), experts and how many a token takes, attention as (heads, score
    and value sizes, values a cached token holds, the keys a query sees at most or None; None: no attention) and the
    values of recurrent state a request keeps."""
    cfg, out = _config(case), []
    if case["model"] == "qwen3":
        w, h, g, d, f = (cfg[k] for k in ("hidden_size", "num_attention_heads", "num_key_value_heads", "head_dim",
                                          "intermediate_size"))
        layer = {"always": w * (h + 2 * g) * d + h * d * w + 3 * w * f, "expert": 0, "experts": 0, "top": 0,
                 "attn": (h, d, d, 2 * g * d, None), "state": 0}
        return [layer] * cfg["num_hidden_layers"]
    w = cfg["width"]

    def softmax(m: dict) -> tuple[int, tuple]:
        h, g, d, v = m["heads"], m.get("kv_heads") or m["heads"], m["dim"], m["vdim"]
        seen = (m.get("mask") or {}).get("size")
        return w * (h * d + g * (d + v)) + h * v * w, (h, d, v, g * (d + v), seen)
    for layer in cfg["layers"]:
        m, kind, state, attn = layer["mixer"], layer["type"], 0, None
        if kind == "attention":
            always, attn = softmax(m)
            if case["model"] == "dopirax":                # values are the keys: no projection of their own
                always -= w * m["kv_heads"] * m["vdim"]
        elif kind == "attention_2":
            h, g, d, v, own = m["heads"], m["kv_heads"], m["dim"], m["vdim"], m.get("kv_from") is None
            always = w * 2 * h * d + h * v * w + (w * g * (2 * d + v) if own else 0)
            attn = (2 * h, d, v, g * (2 * d + v), None)
        elif kind == "latent_attention":
            h, d, v, rot, rank = m["heads"], m["dim"], m["vdim"], m.get("rot_dim", 0), m["kv_rank"]
            q = w * m["q_rank"] + m["q_rank"] * h * d if m.get("q_rank") else w * h * (d + rot)
            always = q + (w * (rank + rot) if m.get("kv_from") is None else 0) + rank * h * (d + v) + h * v * w
            always += w * h * v if case["model"] == "falisun" else 0
            attn = (h, d + rot, v, rank + rot, (m.get("mask") or {}).get("size"))
        elif kind == "mamba2":
            inner = m["heads"] * m["vdim"]
            always = w * (2 * inner + 2 * m["groups"] * m["state"] + m["heads"]) + inner * w
            state = m["heads"] * m["vdim"] * m["state"]
        elif kind in ("mlstm", "delta"):
            always, state = 5 * w * m["heads"] * m["dim"], m["heads"] * m["dim"] * m["vdim"]
        else:                                             # two mixers side by side
            always, attn = softmax(m["left"])
            r = m["right"]
            v = r.get("vdim", r["dim"])
            always += w * r["heads"] * (2 * r["dim"] + 3 * v) + (w * m["left"]["heads"] * m["left"]["vdim"]
                                                                  if case["model"] == "tolurax" else 0)
            state = r["heads"] * r["dim"] * v
        mlp = layer["mlp"]
        gated = 2 if case["model"] in ("dopirax", "nevodra") and mlp["kind"] == "dense" else \
            2 if case["model"] == "sopepel" and mlp["kind"] == "moe" else 3
        if mlp["kind"] == "dense":
            out.append({"always": always + gated * w * mlp["ff"], "expert": 0, "experts": 0, "top": 0, "attn": attn,
                        "state": state})
        else:
            router = mlp["router"]
            out.append({"always": always + gated * w * mlp["shared"]["ff"], "expert": gated * w * mlp["expert"]["ff"],
                        "experts": router["experts"], "top": router["top"], "attn": attn, "state": state})
    return out


def work(case: dict) -> dict:
    """Every step reads the weights that its tokens need once (an expert's as long as a token can have chosen it), the
    cached tokens and the state of its rows, and writes what it adds; products of all tokens, causal attention."""
    item = 4 if case["dtype"] == "float32" else 2
    layers, vocab = _layers(case), _vocab(case)
    width = _config(case)["hidden_size" if case["model"] == "qwen3" else "width"]
    total_bytes = flops = 0.0
    for rows in _steps(case):
        tokens, wanted = sum(n for _, _, n, _ in rows), sum(want for *_, want in rows)
        if wanted:
            total_bytes += vocab * width * item + wanted * vocab * 4
            flops += 2.0 * wanted * vocab * width
        for la in layers:
            total_bytes += (la["always"] + la["expert"] * min(la["experts"], tokens * la["top"])) * item
            total_bytes += 8.0 * la["state"] * len(rows)
            flops += 2.0 * tokens * (la["always"] + la["expert"] * la["top"]) + 4.0 * tokens * la["state"]
            if la["attn"]:
                heads, d, v, kept, seen = la["attn"]
                for _, start, n, _ in rows:
                    keys = min(start + n, seen + n) if seen else start + n
                    total_bytes += keys * kept * item
                    pairs = n * (min(start, seen) if seen else start) + n * min(n, seen or n) / 2
                    flops += 2.0 * heads * (d + v) * pairs
    return {"bytes": total_bytes, "flops": flops}


def tolerance(case: dict) -> dict:
    """Measured: bfloat16 against 64 bits 0.0025 over Relanex (its norms keep every sublayer small), 0.006 to 0.02 over
    the others, a token whose expert a rounding changed up to 0.2 in its own row; float32 1e-6 to 9e-6, Sopepel 1e-5 to
    5e-4 (a norm over a result near nothing)."""
    if case["dtype"] == "float32":
        return {"rel": 2e-3, "max": 0.07} if case["model"] == "sopepel" else {"rel": 4e-5, "max": 4e-4}
    return {"rel": 0.01, "max": 0.08} if case["model"] == "relanex" else {"rel": 0.03, "max": 0.99}


# -- the same in 64 bits, as plain torch gives it --------------------------------------------------------------------
class _Weights:
    """The random weights of a seed by checkpoint name: each from a generator seeded by (seed, name), rounded to
    bfloat16. Laws: `linear` N(0, 0.02), `norm` 1 + N(0, 0.1), `tap` N(0, 0.3), `zero` N(0, 0.5), `unit` [0, 1)."""

    STD = {"linear": 0.02, "tap": 0.3, "zero": 0.5}

    def __init__(self, seed: int) -> None:
        self.seed = seed

    def __call__(self, name: str, *shape: int, law: str = "linear") -> torch.Tensor:
        digest = hashlib.sha256(f"{self.seed}:{name}".encode()).digest()[:8]
        g = torch.Generator(device="cuda").manual_seed(int.from_bytes(digest, "little") & (2 ** 63 - 1))
        if law == "unit":
            x = torch.rand(shape, generator=g, device="cuda", dtype=torch.float32)
        else:
            x = torch.randn(shape, generator=g, device="cuda", dtype=torch.float32)
            x = 1 + 0.1 * x if law == "norm" else self.STD[law] * x
        return x.bfloat16().double()


def _unit(x, eps):
    return x / torch.sqrt(x.square().mean(-1, keepdim=True) + eps)


def _silu(z):
    return z * torch.sigmoid(z)


def _filter(x, taps):
    """x [B, T, C], taps [C, n] (the last one weighs the current token); zeros before the start."""
    n = taps.shape[1]
    padded = torch.cat((x.new_zeros(x.shape[0], n - 1, x.shape[2]), x), dim=1)
    return sum(taps[:, j] * padded[:, j: j + x.shape[1]] for j in range(n))


def _turn(x, rot, neighbours: bool):
    """x [B, T, heads, D]: the first rot.dims dimensions turned, in pairs (i, i + dims / 2) or (2i, 2i + 1)."""
    dims, base, s = rot["dims"], float(rot["base"]), rot.get("scaling")
    i = torch.arange(dims // 2, dtype=torch.float64, device=x.device)
    f, gain = base ** (-2 * i / dims), 1.0
    if s and "low" in s:                                  # by wavelength bands
        wave = 2 * math.pi / f
        mix = ((s["original"] / wave - s["low"]) / (s["high"] - s["low"])).clamp(0, 1)
        f = (1 - mix) * f / s["factor"] + mix * f
    elif s:                                               # YaRN
        def index(turns):
            return dims * math.log(s["original"] / (2 * math.pi * turns)) / (2 * math.log(base))
        lo, hi = max(math.floor(index(s["fast"])), 0), min(math.ceil(index(s["slow"])), dims - 1)
        ramp = ((i - lo) / max(hi - lo, 0.001)).clamp(0, 1)
        f, gain = f / s["factor"] * ramp + f * (1 - ramp), 0.1 * math.log(s["factor"]) + 1
    angle = (torch.arange(x.shape[1], dtype=torch.float64, device=x.device)[:, None] * f)[:, None, :]
    cos, sin = angle.cos() * gain, angle.sin() * gain
    out = x.clone()
    a, b = (slice(0, dims, 2), slice(1, dims, 2)) if neighbours else (slice(0, dims // 2), slice(dims // 2, dims))
    out[..., a] = x[..., a] * cos - x[..., b] * sin
    out[..., b] = x[..., b] * cos + x[..., a] * sin
    return out


def _attend(q, k, v, scale, *, size=None, keep_first=0, chunk=None, cap=None, far=None, sink=None, weigh=None):
    """q [B, T, H, D], k [B, T, G, D], v [B, T, G, V] -> [B, T, H, V]. A query sees the keys up to its own: the last
    `size` and the first `keep_first`, or its own chunk's; `cap` squashes scores, `far` (r1, r2 [H]) takes off
    r1 ln(1 + r2 distance), `sink` [H] is one more term of the denominator, `weigh` replaces the softmax by a weight a
    score."""
    B, T, H, _ = q.shape
    G = k.shape[2]
    out = q.new_empty(B, T, H, v.shape[3])
    for b in range(B):
        kb, vb = k[b].permute(1, 2, 0).contiguous(), v[b].transpose(0, 1).contiguous()      # [G, D, T], [G, T, V]
        for lo in range(0, T, 512):
            i = torch.arange(lo, min(lo + 512, T), device=q.device)[:, None]
            j = torch.arange(T, device=q.device)[None, :]
            seen = j <= i
            if size:
                seen = seen & ((i - j < size) | (j < keep_first))
            if chunk:
                seen = seen & (i // chunk == j // chunk)
            for g in range(G):
                hs = slice(g * (H // G), (g + 1) * (H // G))
                qg = q[b, lo: lo + 512, hs].transpose(0, 1).contiguous()                    # [H / G, rows, D]
                s = torch.matmul(qg, kb[g]) * scale
                if cap:
                    s = cap * torch.tanh(s / cap)
                if far is not None:
                    s = s - far[0][hs, None, None] * torch.log1p(far[1][hs, None, None] * (i - j).clamp(min=0))
                if weigh is not None:
                    p = weigh(s, hs).masked_fill(~seen, 0.0)
                else:
                    s = s.masked_fill(~seen, -math.inf)
                    if sink is not None:
                        s = torch.cat((s, sink[hs, None, None].expand(-1, s.shape[1], 1)), dim=-1)
                    p = torch.softmax(s, dim=-1)[..., :T]
                out[b, lo: lo + 512, hs] = torch.matmul(p, vb[g]).transpose(0, 1)
    return out


def _scan(T, step):
    """Stacks what `step(t)` gives for every t along dimension 1."""
    return torch.stack([step(t) for t in range(T)], dim=1)


def _experts(w, p, mlp, x, choose, gated, act):
    """Sum over a token's experts of weight * down(act(...)), token sets gathered by expert; x [B, T, W].
    `choose(flat x)` -> (indices [n, top], weights [n, top] of the outputs)."""
    W, flat = x.shape[-1], x.reshape(-1, x.shape[-1])
    which, weight = choose(flat)
    out = torch.zeros_like(flat)

    def one(name, ff, rows):
        up = rows @ w(name + "up", ff, W).T
        return act(rows @ w(name + "gate", ff, W).T if gated else None, up) @ w(name + "down", W, ff).T
    for e in range(mlp["router"]["experts"]):
        rows, place = torch.nonzero(which == e, as_tuple=True)
        if len(rows):
            out.index_add_(0, rows, one(f"{p}e{e}.", mlp["expert"]["ff"], flat[rows]) * weight[rows, place][:, None])
    shared = one(p + "shared.", mlp["shared"]["ff"], flat)
    if "sg" in mlp:
        shared = shared * torch.sigmoid(flat @ mlp["sg"].T)
    return (out + shared).view(x.shape)


def _gated(g, u):
    return _silu(g) * u


def _top(z, top, groups=None, rank=None):
    """Indices of the `top` largest z [n, E], only among the `keep` groups of neighbours that `rank` puts first."""
    if groups:
        best = rank(z.view(z.shape[0], groups["count"], -1)).topk(groups["keep"], dim=-1).indices
        open_ = torch.zeros(z.shape[0], groups["count"], dtype=torch.bool, device=z.device).scatter_(1, best, True)
        z = z.masked_fill(~open_.repeat_interleave(z.shape[1] // groups["count"], dim=1), -math.inf)
    return z.topk(top, dim=-1).indices


def _heads(x, heads):
    return x.view(*x.shape[:2], heads, -1)


def _qwen3(w, c, x):
    W, H, G, D, F, eps = (c[k] for k in ("hidden_size", "num_attention_heads", "num_key_value_heads", "head_dim",
                                         "intermediate_size", "rms_norm_eps"))
    rot = {"dims": D, "base": c["rope_theta"]}
    for i in range(c["num_hidden_layers"]):
        p = f"model.layers.{i}."
        a, at = _unit(x, eps) * w(p + "input_layernorm.weight", W, law="norm"), p + "self_attn."
        q = _unit(_heads(a @ w(at + "q_proj.weight", H * D, W).T, H), eps) * w(at + "q_norm.weight", D, law="norm")
        k = _unit(_heads(a @ w(at + "k_proj.weight", G * D, W).T, G), eps) * w(at + "k_norm.weight", D, law="norm")
        v = _heads(a @ w(at + "v_proj.weight", G * D, W).T, G)
        o = _attend(_turn(q, rot, False), _turn(k, rot, False), v, D ** -0.5)
        x = x + o.flatten(2) @ w(at + "o_proj.weight", W, H * D).T
        a = _unit(x, eps) * w(p + "post_attention_layernorm.weight", W, law="norm")
        up = a @ w(p + "mlp.up_proj.weight", F, W).T
        x = x + _gated(a @ w(p + "mlp.gate_proj.weight", F, W).T, up) @ w(p + "mlp.down_proj.weight", W, F).T
    return lambda rows: _unit(rows, eps) * w("model.norm.weight", W, law="norm") @ w("lm_head.weight", c["vocab_size"], W).T, x


def _dense(w, p, W, F, x):
    return _gated(x @ w(p + "gate", F, W).T, x @ w(p + "up", F, W).T) @ w(p + "down", W, F).T


def _tolurax(w, c, x):
    W, eps, B, T = c["width"], c["norm"]["eps"], x.shape[0], x.shape[1]

    def layer_norm(v, name):
        v = v - v.mean(-1, keepdim=True)
        return v / torch.sqrt(v.square().mean(-1, keepdim=True) + eps) * w(name, W, law="norm")

    def left(h, p, m):
        H, G, D = m["heads"], m["kv_heads"], m["dim"]
        q = _unit(_heads(h @ w(p + "q", H * D, W).T, H), eps) * w(p + "q.norm", D, law="norm")
        k = _unit(_heads(h @ w(p + "k", G * D, W).T, G), eps) * w(p + "k.norm", D, law="norm")
        v = _heads(h @ w(p + "v", G * D, W).T, G)
        bias = w(p + "pb", H, law="zero")
        o = _attend(_turn(q, m["rot"], False), _turn(k, m["rot"], False), v, m["scale"], size=m["mask"]["size"],
                    weigh=lambda s, hs: torch.sigmoid(s + bias[hs, None, None]))
        return (o.flatten(2) * torch.sigmoid(h @ w(p + "g", H * D, W).T)) @ w(p + "o", W, H * D).T

    def right(h, p, m):
        H, D, R = m["heads"], m["dim"], m["rank"]
        prev = torch.cat((torch.zeros_like(h[:, :1]), h[:, :-1]), dim=1)
        mixed = {n: h + (prev - h) * w(p + "mu." + n, W, law="unit") for n in "rkvgw"}
        r, k, v = (_heads(mixed[n] @ w(p + n, H * D, W).T, H) for n in "rkv")
        gate = _silu(mixed["g"] @ w(p + "g", H * D, W).T)
        lora = torch.tanh(mixed["w"] @ w(p + "w1", R, W).T) @ w(p + "w2", H * D, R, law="tap").T
        decay = _heads(torch.exp(-torch.exp(lora + w(p + "w0", H * D, law="zero"))), H)
        u, S = w(p + "u", H, D, law="zero")[:, :, None], h.new_zeros(B, H, D, D)

        def step(t):
            nonlocal S
            kv = k[:, t, :, :, None] * v[:, t, :, None, :]
            o = ((S + u * kv) * r[:, t, :, :, None]).sum(2)
            S = decay[:, t, :, :, None] * S + kv
            return o
        o = _unit(_scan(T, step), eps).flatten(2) * w(p + "norm", H * D, law="norm") * gate
        return o @ w(p + "o", W, H * D).T

    def delta(h, p, m):
        H, G, D, V = m["heads"], m["kv_heads"], m["dim"], m["vdim"]
        q, k, v = (_heads(_silu(_filter(h @ w(p + n, g * d, W).T, w(p + n + ".conv", g * d, m["conv"], law="tap"))), g)
                   for n, g, d in (("q", G, D), ("k", G, D), ("v", H, V)))
        q = q / torch.sqrt(q.square().sum(-1, keepdim=True) + 1e-6) * D ** -0.5
        k = k / torch.sqrt(k.square().sum(-1, keepdim=True) + 1e-6)
        q, k = q.repeat_interleave(H // G, dim=2), k.repeat_interleave(H // G, dim=2)
        beta = torch.sigmoid(h @ w(p + "b", H, W).T)
        g = torch.exp(-torch.exp(w(p + "A_log", H, law="zero"))
                      * torch.nn.functional.softplus(h @ w(p + "a", H, W).T + w(p + "dt_bias", H, law="zero")))
        S = h.new_zeros(B, H, D, V)

        def step(t):
            nonlocal S
            S = g[:, t, :, None, None] * S
            kt = k[:, t, :, :, None]
            S = S + kt * (beta[:, t, :, None] * (v[:, t] - (S * kt).sum(2)))[:, :, None, :]
            return (S * q[:, t, :, :, None]).sum(2)
        o = _unit(_scan(T, step), eps) * w(p + "norm", V, law="norm")
        return (o.flatten(2) * _silu(h @ w(p + "g", H * V, W).T)) @ w(p + "o", W, H * V).T
    for i, layer in enumerate(c["layers"]):
        p, m = f"l{i}.", layer["mixer"]
        h = layer_norm(x, p + "norm1")
        h = h + _filter(h, w(p + "canon1", W, c["canon"]["taps"], law="tap"))
        if layer["type"] == "delta":
            x = x + delta(h, p + "mix.", m)
        else:
            x = x + m["left_scale"] * left(h, p + "mix.left.", m["left"]) + m["right_scale"] * right(h, p + "mix.right.", m["right"])
        x = x + _dense(w, p + "mlp.", W, layer["mlp"]["ff"], layer_norm(x, p + "norm2"))
    cap = c["logit_softcap"]
    return lambda rows: cap * torch.tanh(layer_norm(rows, "final.norm") @ w("head", c["vocab"], W).T / cap), x


def _relanex(w, c, x):
    W, eps, mult, B, T = c["width"], c["norm"]["eps"], c["residual_mult"], x.shape[0], x.shape[1]

    def dyt(v, name):
        return torch.tanh(w(name + ".alpha", law="unit") * v) * w(name, W, law="norm") + w(name + ".b", W, law="zero")

    def attention(h, p, m):
        H, G, D = m["heads"], m["kv_heads"], m["dim"]
        q, k, v = (_heads(h @ w(p + n, g * D, W).T + w(p + n + ".b", g * D, law="zero"), g)
                   for n, g in (("q", H), ("k", G), ("v", G)))
        o = _attend(_turn(q, m["rot"], True), _turn(k, m["rot"], True), v, m["scale"], sink=w(p + "sink", H, law="zero"))
        return o.flatten(2) @ w(p + "o", W, H * D).T

    def latent(h, p, m):
        H, D, R, Q = m["heads"], m["dim"], m["kv_rank"], m["q_rank"]
        cq = _unit(h @ w(p + "dq", Q, W).T, eps) * w(p + "dq.norm", Q, law="norm")
        ckv = _unit(h @ w(p + "dkv", R, W).T, eps) * w(p + "dkv.norm", R, law="norm")
        q, k, v = (_heads(a @ w(p + n, H * D, r).T, H) for a, n, r in ((cq, "uq", Q), (ckv, "uk", R), (ckv, "uv", R)))
        return _attend(q, k, v, m["scale"], size=m["mask"]["size"]).flatten(2) @ w(p + "o", W, H * D).T

    def mlstm(h, p, m):
        H, D, cap = m["heads"], m["dim"], m["gate_cap"]
        q, k, v = (_heads(h @ w(p + n, H * D, W).T, H) for n in "qkv")
        q = q * D ** -0.5
        gi, gf = (cap * torch.tanh((h @ w(p + n, H, W).T + w(p + n + ".b", H, law="zero")) / cap) for n in "if")
        gf = torch.nn.functional.logsigmoid(gf)
        S, n, top = h.new_zeros(B, H, D, D), h.new_zeros(B, H, D), h.new_zeros(B, H)

        def step(t):
            nonlocal S, n, top
            new = torch.maximum(gf[:, t] + top, gi[:, t])
            keep, take = torch.exp(gf[:, t] + top - new)[..., None], torch.exp(gi[:, t] - new)[..., None]
            S = keep[..., None] * S + (take * k[:, t])[..., None] * v[:, t, :, None, :]
            n, top = keep * n + take * k[:, t], new
            den = torch.maximum((n * q[:, t]).sum(-1).abs(), torch.exp(-top)) + 1e-6
            return (S * q[:, t, :, :, None]).sum(2) / den[..., None]
        y = _unit(_scan(T, step), eps).flatten(2) * w(p + "norm", H * D, law="norm")
        return (y * torch.sigmoid(h @ w(p + "g", H * D, W).T)) @ w(p + "o", W, H * D).T
    kinds = {"attention": attention, "latent_attention": latent, "mlstm": mlstm}
    x = dyt(x, "embed.norm")
    for i, layer in enumerate(c["layers"]):
        p = f"l{i}."
        x = x + mult * dyt(kinds[layer["type"]](dyt(x, p + "norm1"), p + "mix.", layer["mixer"]), p + "norm1b")
        x = x + mult * dyt(_dense(w, p + "mlp.", W, layer["mlp"]["ff"], dyt(x, p + "norm2")), p + "norm2b")
    return lambda rows: dyt(rows, "final.norm") @ w("head", c["vocab"], W).T, x


def _latent_shared(w, p, m, W, h, c, r, turn):
    """Latent attention's queries, keys (with the turned part all heads share) and values."""
    H, D, V, R, rot = m["heads"], m["dim"], m["vdim"], m["kv_rank"], m["rot_dim"]
    q = _heads(h @ w(p + "q", H * (D + rot), W).T, H)
    q = torch.cat((q[..., :D], turn(q[..., D:])), dim=-1)
    k = torch.cat((_heads(c @ w(p + "uk", H * D, R).T, H), r.expand(-1, -1, H, -1)), dim=-1)
    return q, k, _heads(c @ w(p + "uv", H * V, R).T, H)


def _nevodra(w, c, x):
    W, eps, taps = c["width"], c["norm"]["eps"], c["canon"]["taps"]

    def attention(h, p, m):
        H, G, D = m["heads"], m["kv_heads"], m["dim"]
        q = _heads(_unit(h @ w(p + "q", H * D, W).T, eps) * w(p + "q.norm", H * D, law="norm"), H)
        k = _heads(_unit(h @ w(p + "k", G * D, W).T, eps) * w(p + "k.norm", G * D, law="norm"), G)
        v = _heads(h @ w(p + "v", G * D, W).T, G)
        o = _attend(q, k, v, m["scale"], size=m["mask"]["size"], keep_first=m["mask"]["keep_first"], cap=m["softcap"],
                    far=(w(p + "r1", H, law="unit"), w(p + "r2", H, law="unit")))
        return o.flatten(2) @ w(p + "o", W, H * D).T

    def latent(h, p, m):
        R, rot = m["kv_rank"], m["rot_dim"]
        down = h @ w(p + "dkv", R + rot, W).T
        ckv = _unit(down[..., :R], eps) * w(p + "dkv.norm", R, law="norm")
        q, k, v = _latent_shared(w, p, m, W, h, ckv, _turn(down[:, :, None, R:], m["rot"], True),
                                 lambda u: _turn(u, m["rot"], True))
        o = _attend(q, k, v, m["scale"], sink=w(p + "sink", m["heads"], law="zero"))
        return o.flatten(2) @ w(p + "o", W, m["heads"] * m["vdim"]).T

    def polynorm(h, p, ff):
        z, (a, b, d, e) = h @ w(p + "up", ff, W).T, w(p + "act", 4, law="unit")
        return (a * _unit(z, eps) + b * _unit(z ** 2, eps) + d * _unit(z ** 3, eps) + e) @ w(p + "down", W, ff).T

    def moe(h, p, mlp):
        router = mlp["router"]
        E = router["experts"]

        def choose(rows):
            s = torch.sigmoid(rows @ w(p + "router", E, W).T)
            at = _top(s + w(p + "correction", E, law="zero"), router["top"], router["groups"],
                      lambda z: z.topk(min(2, z.shape[-1]), dim=-1).values.sum(-1))
            return at, s.gather(1, at) * router["scale"]
        return _experts(w, p, mlp, h, choose, True, _gated)
    x = x * c["embedding"]["scale"]
    for i, layer in enumerate(c["layers"]):
        p, mlp = f"l{i}.", layer["mlp"]
        a = _unit(x, eps) * w(p + "norm1", W, law="norm")
        b = _unit(x, eps) * w(p + "norm2", W, law="norm")
        a = a + _filter(a, w(p + "canon1", W, taps, law="tap"))
        b = b + _filter(b, w(p + "canon2", W, taps, law="tap"))
        y = (attention if layer["type"] == "attention" else latent)(a, p + "mix.", layer["mixer"])
        x = x + y + (polynorm(b, p + "mlp.", mlp["ff"]) if mlp["kind"] == "dense" else moe(b, p + "mlp.", mlp))
    return lambda rows: _unit(rows, eps) * w("final.norm", W, law="norm") @ w("head", c["vocab"], W).T, x


def _dopirax(w, c, x):
    W, eps, kept = c["width"], c["norm"]["eps"], {}

    def attention(h, p, m, i):
        H, G, D = m["heads"], m["kv_heads"], m["dim"]
        q = _heads(h @ w(p + "q", H * D, W).T + w(p + "q.b", H * D, law="zero"), H)
        k = _heads(h @ w(p + "k", G * D, W).T + w(p + "k.b", G * D, law="zero"), G)
        o = _attend(_turn(q, m["rot"], False), _turn(k, m["rot"], False), k, m["scale"], cap=m["softcap"],
                    sink=h.new_zeros(H))
        o = o * torch.sigmoid(h @ w(p + "g", H, W).T)[..., None]
        return o.flatten(2) @ w(p + "o", W, H * D).T + w(p + "o.b", W, law="zero")

    def attention_2(h, p, m, i):
        H, G, D, V, diff = m["heads"], m["kv_heads"], m["dim"], m["vdim"], m["diff"]
        if m.get("kv_from") is None:
            k = _unit(_heads(h @ w(p + "k", G * 2 * D, W).T, 2 * G), eps) * w(p + "k.norm", D, law="norm")
            kept[i] = _turn(k, m["rot"], True), _heads(h @ w(p + "v", G * V, W).T, G)
        k, v = kept[i if m.get("kv_from") is None else m["kv_from"]]
        q = _unit(_heads(h @ w(p + "q", H * 2 * D, W).T, 2 * H), eps) * w(p + "q.norm", D, law="norm")
        q = _turn(q, m["rot"], True)
        l1, l2, r1, r2 = (w(p + n, D, law="tap") for n in ("lq1", "lq2", "lk1", "lk2"))
        lam = torch.exp((l1 * r1).sum()) - torch.exp((l2 * r2).sum()) + diff
        one, two = (_attend(q[:, :, s::2], k[:, :, s::2], v, m["scale"]) for s in (0, 1))
        return (_unit(one - lam * two, eps) * (1 - diff)).flatten(2) @ w(p + "o", W, H * V).T

    def moe(h, p, mlp):
        E = mlp["router"]["experts"]

        def choose(rows):
            z = rows @ w(p + "router", E, W).T + w(p + "router.b", E, law="zero")
            at = _top(z, mlp["router"]["top"])
            return at, torch.softmax(z.gather(1, at), dim=-1)
        return _experts(w, p, dict(mlp, sg=w(p + "shared.sg", 1, W)), h, choose, True, _gated)
    x = x * c["embedding"]["scale"]
    for i, layer in enumerate(c["layers"]):
        p, mlp = f"l{i}.", layer["mlp"]
        a = _unit(x, eps) * (1 + w(p + "norm1", W, law="tap"))
        y = (attention if layer["type"] == "attention" else attention_2)(a, p + "mix.", layer["mixer"], i)
        if mlp["kind"] == "dense":
            ff = mlp["ff"]
            y = y + torch.relu(a @ w(p + "mlp.up", ff, W).T).square() @ w(p + "mlp.down", W, ff).T
        else:
            y = y + moe(a, p + "mlp.", mlp)
        x = x + y
    return lambda rows: _unit(rows, eps) * (1 + w("final.norm", W, law="tap")) @ w("head", c["vocab"], W).T, x


def _falisun(w, c, x):
    W, eps, kept, B, T = c["width"], c["norm"]["eps"], {}, x.shape[0], x.shape[1]

    def latent(h, p, m, i):
        R, rot, H, V = m["kv_rank"], m["rot_dim"], m["heads"], m["vdim"]
        if m.get("kv_from") is None:
            down = h @ w(p + "dkv", R + rot, W).T
            kept[i] = (_unit(down[..., :R], eps) * w(p + "dkv.norm", R, law="norm"),
                       _turn(down[:, :, None, R:], m["rot"], False))
        ckv, r = kept[i if m.get("kv_from") is None else m["kv_from"]]
        o = _attend(*_latent_shared(w, p, m, W, h, ckv, r, lambda u: _turn(u, m["rot"], False)), m["scale"])
        return (o.flatten(2) * torch.sigmoid(h @ w(p + "g", H * V, W).T)) @ w(p + "o", W, H * V).T

    def mamba2(h, p, m, i):
        H, V, G, N = m["heads"], m["vdim"], m["groups"], m["state"]
        inner, gn = H * V, G * N
        z, u, b = torch.split(h @ w(p + "in", 2 * inner + 2 * gn + H, W).T, [inner, inner + 2 * gn, H], dim=-1)
        u = _silu(_filter(u, w(p + "conv", inner + 2 * gn, m["conv"], law="tap")) + w(p + "conv.b", inner + 2 * gn, law="zero"))
        v, Bm, Cm = torch.split(u, [inner, gn, gn], dim=-1)
        v, Bm, Cm = _heads(v, H), *(_heads(t, G).repeat_interleave(H // G, dim=2) for t in (Bm, Cm))
        dt = torch.nn.functional.softplus(b + w(p + "dt_bias", H, law="zero"))
        decay = torch.exp(-torch.exp(w(p + "A_log", H, law="zero")) * dt)
        S = h.new_zeros(B, H, N, V)

        def step(t):
            nonlocal S
            S = decay[:, t, :, None, None] * S + (dt[:, t, :, None] * Bm[:, t])[..., None] * v[:, t, :, None, :]
            return (S * Cm[:, t, :, :, None]).sum(2)
        y = _scan(T, step) + w(p + "D", H, law="norm")[:, None] * v
        y = (y.flatten(2) * _silu(z)).view(B, T, m["norm_groups"], -1)
        return (_unit(y, eps).flatten(2) * w(p + "norm", inner, law="norm")) @ w(p + "o", W, inner).T

    def moe(h, p, mlp):
        E, router = mlp["router"]["experts"], mlp["router"]

        def choose(rows):
            z = rows @ w(p + "router", E, W).T
            at = _top(z, router["top"], router["groups"], lambda g: g.amax(-1))
            return at, torch.softmax(z.gather(1, at), dim=-1)
        return _experts(w, p, mlp, h, choose, True, _gated)
    for i, layer in enumerate(c["layers"]):
        p = f"l{i}."
        y = (mamba2 if layer["type"] == "mamba2" else latent)(_unit(x, eps) * w(p + "norm1", W, law="norm"), p + "mix.",
                                                             layer["mixer"], i)
        x = x + _unit(y, eps) * w(p + "norm1b", W, law="norm") * w(p + "ls1", W, law="norm")
        y = moe(_unit(x, eps) * w(p + "norm2", W, law="norm"), p + "mlp.", layer["mlp"])
        x = x + _unit(y, eps) * w(p + "norm2b", W, law="norm") * w(p + "ls2", W, law="norm")
    return lambda rows: _unit(rows, eps) * w("final.norm", W, law="norm") @ w("embed", c["vocab"], W).T, x


def _sopepel(w, c, x):
    W, eps, B, T = c["width"], c["norm"]["eps"], x.shape[0], x.shape[1]

    def left(h, p, m):
        H, G, D = m["heads"], m["kv_heads"], m["dim"]
        q, k, v = (_heads(h @ w(p + n, g * D, W).T + w(p + n + ".b", g * D, law="zero"), g)
                   for n, g in (("q", H), ("k", G), ("v", G)))
        q, k = (_unit(a, eps) * w(p + n + ".norm", D, law="norm") for n, a in (("q", q), ("k", k)))
        o = _attend(_turn(q, m["rot"], False), _turn(k, m["rot"], False), v, m["scale"], chunk=m["mask"]["size"])
        o = o * torch.sigmoid(h @ w(p + "g", H, W).T)[..., None]
        return o.flatten(2) @ w(p + "o", W, H * D).T + w(p + "o.b", W, law="zero")

    def right(h, p, m):
        H, D, V, R = m["heads"], m["dim"], m["vdim"], m["rank"]
        q, k, v = (_heads(h @ w(p + n, H * d, W).T, H) for n, d in (("q", D), ("k", D), ("v", V)))
        q = q * D ** -0.5
        z = h @ w(p + "a1", R, W).T @ w(p + "a2", H * D, R, law="tap").T + w(p + "a2.b", H * D, law="zero")
        alpha, S = _heads(torch.exp(torch.nn.functional.logsigmoid(z) / m["tau"]), H), h.new_zeros(B, H, D, V)

        def step(t):
            nonlocal S
            S = alpha[:, t, :, :, None] * S + k[:, t, :, :, None] * v[:, t, :, None, :]
            return (S * q[:, t, :, :, None]).sum(2)
        o = _unit(_scan(T, step), eps) * w(p + "norm", V, law="norm")
        return (o.flatten(2) * _silu(h @ w(p + "g", H * V, W).T)) @ w(p + "o", W, H * V).T

    def moe(h, p, mlp):
        E = mlp["router"]["experts"]

        def choose(rows):
            s = torch.sigmoid(rows @ w(p + "router", E, W).T)
            at = _top(s, mlp["router"]["top"])
            return at, s.gather(1, at).square()           # relu(W_up s x)^2 = s^2 relu(W_up x)^2
        return _experts(w, p, dict(mlp, sg=w(p + "shared.sg", 1, W)), h, choose, False,
                        lambda _, u: torch.relu(u).square())
    for i, layer in enumerate(c["layers"]):
        p, m, mlp = f"l{i}.", layer["mixer"], layer["mlp"]
        y = m["left_scale"] * left(x, p + "mix.left.", m["left"]) + m["right_scale"] * right(x, p + "mix.right.", m["right"])
        x = x + _unit(y, eps) * w(p + "norm1", W, law="norm")
        if mlp["kind"] == "dense":
            ff = mlp["ff"]
            gate = torch.nn.functional.gelu(x @ w(p + "mlp.gate", ff, W).T, approximate="tanh")
            y = (gate * (x @ w(p + "mlp.up", ff, W).T)) @ w(p + "mlp.down", W, ff).T
        else:
            y = moe(x, p + "mlp.", mlp)
        x = x + _unit(y, eps) * w(p + "norm2", W, law="norm")
    scale = c["logit_scale"]
    return lambda rows: _unit(rows, eps) * w("final.norm", W, law="norm") @ w("embed", c["vocab"], W).T * scale, x


_PLAIN = {"qwen3": _qwen3, "tolurax": _tolurax, "relanex": _relanex, "nevodra": _nevodra, "dopirax": _dopirax,
          "falisun": _falisun, "sopepel": _sopepel}


@torch.no_grad()
def exact(case: dict, seed: int) -> torch.Tensor | None:
    """Every request's whole sequence at once, shorter ones padded behind their end, and the logits of the trace's wanted
    places in its order."""
    w, cfg, tokens = _Weights(seed), _config(case), _tokens(case, seed)
    longest = max(map(len, tokens))
    ids = torch.tensor([t + [0] * (longest - len(t)) for t in tokens], device="cuda")
    width = cfg["hidden_size" if case["model"] == "qwen3" else "width"]
    x = w("model.embed_tokens.weight" if case["model"] == "qwen3" else "embed", _vocab(case), width)[ids]
    if case["model"] == "sopepel":
        pair = cfg["embedding"]["bigram"]
        rows = (ids[:, :-1] * pair["mul_prev"] + ids[:, 1:] * pair["mul_cur"]) % pair["buckets"]
        rows = torch.cat((torch.full_like(ids[:, :1], pair["buckets"]), rows), dim=1)
        x = x + w("bigram", pair["buckets"] + 1, width)[rows]
    head, x = _PLAIN[case["model"]](w, cfg, x)
    places = [(r, start + n - 1) for step in _steps(case) for r, start, n, want in step if want]
    r, t = (torch.tensor(v, device="cuda") for v in zip(*places))
    return head(x[r, t])
