"""Tolurax through the engine against the plain model (`tests/plain/tolurax.py`, written from the design's equations,
no cache, float64): every mechanism alone, every way of cutting a prompt, batches, reused pages and slots, window and
page edges, far keys, long decoding, sizes that are 1 or equal, and greedy generation through the engine's own entry
point. On the CPU the plain twins of the operations stand in for the HIP kernels (this checks configuration, weights,
cache, state and batching); the `gpu` cases run the HIP kernels."""
from __future__ import annotations

import functools
import json
import subprocess
import sys

import numpy as np
import pytest
import torch

from tests import helpers as H
from tests import tolurax_models as M
from tests.plain.ops import TorchKernels

DEVICES = [pytest.param("cpu", id="cpu-twin"), pytest.param("cuda", marks=pytest.mark.gpu, id="hip")]
DTYPES = ["float32", "bfloat16"]
MODELS = {"X": (M.CONFIG_X, 11, False, 8), "Y": (M.CONFIG_Y, 12, False, 16), "Z": (M.CONFIG_Z, 13, False, 4),
          "X-sharp": (M.CONFIG_X, 14, True, 16), "Y-sharp": (M.CONFIG_Y, 15, True, 8),
          "delta": (M.ONLY_DELTA, 16, False, 8), "left": (M.ONLY_LEFT, 17, True, 8), "right": (M.ONLY_RIGHT, 18, False, 8),
          "filter-ffn": (M.ONLY_FILTER_FFN, 19, False, 8), "W-sharp": (M.CONFIG_W, 20, True, 16)}
LENGTHS = (40, 70, 33, 58, 50, 64, 21)
# bfloat16 engine against the float64 plain model, relative rms of the logits: what rounding alone gives on these
# models stays below a third of this; a lost key, state or filter input is far above it on the sharp models.
BF16_RMS = 0.06


@pytest.fixture(scope="module")
def folders(tmp_path_factory):
    root = tmp_path_factory.mktemp("tolurax")
    return {name: M.make_folder(root / name, cfg, seed, sharp) for name, (cfg, seed, sharp, _) in MODELS.items()}


@functools.lru_cache(maxsize=None)
def _plain(folder: str) -> M.PlainTolurax:
    return M.PlainTolurax(folder)


def _requests(name: str, lengths=LENGTHS) -> dict[str, list[int]]:
    return {f"r{i}": H.random_ids(n, MODELS[name][0]["vocab"], 300 + i) for i, n in enumerate(lengths)}


def _replayer(folder, device, dtype, page, cache_tokens, max_seqs=4, max_model_len=256):
    from holon_amd.engine.loading import load_model
    from holon_amd.engine.replay import Replayer
    loaded = load_model(folder, device=device, dtype=dtype, kernels=TorchKernels() if device == "cpu" else None,
                        page_size=page, max_seqs=max_seqs, max_model_len=max_model_len, max_step_tokens=max_model_len,
                        cache_tokens=cache_tokens)
    return Replayer(loaded)


def _check(folder, dtype, requests, got, what):
    want = {r: _plain(str(folder)).logits(ids) for r, ids in requests.items()}
    g, w = H.gather(want, got)
    assert torch.isfinite(g).all(), f"{what}: non-finite logits"
    if dtype == "float32":
        r, m = H.rel_rms(g, w), H.max_over_rms(g, w)
        assert r <= 3e-5 and m <= 3e-4, f"{what}: float32 logits differ: rms {r:.3g}, max {m:.3g}"
    else:
        r = H.rel_rms(g, w)
        assert r <= BF16_RMS, f"{what}: bfloat16 logits differ: rms {r:.3g}"
        worst = ((g - w).square().mean(-1).sqrt() / w.square().mean().sqrt()).max().item()      # no single position far off
        assert worst <= 3 * BF16_RMS, f"{what}: one position differs by {worst:.3g}"


@pytest.mark.parametrize("device", DEVICES)
@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("name", list(MODELS))
def test_every_way_of_cutting(folders, name, dtype, device):
    """Whole prompts (the first tokens of a sequence among them), token-by-token decoding from the second token on and
    after a long prompt, portions of changing size down to two tokens; in a pool that holds only the longest request,
    so that every request uses the pages and the slot of the one before."""
    folder, requests = folders[name], _requests(name)
    page = MODELS[name][3]
    rep = _replayer(folder, device, dtype, page, cache_tokens=-(-max(LENGTHS) // page) * page)
    got = H.run_trace(rep, H.trace_whole({**requests, "one": requests["r0"][:1]}))
    assert len(got) == sum(LENGTHS) + 1
    _check(folder, dtype, {**requests, "one": requests["r0"][:1]}, got, f"{name} {dtype} whole")
    rep.cache.check()
    for rid, tail in (("r2", len(requests["r2"]) - 1), ("r1", 32)):       # everything after the first token; a tail
        got = H.run_trace(rep, H.trace_decode_tail(rid, requests[rid], tail))
        assert len(got) == len(requests[rid])
        _check(folder, dtype, requests, got, f"{name} {dtype} decode tail {rid}")
    for rid, sizes in (("r3", [7, 2, 13, 3, 2, 30, 5]), ("r1", [2, 2, 17, 16, 1 + page, 2]), ("r5", [1, 3, page, 2])):
        got = H.run_trace(rep, H.trace_chunks(rid, requests[rid], sizes))
        assert len(got) == len(requests[rid])
        _check(folder, dtype, requests, got, f"{name} {dtype} portions {rid}")
    rep.cache.check()
    assert all(g.pool.free == g.pool.usable for g in rep.cache.groups)


@pytest.mark.parametrize("device", DEVICES)
@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("name", ["X", "Y-sharp", "Z", "W-sharp"])
def test_mixed_batches_in_a_small_pool(folders, name, dtype, device):
    """Unequal requests side by side (portions beside single tokens, requests left out of steps) against each alone;
    three slots and a pool of the trace's peak, so that pages and slots are given back and used again."""
    folder, requests = folders[name], _requests(name)
    page = MODELS[name][3]
    for seed in (0, 1):
        trace = H.trace_mixed(requests, seed=seed, max_live=3, decode_tail=6 + 5 * seed, max_chunk=19)
        rep = _replayer(folder, device, dtype, page, cache_tokens=H.peak_live_tokens(trace, round_to=page), max_seqs=3)
        got = H.run_trace(rep, trace)
        assert len(got) == sum(LENGTHS)
        _check(folder, dtype, requests, got, f"{name} {dtype} mixed seed {seed}")
        rep.cache.check()
        assert all(g.pool.free == g.pool.usable for g in rep.cache.groups)


@pytest.mark.parametrize("device", DEVICES)
def test_float32_does_not_depend_on_the_cut(folders, device):
    """A position's float32 logits whole, in portions, decoded and in a mixed batch: the same to rounding of the
    sums' order (the kernels fix every order by the position alone: equal on the GPU bit for bit)."""
    folder, requests = folders["Y"], _requests("Y", (45, 38, 27))
    rep = _replayer(folder, device, "float32", 16, cache_tokens=256)
    whole = H.run_trace(rep, H.trace_whole(requests))
    cut = H.run_trace(rep, H.trace_chunks("r0", requests["r0"], [3, 2, 16, 5]))
    tail = H.run_trace(rep, H.trace_decode_tail("r1", requests["r1"], 20))
    mixed = H.run_trace(rep, H.trace_mixed(requests, seed=5, max_live=3, decode_tail=7))
    for other in (cut, tail, mixed):
        for key, row in other.items():
            if device == "cuda":
                assert torch.equal(row, whole[key]), f"{key}: logits depend on how the prompt was cut"
            else:
                assert H.rel_rms(row, whole[key]) < 1e-5


def _needle_model(root, window, page, dim=16):
    """One parallel layer whose attention alone reaches the stream (no rotation, no filter, memory scaled by 0). A
    pair of token ids (query token, key token) whose score is the largest of all, and a filler token whose scores
    with them and with itself are lowest; the head biases are then set so that the pair's weight is sigmoid(3) and
    every other weight in the test's prompts below sigmoid(-4). Returns the folder and the three ids."""
    cfg = {"architecture": "Tolurax", "width": 32, "vocab": 40, "norm": {"eps": 1e-6},
           "layers": [M.parallel(M.left(2, 1, dim, dim, window, 16.0 / dim), 1, 8, 1.0, 0.0)]}
    found = {}

    def edit(t):
        for name in ("l0.mix.left.q.norm", "l0.mix.left.k.norm"):
            t[name] = (t[name].float() * 1.6).bfloat16()
        get = lambda n: t[n].double()                          # noqa: E731
        h = M.plain.layer_norm(get("embed"), get("l0.norm1"), 1e-6)       # every token's mixer input
        q = (h @ get("l0.mix.left.q").T).view(-1, 2, dim)
        k = (h @ get("l0.mix.left.k").T).view(-1, 1, dim)
        q = M.plain.rms_div(q, 1e-6) * get("l0.mix.left.q.norm")
        k = M.plain.rms_div(k, 1e-6) * get("l0.mix.left.k.norm")
        score = torch.einsum("ahd,bd->abh", q, k[:, 0]).amax(-1) * 16.0 / dim    # [query token, key token]
        a, b = divmod(int(score.argmax()), score.shape[1])
        others = torch.stack((score[a], score[:, b], score.diagonal())).amax(0)
        filler = int(others.argmin())
        assert score[a, b] - others[filler] > 7, "the needle does not stand out"
        t["l0.mix.left.pb"] = torch.full((2,), 3.0 - float(score[a, b])).bfloat16()
        found.update(a=a, b=b, filler=filler)
    folder = M.make_folder(root, cfg, 77, sharp=False, edit=edit)
    return folder, found["a"], found["b"], found["filler"]


@pytest.mark.parametrize("device", DEVICES)
@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("window,page,dim", [(21, 8, 16), (16, 16, 16), (35, 16, 64), (70, 32, 128)])
def test_a_key_just_inside_and_just_outside_the_window(tmp_path, window, page, dim, dtype, device):
    """One key whose score stands out, `window - 1` and `window` tokens behind the query, the key on either side of a
    page border: the plain model says the logits differ widely between the two, and the engine follows it both in a
    prompt and when the query is decoded alone."""
    folder, a, b, filler = _needle_model(tmp_path / "needle", window, page, dim)
    plain = M.PlainTolurax(folder)
    for key_at in (page - 1, page, 2 * page + 3):
        inside = [filler] * key_at + [b] + [filler] * (window - 2) + [a, filler]
        outside = [filler] * key_at + [b] + [filler] * (window - 1) + [a, filler]
        qi, qo = key_at + window - 1, key_at + window
        gap = H.rel_rms(plain.logits(inside)[qi], plain.logits(outside)[qo])
        assert gap > 0.3, f"the test's key does not show: {gap}"
        for ids, at, what in ((inside, qi, "inside"), (outside, qo, "outside")):
            rep = _replayer(folder, device, dtype, page, cache_tokens=-(-len(ids) // page) * page, max_model_len=192)
            got = H.run_trace(rep, H.trace_whole({"p": ids}))
            _check(folder, dtype, {"p": ids}, got, f"window {window} key at {key_at} {what}, prompt")
            got = H.run_trace(rep, H.trace_decode_tail("p", ids, len(ids) - at + 2))
            _check(folder, dtype, {"p": ids}, got, f"window {window} key at {key_at} {what}, decoded")
            err = H.rel_rms(got[("p", at)], plain.logits(ids)[at])
            assert err < gap / 8, f"window {window} key at {key_at} {what}: {err} against a gap of {gap}"


@pytest.mark.parametrize("device", DEVICES)
@pytest.mark.parametrize("name", ["delta", "right"])
def test_a_far_token_reaches_through_the_state(tmp_path, name, device):
    """With decays near one, the first token still moves the logits 150 tokens later (the plain model says by how
    much); the engine, in portions and then token by token across many pages, agrees with the plain model."""
    cfg, seed = MODELS[name][0], MODELS[name][1]

    def edit(t):
        for key in t:
            if key.endswith("w0"):
                t[key] = torch.full_like(t[key], -7.0)
            if key.endswith("A_log"):
                t[key] = torch.full_like(t[key], -6.0)
    folder = M.make_folder(tmp_path / name, cfg, seed, edit=edit)
    plain = M.PlainTolurax(folder)
    ids = H.random_ids(151, cfg["vocab"], 9)
    other = [(ids[0] + 1) % cfg["vocab"]] + ids[1:]
    gap = H.rel_rms(plain.logits(ids)[150], plain.logits(other)[150])
    assert gap > 1e-3, f"the first token does not reach the last: {gap}"
    rep = _replayer(folder, device, "float32", 8, cache_tokens=152)
    trace = H.Trace()
    at = 0
    for n in (29, 2, 48, 11):
        trace.add([("f", at, ids[at: at + n], list(range(n)))])
        at += n
    for p in range(at, len(ids)):
        trace.add([("f", p, [ids[p]], [0])], end=["f"] if p == len(ids) - 1 else [])
    got = H.run_trace(rep, trace)
    _check(folder, "float32", {"f": ids}, got, f"{name} far token")
    assert H.rel_rms(got[("f", 150)], plain.logits(ids)[150]) < gap / 20


@pytest.mark.parametrize("device", DEVICES)
@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("name", ["right", "delta", "X"])
def test_long_rows_run_in_pieces(folders, name, dtype, device):
    """Rows long enough for the scans to cut them into pieces that run side by side: a prompt of 700 tokens whole,
    then portions of 300 and 290 beside a short request and a decode row, then the rest token by token."""
    folder = folders[name]
    vocab = MODELS[name][0]["vocab"]
    long_ids, short_ids = H.random_ids(700, vocab, 31), H.random_ids(41, vocab, 32)
    rep = _replayer(folder, device, dtype, 16, cache_tokens=1600, max_model_len=704)
    got = H.run_trace(rep, H.trace_whole({"long": long_ids}))
    _check(folder, dtype, {"long": long_ids}, got, f"pieces, whole {dtype}")
    trace = H.Trace()
    trace.add([("long", 0, long_ids[:300], [0, 127, 128, 255, 256, 299]), ("short", 0, short_ids[:40], [39])])
    trace.add([("long", 300, long_ids[300:590], [0, 100, 289]), ("short", 40, short_ids[40:], [0])], end=["short"])
    for at in range(590, 700):
        trace.add([("long", at, [long_ids[at]], [0])], end=["long"] if at == 699 else [])
    got = H.run_trace(rep, trace)
    _check(folder, dtype, {"long": long_ids, "short": short_ids}, got, f"pieces, portions {dtype}")
    rep.cache.check()


@pytest.mark.parametrize("device", DEVICES)
@pytest.mark.parametrize("dtype", DTYPES)
def test_long_decoding(folders, dtype, device):
    """180 tokens one by one after a prompt of 5: many window lengths, many pages given back on the way."""
    folder, page = folders["X-sharp"], 8
    ids = H.random_ids(185, M.CONFIG_X["vocab"], 21)
    rep = _replayer(folder, device, dtype, page, cache_tokens=192)
    got = H.run_trace(rep, H.trace_decode_tail("d", ids, 180))
    _check(folder, dtype, {"d": ids}, got, f"long decoding {dtype}")
    left_pages = [g for g in rep.cache.groups if g.decl.window > 0]
    assert left_pages and all(g.pool.free == g.pool.usable for g in rep.cache.groups)


def test_configuration_and_weights_are_checked(tmp_path):
    from holon_amd.config.model import ConfigError
    from holon_amd.registry import resolve
    from holon_amd.weights.loader import WeightError
    cfg, spec = resolve(M.CONFIG_X)
    assert [r.layer for r in spec.order] == [0, 0, 0, 1] and cfg.to_dict()["loop"] == M.CONFIG_X["loop"]
    assert [r.layer for r in resolve(M.CONFIG_Z)[1].order] == [0, 1]
    for bad in (M.variant(M.CONFIG_X, loop={"start": 1, "stop": 1, "times": 2}),
                {k: v for k, v in M.CONFIG_X.items() if k != "norm"},
                M.variant(M.CONFIG_X, layers=[{"type": "conv", "mixer": {}, "mlp": None}])):
        with pytest.raises(ConfigError):
            resolve(bad)

    def drop(t):
        del t["l1.mix.right.mu.w"]
        t["l0.mix.q.conv"] = t["l0.mix.q.conv"][:, :2].contiguous()
    folder = M.make_folder(tmp_path / "bad", M.CONFIG_X, 1, edit=drop)
    from holon_amd.engine.loading import load_model
    with pytest.raises(WeightError) as e:
        load_model(folder, device="cpu", dtype="float32", kernels=TorchKernels(), max_model_len=32, max_seqs=2)
    assert "l1.mix.right.mu.w" in str(e.value) and "l0.mix.q.conv" in str(e.value)


@pytest.mark.parametrize("device", DEVICES)
def test_random_weights_from_the_command_line_replay(tmp_path, device):
    """`holon_amd random` writes a Tolurax folder (the decay's rank named in the configuration), and the engine and
    the plain model agree on it."""
    from holon_amd.cli import main
    cfg = M.variant(M.CONFIG_X)
    cfg["layers"][1]["mixer"]["right"]["rank"] = 5
    (tmp_path / "c.json").write_text(json.dumps(cfg))
    assert main(["random", "--config", str(tmp_path / "c.json"), "--seed", "4", "--out", str(tmp_path / "m")]) == 0
    ids = H.random_ids(30, cfg["vocab"], 2)
    rep = _replayer(tmp_path / "m", device, "float32", 8, cache_tokens=32)
    got = H.run_trace(rep, H.trace_chunks("a", ids, [4, 9]))
    _check(tmp_path / "m", "float32", {"a": ids}, got, "random folder")


@pytest.mark.parametrize("device", DEVICES)
@pytest.mark.parametrize("dtype", DTYPES)
def test_greedy_generation_through_the_engine(folders, dtype, device):
    """The engine's own entry point and scheduler: prompts of unequal length generated side by side, with prompt
    portions riding beside decode rows, follow the plain model's most likely token wherever that is clear."""
    from holon_amd.config import EngineConfig, SamplingParams
    from holon_amd.engine.engine import Engine
    folder = folders["Y-sharp"]
    plain = _plain(str(folder))
    prompts = [H.random_ids(n, M.CONFIG_Y["vocab"], 50 + n) for n in (5, 37, 18, 1)]
    cfg = EngineConfig(model=str(folder), device=device, dtype=dtype, page_size=8, max_seqs=3, max_model_len=96,
                       max_step_tokens=40, chunk_with_decode=16, cache_tokens=192)
    engine = Engine(cfg, TorchKernels() if device == "cpu" else None)
    outs = engine.generate(prompts, SamplingParams(temperature=0.0, max_tokens=24, ignore_eos=True))
    held = sum(H.assert_greedy_follows(plain, p, o, margin=0.02 if dtype == "float32" else 0.25)
               for p, o in zip(prompts, outs))
    assert all(len(o) == 24 for o in outs) and held >= (60 if dtype == "float32" else 20)
    engine.cache.check()
    engine.close()


@pytest.mark.gpu
def test_trace_runner_as_a_program(folders, tmp_path):
    """bin/trace_run on a Tolurax folder, as a user runs it."""
    import pathlib

    import numpy as np
    folder, requests = folders["X"], _requests("X", (30, 19))
    trace = H.trace_mixed(requests, seed=3, max_live=2, decode_tail=4)
    exe = pathlib.Path(__file__).resolve().parent.parent / "bin" / "trace_run"
    out = tmp_path / "out"
    run = subprocess.run([sys.executable, str(exe), "--model", str(folder), "--dtype", "float32", "--out", str(out),
                          "--max-tokens", str(H.peak_live_tokens(trace))], input=trace.jsonl(), text=True,
                         capture_output=True, timeout=600)
    assert run.returncode == 0, run.stderr[-2000:]
    got = {}
    for step, expect in zip(trace.steps, trace.expect):
        rows = np.fromfile(out / f"{step['step']}.f32", dtype="<f4").reshape(len(expect), -1)
        for row, key in zip(rows, expect):
            got[key] = torch.from_numpy(row.copy())
    _check(folder, "float32", requests, got, "trace_run")


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("heads,dim", [(3, 64), (2, 16), (2, 40), (1, 128), (1, 200)])
def test_the_memory_in_pieces(heads, dim, dtype):
    """`memory_scan` with rows in pieces against its plain form: rows longer and shorter than a piece, ends inside, at and one
    behind a border of a piece and of a block of 16 tokens, states carried and not, decays near one and near nothing. The
    same products in another order: float32 rounding."""
    from holon_amd.kernels import load_hip
    from holon_amd.kernels.registry import kernel_op
    k, dev = load_hip(), torch.device("cuda")
    gen = torch.Generator().manual_seed(heads * 1000 + dim)
    rn = lambda *s: torch.randn(s, generator=gen).to(dev)                      # noqa: E731
    counts, piece = [385, 256, 17, 1, 300], 128
    t, npc = sum(counts), [-(-n // piece) for n in counts]
    i32 = lambda v: torch.tensor(v, dtype=torch.int32, device=dev)             # noqa: E731
    r, kk, v = (rn(t, heads * dim).to(dtype) for _ in range(3))
    w = torch.exp(-torch.exp(2 * rn(t, heads * dim)))
    u, state = rn(heads, dim), rn(7, heads, dim, dim)
    rows = (i32([6, 1, 2, 0, 4]), i32([5, 0, 9, 3, 0]), i32([sum(counts[:b]) for b in range(6)]), 5, heads)
    one, two = state.clone(), state.clone()
    got = k.memory_scan(r, kk, v, w, u, one, *rows, (piece, max(npc), i32([sum(npc[:b]) for b in range(5)]), sum(npc)))
    want = kernel_op("memory_scan").plain(r.double().float(), kk, v, w, u, two, *rows)
    assert H.rel_rms(got, want) < 2e-6 and H.rel_rms(one, two) < 2e-6


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("dim,shift", [(64, -5), (64, 0), (128, -5), (200, -5)])
def test_the_memory_in_pieces_is_as_near_64_bits_as_token_by_token(dim, shift, dtype):
    """Long sums (decays near one) and short ones: rows in pieces may be at most 1.1 times as far from the recurrence in float64
    as the token-by-token scan of the same row, in results and, where decays are near one, state."""
    import holon_amd.parts  # noqa: F401  (registers the parts' operations)
    from holon_amd.kernels import load_hip
    k, dev, heads, t = load_hip(), torch.device("cuda"), 8, 1000
    gen = torch.Generator().manual_seed(dim + shift)
    rn = lambda *s: torch.randn(s, generator=gen).to(dev)                      # noqa: E731
    i32 = lambda v: torch.tensor(v, dtype=torch.int32, device=dev)             # noqa: E731
    r, kk, v = (rn(t, heads * dim).to(dtype) for _ in range(3))
    w = torch.exp(-torch.exp(rn(t, heads * dim) + shift))
    u, state = rn(heads, dim), rn(2, heads, dim, dim)
    rows = (i32([1]), i32([7]), i32([0, t]), 1, heads)
    S, want = state[1].double(), torch.empty(t, heads, dim, dtype=torch.double, device=dev)
    rd, kd, vd, wd = (x.double().view(t, heads, dim) for x in (r, kk, v, w))
    for i in range(t):
        kv = kd[i][:, :, None] * vd[i][:, None, :]
        want[i] = ((S + u.double()[:, :, None] * kv) * rd[i][:, :, None]).sum(1)
        S = wd[i][:, :, None] * S + kv
    apart = []
    for pieces in (None, (128, 8, i32([0]), 8)):
        held = state.clone()
        got = k.memory_scan(r, kk, v, w, u, held, *rows, pieces).view_as(want)
        apart.append((((got - want).norm() / want.norm()).item(), ((held[1] - S).norm() / S.norm()).item()))
    assert apart[1][0] <= 1.1 * apart[0][0], apart
    if shift < 0:                              # (fast decays: what is left of a state is its last few tokens)
        assert apart[1][1] <= 1.1 * apart[0][1], apart


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("heads,dim", [(2, 24), (2, 64), (1, 128), (1, 200)])
def test_the_memory_in_pieces_keeps_what_is_not_finite_from_earlier_tokens(heads, dim, dtype):
    """A key or value of NaN or infinity: the tokens before it come out bit for bit as without it, those from it on are the
    token-by-token scan's in where they are finite (a value: its own column alone)."""
    import holon_amd.parts  # noqa: F401  (registers the parts' operations)
    from holon_amd.kernels import load_hip
    k, dev, t = load_hip(), torch.device("cuda"), 300
    gen = torch.Generator().manual_seed(dim)
    rn = lambda *s: torch.randn(s, generator=gen).to(dev)                      # noqa: E731
    i32 = lambda v: torch.tensor(v, dtype=torch.int32, device=dev)             # noqa: E731
    r, kk, v = (rn(t, heads * dim).to(dtype) for _ in range(3))
    w = torch.exp(-torch.exp(rn(t, heads * dim) - 2))
    u, state = rn(heads, dim), rn(1, heads, dim, dim)
    cut = (128, 3, i32([0]), 3)
    run = lambda key, val, pieces: k.memory_scan(r, key, val, w, u, state.clone(), i32([0]), i32([7]), i32([0, t]), 1, heads,  # noqa: E731
                                                 pieces).view(t, heads, dim)
    ref = run(kk, v, cut)
    for at, value in ((0, "nan"), (5, "inf"), (37, "-inf"), (140, "nan"), (255, "inf"), (299, "nan")):
        key, val = kk.clone(), v.clone()
        key[at, 3] = float(value)
        val[at, 7] = float(value)
        got = run(key, v, cut)
        assert torch.equal(got[:at], ref[:at]), (at, value)
        assert torch.equal(got.isfinite(), run(key, v, None).isfinite()), (at, value)
        got = run(kk, val, cut)
        assert torch.equal(got[:at], ref[:at]), (at, value)
        assert torch.equal(got.isfinite(), run(kk, val, None).isfinite()), (at, value)
        got[:, 0, 7] = ref[:, 0, 7]
        assert torch.equal(got, ref), (at, value)


@pytest.mark.gpu
@pytest.mark.parametrize("heads,kv,dim,vdim", [(2, 1, 64, 64), (4, 2, 24, 40), (1, 1, 128, 72), (2, 2, 200, 16)])
def test_the_delta_rule_in_pieces_starts_from_a_copy(heads, kv, dim, vdim, monkeypatch):
    """`delta_scan` with rows in pieces against its plain form, carried rows of several pieces among them. The second pass writes
    a row's slot from its last piece while its first one starts, so the first one's start lies in the workspace, in the last
    piece's place."""
    import holon_amd.parts  # noqa: F401  (registers the parts' operations)
    from holon_amd.kernels import load_hip
    from holon_amd.kernels.registry import kernel_op
    k, dev = load_hip(), torch.device("cuda")
    gen = torch.Generator().manual_seed(dim)
    rn = lambda *s: torch.randn(s, generator=gen).to(dev)                      # noqa: E731
    i32 = lambda v: torch.tensor(v, dtype=torch.int32, device=dev)             # noqa: E731
    counts, piece = [513, 256, 1, 257, 300], 256
    t, npc = sum(counts), [-(-n // piece) for n in counts]
    norm = lambda x: x / x.norm(dim=-1, keepdim=True)                          # noqa: E731
    qn, kn = norm(rn(t, kv, dim)), norm(rn(t, kv, dim))
    qkv, beta, g = rn(t, 2 * kv * dim + heads * vdim), torch.rand(t, heads, generator=gen).to(dev), torch.exp(-rn(t, heads).abs() / 20)
    state, base = rn(7, heads, dim, vdim), [sum(npc[:b]) for b in range(5)]
    slots, starts = [6, 1, 2, 0, 4], [5, 0, 9, 3, 0]
    rows = (i32(slots), i32(starts), i32([sum(counts[:b]) for b in range(6)]), 5, heads, vdim)
    one, two, made, empty = state.clone(), state.clone(), [], torch.empty
    with monkeypatch.context() as m:
        m.setattr(torch, "empty", lambda *a, **kw: made.append(empty(*a, **kw)) or made[-1])
        got = k.delta_scan(qn, kn, qkv, beta, g, one, *rows, (piece, max(npc), i32(base), sum(npc)))
    want = kernel_op("delta_scan").plain(qn, kn, qkv, beta, g, two, *rows)
    assert H.rel_rms(got, want) < 1e-5 and H.rel_rms(one, two) < 1e-5
    starts_of = [x for x in made if tuple(x.shape) == (sum(npc), heads, dim, vdim)][-1]
    for b in (0, 3):
        assert torch.equal(starts_of[base[b] + npc[b] - 1], state[slots[b]]), b
    assert not starts_of[base[4] + npc[4] - 1].any()


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("heads,kv,dim,vdim", [(2, 1, 32, 64), (4, 2, 22, 40), (1, 1, 6, 5), (2, 2, 128, 130), (1, 1, 256, 16)])
def test_the_delta_rule_in_blocks_of_tokens(heads, kv, dim, vdim, dtype):
    """`delta_scan` over rows of one token, of a block of 16, of one more and less, whole and in pieces of two blocks, against its plain
    form (the same formulas in float32: sums of up to 256 terms, so 1e-5 leaves a factor of ten). A key or value of NaN or infinity:
    the tokens before it bit for bit as without it, those from it on finite where the token-by-token scan's are."""
    import holon_amd.parts  # noqa: F401  (registers the parts' operations)
    from holon_amd.kernels import load_hip
    from holon_amd.kernels.registry import kernel_op
    k, dev = load_hip(), torch.device("cuda")
    gen = torch.Generator().manual_seed(dim)
    rn = lambda *s: torch.randn(s, generator=gen).to(dev)                      # noqa: E731
    i32 = lambda v: torch.tensor(v, dtype=torch.int32, device=dev)             # noqa: E731
    counts = [1, 15, 16, 17, 33, 47]
    t, n = sum(counts), len(counts)
    norm = lambda x: x / x.norm(dim=-1, keepdim=True)                          # noqa: E731
    qn, kn = norm(rn(t, kv, dim)), norm(rn(t, kv, dim))
    qkv = rn(t, 2 * kv * dim + heads * vdim).to(dtype)
    beta, g = torch.rand(t, heads, generator=gen).to(dev), torch.exp(-rn(t, heads).abs())
    g[5], beta[7] = 0.0, 0.0
    state = rn(n + 1, heads, dim, vdim)
    rows = (i32([6, 1, 2, 0, 4, 5]), i32([5, 0, 9, 3, 0, 1]), i32([sum(counts[:b]) for b in range(n + 1)]), n, heads, vdim)

    def run(piece, key=kn, val=qkv, scan=k.delta_scan):
        npc = [-(-c // piece) for c in counts] if piece else []
        pieces = (piece, max(npc), i32([sum(npc[:b]) for b in range(n)]), sum(npc)) if piece else None
        held = state.clone()
        return scan(qn, key, val, beta, g, held, *rows, pieces), held
    want, after = run(0, scan=kernel_op("delta_scan").plain)
    for piece in (32, 48):
        got, held = run(piece)
        assert H.rel_rms(got, want) < 1e-5 and H.rel_rms(held, after) < 1e-5, piece
    ref, last = run(48)[0], sum(counts[:5])
    for at, value in ((last, "nan"), (last + 5, "inf"), (last + 16, "-inf"), (last + 46, "nan")):
        key, val = kn.clone(), qkv.clone()
        key[at, 0, 3] = float(value)
        val[at, 2 * kv * dim + 1] = float(value)
        for kk, vv in ((key, qkv), (kn, val)):
            got = run(48, kk, vv)[0]
            assert torch.equal(got[:at], ref[:at]), (at, value)
            assert torch.equal(got.isfinite(), run(0, kk, vv)[0].isfinite()), (at, value)


def _step_of(counts, device="cpu"):
    """What the scans read of a step whose rows have these numbers of tokens."""
    from types import SimpleNamespace
    return SimpleNamespace(h_counts=np.array(counts, dtype=np.int32), n_tokens=sum(counts), slots=torch.zeros(1, device=device),
                           rows=SimpleNamespace(max_chunk_query=max([c for c in counts if c > 1], default=0)))


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("columns", [64, 2048, 4096])
def test_a_rows_pieces_do_not_depend_on_the_rows_beside_it(dtype, columns):
    """`delta_pieces` gives every row of a step the tokens a piece that it has alone (none below the block form's border), and
    each row's pieces places of their own in order."""
    from holon_amd.parts.recurrent import DELTA_FROM, delta_pieces
    least = DELTA_FROM[dtype]
    counts = [1, 2, least - 1, least, 511, 512, 513, 1281, 2560, 2561, 9000, 1]

    def form(counts):
        got = delta_pieces(_step_of(counts), columns, dtype)
        if got is None:
            return [0] * len(counts), None
        tokens, most, base, total, each = got
        return ([tokens] * len(counts) if each is None else each.tolist()), (tokens, most, base.tolist(), total)
    each, (tokens, most, base, total) = form(counts)
    assert each == [form([c])[0][0] for c in counts] and all(e in ((256, 512) if c >= least else (0,)) for c, e in zip(counts, each))
    pieces = [-(-c // e) if e else 0 for c, e in zip(counts, each)]
    assert (tokens, most, total) == (max(each), max(pieces), sum(pieces)) and base == [sum(pieces[:b]) for b in range(len(counts))]
    assert form([1, 1, least - 1])[1] is None


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("heads,kv,dim,vdim", [(2, 1, 32, 64), (1, 1, 128, 72)])
def test_the_delta_rule_of_a_row_does_not_depend_on_the_rows_beside_it(heads, kv, dim, vdim, dtype):
    """Rows of one token to several pieces in one step, bit for bit what each of them is alone: below the block form's border, at it,
    in one piece and in several, carried and not."""
    import holon_amd.parts  # noqa: F401  (registers the parts' operations)
    from holon_amd.kernels import load_hip
    from holon_amd.parts.recurrent import delta_pieces
    k, dev = load_hip(), torch.device("cuda")
    gen = torch.Generator().manual_seed(dim)
    rn = lambda *s: torch.randn(s, generator=gen).to(dev)                      # noqa: E731
    i32 = lambda v: torch.tensor(v, dtype=torch.int32, device=dev)             # noqa: E731
    counts, starts = [1, 20, 63, 64, 300, 511, 600, 1, 512], [9, 0, 4, 1, 0, 2, 3, 0, 5]
    t, n = sum(counts), len(counts)
    norm = lambda x: x / x.norm(dim=-1, keepdim=True)                          # noqa: E731
    qn, kn = norm(rn(t, kv, dim)), norm(rn(t, kv, dim))
    qkv = rn(t, 2 * kv * dim + heads * vdim).to(dtype)
    beta, g = torch.rand(t, heads, generator=gen).to(dev), torch.exp(-rn(t, heads).abs())
    state = rn(n, heads, dim, vdim)
    together, lo = state.clone(), 0
    out = k.delta_scan(qn, kn, qkv, beta, g, together, i32(list(range(n))), i32(starts), i32([sum(counts[:b]) for b in range(n + 1)]), n,
                       heads, vdim, delta_pieces(_step_of(counts, dev), heads * vdim, dtype))
    for b, c in enumerate(counts):
        alone, own = state.clone(), slice(lo, lo + c)
        got = k.delta_scan(qn[own].contiguous(), kn[own].contiguous(), qkv[own].contiguous(), beta[own].contiguous(), g[own].contiguous(),
                           alone, i32([b]), i32([starts[b]]), i32([0, c]), 1, heads, vdim,
                           delta_pieces(_step_of([c], dev), heads * vdim, dtype))
        assert torch.equal(got, out[own]) and torch.equal(alone[b], together[b]), (b, c)
        lo += c


@pytest.mark.gpu
@pytest.mark.parametrize("heads,kv,dim,vdim", [(2, 1, 32, 64), (1, 1, 6, 5), (1, 1, 128, 72)])
def test_an_infinite_value_of_a_rows_last_token_is_infinite_in_its_state(heads, kv, dim, vdim):
    """`delta_scan` in blocks of tokens, a row's last token with a value of infinity: its column of the state is what the
    token-by-token scan leaves there (infinities of the key's signs), every other column what it is without it; rows that end with a
    block, inside one, and of one token."""
    import holon_amd.parts  # noqa: F401  (registers the parts' operations)
    from holon_amd.kernels import load_hip
    k, dev = load_hip(), torch.device("cuda")
    gen = torch.Generator().manual_seed(dim)
    rn = lambda *s: torch.randn(s, generator=gen).to(dev)                      # noqa: E731
    i32 = lambda v: torch.tensor(v, dtype=torch.int32, device=dev)             # noqa: E731
    counts = [1, 16, 33, 47]
    t, n = sum(counts), len(counts)
    base = [sum(counts[:b]) for b in range(n + 1)]
    norm = lambda x: x / x.norm(dim=-1, keepdim=True)                          # noqa: E731
    qn, kn = norm(rn(t, kv, dim)), norm(rn(t, kv, dim))
    qkv, beta, g = rn(t, 2 * kv * dim + heads * vdim), 0.1 + torch.rand(t, heads, generator=gen).to(dev), torch.exp(-rn(t, heads).abs())
    state, at = rn(n, heads, dim, vdim), 2 * kv * dim + 3                      # (the first head's column 3)
    for sign in (1.0, -1.0):
        val = qkv.clone()
        val[[b - 1 for b in base[1:]], at] = sign * float("inf")
        after = []
        for v, pieces in ((val, None), (val, (48, 1, i32([0, 1, 2, 3]), 4)), (qkv, (48, 1, i32([0, 1, 2, 3]), 4))):
            held = state.clone()
            k.delta_scan(qn, kn, v, beta, g, held, i32(list(range(n))), i32([1] * n), i32(base), n, heads, vdim, pieces)
            after.append(held)
        tokens, blocks, without = after
        assert torch.equal(blocks[:, 0, :, 3], tokens[:, 0, :, 3]) and blocks[:, 0, :, 3].isinf().all()
        blocks[:, 0, :, 3] = without[:, 0, :, 3]
        assert torch.equal(blocks, without)


def test_sigmoid_decode_rows_keep_few_waves_where_units_have_several_blocks():
    """`decode_waves`: a wave for every 32 keys only up to 256 (row, kv head) pairs, and then one for every 128, never more than four."""
    from holon_amd.parts.sigmoid_attention import decode_blocks, decode_waves
    assert [decode_waves(4, n, 1) for n in (1, 32, 33, 128, 256, 257, 1023, 1024, 5000)] == [1, 1, 2, 4, 4, 5, 5, 8, 8]
    assert [decode_waves(257, n, 1) for n in (1, 128, 129, 300, 400, 512, 5000)] == [1, 1, 2, 3, 4, 4, 4]
    for pairs in (1, 16, 64, 128):
        assert all(decode_waves(pairs, n, decode_blocks(pairs, n)) == min(4, -(-(-(-n // decode_blocks(pairs, n))) // 32)) for n in (257, 700, 9000))
