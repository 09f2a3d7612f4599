"""Each HIP kernel alone against its plain twin (tests/plain/ops.py) on the same inputs, at sizes other than the tiny
models': the reference's own test shapes (plugins/tests/test_op_kernels.py:28-72, test_attention_kernels.py:20-66)
and awkward ones (widths that are no power of two, head sizes in steps of 16, page sizes from 1 up)."""
from __future__ import annotations

import numpy as np
import pytest
import torch

import holon_amd.parts  # noqa: F401  (registers the parts' operations)
from holon_amd.kernels.api import AttnRows
from tests import helpers as H
from tests.plain.ops import TorchKernels

pytestmark = pytest.mark.gpu
DTYPES = [torch.float32, torch.bfloat16]
PLAIN = TorchKernels()


@pytest.fixture(scope="module")
def hip():
    from holon_amd.kernels import load_hip
    return load_hip()


def _randn(*shape, dtype, seed=0, scale=1.0):
    g = torch.Generator().manual_seed(seed)
    return (torch.randn(*shape, generator=g) * scale).to(dtype).cuda()


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("shape", [(37, 4096), (37, 8, 128), (5, 100), (3, 7, 48), (1, 12288), (130, 16)])
def test_rmsnorm_and_add(hip, dtype, shape):
    x, r = _randn(*shape, dtype=dtype, seed=1), _randn(*shape, dtype=dtype, seed=2)
    w = (1 + 0.1 * torch.randn(shape[-1], generator=torch.Generator().manual_seed(3))).to(dtype).cuda()
    x0 = x.clone()
    for eps in (1e-6, 1e-2):
        got, want = hip.rmsnorm(x, w, eps), PLAIN.rmsnorm(x.double(), w.double(), eps)
        assert torch.equal(x, x0), "rmsnorm wrote its input"
        assert H.op_budget_usage(got, want, dtype, shape[-1]) <= 1
    x2, r_hip, r_ref = x.reshape(-1, shape[-1]), r.reshape(-1, shape[-1]).clone(), r.reshape(-1, shape[-1]).clone()
    got = hip.add_rmsnorm(x2, r_hip, w, 1e-6)
    want = PLAIN.add_rmsnorm(x2, r_ref, w, 1e-6)
    assert torch.equal(r_hip, r_ref), "the residual sum is one rounding of x + r"
    assert H.op_budget_usage(got, want.float(), dtype, shape[-1]) <= 1


@pytest.mark.parametrize("dtype", DTYPES)
def test_embedding_and_silu_mul(hip, dtype):
    table = _randn(1000, 120, dtype=dtype, seed=4)
    ids = torch.tensor([0, 999, 5, 5, 123], dtype=torch.int32).cuda()
    assert torch.equal(hip.embedding(ids, table), table[ids.long()])
    table = _randn(333, 4096, dtype=dtype, seed=5)
    assert torch.equal(hip.embedding(ids[2:], table), table[ids[2:].long()])
    # tokens that the last step drew and left on the device: kept by slot, taken where a row says so
    last = torch.zeros(9, dtype=torch.int32).cuda()
    hip.store_tokens(last, torch.tensor([7, 2, 5], dtype=torch.int32).cuda(), torch.tensor([330, 11, 0], dtype=torch.int32).cuda())
    assert last.tolist() == [0, 0, 11, 0, 0, 0, 0, 330, 0]
    take = torch.tensor([-1, 7, -1, 2, 5], dtype=torch.int32).cuda()
    want = table[torch.tensor([0, 330, 5, 11, 0])]
    assert torch.equal(hip.embedding(ids, table, (take, last)), want)
    assert torch.equal(PLAIN.embedding(ids, table, (take, last)), want)
    for t, inter in ((17, 12288), (3, 100), (1, 7)):
        gu = _randn(t, 2 * inter, dtype=dtype, seed=6, scale=3.0)
        got, want = hip.silu_mul(gu), PLAIN.silu_mul(gu.double())
        assert H.op_budget_usage(got, want, dtype, 1) <= 1
    gu = torch.zeros(2, 8, dtype=dtype).cuda()
    gu[:, 4:] = 1
    assert torch.equal(hip.silu_mul(gu), torch.zeros(2, 4, dtype=dtype).cuda())


def test_silu_is_rounded_before_the_multiply(hip):
    """The reference multiplies silu(gate), rounded to the activation dtype, by up (std/holon_std/ffn/reference.py:
    7-12). Where rounding first and rounding only the product give different bfloat16 results, the kernels give the
    first: alone and fused into the gated product."""
    bf = torch.bfloat16
    g = torch.Generator().manual_seed(60)
    gate = (torch.randn(64, 4096, generator=g) * 2).to(bf)
    up = torch.randn(64, 4096, generator=g).to(bf)
    s64 = gate.double() * torch.sigmoid(gate.double())
    first = (s64.to(bf).float() * up.float()).to(bf)                   # rounded, then multiplied (one more rounding)
    late = (s64 * up.double()).to(bf)                                  # only the product rounded
    half_ulp = torch.exp2(torch.frexp(s64.to(bf).double())[1].double() - 1 - 8)      # of silu's bfloat16 neighbour
    edge = half_ulp - (s64 - s64.to(bf).double()).abs() < 1e-2 * half_ulp            # silu on a rounding edge: skip
    tell = (first != late) & ~edge
    assert tell.sum() > 10000                                          # the two orders differ in thousands of places
    got = hip.silu_mul(torch.cat((gate, up), dim=-1).cuda()).cpu()
    assert torch.equal(got[tell], first[tell])
    # the gated product: weights that copy x into gate and up make the product exact, the activation is what is left
    k = 256
    x = torch.cat((gate[:16, :128], up[:16, :128]), dim=-1).contiguous()                 # [16, 256]
    w = torch.zeros(256, k)
    w[:128, :128] = torch.eye(128)                                     # gate_i = x_i
    w[128:, 128:] = torch.eye(128)                                     # up_i = x_(128 + i)
    fused = hip.linear_silu_mul(x.cuda(), w.to(bf).cuda()).cpu()
    t = tell[:16, :128]
    assert t.sum() > 20 and torch.equal(fused[t], first[:16, :128][t])


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize(("head_dim", "rotary_dim", "theta"), [(128, 128, 1e6), (256, 64, 1e7), (48, 48, 1e4), (16, 8, 1e4)])
def test_rope(hip, dtype, head_dim, rotary_dim, theta):
    from holon_amd.parts.positions import rope_table
    table = rope_table(8192, rotary_dim, theta).cuda()
    pos = torch.tensor([0, 1, 2, 15, 16, 1000, 4095, 8191] + list(range(100, 121)), dtype=torch.int32).cuda()
    q = _randn(29, 24, head_dim, dtype=dtype, seed=7)
    want = q.clone()
    PLAIN.rope(want, pos, table)
    got = q.clone()
    hip.rope(got, pos, table)
    assert H.op_budget_usage(got, want, dtype, 2) <= 1
    assert torch.equal(got[..., rotary_dim:], q[..., rotary_dim:])          # the rest passes through untouched
    assert torch.equal(got[0], q[0])                                         # position 0: identity
    # against the formula itself, in float64, half-split pairing
    inv = theta ** (-torch.arange(0, rotary_dim, 2, dtype=torch.float64) / rotary_dim)
    ang = pos.double().cpu()[:, None] * inv
    a, b = q[..., : rotary_dim // 2].double().cpu(), q[..., rotary_dim // 2: rotary_dim].double().cpu()
    ref = torch.cat((a * ang.cos()[:, None] - b * ang.sin()[:, None], b * ang.cos()[:, None] + a * ang.sin()[:, None]), -1)
    assert (got[..., :rotary_dim].double().cpu() - ref).abs().max() < (4e-3 if dtype == torch.float32 else 4e-2)


def _paged_case(rows, heads, kv_heads, head_dim, page, dtype, seed=0, max_seqs=8, scale_q=1.0):
    """rows: (tokens before this step, tokens this step). A shuffled block table with spare pages."""
    g = torch.Generator().manual_seed(seed)
    rng = np.random.default_rng(seed)
    assert len(rows) <= max_seqs
    slots = rng.permutation(max_seqs)[: len(rows)].astype(np.int32)
    max_pages = -(-max(s + n for s, n in rows) // page)
    units = max_seqs * max_pages + 7
    table = torch.from_numpy(rng.permutation(units)[: max_seqs * max_pages].reshape(max_seqs, max_pages).astype(np.int32))
    pages = torch.randn(units, 2, kv_heads, page * head_dim, generator=g).to(dtype).cuda()
    counts = np.array([n for _, n in rows])
    lens = np.array([s + n for s, n in rows])
    qstart = np.concatenate([[0], np.cumsum(counts)]).astype(np.int32)
    q = (torch.randn(int(counts.sum()), heads, head_dim, generator=g) * scale_q).to(dtype).cuda()
    dec, chk = np.flatnonzero(counts == 1), np.flatnonzero(counts > 1)
    i32 = lambda a: torch.as_tensor(np.asarray(a, dtype=np.int32)).cuda()
    attn = AttnRows(slots=i32(slots), lens=i32(lens), query_start=i32(qstart), decode_rows=i32(dec), chunk_rows=i32(chk),
                    n_decode=len(dec), n_chunk=len(chk), max_decode_len=int(lens[dec].max()) if len(dec) else 0,
                    max_chunk_query=int(counts[chk].max()) if len(chk) else 0,
                    max_chunk_len=int(lens[chk].max()) if len(chk) else 0, in_order=len(chk) == 0)
    return q, pages, table.cuda(), attn


GEOMETRIES = [(32, 8, 128), (16, 4, 256), (16, 8, 64), (6, 3, 32), (4, 1, 16), (5, 5, 48), (12, 2, 80),
              (10, 2, 64), (40, 2, 128), (7, 7, 64), (6, 1, 128), (48, 2, 64),   # groups of 5, 20, 1, 6 and 24 heads
              (40, 1, 128), (66, 1, 64),                                         # and of more heads than a tile has rows
              (64, 8, 128)]                                                      # groups of 8 at head_dim 128
ROWSETS = [[(0, 1), (0, 17), (5, 16), (31, 33), (0, 64), (100, 7), (16, 16)],
           [(0, 1), (15, 1), (16, 1), (99, 1), (999, 1), (4096, 1)],
           [(63, 1), (200, 2), (17, 1), (0, 130), (1, 1)]]


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("page", [16, 8, 64, 1, 5])
@pytest.mark.parametrize("geometry", GEOMETRIES)
def test_paged_attention(hip, dtype, page, geometry):
    heads, kv_heads, head_dim = geometry
    for seed, rows in enumerate(ROWSETS):
        if page < 8:
            rows = [(min(s, 300), n) for s, n in rows]
        q, pages, table, attn = _paged_case(rows, heads, kv_heads, head_dim, page, dtype, seed)
        scale = head_dim ** -0.5
        want = PLAIN.paged_attention(q.double(), pages.double(), table, attn, page, scale, 0)
        got = hip.paged_attention(q, pages, table, attn, page, scale, 0)
        again = hip.paged_attention(q, pages, table, attn, page, scale, 0)
        assert torch.equal(got, again), "two runs differ"
        # sums over head_dim (scores) and over the keys (softmax, values)
        assert H.op_budget_usage(got, want, dtype, head_dim + max(s + n for s, n in rows)) <= 1, (geometry, page, rows)


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("geometry", [(32, 8, 128), (6, 3, 32), (8, 2, 64), (32, 1, 64)])
def test_attention_never_touches_what_lies_beyond_a_row(hip, dtype, geometry):
    """Every cache slot that no row of the step holds a token in (the rest of a row's last page, pages of other
    requests, spare pages) is filled with NaN: a kernel that lets such a slot into a product, even with weight zero,
    gives NaN. Decode rows, short portions and portions long enough for the kernels that stage through LDS."""
    heads, kv_heads, head_dim = geometry
    page = 16
    for rows in ([(0, 1), (14, 1), (16, 1), (99, 1), (1000, 1)], [(0, 17), (5, 16), (31, 33), (100, 7)],
                 [(3, 700), (0, 530)]):
        q, pages, table, attn = _paged_case(rows, heads, kv_heads, head_dim, page, dtype, seed=len(rows))
        held = torch.zeros(pages.shape[0], page, dtype=torch.bool)
        for slot, (s, n) in zip(attn.slots.tolist(), rows):
            pos = torch.arange(s + n)
            held[table[slot, pos // page].cpu().long(), pos % page] = True
        kp, vp = pages[:, 0].view(-1, kv_heads, page, head_dim), pages[:, 1].view(-1, kv_heads, head_dim, page)
        free = (~held).cuda()
        kp.masked_fill_(free[:, None, :, None], float("nan"))
        vp.masked_fill_(free[:, None, None, :], float("nan"))
        want = PLAIN.paged_attention(q.double(), pages.double(), table, attn, page, head_dim ** -0.5, 0)
        got = hip.paged_attention(q, pages, table, attn, page, head_dim ** -0.5, 0)
        assert torch.isfinite(got.float()).all(), (geometry, rows)
        assert H.op_budget_usage(got, want, dtype, head_dim + max(s + n for s, n in rows)) <= 1


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("geometry", [(32, 8, 128), (8, 2, 64)])
def test_sixty_four_decode_rows(hip, dtype, geometry):
    """A decode step of 64 rows of unequal lengths (one key to 4,096, on and off page edges), with the launch shaped
    for a longer row than any has (as a graph's length bucket shapes it), and again with 11 of the rows empty rows on
    a table row of one page (as a graph's padding rows are)."""
    heads, kv_heads, head_dim = geometry
    rng = np.random.default_rng(5)
    longest = 4095 if head_dim == 64 else 1030
    rows = [(int(n), 1) for n in rng.integers(0, longest, 60)] + [(0, 1), (15, 1), (16, 1), (longest, 1)]
    q, pages, table, attn = _paged_case(rows, heads, kv_heads, head_dim, 16, dtype, seed=9, max_seqs=64)
    scale = head_dim ** -0.5
    want = PLAIN.paged_attention(q.double(), pages.double(), table, attn, 16, scale, 0)
    got = hip.paged_attention(q, pages, table, attn, 16, scale, 0)
    assert H.op_budget_usage(got, want, dtype, head_dim + longest) <= 1
    attn.max_decode_len = 1 << (longest).bit_length()                   # the bucket's length, not the rows'
    assert H.op_budget_usage(hip.paged_attention(q, pages, table, attn, 16, scale, 0), want, dtype,
                             head_dim + longest) <= 1
    lens = attn.lens.clone()
    lens[53:] = 0                                                       # rows that hold nothing give zeros
    attn.lens = lens
    got = hip.paged_attention(q, pages, table, attn, 16, scale, 0)
    assert not got[53:].any() and H.op_budget_usage(got[:53], want[:53], dtype, head_dim + longest) <= 1


@pytest.mark.parametrize("geometry", [(32, 8, 128), (64, 8, 128), (16, 8, 64), (16, 4, 256), (40, 1, 128), (7, 7, 64)])
@pytest.mark.parametrize("norm,rope", [(True, True), (False, True), (True, False), (False, False)])
def test_decode_attention_from_the_raw_projection(hip, geometry, norm, rope):
    """A step of decode rows alone, from the raw q/k/v projection: per-head norm, rotation and the cache write of each
    row's new token inside the attention kernel, against the three operations one after the other in float64. The
    cache afterwards holds what the separate write would have stored (every page compared: nothing else is touched),
    the rest of each row's last page holds NaN (the new key is read back, its neighbours never), rows differ in
    length (one key, page edges, thousands), one row holds nothing, and a window."""
    from holon_amd.parts.positions import rope_table
    heads, kv_heads, head_dim = geometry
    bf, page = torch.bfloat16, 16
    for seed, (starts, window) in enumerate((([0, 15, 16, 99, 1000, 4100, 31], 0), ([0, 5, 300, 2049], 64))):
        rows = [(s0, 1) for s0 in starts]
        _, pages, table, attn = _paged_case(rows, heads, kv_heads, head_dim, page, bf, seed=40 + seed)
        t = len(rows)
        held = torch.zeros(pages.shape[0], page, dtype=torch.bool)
        wp, wo = [], []
        for slot, (s0, _) in zip(attn.slots.tolist(), rows):
            pos = torch.arange(s0)                                    # the tokens before this step's
            held[table[slot, pos // page].cpu().long(), pos % page] = True
            wp.append(int(table[slot, s0 // page]))
            wo.append(s0 % page)
        kp, vp = pages[:, 0].view(-1, kv_heads, page, head_dim), pages[:, 1].view(-1, kv_heads, head_dim, page)
        free = (~held).cuda()
        kp.masked_fill_(free[:, None, :, None], float("nan"))
        vp.masked_fill_(free[:, None, None, :], float("nan"))
        i32 = lambda a: torch.tensor(a, dtype=torch.int32).cuda()
        wp, wo, pos = i32(wp), i32(wo), i32(starts)
        qkv = _randn(t, (heads + 2 * kv_heads) * head_dim, dtype=bf, seed=50 + seed)
        qw = (_randn(head_dim, dtype=bf, seed=51) + 1) if norm else None
        kw = (_randn(head_dim, dtype=bf, seed=52) + 1) if norm else None
        tab = rope_table(8192, head_dim, 1e4).cuda() if rope else None
        scale = head_dim ** -0.5
        pages_plain = pages.double()
        want = PLAIN.qkv_attention(qkv.double(), heads, kv_heads, head_dim, qw.double() if norm else None,
                                   kw.double() if norm else None, 1e-6, tab, pos, pages_plain, table, wp, wo, attn, page,
                                   scale, window)
        stored = pages.clone()
        ref_q = hip.qk_norm_rope_write(qkv, heads, kv_heads, head_dim, qw, kw, 1e-6, tab, pos, stored, wp, wo, page)
        unfused = hip.paged_attention(ref_q, stored, table, attn, page, scale, window)
        got = hip.qkv_attention(qkv, heads, kv_heads, head_dim, qw, kw, 1e-6, tab, pos, pages, table, wp, wo, attn, page,
                                scale, window)
        assert torch.isfinite(got.float()).all(), (geometry, starts)
        same = (pages == stored) | (pages.isnan() & stored.isnan())
        assert same.all(), "the cache differs from what the separate write stores"
        assert H.op_budget_usage(got, want, bf, head_dim + max(starts) + 1) <= 1, (geometry, starts, window)
        assert H.op_budget_usage(got, unfused.double(), bf, head_dim + max(starts) + 1) <= 1
        attn.lens = attn.lens.clone()
        attn.lens[1] = 0                                              # a row that holds nothing gives zeros, writes nothing
        before = pages.clone()
        got = hip.qkv_attention(qkv, heads, kv_heads, head_dim, qw, kw, 1e-6, tab, pos, pages, table, wp, wo, attn, page,
                                scale, window)
        assert not got[1].any() and ((pages == before) | before.isnan()).all()
        assert H.op_budget_usage(torch.cat((got[:1], got[2:])), torch.cat((want[:1], want[2:])), bf,
                                 head_dim + max(starts) + 1) <= 1


@pytest.mark.parametrize("geometry", [(32, 8, 128), (16, 8, 64), (8, 1, 128), (7, 7, 64), (6, 2, 64), (5, 1, 128),
                                      (24, 1, 64), (32, 1, 128), (40, 1, 128), (66, 1, 64), (80, 2, 64)])
def test_long_prompt_portions_two_tiles_a_wave(hip, geometry):
    """Portions long enough for the kernels that stage keys and values through LDS (tiles of 32 rows, one or two a
    wave, for groups of up to 32 heads; tiles of 16 rows, one or two a wave, for larger groups): one row of 4,500 tokens from position 0, two
    rows continuing earlier tokens (so the keys start before the queries), and a window. Groups of 1, 3, 5, 24, 32
    (tiles that hold one position or several, whole or in part), 40 and 66 heads."""
    heads, kv_heads, head_dim = geometry
    bf = torch.bfloat16
    for rows, window in (([(0, 4500)], 0), ([(300, 4200), (77, 2300)], 0), ([(1000, 4100)], 600)):
        q, pages, table, attn = _paged_case(rows, heads, kv_heads, head_dim, 16, bf, seed=len(rows) + window)
        scale = head_dim ** -0.5
        want = PLAIN.paged_attention(q.double(), pages.double(), table, attn, 16, scale, window)
        # one tile of 32 rows a wave, its stages copied into LDS by the memory pipeline (head_dim 128) or through
        # registers, and two tiles a wave (groups of up to 32 heads)
        for form, direct in ((0, 1), (0, 0), (2, 0)):
            before = hip.lib.holon_attention_prefill_form(form)
            copies = hip.lib.holon_attention_prefill_copies(direct)
            try:
                got = hip.paged_attention(q, pages, table, attn, 16, scale, window)
                again = hip.paged_attention(q, pages, table, attn, 16, scale, window)
            finally:
                hip.lib.holon_attention_prefill_form(before)
                hip.lib.holon_attention_prefill_copies(copies)
            # rows that see few keys are averages of few values and much larger than rows that see thousands: each
            # stretch of rows is held to the budget of its own size and of the keys it sees
            at = 0
            for start, n in rows:
                for lo, hi in ((0, 64), (64, 512), (512, n)):
                    part = slice(at + lo, at + min(hi, n))
                    span = head_dim + (min(window, start + hi) if window else start + min(hi, n))
                    assert H.op_budget_usage(got[part], want[part], bf, span) <= 1, (geometry, rows, window, lo, form, direct)
                at += n
            assert torch.equal(got, again)


@pytest.mark.parametrize("geometry", [(32, 1), (5, 1), (6, 2), (4, 4)])
def test_prompt_portions_of_wide_heads(hip, geometry):
    """Heads of 256 with stages copied into LDS (rows of more than 192 tokens), and straight from the cache: whole prompts, rows
    behind earlier tokens, a window, last stages of 1 to 32 keys; every stretch of rows within the budget of the keys it sees."""
    (heads, kv_heads), bf, head_dim = geometry, torch.bfloat16, 256
    for rows, window in (([(0, 193)], 0), ([(0, 417), (300, 33)], 0), ([(415, 129), (0, 224), (31, 16)], 100), ([(1000, 17)], 0)):
        q, pages, table, attn = _paged_case(rows, heads, kv_heads, head_dim, 16, bf, seed=len(rows) + window)
        want = PLAIN.paged_attention(q.double(), pages.double(), table, attn, 16, head_dim ** -0.5, window)
        for direct in (1, 0):
            copies = hip.lib.holon_attention_prefill_copies(direct)
            try:
                got = hip.paged_attention(q, pages, table, attn, 16, head_dim ** -0.5, window)
            finally:
                hip.lib.holon_attention_prefill_copies(copies)
            at = 0
            for start, n in rows:
                for lo, hi in ((0, 64), (64, n)):
                    part = slice(at + lo, at + min(hi, n))
                    if lo < n:
                        span = head_dim + (min(window, start + hi) if window else start + min(hi, n))
                        assert H.op_budget_usage(got[part], want[part], bf, span) <= 1, (geometry, rows, window, lo, direct)
                at += n


@pytest.mark.parametrize("head_dim,changed", [(256, False), (128, True)])
def test_prompt_portions_over_staged_keys_and_values_that_are_not_finite(hip, head_dim, changed):
    """Stages copied into LDS: what lies past a row's end, and before the window of all of a portion's tokens, may be anything; a value
    that is not finite among the keys that some tokens see stays out of every tile of 32 rows whose tokens see none of its stage of 32."""
    bf, kv, window, page = torch.bfloat16, 36, 70, 16
    rows = [(0, 401), (333, 300), (37, 201)]
    q, pages, table, attn = _paged_case(rows, kv, kv, head_dim, page, bf, seed=head_dim)
    bias = (torch.rand(kv, generator=torch.Generator().manual_seed(1)).cuda(), torch.rand(kv, generator=torch.Generator().manual_seed(2)).cuda())
    how = dict(softcap=5.0, dist=bias) if changed else {}

    def run(pages, direct):
        was = hip.lib.holon_attention_prefill_copies(direct)
        try:
            return hip.paged_attention(q, pages, table, attn, page, head_dim ** -0.5, window, **how)
        finally:
            hip.lib.holon_attention_prefill_copies(was)
    clean = run(pages, 1)
    assert not torch.equal(clean, run(pages, 0))                      # (the staged form it is)
    bad, slots = pages.clone(), attn.slots.tolist()
    for slot, (start, n) in zip(slots, rows):
        for key in list(range(max(0, start - window + 1) // 32 * 32)) + list(range(start + n, table.shape[1] * page)):
            at = table[slot, key // page]
            bad[at, 0].view(kv, page, head_dim)[:, key % page] = float("nan")
            bad[at, 1].view(kv, head_dim, page)[:, :, key % page] = float("inf")
    assert torch.equal(run(bad, 1), clean)
    ends = np.cumsum([n for _, n in rows])
    for (start, n), end, slot, key in zip(rows, ends, slots, (130, 400, 60)):
        bad = pages.clone()
        bad[table[slot, key // page], 1].view(kv, head_dim, page)[:, 3, key % page] = float("nan")
        got = run(bad, 1)
        first = key // 32 * 32                                         # of the key's stage
        sees = torch.tensor([any(first <= p and p - window < first + 32 for p in range(start + t // 32 * 32, start + min(n, t // 32 * 32 + 32)))
                             for t in range(n)])
        mine = torch.arange(end - n, end)
        assert sees.any() and not sees.all()
        assert torch.equal(got[mine[~sees].cuda()], clean[mine[~sees].cuda()]), (start, key)
        others = torch.ones(len(q), dtype=torch.bool)
        others[mine] = False
        assert torch.equal(got[others.cuda()], clean[others.cuda()])
        seen = torch.tensor([start + t >= key > start + t - window for t in range(n)])
        assert got[mine[seen].cuda()][..., 3].isnan().all()


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("window", [1, 7, 16, 100])
def test_paged_attention_window(hip, dtype, window):
    for geometry, page in (((16, 8, 64), 16), ((6, 3, 32), 8), ((32, 8, 128), 16)):
        heads, kv_heads, head_dim = geometry
        q, pages, table, attn = _paged_case(ROWSETS[0] + [(300, 1), (98, 1)], heads, kv_heads, head_dim, page, dtype, 3,
                                            max_seqs=12)
        want = PLAIN.paged_attention(q.double(), pages.double(), table, attn, page, head_dim ** -0.5, window)
        got = hip.paged_attention(q, pages, table, attn, page, head_dim ** -0.5, window)
        assert H.op_budget_usage(got, want, dtype, head_dim + window) <= 1, (geometry, window)


@pytest.mark.parametrize("dtype", DTYPES)
def test_attention_finds_a_far_key(hip, dtype):
    """One key among thousands carries the weight: its query is aligned with it and scaled up. A kernel that skips or
    misplaces a page, a tile edge or the last key shows here."""
    heads, kv_heads, head_dim, page = 8, 2, 64, 16
    for n, target in ((4097, 0), (4097, 4096), (1000, 511), (1000, 512), (2049, 1023), (130, 64), (130, 63)):
        q, pages, table, attn = _paged_case([(n - 1, 1)], heads, kv_heads, head_dim, page, dtype, seed=n + target)
        slot = int(attn.slots[0])
        unit, off = int(table[slot, target // page]), target % page
        kp = pages[:, 0].view(-1, kv_heads, page, head_dim)
        for h in range(heads):
            q[0, h] = kp[unit, h // (heads // kv_heads), off].float().mul(4.0).to(dtype)
        want = PLAIN.paged_attention(q.double(), pages.double(), table, attn, page, head_dim ** -0.5, 0)
        vp = pages[:, 1].view(-1, kv_heads, head_dim, page)
        assert (want[0, 0] - vp[unit, 0, :, off].double()).abs().max() < 0.05       # the test itself singles the key out
        got = hip.paged_attention(q, pages, table, attn, page, head_dim ** -0.5, 0)
        assert H.op_budget_usage(got, want, dtype, head_dim + n) <= 1, (n, target)


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("geometry", [(32, 8, 128, 16), (6, 3, 32, 8), (4, 1, 16, 16), (5, 5, 48, 4), (16, 4, 256, 32)])
def test_fused_norm_rope_write_is_the_three_ops(hip, dtype, geometry):
    from holon_amd.parts.positions import rope_table
    heads, kv_heads, head_dim, page = geometry
    table = rope_table(4096, head_dim, 1e6).cuda()
    rng = np.random.default_rng(0)
    qw, kw = _randn(head_dim, dtype=dtype, seed=9), _randn(head_dim, dtype=dtype, seed=10)
    # few tokens at scattered places; many tokens at consecutive places (whole pages and ragged ends); many scattered
    layouts = [(45, rng.permutation(40 * page)[:45]), (200, np.arange(200) + 3 * page), (130, np.arange(130) + 5),
               (100, rng.permutation(40 * page)[:100]), (300, np.arange(300) + 2 * page + 3),
               (260, rng.permutation(80 * page)[:260])]      # from 256 tokens on a block walks all heads of its token
    for t, where in layouts:
        units = int(where.max()) // page + 2
        qkv = _randn(t, (heads + 2 * kv_heads) * head_dim, dtype=dtype, seed=8)
        pos = torch.as_tensor(rng.integers(0, 4096, t).astype(np.int32)).cuda()
        wp, wo = (torch.as_tensor((where // page).astype(np.int32)).cuda(), torch.as_tensor((where % page).astype(np.int32)).cuda())
        for use_norm, use_rope in ((True, True), (False, True), (True, False), (False, False)):
            pages_h = torch.zeros(units, 2, kv_heads, page * head_dim, dtype=dtype).cuda()
            pages_p = pages_h.clone()
            args = (heads, kv_heads, head_dim, qw if use_norm else None, kw if use_norm else None, 1e-6,
                    table if use_rope else None, pos)
            got = hip.qk_norm_rope_write(qkv, *args, pages_h, wp, wo, page)
            want = PLAIN.qk_norm_rope_write(qkv, *args, pages_p, wp, wo, page)
            assert H.op_budget_usage(got, want, dtype, head_dim) <= 1
            assert H.op_budget_usage(pages_h, pages_p, dtype, head_dim) <= 1
            assert torch.equal(pages_h == 0, pages_p == 0), "a cache entry outside the written ones changed"
            assert torch.equal(pages_h[:, 1], pages_p[:, 1]), "values are copied bit for bit"
    t, where = layouts[0]
    units = 42
    qkv = _randn(t, (heads + 2 * kv_heads) * head_dim, dtype=dtype, seed=8)
    pos = torch.as_tensor(rng.integers(0, 4096, t).astype(np.int32)).cuda()
    wp, wo = (torch.as_tensor((where // page).astype(np.int32)).cuda(), torch.as_tensor((where % page).astype(np.int32)).cuda())
    # queries only (a run that reads another run's cache)
    got = hip.qk_norm_rope_write(qkv, heads, kv_heads, head_dim, qw, kw, 1e-6, table, pos, None, None, None, page)
    want = PLAIN.qk_norm_rope_write(qkv, heads, kv_heads, head_dim, qw, kw, 1e-6, table, pos, None, None, None, page)
    assert H.op_budget_usage(got, want, dtype, head_dim) <= 1
    # the unfused write
    k, v = _randn(t, kv_heads, head_dim, dtype=dtype, seed=11), _randn(t, kv_heads, head_dim, dtype=dtype, seed=12)
    pages_h, pages_p = torch.zeros_like(pages_h), torch.zeros_like(pages_p)
    hip.kv_write(k, v, pages_h, wp, wo, page)
    PLAIN.kv_write(k, v, pages_p, wp, wo, page)
    assert torch.equal(pages_h, pages_p)


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("geometry", [(32, 8, 128, 16), (16, 4, 256, 32), (6, 2, 64, 16)])
def test_values_of_many_tokens_are_written_16_tokens_a_block(hip, dtype, geometry):
    """From 256 tokens on, the norm + rotation + write kernel's launch has blocks behind the tokens' own that write the
    values, 16 tokens of one kv head each, transposed through LDS: whole groups inside one page, groups that straddle
    pages or start off a multiple of 8, a ragged last group, scattered places. Values bit for bit, nothing else touched,
    queries and keys within the budget."""
    from holon_amd.parts.positions import rope_table
    heads, kv_heads, head_dim, page = geometry
    table = rope_table(4096, head_dim, 1e6).cuda()
    rng = np.random.default_rng(1)
    qw, kw = _randn(head_dim, dtype=dtype, seed=9), _randn(head_dim, dtype=dtype, seed=10)
    for t, where in ((530, np.arange(530) + page + 5), (1040, np.arange(1040) + 2 * page),
                     (257, rng.permutation(60 * page)[:257]), (300, np.arange(300) * 2)):
        units = int(where.max()) // page + 2
        qkv = _randn(t, (heads + 2 * kv_heads) * head_dim, dtype=dtype, seed=t)
        pos = torch.as_tensor(rng.integers(0, 4096, t).astype(np.int32)).cuda()
        wp, wo = (torch.as_tensor((where // page).astype(np.int32)).cuda(), torch.as_tensor((where % page).astype(np.int32)).cuda())
        pages_h = torch.zeros(units, 2, kv_heads, page * head_dim, dtype=dtype).cuda()
        pages_p = pages_h.clone()
        got = hip.qk_norm_rope_write(qkv, heads, kv_heads, head_dim, qw, kw, 1e-6, table, pos, pages_h, wp, wo, page)
        want = PLAIN.qk_norm_rope_write(qkv, heads, kv_heads, head_dim, qw, kw, 1e-6, table, pos, pages_p, wp, wo, page)
        assert torch.equal(pages_h[:, 1], pages_p[:, 1]), (geometry, t, "values are copied bit for bit")
        assert torch.equal(pages_h == 0, pages_p == 0), "a cache entry outside the written ones changed"
        assert H.op_budget_usage(got, want, dtype, head_dim) <= 1
        assert H.op_budget_usage(pages_h[:, 0], pages_p[:, 0], dtype, head_dim) <= 1


@pytest.mark.parametrize("dtype", DTYPES)
def test_linear(hip, dtype):
    # up to 16 rows the few-row kernel runs (bfloat16, K >= 256), above that the vendor library's product
    for t, k, n in ((1, 4096, 6144), (8, 4096, 1000), (17, 100, 333), (64, 12288, 4096), (300, 120, 1000), (2, 96, 384),
                    (1, 4096, 4096), (16, 12288, 4096), (3, 4096, 24576), (9, 512, 208), (33, 1024, 4096),
                    (48, 4096, 512), (5, 12288, 151936 // 8), (65, 4096, 512),
                    (1, 8192, 5120), (12, 4096, 8192),                   # 320 and 512 tiles: two tiles a block
                    (5, 512, 80_000), (12, 512, 80_000), (16, 256, 65_568)):  # a vocabulary's worth: two from ten rows up
        x, w = _randn(t, k, dtype=dtype, seed=13), _randn(n, k, dtype=dtype, seed=14, scale=0.05)
        want = x.double() @ w.double().T
        got = hip.linear(x, w)
        assert got.dtype == dtype and H.op_budget_usage(got, want, dtype, k) <= 1, (t, k, n)
        got32 = hip.linear(x, w, torch.float32)
        assert got32.dtype == torch.float32 and H.op_budget_usage(got32, want, dtype, k) <= 1
        assert torch.equal(got32, got.float())         # one rule for every number of rows: the product, then the cast
        tiled = hip.tile_weight(w)
        assert (tiled is None) == (dtype != torch.bfloat16 or n % 16 != 0 or k % 32 != 0 or k < 256)
        if tiled is not None:                          # the tile layout is a permutation: the same bits come out
            assert torch.equal(hip.linear(x, w, None, tiled), got)
            assert torch.equal(hip.linear(x, w, torch.float32, tiled), got32)
    # exact arithmetic: activations in {-1, 0, 1} and weights in {-1, 0, 1} / 8 make every partial sum exact, so any
    # order of summation gives the same bits (plugins/tests/test_attention_kv_quant.py:244-261)
    g = torch.Generator().manual_seed(15)
    x = torch.randint(-1, 2, (5, 512), generator=g).to(dtype).cuda()
    for n in (200, 208, 4096):
        w = (torch.randint(-1, 2, (n, 512), generator=g).float() / 8).to(dtype).cuda()
        assert torch.equal(hip.linear(x, w).float(), x.float() @ w.float().T)
    # a row's result does not depend on the rows beside it, beyond rounding
    x = _randn(64, 4096, dtype=dtype, seed=16)
    w = _randn(512, 4096, dtype=dtype, seed=17, scale=0.02)
    assert H.op_budget_usage(hip.linear(x[:1].contiguous(), w), hip.linear(x, w)[:1].float(), dtype, 4096) <= 1


def test_product_for_17_to_64_rows_over_many_tiles(hip):
    """Steps of 17 to 64 rows over weights with at least 1,024 tiles of 16 rows read the tiled copy through the kernel
    that shares the rows through LDS: plain, with a float32 result (the bfloat16 one cast up), and gated; against
    float64 and against the same product over the rows as they are. A row's result is bit for bit the same whatever
    rows lie beside it, and fewer tiles, other row counts and other K stay where they were."""
    bf = torch.bfloat16
    for m, k, n in ((17, 256, 16384), (64, 4096, 24576), (33, 1024, 16512), (48, 512, 65536), (64, 768, 65664), (20, 256, 131072)):
        x, w = _randn(m, k, dtype=bf, seed=80), _randn(n, k, dtype=bf, seed=81, scale=0.05)
        tiled = hip.tile_weight(w)
        timed = hip.configured("timed")
        assert timed.serves_rows(m, w, tiled)                                          # outside an engine's start: untimed, ours
        assert timed.plan.how == {f"rows:{n}x{k}:{32 if m <= 32 else 64}": "untimed"}
        timed = hip.configured("timed")
        timed.plan.resolving = True                                                    # as while an engine starts: timed once
        timed.serves_rows(m, w, tiled)
        bucket = 32 if m <= 32 else 64
        assert timed.plan.how == {f"rows:{n}x{k}:{bucket}": "timed"} and timed.plan.seconds > 0
        assert timed.plan.report()[f"rows:{n}x{k}:{32 if m <= 32 else 64}"] in ("rows", "vendor")
        assert not hip.configured("vendor").serves_rows(m, w, tiled)
        assert hip.serves_rows(m, w, tiled) and not hip.serves_rows(16, w, tiled) and not hip.serves_rows(65, w, tiled)
        want = x.double() @ w.double().T
        got = hip.linear(x, w, None, tiled)
        assert got.dtype == bf and H.op_budget_usage(got, want, bf, k) <= 1, (m, k, n)
        assert H.op_budget_usage(got, hip.linear(x, w).double(), bf, k) <= 1          # the vendor library's, over the rows
        assert torch.equal(hip.linear(x, w, torch.float32, tiled), got.float())
        fewer = hip.linear(x[3:21].contiguous(), w, None, tiled)                       # 18 rows, other places
        assert torch.equal(fewer, got[3:21]) if m >= 21 else True
    for m, k, inter in ((64, 4096, 12288), (17, 256, 8192), (40, 1024, 8320), (33, 512, 16384), (64, 768, 16512)):   # the last two: eight waves a block
        x, w = _randn(m, k, dtype=bf, seed=82), _randn(2 * inter, k, dtype=bf, seed=83, scale=0.05)
        tiled = hip.tile_weight(w)
        assert hip.serves_rows(m, w, tiled, gated=True)
        pinned = hip.configured("own", {f"glu:{2 * inter}x{k}:{32 if m <= 32 else 64}": "vendor"})
        assert not pinned.serves_rows(m, w, tiled, gated=True) and pinned.plan.how.popitem()[1] == "pinned"
        exact = PLAIN.silu_mul(PLAIN.linear(x.double(), w.double()))
        got = hip.linear_silu_mul(x, w, tiled)
        assert got is not None and got.shape == (m, inter) and H.op_budget_usage(got, exact, bf, k) <= 1, (m, k, inter)
        two = hip.silu_mul(hip.linear(x, w))                                           # the same roundings in two kernels
        assert (got != two).float().mean() < 0.02
    w = _randn(4096, 4096, dtype=bf, seed=84)
    tiled = hip.tile_weight(w)
    assert not hip.serves_rows(32, w, tiled) and not hip.serves_rows(32, w, None)      # 256 tiles: the vendor library's
    w = _randn(16384, 384, dtype=bf, seed=85)
    assert not hip.serves_rows(32, w, hip.tile_weight(w))                              # K no multiple of 256


def test_product_in_shares_of_k_for_narrow_weights(hip):
    """Steps of 17 to 64 rows over narrow weights (a few hundred tiles: output and down projections) may have K split
    over blocks: float32 sums of every share, which the residual add + norm kernel (or `sum_parts`) adds up in order.
    Every share against float64 over its columns; the sum, rounded once, against the whole product; the norm that
    reads the parts against the norm over their rounded sum (the residual rows bit for bit), in both of its kernels
    (rows of 1,024 values and more, and narrower ones); a row's result whatever rows lie beside it; and the timed
    choice."""
    from holon_amd.kernels.hip import KernelError
    bf = torch.bfloat16
    for m, k, n in ((64, 4096, 4096), (17, 12288, 4096), (33, 1024, 5120), (48, 25600, 5120), (40, 512, 320), (64, 256, 64),
                    (65, 4096, 4096), (100, 12288, 4096), (128, 1024, 5120), (90, 256, 64), (113, 2560, 1024)):
        x, w = _randn(m, k, dtype=bf, seed=90), _randn(n, k, dtype=bf, seed=91, scale=0.05)
        tiled = hip.tile_weight(w)
        splits = hip.lib.holon_gemm_rows_splits(m, n, k)
        assert splits in (2, 4, 8) and k % (128 * splits) == 0, (m, k, n, splits)
        parts = hip._rows_parts(x, w, tiled, splits)
        assert parts.shape == (splits, m, n) and parts.dtype == torch.float32
        share = k // splits
        for s in range(splits):
            want = x[:, s * share:(s + 1) * share].double() @ w[:, s * share:(s + 1) * share].double().T
            assert H.op_budget_usage(parts[s], want, torch.float32, share) <= 1, (m, k, n, s)
        total = hip.sum_parts(parts)
        in_order = parts[0].clone()
        for s in range(1, splits):
            in_order += parts[s]
        assert torch.equal(total, in_order.to(bf))
        assert H.op_budget_usage(total, x.double() @ w.double().T, bf, k) <= 1
        assert H.op_budget_usage(total, hip.linear(x, w).double(), bf, k) <= 1           # the vendor library's product
        fewer = hip._rows_parts(x[3:21].contiguous(), w, tiled, splits) if m >= 21 else None
        assert fewer is None or torch.equal(fewer, parts[:, 3:21])
        weight, eps = _randn(n, dtype=bf, seed=92) + 1, 1e-5
        res_a, res_b = _randn(m, n, dtype=bf, seed=93), _randn(m, n, dtype=bf, seed=93)
        normed_a = hip.add_rmsnorm(parts, res_a, weight, eps)                             # reads the parts itself
        normed_b = hip.add_rmsnorm(total, res_b, weight, eps)
        assert torch.equal(res_a, res_b), (m, k, n)                                       # the same sums, bit for bit
        assert H.op_budget_usage(normed_a, normed_b.double(), bf, 1) <= 1, (m, k, n)      # (squares summed in another order)
        plain_res = _randn(m, n, dtype=bf, seed=93)
        plain_normed = PLAIN.add_rmsnorm(parts, plain_res, weight, eps)                   # the twin takes parts as well
        assert torch.equal(plain_res, res_a) and H.op_budget_usage(normed_a, plain_normed.double(), bf, 1) <= 1
    x, w = _randn(32, 4096, dtype=bf, seed=94), _randn(4096, 4096, dtype=bf, seed=95, scale=0.05)
    tiled = hip.tile_weight(w)
    timed = hip.configured("timed")
    timed.plan.resolving = True
    got = timed.linear_parts(x, w, tiled)                                                 # timed once, then kept
    assert timed.plan.report()["parts:4096x4096:32"] in ("parts", "vendor")
    assert (got is None) == (timed.plan.report()["parts:4096x4096:32"] == "vendor")
    assert hip.configured("vendor").linear_parts(x, w, tiled) is None
    assert hip.configured("vendor", {"parts:4096x4096:32": "parts"}).linear_parts(x, w, tiled).shape == (8, 32, 4096)
    assert hip.linear_parts(x, w, tiled).shape == (8, 32, 4096)
    assert hip.linear_parts(x[:16].contiguous(), w, tiled) is None and hip.linear_parts(x, w, None) is None
    assert hip.linear_parts(_randn(129, 4096, dtype=bf, seed=99), w, tiled) is None            # beyond 128 rows, K < 2 N
    assert hip.linear_parts(_randn(32, 4096, dtype=torch.float32, seed=96), w.float(), tiled) is None          # float32 rows: not this path
    w = _randn(4096, 4224, dtype=bf, seed=97)                                             # K = 33 x 128: no equal shares
    assert hip.linear_parts(_randn(32, 4224, dtype=bf, seed=98), w, hip.tile_weight(w)) is None
    with pytest.raises(KernelError):
        hip._rows_parts(x, w[:, :4096].contiguous(), tiled, 3)                            # 4096 / 128 = 32 chunks, not by 3
    with pytest.raises(KernelError):
        hip._rows_parts(x.cpu(), w[:, :4096].contiguous(), tiled, 8)
    with pytest.raises(KernelError):
        hip.add_rmsnorm(torch.zeros(8, 32, 4000, device="cuda"), _randn(32, 4096, dtype=bf), _randn(4096, dtype=bf), 1e-5)


def test_choices_are_timed_over_the_same_shaped_weights_of_other_layers(hip):
    """Every weight that got a tiled copy is known by shape (weakly: a weight that is gone is forgotten), and a timing
    calls its candidates on them in turn, the given one first, up to 16 of them or a gigabyte: one weight called over
    and over would be read from the memory-side cache, which a step's weights never are."""
    import gc
    bf = torch.bfloat16
    ws = [_randn(2048, 512, dtype=bf, seed=300 + i) for i in range(5)]
    ts = [hip.tile_weight(w) for w in ws]
    pairs = hip._alike(ws[2], ts[2])
    assert pairs[0][0] is ws[2] and pairs[0][1] is ts[2] and len(pairs) == 5
    assert {id(w) for w, _ in pairs} == {id(w) for w in ws} and all(t is ts[[id(x) for x in ws].index(id(w))] for w, t in pairs)
    assert all(t is None for _, t in hip._alike(ws[0], None)) and len(hip._alike(ws[0], None)) == 5
    assert len(hip._alike(ws[0], ts[0], most=3)) == 3 and len(hip._alike(ws[0], ts[0], most_bytes=2 * 2048 * 512 * 2)) == 2
    folded = hip.tile_weight(ws[1], _randn(512, dtype=bf, seed=310))      # a new copy of a known weight replaces the old
    assert [t for w, t in hip._alike(ws[0], ts[0]) if w is ws[1]] == [folded]
    del pairs, ws[3:], ts[3:]
    gc.collect()
    assert len(hip._alike(ws[0], ts[0])) == 3
    calls = hip._in_turn(hip._alike(ws[0], ts[0]), lambda w, t: (w, t))
    assert len(calls) == 9 and calls[0]()[0] is ws[0] and calls[3]()[0] is ws[0]          # three rounds over three weights
    assert {id(c()[0]) for c in calls[:3]} == {id(w) for w in ws}
    x = _randn(32, 512, dtype=bf, seed=311)
    ms = hip._graph_time(hip._in_turn(hip._alike(ws[0], ts[0]), lambda w, t: torch.matmul(x, w.t())))
    assert 0 < ms < 5


def test_vendor_product_forms_for_steps_of_17_to_64_rows(hip):
    """Steps of 17 to 64 bfloat16 rows (over deep weights also prompt portions of up to 1,024 rows) take the vendor
    library's product in the fastest of three forms, timed once per weight shape and row bucket: each is the product
    rounded once, whichever is kept, and the float32 output is the bfloat16 one cast up."""
    bf = torch.bfloat16
    for m, k, n in ((32, 25600, 5120), (24, 4096, 6144), (64, 1024, 512), (300, 25600, 5120), (1000, 8192, 512)):
        x, w = _randn(m, k, dtype=bf, seed=70), _randn(n, k, dtype=bf, seed=71, scale=0.02)
        want = x.double() @ w.double().T
        key = f"vendor:{n}x{k}:{32 if m <= 32 else 1 << (m - 1).bit_length()}"
        timed = hip.configured("timed")
        timed.plan.resolving = True
        got = timed.linear(x, w)
        assert timed.plan.report()[key] in ("bf16", "f32", "f32x2")       # timed and kept
        for form in ("bf16", "f32", "f32x2"):
            y = hip.configured("own", {key: form}).linear(x, w)
            assert y.dtype == bf and H.op_budget_usage(y, want, bf, k) <= 1, (m, k, n, form)
            assert torch.equal(hip.configured("own", {key: form}).linear(x, w, torch.float32), y.float())
        assert torch.equal(hip.linear(x, w), hip.configured("vendor").linear(x, w))          # both: the plain form
        assert H.op_budget_usage(got, want, bf, k) <= 1
    timed = hip.configured("timed")
    timed.plan.resolving = True
    timed.linear(_randn(300, 4096, dtype=bf, seed=72), _randn(512, 4096, dtype=bf, seed=73))    # a shallow weight, and
    timed.linear(_randn(1025, 8192, dtype=bf, seed=74), _randn(512, 8192, dtype=bf, seed=75))   # more rows: no choice
    assert timed.plan.report() == {}


def test_float32_product_is_true_32_bit_and_its_order_is_fixed(hip):
    """The 32-bit path's own product: close to the float64 product as only true float32 arithmetic is (a
    reduced-precision matrix mode would be a thousand times off), at odd sizes (K no multiple of 4 or 32, N and M
    off the tile edges), and bit for bit independent of the rows beside a row and of the row's place in the batch."""
    f32 = torch.float32
    for m, k, n in ((1, 64, 256), (5, 30, 97), (33, 33, 65), (70, 200, 120), (64, 4096, 64), (130, 72, 1000),
                    (3, 12288, 4096), (257, 4096, 192)):
        x, w = _randn(m, k, dtype=f32, seed=40), _randn(n, k, dtype=f32, seed=41, scale=0.05)
        got, want = hip.linear(x, w), x.double() @ w.double().T
        assert got.dtype == f32 and H.op_budget_usage(got, want, f32, k) <= 1, (m, k, n)
        rel = ((got.double() - want).abs().max() / want.abs().max()).item()
        assert rel < 2e-6 * max(1.0, (k / 64) ** 0.5), (m, k, n, rel)            # bfloat16 or tf32 operands give 1e-3
        rows = torch.tensor(sorted({0, m // 2, m - 1}))
        alone = hip.linear(x[rows.cuda()].contiguous(), w)                        # other company, other places
        assert torch.equal(alone, got[rows.cuda()]), (m, k, n)
        if m > 1:
            shifted = hip.linear(torch.cat((x[-1:], x)).contiguous(), w)          # every row one place further down
            assert torch.equal(shifted[1:], got), (m, k, n)
    x = torch.randint(-1, 2, (7, 100), generator=torch.Generator().manual_seed(42)).float().cuda()
    w = (torch.randint(-1, 2, (50, 100), generator=torch.Generator().manual_seed(43)).float() / 8).cuda()
    assert torch.equal(hip.linear(x, w), x @ w.T)                                 # exact arithmetic: any order, same bits


@pytest.mark.parametrize("m", (16, 17, 33, 64, 65, 96, 130, 300))
def test_float32_product_across_its_tiles(hip, m):
    """Every tile the float32 product chooses between, at the edges of its rows, columns, shares and chunks of K: against
    the float64 product, and each row bit for bit what it is alone. A sum of
    max(64, K / 16 up to a multiple of 32) products a share, then 16 shares (or one of K, where K >= 4,096 and N > K): its error
    stays below that many times 2^-24 sum |x w|."""
    for k, n in ((30, 97), (32, 16), (36, 200), (512, 48), (544, 1000), (2080, 64), (1100, 3072), (256, 16384),
                 (4096, 4096), (4096, 4112), (4101, 4200)):
        x, w = _randn(m, k, dtype=torch.float32, seed=44), _randn(n, k, dtype=torch.float32, seed=45)
        got, want = hip.linear(x, w), x.double() @ w.double().T
        longest = k if k >= 4096 and n > k else max(64, -(-k // 512) * 32) + 16
        bound = longest * 2.0 ** -24 * (x.double().abs() @ w.double().abs().T)
        assert ((got.double() - want).abs() <= bound).all(), (m, k, n)
        for row in (0, 15, m - 1):
            assert torch.equal(hip.linear(x[row: row + 1].contiguous(), w)[0], got[row]), (m, k, n, row)
        odd = torch.empty(m * k + 1, device=x.device)[1:].view(m, k)              # rows that start on no 16-byte border
        odd.copy_(x)
        assert torch.equal(hip.linear(odd, w), got), (m, k, n)


def test_norm_folded_into_the_product(hip):
    """The norm's weight folded into the tiled copy, the rows scaled inside the product from statistics another kernel
    left: against norm then product in float64, within the budget of the two operations; the statistics from the
    residual add's kernel, from the embedding and from `row_sumsq` are the rows' sums of squares; the gated form too."""
    bf = torch.bfloat16
    for m, k, n in ((1, 4096, 6144), (8, 4096, 1024), (16, 512, 208), (5, 12288, 4096), (3, 4096, 24576)):
        h = _randn(m, k, dtype=bf, seed=50, scale=2.0)
        g = (1 + 0.2 * torch.randn(k, generator=torch.Generator().manual_seed(51))).to(bf).cuda()
        w = _randn(n, k, dtype=bf, seed=52, scale=0.05)
        eps = 1e-5
        exact = PLAIN.rmsnorm(h.double(), g.double(), eps) @ w.double().T
        composed = hip.linear(hip.rmsnorm(h, g, eps), w)
        folded = hip.tile_weight(w, g)
        assert hip.folds_norm(m, w, folded)
        stats = hip.row_sumsq(h)
        assert stats.shape == (1, 16)
        assert torch.allclose(stats[0, :m], h.float().pow(2).sum(-1), rtol=1e-5)
        got = hip.linear(h, w, None, folded, row_scale=(stats, eps))
        assert got.dtype == bf and H.op_budget_usage(got, exact, bf, 2 * k) <= 1, (m, k, n)
        assert H.rel_rms(got, exact) <= 1.5 * H.rel_rms(composed, exact) + 1e-4          # no worse than norm, then product
        split = torch.zeros(7, 16, device="cuda")                                      # the same sums in seven parts
        split[:, :m] = (h.float().pow(2).sum(-1) / 7)[None, :]
        assert H.op_budget_usage(hip.linear(h, w, None, folded, row_scale=(split, eps)), exact, bf, 2 * k) <= 1
        got32 = hip.linear(h, w, torch.float32, folded, row_scale=(stats, eps))
        assert torch.equal(got32, got.float())
        if n % 32 == 0 and k % 128 == 0:                                               # the gated form
            want = PLAIN.silu_mul((PLAIN.rmsnorm(h.double(), g.double(), eps) @ w.double().T))
            glu = hip.linear_silu_mul(h, w, folded, row_scale=(stats, eps))
            assert glu.shape == (m, n // 2) and H.op_budget_usage(glu, want, bf, 2 * k) <= 1, (m, k, n)
    # the residual add leaves the statistics of the rows it wrote, one part per 16 columns
    for m, k, n in ((8, 4096, 4096), (1, 12288, 4096), (16, 512, 208), (7, 8192, 5120), (16, 1024, 6144)):
        x, r = _randn(m, k, dtype=bf, seed=53), _randn(m, n, dtype=bf, seed=54)
        w = _randn(n, k, dtype=bf, seed=55, scale=0.05)
        tiled = hip.tile_weight(w)
        want = r.clone()
        assert hip.linear_add(x, w, tiled, want) is True
        stats = hip.linear_add(x, w, tiled, r, want_stats=True)
        assert torch.equal(r, want) and stats.shape == (n // 16, 16)
        assert torch.allclose(stats.sum(0)[:m], r.float().pow(2).sum(-1), rtol=1e-5) and not stats[:, m:].any()
    table = _randn(500, 4096, dtype=bf, seed=56)
    ids = torch.tensor([3, 499, 0, 3, 77], dtype=torch.int32).cuda()
    rows, stats = hip.embedding(ids, table, None, want_stats=True)
    assert torch.equal(rows, table[ids.long()]) and torch.allclose(stats[0, :5], rows.float().pow(2).sum(-1), rtol=1e-5)
    rows, stats = hip.embedding(torch.zeros(40, dtype=torch.int32).cuda(), table, None, want_stats=True)
    assert stats is None                                                               # more rows than a folded norm serves


def test_fused_gate_up_is_the_two_kernels(hip, monkeypatch):
    for m, k, inter in ((1, 4096, 12288), (8, 4096, 12288), (16, 512, 208), (3, 1024, 1024), (5, 256, 48)):
        x = _randn(m, k, dtype=torch.bfloat16, seed=30)
        w = _randn(2 * inter, k, dtype=torch.bfloat16, seed=31, scale=0.05)
        exact = PLAIN.silu_mul(PLAIN.linear(x.double(), w.double()))
        want = hip.silu_mul(hip.linear(x, w))
        assert H.op_budget_usage(want, exact, torch.bfloat16, k) <= 1
        both = []
        for tiled in (None, hip.tile_weight(w)):
            got = hip.linear_silu_mul(x, w, tiled)
            assert got is not None and H.op_budget_usage(got, exact, torch.bfloat16, k) <= 1, (m, k, inter)
            # the same roundings as the two kernels; the sums over K may be split differently
            assert (got != want).float().mean() < 0.02
            both.append(got)
        assert torch.equal(both[0], both[1])           # the tile layout is a permutation of the same reads
    assert hip.linear_silu_mul(_randn(40, 256, dtype=torch.bfloat16), _randn(64, 256, dtype=torch.bfloat16)) is None
    assert hip.linear_silu_mul(_randn(4, 256, dtype=torch.float32), _randn(64, 256, dtype=torch.float32)) is None


def test_product_added_into_the_residual(hip):
    """`linear_add` = the few-row product, rounded, added into the residual, rounded: the bits of the two kernels one
    after the other, since the product is the same kernel's."""
    from holon_amd.kernels.hip import KernelError
    bf = torch.bfloat16
    for m, k, n in ((1, 4096, 6144), (8, 4096, 4096), (16, 12288, 4096), (3, 256, 48), (5, 1024, 208), (2, 4096, 24576)):
        x, w = _randn(m, k, dtype=bf, seed=50), _randn(n, k, dtype=bf, seed=51, scale=0.05)
        tiled = hip.tile_weight(w)
        res = _randn(m, n, dtype=bf, seed=53, scale=2.0)
        exact = res.double() + (x.double() @ w.double().T).to(bf).double()
        want = (res.float() + hip.linear(x, w, None, tiled).float()).to(bf)
        mine = res.clone()
        assert hip.linear_add(x, w, tiled, mine) is True
        assert torch.equal(mine, want), (m, k, n)
        assert H.op_budget_usage(mine, exact, bf, k) <= 1, (m, k, n)
    # what is not served is left to the kernels one after the other, and nothing is touched
    w = _randn(512, 4096, dtype=bf, seed=55, scale=0.02)
    tiled = hip.tile_weight(w)
    res = _randn(17, 512, dtype=bf)
    keep = res.clone()
    assert hip.linear_add(_randn(17, 4096, dtype=bf), w, tiled, res) is False and torch.equal(res, keep)
    assert hip.linear_add(_randn(4, 4096, dtype=bf), w, None, res[:4].contiguous()) is False
    f32 = torch.float32
    assert hip.linear_add(_randn(4, 256, dtype=f32), _randn(64, 256, dtype=f32), None, _randn(4, 64, dtype=f32)) is False
    with pytest.raises(KernelError):
        hip.linear_add(_randn(16, 4096, dtype=bf), w, tiled, _randn(16, 500, dtype=bf))


def test_logprobs_kernel(hip):
    g = torch.Generator().manual_seed(40)
    for rows, vocab, k in ((3, 151_936, 20), (5, 97, 5), (2, 40, 0), (1, 33, 32)):
        logits = (torch.randn(rows, vocab, generator=g) * 3).cuda()
        logits[0, 7] = logits[0, 3] = logits[0].max() + 1                 # a tie at the top: the lower id first
        tokens = torch.randint(0, vocab, (rows,), generator=g).to(torch.int32).cuda()
        lp, ids, top = hip.logprobs(logits, tokens, k)
        want_lp, want_ids, want_top = PLAIN.logprobs(logits.double(), tokens, k)
        assert ids.tolist() == want_ids.tolist()
        torch.testing.assert_close(lp.double(), want_lp.double(), rtol=1e-5, atol=1e-5)
        torch.testing.assert_close(top.double(), want_top.double(), rtol=1e-5, atol=1e-5)


def test_argmax_and_sampling(hip):
    from tests.plain import sampling as S
    g = torch.Generator().manual_seed(20)
    logits = (torch.randn(9, 151_936, generator=g) * 3).cuda()
    logits[3, 777] = logits[3, 90_000] = 50.0                     # a tie: the first index wins
    assert hip.argmax(logits).tolist() == logits.argmax(-1).tolist()
    assert int(hip.argmax(logits)[3]) == 777
    # wide rows are searched in pieces of 4,096: ties across pieces, rows of -inf and of NaN, widths that are no
    # multiple of 4 (or of the piece), a best value at a piece's first and last place
    for rows, vocab in ((3, 16_385), (70, 20_001), (2, 16_384), (5, 9_001)):
        x = torch.randn(rows, vocab, generator=g).cuda()
        x[0, 4095] = x[0, 4096] = x[0, vocab - 1] = 9.0
        x[1, :] = float("-inf")
        x[1, 5000:5003] = float("nan")
        if rows > 2:
            x[2, :] = float("nan")
        if rows > 3:
            x[3, :4100] = float("nan")
            x[3, 4100:] = float("-inf")
            x[4, 8192] = 30.0
        got = hip.argmax(x).tolist()
        want = torch.where(x.isnan(), torch.full_like(x, float("-inf")), x).cpu().argmax(-1).tolist()
        if rows > 2:
            want[2] = 0                        # nothing to choose from: the first token
        if rows > 3:
            want[3] = 4100                     # the first value that is a number
        assert got == want, (rows, vocab, got[:5], want[:5])
        assert got[0] == 4095 and got[1] == 0
    # the law, by counting: one row of 40 logits drawn 100,000 times at consecutive positions
    v, n = 40, 100_000
    row = torch.randn(v, generator=torch.Generator().manual_seed(0)) * 2
    row[7] = row[11]                                              # equal logits straddling a top-k edge
    cases = [(0.7, 0, 1.0, 0.0), (1.0, 5, 1.0, 0.0), (1.0, 0, 0.8, 0.0), (1.3, 0, 1.0, 0.1), (0.9, 12, 0.9, 0.02),
             (1.0, 1, 1.0, 0.0), (1.0, 0, 1e-6, 0.0)]
    for temp, top_k, top_p, min_p in cases:
        f = lambda x, dt: torch.full((n,), x, dtype=dt).cuda()
        tokens = hip.sample(row.expand(n, v).contiguous().cuda(), f(temp, torch.float32), f(top_k, torch.int32),
                            f(top_p, torch.float32), f(min_p, torch.float32), f(1234, torch.int64),
                            torch.arange(n, dtype=torch.int64).cuda())
        freq = torch.bincount(tokens.long().cpu(), minlength=v).double() / n
        p = S.probs(row, temp, top_k, top_p, min_p)
        assert (freq[p == 0] == 0).all(), (temp, top_k, top_p, min_p, "a filtered token was drawn")
        assert 0.5 * (freq - p).abs().sum() < 0.02, (temp, top_k, top_p, min_p)
    # a draw depends on (seed, position) only: not on the row's place in the batch or on the other rows
    logits = torch.randn(6, v, generator=torch.Generator().manual_seed(1)).cuda()
    one = lambda x, dt, r: torch.full((r,), x, dtype=dt).cuda()
    seeds = torch.tensor([100, 101, 102, 103, 100, 101], dtype=torch.int64).cuda()
    pos = torch.tensor([5, 5, 5, 5, 9, 9], dtype=torch.int64).cuda()
    together = hip.sample(logits, one(1.0, torch.float32, 6), one(0, torch.int32, 6), one(1.0, torch.float32, 6),
                          one(0.0, torch.float32, 6), seeds, pos)
    alone = hip.sample(logits[[1, 5]].contiguous(), one(1.0, torch.float32, 2), one(0, torch.int32, 2),
                       one(1.0, torch.float32, 2), one(0.0, torch.float32, 2), seeds[[1, 5]].contiguous(),
                       pos[[1, 5]].contiguous())
    assert together[[1, 5]].tolist() == alone.tolist()
    # the draw is the inverse CDF at the hashed uniform, in vocabulary order, at the full vocabulary
    big = (torch.randn(4, 151_936, generator=g) * 3).cuda()
    toks = hip.sample(big, one(1.0, torch.float32, 4), one(0, torch.int32, 4), one(1.0, torch.float32, 4),
                      one(0.0, torch.float32, 4), one(77, torch.int64, 4), torch.arange(4, dtype=torch.int64).cuda())
    for r in range(4):
        cdf = big[r].double().softmax(-1).cumsum(0).cpu()
        u, t = S.uniform(77, r), int(toks[r])
        assert (cdf[t - 1] if t else 0.0) - 1e-5 <= u < cdf[t] + 1e-5
    # temperature 0 rows take the argmax beside sampled rows
    mixed_t = torch.tensor([0.0, 1.0, 0.0, 1.0], dtype=torch.float32).cuda()
    toks = hip.sample(big, mixed_t, one(0, torch.int32, 4), one(1.0, torch.float32, 4), one(0.0, torch.float32, 4),
                      one(5, torch.int64, 4), torch.arange(4, dtype=torch.int64).cuda())
    assert toks[[0, 2]].tolist() == big[[0, 2]].argmax(-1).tolist()


def test_temperature_divides_the_logits_as_the_reference_does(hip):
    """logit / t and logit * (1 / t) differ in the last place for some values, and with them which of two nearly equal
    logits count as equal at a filter's edge (equal ones go by index). Two such pairs, found by search: one that is a
    tie only under division, one only under multiplication; top-k = 1 then keeps the token the division says
    (std/holon_std/sampling/sampler.py:137 divides)."""
    from tests.plain import sampling as S
    g = torch.Generator().manual_seed(3)
    t = torch.tensor(1.7, dtype=torch.float32)
    inv = torch.tensor(1.0, dtype=torch.float32) / t
    a = torch.rand(200_000, generator=g) * 8 + 4
    b = torch.nextafter(a, torch.tensor(0.0))                        # the float just below
    tie_div, tie_mul = (a / t) == (b / t), (a * inv) == (b * inv)
    only_div, only_mul = int((tie_div & ~tie_mul).nonzero()[0]), int((tie_mul & ~tie_div).nonzero()[0])
    for at, first in ((only_div, 3), (only_mul, 9)):                 # b sits at index 3, a (larger) at index 9
        row = torch.full((1000,), -30.0)
        row[3], row[9] = b[at], a[at]
        f = lambda x, dt: torch.full((16,), x, dtype=dt).cuda()
        got = hip.sample(row.expand(16, 1000).contiguous().cuda(), f(1.7, torch.float32), f(1, torch.int32),
                         f(1.0, torch.float32), f(0.0, torch.float32), f(5, torch.int64), torch.arange(16).cuda())
        assert got.tolist() == [first] * 16, (at, got.tolist())      # a tie: the lower index; no tie: the larger value
        assert int(S.probs(row, 1.7, 1).argmax()) == first and int(PLAIN.sample(
            row[None].cuda(), f(1.7, torch.float32)[:1], f(1, torch.int32)[:1], f(1.0, torch.float32)[:1],
            f(0.0, torch.float32)[:1], f(5, torch.int64)[:1], torch.arange(1).cuda())[0]) == first


def _at_uniform(law, order, token, u, slack=2e-5):
    """Whether `token` is where the inverse CDF of `law`, walked in `order` (None: as it lies), puts the uniform `u`."""
    walk = law if order is None else law[order]
    at = token if order is None else int((order == token).nonzero()[0])
    cdf = walk.cumsum(0)
    return (cdf[at - 1] if at else 0.0) - slack <= u < cdf[at] + slack


def test_sampling_filters_at_the_full_vocabulary(hip):
    """Every draw is the plain sampler's (float64 law, inverse CDF at the hashed uniform, a filtered row walked in
    sorted order) at 151,936 tokens: peaked
    rows whose kept set is small (the fast form: candidates collected and sorted), flat rows and a large k (the
    general form), ties at the edge of top-k and of top-p, k = 1, a tiny top-p."""
    from tests.plain import sampling as S
    v = 151_936
    g = torch.Generator().manual_seed(60)
    peaked = torch.randn(v, generator=g) * 3
    flat = torch.randn(v, generator=g) * 0.3
    tied = peaked.clone()
    order = peaked.argsort(descending=True)
    tied[order[45:55]] = peaked[order[49]]                       # ten equal values around the 50th place
    tied[order[2:5]] = peaked[order[3]]
    plateau = peaked.clone()
    plateau[order[:6000]] = peaked[order[0]]
    coarse = (torch.randn(v, generator=g) * 0.4).round() / 4     # five values, tens of thousands of each; +0 and -0 are one
    assert (coarse == 0).sum() > 50_000 and ((coarse == 0) & coarse.signbit()).sum() > 10_000
    cases = [(peaked, 0.8, 50, 1.0, 0.0), (peaked, 0.8, 0, 0.9, 0.0), (peaked, 1.0, 50, 0.9, 0.02), (peaked, 0.7, 0, 1.0, 0.05),
             (peaked, 1.0, 1, 1.0, 0.0), (peaked, 1.0, 0, 1e-6, 0.0), (peaked, 1.2, 2048, 0.99, 0.0), (peaked, 1.0, 5000, 1.0, 0.0),
             (flat, 1.0, 0, 0.9, 0.0), (flat, 1.0, 300, 0.5, 0.0), (tied, 1.0, 50, 1.0, 0.0), (tied, 1.0, 48, 0.95, 0.0),
             (tied, 0.9, 4, 1.0, 0.0), (tied, 1.0, 0, 0.5, 0.0), (peaked, 1.0, 0, 1.0, 0.0),
             (peaked * 8, 1.0, 50, 1.0, 0.0), (peaked * 8, 1.0, 0, 0.999, 0.0), (peaked * 8, 0.5, 20, 0.9, 0.0),
             (peaked * 40, 1.0, 50, 0.9, 0.0),      # sharp rows: the 50th token lies tens, or hundreds, below the first
             (flat, 1.0, 0, 1.0, 0.2), (peaked, 1.0, 200_000, 1.0, 0.0),   # kept sets too long to collect: min-p alone, all
             (plateau, 1.0, 0, 0.5, 0.0), (plateau, 1.0, 0, 1.0, 0.5), (plateau, 1.0, 7000, 1.0, 0.0),   # 6,000 equal values
             (flat, 0.8, 50, 0.9, 0.0), (flat, 0.8, 20, 0.95, 0.05), (peaked, 1.0, 5000, 0.9, 0.01),    # cuts found by halving
             (plateau, 1.0, 3000, 1.0, 0.0), (peaked * 40, 1.0, 5000, 1.0, 0.0),   # a cut inside equal values; k beyond what weighs
             (coarse, 0.3, 0, 0.9, 0.0), (coarse, 1.0, 0, 0.5, 0.0), (coarse, 1.0, 70_000, 1.0, 0.0), (coarse, 0.3, 0, 1.0, 0.15)]
    n = 48
    for at, (row, temp, top_k, top_p, min_p) in enumerate(cases):
        f = lambda x, dt: torch.full((n,), x, dtype=dt).cuda()
        seed = 900 + at
        tokens = hip.sample(row.expand(n, v).contiguous().cuda(), f(temp, torch.float32), f(top_k, torch.int32),
                            f(top_p, torch.float32), f(min_p, torch.float32), f(seed, torch.int64),
                            torch.arange(n, dtype=torch.int64).cuda()).tolist()
        law = S.probs(row, temp, top_k, top_p, min_p)
        order = S.drawing_order(row, temp, top_k, top_p, min_p)
        assert (order is None) == (top_k == 0 and top_p == 1.0 and min_p == 0.0)
        assert all(law[t] > 0 for t in tokens), (at, "a filtered token was drawn")
        for pos, t in enumerate(tokens):                   # the inverse CDF at the hashed uniform, to float32 rounding
            assert _at_uniform(law, order, t, S.uniform(seed, pos)), (at, pos, t)
        if row is not flat and row is not coarse and top_k < v:   # few tokens carry the mass: a draw then sits well inside its token's share
            want = [S.draw(law, S.uniform(seed, pos), order) for pos in range(n)]
            assert sum(a != b for a, b in zip(tokens, want)) <= 1, (at, temp, top_k, top_p, min_p)
    # rows of one batch with different settings do not disturb each other
    rows = torch.stack([peaked, flat, tied, peaked]).cuda()
    t = torch.tensor([0.8, 1.0, 0.0, 1.0], dtype=torch.float32).cuda()
    k = torch.tensor([50, 0, 0, 1], dtype=torch.int32).cuda()
    p = torch.tensor([1.0, 0.9, 1.0, 1.0], dtype=torch.float32).cuda()
    m = torch.zeros(4, dtype=torch.float32).cuda()
    got = hip.sample(rows, t, k, p, m, torch.full((4,), 5, dtype=torch.int64).cuda(), torch.arange(4).cuda()).tolist()
    assert got[0] == S.draw(S.probs(peaked, 0.8, 50), S.uniform(5, 0), S.drawing_order(peaked, 0.8, 50))
    assert _at_uniform(S.probs(flat, 1.0, 0, 0.9), S.drawing_order(flat, 1.0, 0, 0.9), got[1], S.uniform(5, 1))
    assert got[2] == int(tied.argmax()) and got[3] == int(peaked.argmax())


def test_sampling_under_random_settings(hip):
    """Many rows with settings drawn at random, a row each its own: vocabularies of 1,000 to 33,000, flat to sharp
    rows, every filter alone and together, k beyond what is collected. A drawn token lies in the plain law's kept set
    and at the hashed uniform of the plain CDF."""
    import random
    from tests.plain import sampling as S
    rng = random.Random(7)
    for vocab in (1000, 5003, 33000):
        g = torch.Generator().manual_seed(vocab)
        rows = 48
        scales = [rng.choice([0.3, 1.0, 3.0, 10.0]) for _ in range(rows)]
        logits = torch.randn(rows, vocab, generator=g) * torch.tensor(scales)[:, None]
        temp = [rng.choice([0.3, 0.7, 1.0, 1.5]) for _ in range(rows)]
        top_k = [rng.choice([0, 0, 1, 5, 50, 500, 3000, 5000]) for _ in range(rows)]
        top_p = [rng.choice([1.0, 1.0, 0.99, 0.9, 0.5, 0.1]) for _ in range(rows)]
        min_p = [rng.choice([0.0, 0.0, 0.01, 0.2]) for _ in range(rows)]
        t = lambda v, dt: torch.tensor(v, dtype=dt).cuda()
        got = hip.sample(logits.cuda(), t(temp, torch.float32), t(top_k, torch.int32), t(top_p, torch.float32),
                         t(min_p, torch.float32), t([11] * rows, torch.int64), torch.arange(rows).cuda()).tolist()
        for r in range(rows):
            law = S.probs(logits[r], temp[r], top_k[r], top_p[r], min_p[r])
            case = (vocab, r, scales[r], temp[r], top_k[r], top_p[r], min_p[r])
            assert law[got[r]] > 0, case
            order = S.drawing_order(logits[r], temp[r], top_k[r], top_p[r], min_p[r])
            assert _at_uniform(law, order, got[r], S.uniform(11, r)), case


def test_product_in_shares_of_k_for_prompt_portions(hip):
    """129 to 1,024 rows over a weight whose K is at least twice its N (a feed-forward's second product): blocks of
    128 rows against 256 columns, K in shares. Every share against float64 over its columns, for every number of
    shares the kernel takes; the sum against the whole product and the vendor library's; rows whatever rows lie beside
    them (another number of row blocks); the norm that reads the parts; what the kernel does not take."""
    from holon_amd.kernels.hip import KernelError
    bf = torch.bfloat16
    for m, k, n in ((129, 512, 256), (200, 1024, 512), (512, 12288, 4096), (1000, 2048, 512), (1024, 1536, 768),
                    (300, 25600, 5120), (640, 9728, 2560), (256, 9728, 2560), (400, 9728, 2560)):
        x, w = _randn(m, k, dtype=bf, seed=190), _randn(n, k, dtype=bf, seed=191, scale=0.05)
        tiled = hip.tile_weight(w)
        auto = hip.lib.holon_gemm_tiles_splits(m, n, k)
        assert auto in (0, 1, 2, 4, 8) and (auto > 0 or n <= 512), (m, k, n, auto)    # (0: too few blocks to be worth taking)
        whole = x.double() @ w.double().T
        for splits in (1, 2, 4, 8):
            if not hip.lib.holon_gemm_tiles_parts_supported(m, n, k, splits):
                assert splits != auto
                continue
            parts = hip._rows_parts(x, w, tiled, splits)
            assert parts.shape == (splits, m, n) and parts.dtype == torch.float32
            share = k // splits
            for s in range(splits):
                want = x[:, s * share:(s + 1) * share].double() @ w[:, s * share:(s + 1) * share].double().T
                assert H.op_budget_usage(parts[s], want, torch.float32, share) <= 1, (m, k, n, splits, s)
            total = hip.sum_parts(parts)
            assert H.op_budget_usage(total, whole, bf, k) <= 1
            if splits == (auto or 2):
                assert H.op_budget_usage(total, hip.linear(x, w).double(), bf, k) <= 1       # the vendor library's product
                some = hip._rows_parts(x[5:200].contiguous(), w, tiled, splits) if m >= 200 else None
                assert some is None or torch.equal(some, parts[:, 5:200])
                odd = torch.empty(x.numel() + 1, dtype=bf, device="cuda")[1:].view(x.shape).copy_(x)      # off a border of 16 bytes
                assert torch.equal(hip._rows_parts(odd, w, tiled, splits), parts)
                weight, eps = _randn(n, dtype=bf, seed=192) + 1, 1e-5
                res_a, res_b = _randn(m, n, dtype=bf, seed=193), _randn(m, n, dtype=bf, seed=193)
                normed_a = hip.add_rmsnorm(parts, res_a, weight, eps)
                normed_b = hip.add_rmsnorm(total, res_b, weight, eps)
                assert torch.equal(res_a, res_b), (m, k, n)
                assert H.op_budget_usage(normed_a, normed_b.double(), bf, 1) <= 1, (m, k, n)
    x, w = _randn(512, 12288, dtype=bf, seed=194), _randn(4096, 12288, dtype=bf, seed=195, scale=0.05)
    tiled = hip.tile_weight(w)
    assert hip.linear_parts(x, w, tiled).shape == (8, 512, 4096)                            # mode `own`
    # which of the two kernels of such parts a call takes: 256 x 256 tiles where they serve, these blocks elsewhere
    for m, k, n, whole in ((512, 12288, 4096, True), (256, 9728, 2560, False), (400, 9728, 2560, False), (640, 9728, 2560, True)):
        a, b = _randn(m, k, dtype=bf, seed=199), _randn(n, k, dtype=bf, seed=200, scale=0.05)
        t, splits = hip.tile_weight(b), (hip.lib.holon_gemm_block_parts_splits if whole else hip.lib.holon_gemm_tiles_splits)(m, n, k)
        assert bool(hip.lib.holon_gemm_block_parts_splits(m, n, k)) == whole and splits
        assert torch.equal(hip.linear_parts(a, b, t), hip._rows_parts(a, b, t, splits, whole)), (m, k, n)
    assert hip.configured("vendor").linear_parts(x, w, tiled) is None
    assert hip.configured("vendor", {"parts:4096x12288:512": "parts"}).linear_parts(x, w, tiled).shape == (8, 512, 4096)
    assert hip.linear_parts(_randn(1025, 12288, dtype=bf, seed=196), w, tiled) is None     # beyond 1,024 rows
    wide = _randn(8192, 4096, dtype=bf, seed=197)
    assert hip.linear_parts(_randn(512, 4096, dtype=bf, seed=198), wide, hip.tile_weight(wide)) is None   # K < 2 N
    with pytest.raises(KernelError):
        hip._rows_parts(x, w, tiled, 5)
    with pytest.raises(KernelError):
        hip._rows_parts(x, w[:4000].contiguous(), hip.tile_weight(w[:4000].contiguous()), 4)   # 4,000 columns: no whole blocks


def test_products_of_17_to_47_rows_over_narrow_weights(hip):
    """A block a tile of 16 columns, K over its waves: against float64, results in either type, rows whatever lies beside them, at the
    edges of what the kernel takes; rows that start on no border of 16 bytes."""
    from holon_amd.kernels.hip import KernelError
    bf, served = torch.bfloat16, lambda m, n, k: bool(hip.lib.holon_gemm_rows_supported(m, n, k, 0))     # noqa: E731
    assert [served(m, 2048, 2048) for m in (16, 17, 47, 48, 64)] == [False, True, True, False, False]
    assert [served(32, n, k) for n, k in ((1008, 2048), (1024, 768), (1024, 1280), (4112, 2048), (4096, 2304), (1032, 1280))] == \
        [False, False, True, False, False, False]
    for n, k in ((1024, 1536), (1040, 1280), (4096, 2048), (2064, 1792)):
        w = _randn(n, k, dtype=bf, seed=185, scale=0.05)
        tiled, x = hip.tile_weight(w), _randn(47, k, dtype=bf, seed=186)
        want, whole = x.double() @ w.double().T, hip.linear(x, w, tiled=tiled)
        assert H.op_budget_usage(whole, want, bf, k) <= 1, (n, k)
        for m in (17, 32, 33, 40):
            assert torch.equal(hip.linear(x[:m].contiguous(), w, tiled=tiled), whole[:m]), (m, n, k)
        assert torch.equal(hip.linear(x, w, torch.float32, tiled), whole.float()), (n, k)
        odd = torch.empty(x.numel() + 1, dtype=bf, device="cuda")[1:].view(x.shape).copy_(x)
        assert torch.equal(hip.linear(odd, w, tiled=tiled), whole), (n, k)
        y = torch.empty_like(whole)
        with pytest.raises(KernelError):                                              # (the entry point itself takes no such rows)
            hip._call(hip.lib.holon_gemm_rows_bf16, odd.data_ptr(), tiled.data_ptr(), y.data_ptr(), 47, n, k, 0, hip._stream())


def test_products_on_tiles_of_256_rows(hip):
    """Tiles of 256 x 256 with up to 16 rows more in the last one: a gated first product against float64 (three roundings to bfloat16 of
    2^-9 each: gate and up, the activation, the result) in either activation, products in shares of K against float64 shares; rows whatever
    lies beside them; which calls take them."""
    from holon_amd.kernels.hip import KernelError, glu_block_pays
    bf = torch.bfloat16
    for m, inter, k in ((1, 16, 128), (17, 128, 256), (256, 112, 128), (257, 144, 384), (272, 272, 256), (273, 128, 640), (520, 400, 256),
                        (769, 256, 128)):
        x, w = _randn(m, k, dtype=bf, seed=180), _randn(2 * inter, k, dtype=bf, seed=181, scale=2 * k ** -0.5)
        z = x.double() @ w.double().T
        outs = []
        for act, fn in ((0, torch.nn.functional.silu), (1, lambda v: torch.nn.functional.gelu(v, approximate="tanh"))):
            y = torch.empty(m, inter, dtype=bf, device="cuda")
            hip._call(hip.lib.holon_gemm_block_glu_bf16, x.data_ptr(), w.data_ptr(), y.data_ptr(), m, inter, k, act, hip._stream())
            assert H.rel_rms(y, fn(z[:, :inter]) * z[:, inter:]) < 3 * 2.0 ** -9, (m, inter, k, act)
            outs.append(y)
        one = torch.empty(1, inter, dtype=bf, device="cuda")
        for row in {0, m // 2, m - 1}:
            hip._call(hip.lib.holon_gemm_block_glu_bf16, x[row:].data_ptr(), w.data_ptr(), one.data_ptr(), 1, inter, k, 0, hip._stream())
            assert torch.equal(one[0], outs[0][row]), (m, inter, k, row)
    for m, n, k, splits in ((1, 16, 128, 1), (257, 272, 512, 2), (272, 256, 1024, 8), (300, 512, 768, 3), (520, 256, 256, 1), (529, 48, 512, 4)):
        x, w = _randn(m, k, dtype=bf, seed=182), _randn(n, k, dtype=bf, seed=183, scale=0.05)
        parts = torch.empty(splits, m, n, dtype=torch.float32, device="cuda")
        hip._call(hip.lib.holon_gemm_block_parts_bf16, x.data_ptr(), w.data_ptr(), parts.data_ptr(), m, n, k, splits, hip._stream())
        for s in range(splits):
            part = slice(s * k // splits, (s + 1) * k // splits)
            want = x[:, part].double() @ w[:, part].double().T
            assert H.op_budget_usage(parts[s], want, torch.float32, k // splits) <= 1, (m, n, k, s)
    assert [glu_block_pays(m, 12288, 4096) for m in (128, 520, 600, 768, 1024, 4096)] == [False, True, False, False, True, True]
    x, w = _randn(520, 256, dtype=bf), _randn(2 * 16384, 256, dtype=bf, scale=0.1)
    assert torch.equal(hip.linear_silu_mul(x, w), hip._glu_block(x, w)) and hip.configured("vendor").linear_silu_mul(x, w) is None
    with pytest.raises(KernelError):                                                   # K of whole pairs of chunks alone
        hip._call(hip.lib.holon_gemm_block_parts_bf16, x.data_ptr(), w.data_ptr(), x.data_ptr(), 16, 16, 192, 1, hip._stream())
    with pytest.raises(KernelError):
        hip._call(hip.lib.holon_gemm_block_parts_bf16, x.data_ptr(), w.data_ptr(), x.data_ptr(), 16, 16, 256, 4, hip._stream())


@pytest.mark.parametrize("act", [0, 1])
def test_gated_products_on_tiles_of_256_rows_are_a_product_choice(hip, act):
    """In either activation: the mode `vendor`, a pin of the kind, and a pinned form of the library's product keep that product, at any
    number of rows; what was taken is recorded; mode `timed` times it only where a start does (here against the library's best form,
    K being long enough for one)."""
    x, w = _randn(2048, 256, dtype=torch.bfloat16), _randn(2 * 16384, 256, dtype=torch.bfloat16, scale=0.1)
    for m, bucket in ((520, 768), (2048, 2048)):
        for mode, pins, taken in (("own", {}, "rows"), ("vendor", {}, "vendor"), ("own", {f"glu:32768x256:{bucket}": "vendor"}, "vendor"),
                                  ("vendor", {f"glu:32768x256:{bucket}": "rows"}, "rows"),
                                  ("own", {f"vendor:32768x256:{bucket}": "f32"}, "vendor"), ("timed", {}, "rows")):
            k = hip.configured(mode, pins)
            got = k.linear_glu(x[:m], w, act)
            assert (got is not None) == (taken == "rows"), (m, mode, pins)
            by_rule = m > 1024 and not pins                 # (never timed: recorded only where it is pinned)
            assert k.plan.report() == ({} if by_rule else {f"glu:32768x256:{bucket}": taken}), (m, mode, pins)
            if got is not None and mode == "own":
                assert torch.equal(got, hip._glu_block(x[:m], w, act))
                z = x[:m].double() @ w.double().T
                gate = torch.nn.functional.gelu(z[:, :16384], approximate="tanh") if act else torch.nn.functional.silu(z[:, :16384])
                assert H.rel_rms(got, gate * z[:, 16384:]) < 3 * 2.0 ** -9
    deep = torch.zeros(2 * 16384, 8192, dtype=torch.bfloat16, device="cuda")
    timed = hip.configured("timed")
    timed.plan.resolving = True
    timed.linear_glu(_randn(520, 8192, dtype=torch.bfloat16), deep, act)
    assert timed.plan.how == {"glu:32768x8192:768": "timed"}


def test_kernels_refuse_what_they_do_not_serve(hip):
    from holon_amd.kernels.hip import KernelError
    with pytest.raises(KernelError):
        hip.rmsnorm(torch.zeros(4, 8), torch.ones(8), 1e-6)                         # a CPU tensor: no fallback
    with pytest.raises(KernelError):
        hip.rmsnorm(torch.zeros(4, 8, dtype=torch.float16).cuda(), torch.ones(8, dtype=torch.float16).cuda(), 1e-6)
    q, pages, table, attn = _paged_case([(0, 4)], 2, 1, 12, 16, torch.float32)     # head_dim 12: not a multiple of 8
    with pytest.raises(KernelError, match="head_dim"):
        hip.paged_attention(q, pages, table, attn, 16, 1.0, 0)
    # the products run on raw pointers: an operand off the GPU, or a tiled copy that is not this weight's, is refused
    bf = torch.bfloat16
    w, other = _randn(512, 1024, dtype=bf, seed=1), _randn(256, 1024, dtype=bf, seed=2)
    tiled = hip.tile_weight(w)
    big = _randn(16384, 256, dtype=bf, seed=3)
    for rows, weight in ((4, w), (32, big)):
        with pytest.raises(KernelError):
            hip.linear(torch.zeros(rows, weight.shape[1], dtype=bf), weight, None, hip.tile_weight(weight))   # rows on the CPU
    with pytest.raises(KernelError, match="tiled"):
        hip.linear(_randn(32, 256, dtype=bf), big, None, hip.tile_weight(_randn(8192, 256, dtype=bf)))
    with pytest.raises(KernelError, match="tiled"):
        hip.linear(_randn(4, 1024, dtype=bf), w, None, hip.tile_weight(other))
    with pytest.raises(KernelError, match="tiled"):
        hip.linear_add(_randn(4, 1024, dtype=bf), w, hip.tile_weight(other), _randn(4, 512, dtype=bf))
    with pytest.raises(KernelError):
        hip.linear_add(_randn(4, 1024, dtype=bf), w, tiled, torch.zeros(4, 512, dtype=bf))   # residual on the CPU


def test_nothing_is_collected_while_a_graph_is_recorded():
    """Python's garbage collector is off inside a recording (what a collection destroys may make calls that a recording
    does not allow) and on again behind it, also behind one that fails."""
    import gc

    from holon_amd.kernels.hip import capture
    x = torch.ones(64, device="cuda")
    y = x * 2
    graph = torch.cuda.CUDAGraph()
    assert gc.isenabled()
    with capture(graph):
        assert not gc.isenabled()
        y = x * 2
    assert gc.isenabled()
    for i in range(3):
        x.fill_(float(i))
        graph.replay()
        assert torch.equal(y, torch.full_like(y, 2.0 * i))
    with pytest.raises(RuntimeError, match="stop here"):
        with capture(torch.cuda.CUDAGraph()):
            raise RuntimeError("stop here")
    assert gc.isenabled()


def _moe_few(hip, x, weights, up_t, down_t, experts, ff, shared, gated, shared_weight=False):
    """The two products of a mixture's step of few rows as a model runs them; None where they are not served."""
    from holon_amd.parts.products import ExpertsDown
    act = hip.moe_up_few(x, weights, up_t, down_t, experts, ff, shared, gated, shared_weight=shared_weight)
    return None if act is None else ExpertsDown(hip, act, weights, down_t, experts, ff, shared).alone()


@pytest.mark.parametrize("hidden,experts,ff,shared,top,gated,own_gate", [
    (256, 8, 32, 0, 1, True, False), (384, 8, 160, 64, 2, True, True), (512, 70, 544, 32, 6, False, False),
    (288, 5, 96, 0, 2, False, False), (2048, 8, 2048, 2048, 2, True, True)])
def test_chosen_experts_alone(hip, hidden, experts, ff, shared, top, gated, own_gate):
    """The two products over the chosen experts: bit for bit the products over all experts with the activation between them, and
    against float64 five roundings to bfloat16 (gate, up, their activation, the product, the result), of 2^-9 each at most. No
    row's result depends on the rows beside it."""
    bf, cols = torch.bfloat16, experts * ff + shared
    up_w = _randn((2 if gated else 1) * cols, hidden, dtype=bf, seed=60, scale=hidden ** -0.5)
    down_w = _randn(hidden, cols, dtype=bf, seed=61, scale=ff ** -0.5)
    up_t, down_t = hip.tile_weight(up_w), hip.tile_weight(down_w)
    g = torch.Generator().manual_seed(62)
    for m in (1, 2, 7, 16):
        x = _randn(m, hidden, dtype=bf, seed=63 + m)
        weights = torch.zeros(m, experts + int(own_gate))
        for row in range(m):
            weights[row, torch.randperm(experts, generator=g)[:top]] = torch.rand(top, generator=g) + 0.2
        weights[:, experts:] = 0.7
        if m == 7:
            weights[:, 1:experts] = 0          # one expert or none
        weights = weights.cuda()
        garbage = torch.full((m, cols), float("nan"), dtype=bf, device="cuda")
        del garbage                            # what no row chose must not be read
        got = _moe_few(hip, x, weights, up_t, down_t, experts, ff, shared, gated, shared_weight=own_gate)
        between = hip.moe_gate if gated else hip.moe_relu2
        whole = hip.linear(between(hip.linear(x, up_w, tiled=up_t), weights, ff, shared, shared_weight=own_gate), down_w,
                           tiled=down_t)
        assert torch.equal(got, whole), m
        z = x.double() @ up_w.double().T
        act = torch.nn.functional.silu(z[:, :cols]) * z[:, cols:] if gated else torch.relu(z).square()
        each = weights[:, :experts].double().repeat_interleave(ff, 1)
        last = weights[:, experts:].double() if own_gate else torch.ones(m, 1, dtype=torch.double, device="cuda")
        want = (act * torch.cat((each, last.expand(m, shared)), 1)) @ down_w.double().T
        apart = H.rel_rms(got, want) if want.any() else got.abs().max().item()
        assert apart < 5 * 2.0 ** -9, (m, apart)
        for row in (0, m // 2, m - 1):
            alone = _moe_few(hip, x[row: row + 1].contiguous(), weights[row: row + 1].contiguous(), up_t, down_t, experts, ff, shared,
                             gated, shared_weight=own_gate)
            assert torch.equal(alone[0], got[row]), (m, row)
    assert _moe_few(hip, _randn(17, hidden, dtype=bf), weights, up_t, down_t, experts, ff, shared, gated) is None


@pytest.mark.parametrize("hidden,experts,ff,shared,top,gated,own_gate", [
    (128, 1, 128, 0, 1, True, False), (256, 8, 128, 256, 2, True, True), (384, 5, 384, 0, 3, False, False),
    (640, 70, 128, 128, 6, True, False), (256, 130, 256, 128, 2, False, False), (2048, 8, 1024, 2048, 4, True, True)])
def test_every_expert_over_its_own_rows(hip, hidden, experts, ff, shared, top, gated, own_gate):
    """Against float64 five roundings to bfloat16 (gate, up, their activation, the product, the result), of 2^-9 each at most; and no
    row's result depends on the rows beside it, nor on which tile of its expert's rows it lies in."""
    bf, cols = torch.bfloat16, experts * ff + shared
    up_w = _randn((2 if gated else 1) * cols, hidden, dtype=bf, seed=64, scale=hidden ** -0.5)
    down_w = _randn(hidden, cols, dtype=bf, seed=65, scale=ff ** -0.5)
    g = torch.Generator().manual_seed(66)
    for m in (1, 17, 256, 257, 1030):
        x = _randn(m, hidden, dtype=bf, seed=67 + m)
        weights = torch.zeros(m, experts + int(own_gate))
        for row in range(m):
            weights[row, torch.randperm(experts, generator=g)[:top]] = torch.rand(top, generator=g) + 0.2
        weights[:, experts:] = 0.7
        if m == 257:
            weights[:, 1:experts] = 0          # one expert for all that chose it, none for the others
            weights[3:5] = 0                   # rows of no expert, the shared one's gate closed too
        weights = weights.cuda()
        got = hip.moe_rows(x, weights, up_w, down_w, experts, top, ff, shared, gated, shared_weight=own_gate)
        z = x.double() @ up_w.double().T
        act = torch.nn.functional.silu(z[:, :cols]) * z[:, cols:] if gated else torch.relu(z).square()
        each = weights[:, :experts].double().repeat_interleave(ff, 1)
        last = weights[:, experts:].double() if own_gate else torch.ones(m, 1, dtype=torch.double, device="cuda")
        want = (act * torch.cat((each, last.expand(m, shared)), 1)) @ down_w.double().T
        apart = H.rel_rms(got, want) if want.any() else got.abs().max().item()
        assert apart < 5 * 2.0 ** -9, (m, apart)
        if m == 257 and (own_gate or not shared):
            assert not got[3:5].any()
        for row in {0, m // 2, m - 1}:
            alone = hip.moe_rows(x[row: row + 1].contiguous(), weights[row: row + 1].contiguous(), up_w, down_w, experts, top, ff,
                                 shared, gated, shared_weight=own_gate)
            assert torch.equal(alone[0], got[row]), (m, row)
    assert hip.moe_rows(_randn(4, hidden, dtype=torch.float32), weights[:4], up_w, down_w, experts, top, ff, shared, gated) is None


@pytest.mark.parametrize("op,dtype", [("moe_rows", torch.bfloat16), ("moe_f32", torch.float32)])
def test_rows_that_are_not_finite_among_the_rows_of_an_expert(hip, op, dtype):
    """A row with a NaN or an infinity changes no other row's result, whichever experts they share, and is not finite itself; weights that
    are not finite, or more of them than a row may choose, write nothing out of place."""
    hidden, experts, ff, shared, top = 256, 6, 128, 128, 2
    cols, g = experts * ff + shared, torch.Generator().manual_seed(69)
    up, down = _randn(2 * cols, hidden, dtype=dtype, seed=70, scale=hidden ** -0.5), _randn(hidden, cols, dtype=dtype, seed=71, scale=ff ** -0.5)
    for m in (5, 70, 600):
        x = _randn(m, hidden, dtype=dtype, seed=72 + m)
        weights = torch.zeros(m, experts)
        for row in range(m):
            weights[row, torch.randperm(experts, generator=g)[:top]] = torch.rand(top, generator=g) + 0.2
        weights = weights.cuda()
        run = lambda x, w: getattr(hip, op)(x, w, up, down, experts, top, ff, shared, True)      # noqa: E731
        clean, spoilt, wrong = run(x, weights), x.clone(), weights.clone()
        rows = [1, m // 2, m - 1]
        for row, value in zip(rows, (float("nan"), float("inf"), -float("inf"))):
            spoilt[row, 7] = value
        wrong[rows[0]], wrong[rows[1]] = float("nan"), 0.3
        others = torch.tensor([r for r in range(m) if r not in rows], device="cuda")
        assert torch.isfinite(clean).all()
        got = run(spoilt, weights)
        assert torch.equal(got[others], clean[others]) and not torch.isfinite(got[rows]).all(1).any(), m
        assert torch.equal(run(spoilt, wrong)[others], clean[others]), m


def test_experts_whose_operands_start_on_no_border_of_16_bytes_stay_with_the_products_over_all(hip):
    """The kernels over an expert's own rows read 16 bytes at a time: elsewhere they serve nothing, whichever operand it is."""
    from holon_amd.kernels.hip import KernelError
    for op, dtype in ((hip.moe_rows, torch.bfloat16), (hip.moe_f32, torch.float32)):
        rows, hidden, experts, ff = 64, 128, 4, 128
        weights = torch.zeros(rows, experts, device="cuda")
        weights[:, 0] = 1
        operands = [_randn(n, k, dtype=dtype, seed=68) for n, k in ((rows, hidden), (experts * ff, hidden), (hidden, experts * ff))]
        for at in (None, 0, 1, 2):
            x, up, down = (torch.empty(v.numel() + 1, dtype=dtype, device="cuda")[1:].view(v.shape).copy_(v) if i == at else v
                           for i, v in enumerate(operands))
            assert (op(x, weights, up, down, experts, 1, ff, 0, False) is None) == (at is not None), (dtype, at)
            if at is not None:                     # (the entry points refuse them)
                scratch = [torch.empty(rows * (experts + 2) * (hidden + ff), dtype=dt, device="cuda")
                           for dt in (torch.int32, dtype, torch.float32, dtype)]
                with pytest.raises(KernelError, match="not served"):
                    hip._call(hip.lib.holon_moe_f32 if dtype == torch.float32 else hip.lib.holon_moe_rows_bf16, x.data_ptr(), up.data_ptr(),
                              down.data_ptr(), scratch[3].data_ptr(), scratch[0].data_ptr(), scratch[1].data_ptr(), scratch[2].data_ptr(),
                              rows, hidden, experts, 1, ff, 0, 0, weights.data_ptr(), experts, -1, hip._stream())


@pytest.mark.parametrize("hidden,experts,ff,shared,top,gated,own_gate", [
    (16, 1, 16, 0, 1, True, False), (272, 8, 80, 48, 2, True, True), (400, 5, 384, 0, 3, False, False),
    (128, 70, 32, 16, 6, True, False), (2048, 8, 1024, 2048, 4, False, True)])
def test_float32_experts_over_the_rows_that_chose_them(hip, hidden, experts, ff, shared, top, gated, own_gate):
    """Few rows and many, against float64: sums of K and of the experts' columns in float32, 2^-24 of the larger of the two's shares and
    their additions; a row the same bits alone, in a few and among many."""
    cols = experts * ff + shared
    up_w = _randn((2 if gated else 1) * cols, hidden, dtype=torch.float32, seed=74, scale=hidden ** -0.5)
    down_w = _randn(hidden, cols, dtype=torch.float32, seed=75, scale=ff ** -0.5)
    g = torch.Generator().manual_seed(76)
    for m in (1, 2, 16, 17, 64, 65, 300):
        x = _randn(m, hidden, dtype=torch.float32, seed=77 + m)
        weights = torch.zeros(m, experts + int(own_gate))
        for row in range(m):
            weights[row, torch.randperm(experts, generator=g)[:top]] = torch.rand(top, generator=g) + 0.2
        weights[:, experts:] = 0.7
        if m in (16, 65):
            weights[:, 1:experts] = 0          # one expert for all that chose it, none for the others
            weights[3:5] = 0                   # rows of no expert, the shared one's gate closed too
        weights = weights.cuda()
        got = hip.moe_f32(x, weights, up_w, down_w, experts, top, ff, shared, gated, shared_weight=own_gate)
        z = x.double() @ up_w.double().T
        act = torch.nn.functional.silu(z[:, :cols]) * z[:, cols:] if gated else torch.relu(z).square()
        each = weights[:, :experts].double().repeat_interleave(ff, 1)
        last = weights[:, experts:].double() if own_gate else torch.ones(m, 1, dtype=torch.double, device="cuda")
        want = (act * torch.cat((each, last.expand(m, shared)), 1)) @ down_w.double().T
        apart = H.rel_rms(got, want) if want.any() else got.abs().max().item()
        assert apart < 2e-6, (m, apart)
        for row in {0, m // 2, m - 1}:
            alone = hip.moe_f32(x[row: row + 1].contiguous(), weights[row: row + 1].contiguous(), up_w, down_w, experts, top, ff,
                                shared, gated, shared_weight=own_gate)
            assert torch.equal(alone[0], got[row]), (m, row)
    assert hip.moe_f32(x.bfloat16(), weights, up_w, down_w, experts, top, ff, shared, gated) is None


def test_float32_products_of_few_rows_by_half_tiles(hip):
    """Up to 128 tiles of columns a block takes half a tile: the same bits as whole tiles (a row among more than 16), any K and N."""
    for n, k in ((2048, 2048), (2047, 1000), (9, 31), (16, 64), (24, 4100), (1030, 513)):
        x, w = _randn(17, k, dtype=torch.float32, seed=145), _randn(n, k, dtype=torch.float32, seed=146)
        whole = hip.linear(x, w)
        for m in (1, 5, 16):
            assert torch.equal(hip.linear(x[:m].contiguous(), w), whole[:m]), (m, n, k)


@pytest.mark.parametrize("dtype", DTYPES)
def test_router_of_few_experts(hip, dtype):
    """Both routers up to 64 experts, on either side of 256 rows: the plain form's choice but for rows of a close call, and a
    row alone what it is among others."""
    for experts, top, width, groups, keep in ((1, 1, 40, 1, 1), (8, 2, 2048, 1, 1), (17, 5, 250, 1, 1), (64, 6, 1024, 8, 3),
                                              (12, 4, 37, 6, 2), (64, 64, 128, 64, 64)):
        for rows in (1, 256, 257, 1030):
            x = _randn(rows, width, dtype=dtype, seed=70)
            router = _randn(experts + 1, width, dtype=torch.float32, seed=71, scale=width ** -0.5)
            bias = _randn(experts, dtype=torch.float32, seed=72, scale=0.2)
            from holon_amd.kernels.registry import kernel_op
            cases = [("moe_router", (x, router[:experts], bias, top, groups, keep, 1.7), {}),
                     ("moe_router", (x, router[:experts], None, top, groups, keep, 0.5), {})]
            cases += [("moe_router_top", (x, router, bias, experts, top, groups, keep), dict(score=how))
                      for how in ("softmax", "sigmoid", "sigmoid_squared")]
            for name, args, how in cases:
                op = getattr(hip, name)
                got, want = op(*args, **how), kernel_op(name).plain(*args, **how)
                close = ((got != 0) != (want != 0)).any(1)
                assert close.sum() <= 1 + rows // 500 and torch.allclose(got[~close], want[~close], atol=2e-5), (name, how, experts, rows)
                alone = op(x[-1:].contiguous(), *args[1:], **how)
                assert torch.equal(alone[0], got[-1]), (name, how, experts, rows)


@pytest.mark.parametrize("dtype", DTYPES)
def test_stream_norm_across_its_widths(hip, dtype):
    """The residual sum in float32 and its norm, at the edges of the widths a thread's registers are cut for, with operands on
    and off 16-byte borders and terms of either type."""
    from holon_amd.kernels.registry import kernel_op
    plain = kernel_op("stream_norm").plain
    for dim in (4, 1024, 1028, 2044, 2048, 2052, 4096, 4100, 8192, 8196, 1030):
        weight = 1 + 0.2 * _randn(dim, dtype=dtype, seed=80)
        for kinds in ((), (dtype,), (torch.bfloat16, torch.bfloat16), (torch.float32, torch.bfloat16)):
            for off in (0, 1):
                x = torch.empty(3 * dim + off, device="cuda")[off:].view(3, dim)
                x.copy_(_randn(3, dim, dtype=torch.float32, seed=81))
                terms = [(_randn(3, dim, dtype=kind, seed=82 + i), 0.5 + i) for i, kind in enumerate(kinds)]
                ref = x.double()
                got = hip.stream_norm(x, terms, weight, 1e-5, dtype)
                for term, factor in terms:
                    ref = ref + term.double() * factor
                assert (x.double() - ref).abs().max() <= 4 * 2.0 ** -24 * ref.abs().max() + 1e-6, (dim, kinds)
                want = plain(ref, [], weight.double(), 1e-5, torch.float64)
                assert H.op_budget_usage(got, want, dtype, dim) <= 1, (dim, kinds, off)


@pytest.mark.parametrize("shared", (64, 512))
@pytest.mark.parametrize("gated", (True, False))
def test_a_shared_expert_whose_gate_is_shut(hip, gated, shared):
    """A shared expert's weight of exactly 0 (the sigmoid of anything below -88 or so) for every row of a step, and for some of
    them: bit for bit the products over all experts, whatever the memory of the activations held before."""
    bf, hidden, experts, ff = torch.bfloat16, 256, 4, 96
    cols = experts * ff + shared
    up_w = _randn((2 if gated else 1) * cols, hidden, dtype=bf, seed=90, scale=hidden ** -0.5)
    down_w = _randn(hidden, cols, dtype=bf, seed=91, scale=ff ** -0.5)
    up_t, down_t = hip.tile_weight(up_w), hip.tile_weight(down_w)
    between = hip.moe_gate if gated else hip.moe_relu2
    for m, open_rows in ((1, 0), (3, 0), (16, 0), (1, 1), (16, 5)):
        x = _randn(m, hidden, dtype=bf, seed=92 + m)
        weights = torch.zeros(m, experts + 1)
        weights[:, 1] = 0.4
        weights[:open_rows, experts] = 0.7
        weights = weights.cuda()
        garbage = torch.full((m, cols), float("nan"), dtype=bf, device="cuda")
        del garbage                            # what the next allocation of this size finds
        got = _moe_few(hip, x, weights, up_t, down_t, experts, ff, shared, gated, shared_weight=True)
        whole = hip.linear(between(hip.linear(x, up_w, tiled=up_t), weights, ff, shared, shared_weight=True), down_w,
                           tiled=down_t)
        assert torch.equal(got, whole), (m, open_rows)


@pytest.mark.parametrize("dtype", DTYPES)
def test_general_attention_with_keys_that_are_not_finite(hip, dtype):
    """Keys of NaN and of -inf in different tiles of 64, alone in their tile and among others: a NaN score makes the results of
    every query that sees its key NaN and no others', a score of -inf weighs nothing."""
    page, d, n = 16, 48, 700                    # (48: a size the matrix-core kernels do not serve)
    most = -(-n // page)
    pages = _randn(most, 2, 1, page * d, dtype=dtype, seed=95)
    table = torch.arange(most, dtype=torch.int32, device="cuda")[None]
    i32 = lambda v: torch.tensor(v, dtype=torch.int32, device="cuda")            # noqa: E731
    rows = AttnRows(slots=i32([0]), lens=i32([n]), query_start=i32([0, n]), decode_rows=None, chunk_rows=i32([0]), n_decode=0,
                    n_chunk=1, max_decode_len=0, max_chunk_query=n, max_chunk_len=n)
    q = _randn(n, 2, d, dtype=dtype, seed=96).abs() + 0.1
    for at, count, value in ((64, 1, "nan"), (320, 64, "nan"), (640, 60, "nan"), (699, 1, "nan"), (130, 1, "-inf"),
                             (320, 64, "-inf"), (0, 1, "-inf")):
        held = pages.clone()
        for key in range(at, at + count):
            pages[key // page, 0, 0, key % page * d: (key % page + 1) * d] = float(value)
        got = hip.paged_attention(q, pages, table, rows, page, d ** -0.5, 0).cpu()
        want = TorchKernels().paged_attention(q.float().cpu(), pages.float().cpu(), table.cpu(), AttnRows(
            **{k: v.cpu() if torch.is_tensor(v) else v for k, v in rows.__dict__.items()}), page, d ** -0.5, 0)
        gone = torch.isnan(want)
        assert torch.equal(torch.isnan(got), gone) and gone.any() == (value == "nan" or at == 0), (at, value)
        assert H.rel_rms(got[~gone], want[~gone]) < (1e-5 if dtype == torch.float32 else 1e-2), (at, value)
        pages.copy_(held)


def test_general_attention_with_more_heads_than_a_grid_has_rows(hip):
    """65,537 heads (a grid's second number ends at 65,535), each with keys and values of its own, and 131,074 on as many pairs."""
    page, d = 4, 8
    i32 = lambda v: torch.tensor(v, dtype=torch.int32, device="cuda")            # noqa: E731
    rows = AttnRows(slots=i32([0]), lens=i32([3]), query_start=i32([0, 1]), decode_rows=i32([0]), chunk_rows=None, n_decode=1,
                    n_chunk=0, max_decode_len=3, max_chunk_query=0, max_chunk_len=0)
    for heads, kv in ((65537, 65537), (131074, 65537)):
        pages, q = _randn(1, 2, kv, page * d, dtype=torch.float32, seed=97), _randn(1, heads, d, dtype=torch.float32, seed=98)
        args = (torch.zeros(1, 1, dtype=torch.int32, device="cuda"), rows, page, 0.5, 0)
        assert H.rel_rms(hip.paged_attention(q, pages, *args), TorchKernels().paged_attention(q, pages, *args)) < 1e-5


@pytest.mark.parametrize("dim", (1028, 2052, 4100))
def test_stream_norm_of_rows_within_a_tensor(hip, dim):
    """Rows of bfloat16 whose width is a multiple of 4 and not of 8 (every other one starts on no 16-byte border): each row comes out
    bit for bit the same whichever row a call starts from."""
    bf = torch.bfloat16
    x, weight = _randn(6, dim, dtype=torch.float32, seed=99), 1 + 0.2 * _randn(dim, dtype=bf, seed=100)
    terms = [(_randn(6, dim, dtype=bf, seed=101 + i), 0.5 + i) for i in range(2)]
    whole = x.clone()
    want = hip.stream_norm(whole, terms, weight, 1e-5, bf)
    for at in range(1, 6):
        part = x[at:].clone()
        got = hip.stream_norm(part, [(term[at:], factor) for term, factor in terms], weight, 1e-5, bf)
        assert torch.equal(got, want[at:]) and torch.equal(part, whole[at:]), at


@pytest.mark.parametrize("dtype", DTYPES)
def test_routers_wherever_their_rows_lie(hip, dtype):
    """Rows that start on no border of 16 bytes or of four values: a token's weights are bit for bit the same in every kernel (up to 256
    rows and more) and wherever its row lies."""
    for width, off in ((1028, 0), (1028, 1), (2052, 2), (1026, 1), (2050, 3)):
        rows, experts, top = 300, 24, 3
        x = torch.empty(rows * width + off, dtype=dtype, device="cuda")[off:].view(rows, width)
        x.copy_(_randn(rows, width, dtype=dtype, seed=110))
        router = _randn(experts + 1, width, dtype=torch.float32, seed=111, scale=width ** -0.5)
        bias = _randn(experts, dtype=torch.float32, seed=112, scale=0.2)
        for op, args, how in ((hip.moe_router, (router[:experts], bias, top, 1, 1, 1.7), {}),
                              (hip.moe_router_top, (router, bias, experts, top, 1, 1), dict(score="softmax"))):
            want = op(x.clone(), *args, **how)
            for first, count in ((0, 300), (1, 299), (1, 256), (7, 257), (3, 1)):
                assert torch.equal(op(x[first: first + count], *args, **how), want[first: first + count]), (width, off, first, count)


def test_few_row_products_with_few_tiles_take_one_a_block(hip):
    """A block owns one tile of 16 columns where there are at most 256, also where K is no multiple of 512 and eight waves share a
    tile (two would leave half the compute units without a block); the results across those sizes against float64."""
    for n, k in ((4096, 11008), (2816, 2816), (1024, 768), (4096, 2304)):
        assert [hip.lib.holon_gemm_skinny_tiles(m, n, k) for m in (1, 8, 16)] == [1, 1, 1], (n, k)
    assert [hip.lib.holon_gemm_skinny_tiles(m, 6144, 4096) for m in (1, 8, 16)] == [2, 2, 2]
    assert [hip.lib.holon_gemm_skinny_tiles(m, 8192, 4096) for m in (1, 8, 16)] == [1, 1, 1]
    for n, k in ((4096, 2816), (4112, 768), (5088, 1280), (5104, 1280), (5120, 1280)):
        x, w = _randn(16, k, dtype=torch.bfloat16, seed=120), _randn(n, k, dtype=torch.bfloat16, seed=121)
        tiled, want = hip.tile_weight(w), x.double() @ w.double().T
        for m in (1, 9, 16):
            got = hip.linear(x[:m].contiguous(), w, tiled=tiled)
            assert H.op_budget_usage(got, want[:m], torch.bfloat16, k) <= 1, (m, n, k)
            assert torch.equal(got, hip.linear(x, w, tiled=tiled)[:m]), (m, n, k)


def test_float32_product_of_short_sums(hip):
    """Rows many enough for 64 x 64 tiles over short K, quarters of K side by side and one after the other: at K's borders against the
    float64 product, each row bit for bit what it is alone; and the time follows K (a block does not walk what is not there)."""
    for k in (1, 31, 32, 33, 64, 65, 100, 128, 255, 256, 257, 320, 512, 700, 768, 1000, 1024, 1056):
        for m, n in ((65, 1100), (300, 1024), (830, 4160)):
            x, w = _randn(m, k, dtype=torch.float32, seed=130), _randn(n, k, dtype=torch.float32, seed=131)
            got, want = hip.linear(x, w), x.double() @ w.double().T
            bound = (max(64, -(-k // 512) * 32) + 16) * 2.0 ** -24 * (x.double().abs() @ w.double().abs().T)
            assert ((got.double() - want).abs() <= bound).all(), (m, k, n)
            for row in (0, m - 1):
                assert torch.equal(hip.linear(x[row: row + 1].contiguous(), w)[0], got[row]), (m, k, n, row)

    def us(k):
        x, w, took = _randn(2048, k, dtype=torch.float32), _randn(8192, k, dtype=torch.float32), []
        for _ in range(8):
            begin, end = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
            begin.record()
            for _ in range(4):
                hip.linear(x, w)
            end.record()
            end.synchronize()
            took.append(begin.elapsed_time(end) * 250)
        return min(took)
    assert us(64) < 0.4 * us(1024)


def test_float32_product_of_long_sums_takes_the_form_that_is_done_first(hip):
    """Some hundred rows over K beyond 4,096 take staged tiles, 32 x 64 a block where 64 x 64 would leave a last round mostly empty, else
    64 x 64 with the quarters of K side by side or one after the other; few rows narrow tiles straight from memory, wide weights one
    running sum. Each of these forms against the float64 product, each row bit for bit what it is alone."""
    form = hip.lib.holon_gemm_f32_form
    assert [form(m, 2048, 18432) for m in (1, 17, 704)] == [0, 0, 6]
    assert [form(704, 2048, 9248), form(500, 3072, 12288), form(300, 4096, 18432), form(2048, 2048, 2048)] == [6, 6, 6, 5]
    assert [form(m, n, k) for m, n, k in ((1, 6144, 4096), (704, 4097, 4096), (704, 4096, 4096))] == [-1, -1, 5]
    # few tiles of weights that come from memory: not staged (back to back over weights in a cache blocks of 32 rows looked as fast)
    assert [form(m, n, k) for m, n, k in ((145, 2048, 2048), (145, 3072, 2048), (92, 4096, 2048), (295, 1024, 2048))] == [3, 3, 3, 3]
    for m, n, k, taken in ((130, 2048, 4608, 3), (400, 2048, 5120, 4), (300, 1056, 9248, 3), (67, 4096, 6150, 3), (500, 3072, 4160, 6)):
        assert form(m, n, k) == taken, (m, n, k)
        x, w = _randn(m, k, dtype=torch.float32, seed=140), _randn(n, k, dtype=torch.float32, seed=141)
        got, want = hip.linear(x, w), x.double() @ w.double().T
        bound = (-(-k // 512) * 32 + 16) * 2.0 ** -24 * (x.double().abs() @ w.double().abs().T)
        assert ((got.double() - want).abs() <= bound).all(), (m, n, k)
        for row in (0, 64, m - 1):
            assert torch.equal(hip.linear(x[row: row + 1].contiguous(), w)[0], got[row]), (m, n, k, row)


@pytest.mark.parametrize("m,n,k,form", [(33, 4160, 64, 6), (825, 16384, 64, 5), (97, 16384, 160, 5), (500, 2100, 288, 6), (705, 16384, 416, 5),
                                        (65, 9248, 512, 6), (705, 3072, 544, 6), (300, 3072, 704, 4), (33, 9248, 800, 4), (825, 3072, 1024, 6),
                                        (97, 4160, 1056, 4), (705, 2049, 2016, 6), (1030, 9248, 2016, 5), (700, 2048, 2048, 6), (300, 2048, 4128, 4)])
def test_float32_products_copied_straight_into_lds(hip, m, n, k, form):
    """Each of the staged forms (blocks of 64 and of 32 rows, the quarters of K side by side where it is long enough for that), edges of
    their tiles, K that ends in each quarter: bit for bit what operands give that pass registers (those off a border of 16 bytes) and what
    a row is alone; against the float64 product."""
    assert hip.lib.holon_gemm_f32_form(m, n, k) == form
    x, w = _randn(m, k, dtype=torch.float32, seed=142), _randn(n, k, dtype=torch.float32, seed=143)
    got, want = hip.linear(x, w), x.double() @ w.double().T
    bound = (max(64, -(-k // 512) * 32) + 16) * 2.0 ** -24 * (x.double().abs() @ w.double().abs().T)
    assert ((got.double() - want).abs() <= bound).all()
    off = torch.empty(m * k + 1, dtype=torch.float32, device="cuda")[1:].view(m, k).copy_(x)
    assert off.data_ptr() % 16 and torch.equal(hip.linear(off, w), got)
    for row in (0, 31, m - 1):
        assert torch.equal(hip.linear(x[row: row + 1].contiguous(), w)[0], got[row]), row


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("heads,kv,d", [(6, 2, 48), (8, 8, 24), (4, 1, 272), (4, 2, 80)])
def test_general_attention_of_short_rows(hip, dtype, heads, kv, d):
    """A block has as many waves as the longest row has tiles of 64 keys, eight at most: rows around the borders at which that
    changes come out bit for bit as with eight waves (a bound that says nothing), within a window of either kind too, and a bound that
    is too short still leaves no key out."""
    page, i32 = 16, lambda v: torch.tensor(v, dtype=torch.int32, device="cuda")            # noqa: E731
    for n, window in ((1, 0), (63, 0), (64, 0), (65, 0), (128, 0), (129, 0), (256, 0), (257, 0), (300, 64), (300, 65), (300, -64), (300, -130)):
        count = -(-300 // n)                    # more blocks than compute units, whatever the heads share
        lens, starts = [n] * count, [n * b for b in range(count + 1)]
        most = -(-n // page)
        pages = _randn(most * count, 2, kv, page * d, dtype=dtype, seed=150)
        table = torch.arange(most * count, dtype=torch.int32, device="cuda").view(count, most)
        q = _randn(n * count, heads, d, dtype=dtype, seed=151)

        def rows(bound):
            return AttnRows(slots=i32(list(range(count))), lens=i32(lens), query_start=i32(starts), decode_rows=None,
                            chunk_rows=i32(list(range(count))), n_decode=0, n_chunk=count, max_decode_len=0, max_chunk_query=n,
                            max_chunk_len=bound)
        got = hip.paged_attention(q, pages, table, rows(n), page, d ** -0.5, window)
        assert torch.equal(got, hip.paged_attention(q, pages, table, rows(1000), page, d ** -0.5, window)), (n, window)
        want = TorchKernels().paged_attention(q.float(), pages.float(), table, rows(n), page, d ** -0.5, window)
        tight = 1e-5 if dtype == torch.float32 else 1e-2
        assert H.rel_rms(got, want) < tight and H.rel_rms(hip.paged_attention(q, pages, table, rows(1), page, d ** -0.5, window), want) < tight


@pytest.mark.parametrize("heads,kv,window,steps", [
    (16, 1, 0, ((0, (540, 530)), (37, (641, 17)), (560, (25, 300)))), (16, 1, 200, ((0, (1030, 97)), (37, (1100, 17)))), (20, 1, 0, ((0, (577, 97)),)),
    (8, 2, 0, ((0, (577, 97)), (490, (130, 300)))), (6, 2, -160, ((0, (2700, 60)),)), (34, 1, 0, ((37, (641, 17)),)), (34, 1, 128, ((0, (1100, 17)),)),
    (3, 3, 0, ((0, (641, 500)),)), (3, 3, 128, ((0, (5600, 40)),)), (3, 3, 513, ((600, (5600, 900)),)),
    (16, 1, 1024, ((1200, (304, 25)), (1500, (17, 20)))), (32, 8, -768, ((900, (300, 17)),)), (34, 1, 600, ((700, (65, 20)),))])
def test_heads_of_256_staged_are_the_bits_of_short_portions(hip, heads, kv, window, steps):
    """Two prompts in one step that takes its stages through LDS, behind cached tokens or not: every row bit for bit what portions give
    that are too short for it, under sinks and windows of either kind, whatever later tokens' values are."""
    d, page, bf = 256, 16, torch.bfloat16
    i32 = lambda v: torch.tensor(v, dtype=torch.int32, device="cuda")                      # noqa: E731
    hip = hip.configured()
    hip.settled = True
    short = 16 // min(heads // kv, 16) * 15                                                # (15 tiles of 16 rows)
    sink = _randn(heads, dtype=torch.float32, seed=172)
    for behind, lens in steps:
        total = [behind + n for n in lens]
        staged = hip.lib.holon_attention_prefill_one_order_staged
        assert staged(heads, kv, 2, max(lens), max(total), page, window, sum(lens)) and not staged(heads, kv, 1, short, max(total), page, window, short)
        pages_each = -(-max(total) // page)
        pages = _randn(2 * pages_each, 2, kv, page * d, dtype=bf, seed=170)
        table = torch.arange(2 * pages_each, dtype=torch.int32, device="cuda").flip(0).view(2, pages_each).contiguous()
        q = _randn(sum(lens), heads, d, dtype=bf, seed=171)
        rows = AttnRows(slots=i32([0, 1]), lens=i32(total), query_start=i32([0, lens[0], sum(lens)]), decode_rows=None,
                        chunk_rows=i32([0, 1]), n_decode=0, n_chunk=2, max_decode_len=0, max_chunk_query=max(lens),
                        max_chunk_len=max(total))
        last = total[0] - 1                                                                # (rows of its own tile weigh it by zero: left out below)
        pages[table[0, last // page].long(), 1].view(kv, d, page)[:, :, last % page] = torch.inf
        got = hip.paged_attention(q, pages, table, rows, page, d ** -0.5, window, sink=sink)
        for b, first in ((0, 0), (1, lens[0])):
            for s in range(0, lens[b], short):
                n = min(short, lens[b] - s)
                one = AttnRows(slots=i32([b]), lens=i32([behind + s + n]), query_start=i32([0, n]), decode_rows=None, chunk_rows=i32([0]),
                               n_decode=0, n_chunk=1, max_decode_len=0, max_chunk_query=n, max_chunk_len=behind + s + n)
                part = slice(first + s, first + s + n)
                want = hip.paged_attention(q[part].contiguous(), pages, table, one, page, d ** -0.5, window, sink=sink)
                mine = slice(0, max(0, n - 16) if b == 0 and s + n == lens[0] else n)
                assert torch.equal(got[part][mine], want[mine]) and torch.isfinite(want[mine]).all(), (behind, b, s)


def test_which_portions_of_heads_of_256_go_through_lds(hip):
    """Both sides of the lines: keys without a window, tiles for the SIMDs, windows that are narrow, wide or wider than the rows, groups of more
    heads than a tile has rows, a long portion among short ones, rows of more pages than LDS holds."""
    staged = hip.lib.holon_attention_prefill_one_order_staged

    def of(lens, heads, kv, window=0, behind=0, known=True, page=16):
        return staged(heads, kv, len(lens), max(lens), behind + max(lens), page, window, sum(lens) if known else 0)
    assert [of([n], 16, 1) for n in (511, 575, 576)] == [0, 0, 1] and [of([512] * n, 16, 1) for n in (2, 3)] == [0, 1]
    assert [of([n], 16, 16, behind=600) for n in (240, 241)] == [0, 1]                      # (fewer than 16 tiles)
    assert [of([n], 16, 1, w) for n, w in ((1024, 128), (1025, 128), (1100, 99), (1100, 512), (1024, 512))] == [0, 1, 1, 1, 0]
    assert [of([304], 16, 1, w, behind=1200) for w in (384, 440, 480, 512, 1024, -1024)] == [0, 0, 1, 1, 1, 1]
    assert [of([n], 16, 1, 512, behind=600) for n in (816, 820, 1024, 1028)] == [1, 0, 0, 1] and [of([576], 16, 1, w) for w in (128, 576, 600)] == [0, 1, 1]
    assert [of([n], 34, 1, 128, behind=300) for n in (341, 342)] == [0, 1] and of([600], 34, 1, -512) == 1 and of([1500] + [40] * 12, 32, 8, 128) == 0
    assert [of([n] + [40] * 7, 16, 1, 128) for n in (300, 600, 1500)] == [0, 1, 1]
    assert [of([600] + [17] * 7, 16, 1, 128, known=k) for k in (True, False)] == [0, 1]
    assert of([64], 16, 1, behind=65536 - 64) == 1 and of([64], 16, 1, behind=65536 - 63) == 0 and of([64], 16, 1, behind=65536 - 63, page=32) == 1


def test_few_row_products_whose_steps_leave_a_rest(hip):
    """A wave's steps of 32 are multiplied in sets of 2, 4 or 8, and what is left over in a set by itself: every remainder of each, none
    among them, fewer steps than a set, for each number of waves a tile, both weight layouts and the gated form, against float64; a
    row bit for bit what it is alone."""
    bf = torch.bfloat16
    for n, k in ((48, 288), (48, 352), (64, 416), (32, 480), (16, 544), (48, 320), (64, 448), (80, 576), (48, 704), (8224, 704), (64, 832),
                 (48, 384), (64, 640), (80, 896), (48, 1152), (4112, 1664), (48, 256), (64, 768), (2064, 768), (80, 1280), (48, 1792),
                 (64, 2304), (5136, 1152), (5120, 1280), (5136, 1792), (16400, 2816), (5120, 256), (48, 512), (64, 1024), (64, 1536),
                 (80, 2048), (80, 2560), (48, 3584), (32, 4608)):
        x, w = _randn(16, k, dtype=bf, seed=160), _randn(n, k, dtype=bf, seed=161)
        tiled, want = hip.tile_weight(w), x.double() @ w.double().T
        for held in (tiled, None):
            for m in (1, 9, 16):
                got = hip.linear(x[:m].contiguous(), w, tiled=held)
                assert H.op_budget_usage(got, want[:m], bf, k) <= 1, (m, n, k)
                assert torch.equal(got[:1], hip.linear(x[:1].contiguous(), w, tiled=held)), (m, n, k)
    for i, k in ((64, 256), (48, 384), (80, 512), (48, 640), (64, 768), (48, 896), (80, 1024), (64, 1280), (8208, 256), (8192, 384), (8208, 640)):
        x, w = _randn(16, k, dtype=bf, seed=162, scale=0.5), _randn(2 * i, k, dtype=bf, seed=163, scale=2 * k ** -0.5)
        tiled = hip.tile_weight(w)
        for held in (tiled, None):
            whole = hip.linear_silu_mul(x, w, tiled=held)
            assert torch.equal(whole[:1], hip.linear_silu_mul(x[:1].contiguous(), w, tiled=held)), (i, k)
            assert H.rel_rms(whole, torch.nn.functional.silu(x.double() @ w[:i].double().T) * (x.double() @ w[i:].double().T)) < 1e-2, (i, k)


@pytest.mark.parametrize("heads,kv,dim,vdim", [(3, 1, 204, 204), (2, 2, 128, 255), (2, 2, 128, 256), (14, 1, 64, 64)])
def test_whole_norm_prepare_around_its_block_sizes(hip, heads, kv, dim, vdim):
    """Rows of 1,020 to 1,024 values, steps of up to 256 tokens and more: blocks of 256 and of 1,024 threads leave the same bits, which are
    the plain form's within a rounding."""
    from holon_amd.kernels.registry import kernel_op
    width, bf, page = (heads + kv) * dim + kv * vdim, torch.bfloat16, 16
    x, qw, kw = _randn(257, width, dtype=bf, seed=170), 1 + _randn(heads * dim, dtype=bf, seed=171, scale=0.1), 1 + _randn(kv * dim, dtype=bf, seed=172, scale=0.1)
    at = torch.arange(257, dtype=torch.int32, device="cuda")
    held = {}
    for t in (1, 256, 257):
        pages = torch.zeros(17, kv * page * (dim + vdim), dtype=bf, device="cuda")
        held[t] = hip.whole_norm_prepare(x[:t].contiguous(), heads, kv, dim, vdim, qw, kw, 1e-5, pages, at[:t] // page, at[:t] % page, page), pages
    plain = torch.zeros_like(pages)
    want = kernel_op("whole_norm_prepare").plain(x, heads, kv, dim, vdim, qw, kw, 1e-5, plain, at // page, at % page, page)
    assert H.rel_rms(held[257][0], want) < 3e-3 and H.rel_rms(held[257][1], plain) < 3e-3
    assert torch.equal(held[256][0], held[257][0][:256]) and torch.equal(held[256][1][:16], held[257][1][:16])
    assert torch.equal(held[1][0], held[257][0][:1])


@pytest.mark.gpu
@pytest.mark.parametrize("rows", [1, 5, 16])
@pytest.mark.parametrize("sizes", [[(2048, 2048), (64, 2048), (16, 512)], [(2064, 512), (5136, 512), (48, 1184), (80, 288), (32, 256)],
                                   [(128, 2048), (144, 8192), (528, 352)] * 3, [(8192, 256)] * 2 + [(40, 256)]])
def test_products_in_one_launch_are_the_products(hip, rows, sizes):
    """`linear_group`, in every output form, bit for bit against each product by itself: tiles of 16, 8, 4, 2 and 1 waves, tiles that do
    not fill a block, short and long runs of K with and without a rest, more products than a launch takes, one that is not served."""
    from holon_amd.parts.products import Product
    k, gen = hip, torch.Generator(device="cuda").manual_seed(rows)

    class Weights:                                # what a projection holds
        folded, kernels = None, hip

        def __init__(self, n, kk):
            self.weight = (0.05 * torch.randn(n, kk, generator=gen, device="cuda")).bfloat16()
            self.tiled = k.tile_weight(self.weight)

        def __call__(self, x, dtype=None):
            return k.linear(x, self.weight, dtype, self.tiled)
    products = [Product(Weights(n, kk), torch.randn(rows, kk, generator=gen, device="cuda").bfloat16(),
                        **({}, {"dtype": torch.float32}, {"relu2": True})[i % 3]) for i, (n, kk) in enumerate(sizes)]
    for p, got in zip(products, k.linear_group(products)):
        want = p.alone()
        assert got.dtype == want.dtype and torch.equal(got, want), (p.linear.weight.shape, p.dtype, p.relu2)


@pytest.mark.gpu
@pytest.mark.parametrize("act", [0, 1])
@pytest.mark.parametrize("m,inter,k", [(1, 16, 128), (255, 96, 256), (256, 112, 128), (272, 192, 384), (273, 208, 256), (520, 400, 640)])
def test_gated_tiles_of_both_widths(hip, act, m, inter, k):
    """A gated first product on tiles of 96 gates and their ups is the one on tiles of 128, bit for bit: columns that end inside a tile,
    at its end and in its first sixteen, rows up to 16 beyond the last tile's 256."""
    x, w = _randn(m, k, dtype=torch.bfloat16, seed=190), _randn(2 * inter, k, dtype=torch.bfloat16, seed=191, scale=2 * k ** -0.5)
    outs = []
    for width in (128, 96):
        y = torch.full((m + 1, inter), 7.0, dtype=torch.bfloat16, device="cuda")
        hip._call(hip.lib.holon_gemm_block_glu_width_bf16, x.data_ptr(), w.data_ptr(), y.data_ptr(), m, inter, k, act, width, hip._stream())
        outs.append(y)
    assert torch.equal(outs[0], outs[1]) and (outs[1][m] == 7.0).all()


@pytest.mark.gpu
@pytest.mark.parametrize("dim,page", [(64, 16), (128, 32)])
@pytest.mark.parametrize("window", [0, 40, 1024])
def test_sigmoid_decode_rows_over_blocks(hip, dim, page, window):
    """Sigmoid-weighted decode rows with their keys over one block and over several: float32 sums of up to 1,024 bfloat16 products in
    another order, rounded once (2^-9)."""
    from holon_amd.kernels.registry import kernel_op
    from holon_amd.parts import sigmoid_attention as sa
    heads, kv, lens = 4, 2, [1, 33, 256, 257, 700, 1300]
    n, per = len(lens), -(-max(lens) // page)
    pages = _randn(n * per + 1, kv * page * 2 * dim, dtype=torch.bfloat16, seed=192)
    table = torch.arange(1, n * per + 1, dtype=torch.int32, device="cuda").view(n, per)
    i32 = lambda v: torch.tensor(v, dtype=torch.int32, device="cuda")          # noqa: E731
    q, gate = _randn(n, heads, dim, dtype=torch.bfloat16, seed=193), _randn(n, heads * dim, dtype=torch.bfloat16, seed=194)
    bias, order = _randn(heads, dtype=torch.float32, seed=195), i32(list(range(n)))
    rows = AttnRows(slots=order, lens=i32(lens), query_start=i32(list(range(n + 1))), decode_rows=order, chunk_rows=i32([]), n_decode=n,
                    n_chunk=0, max_decode_len=max(lens), max_chunk_query=0, max_chunk_len=0, in_order=True)
    args = (q, pages, table, rows, order, i32([v - 1 for v in lens]), kv, dim, page, bias, dim ** -0.5, window, gate)
    want, got = kernel_op("sigmoid_attention").plain(*args), []
    for blocks in (1, 2, 11):
        with pytest.MonkeyPatch.context() as m:
            m.setattr(sa, "decode_blocks", lambda pairs, span: blocks)
            got.append(hip.sigmoid_attention(*args))
        assert H.rel_rms(got[-1], want) < 2.0 ** -8, blocks
        assert H.rel_rms(got[-1], got[0]) < 2.0 ** -9, blocks


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("tokens,channels,rank", [(1, 2048, 64), (17, 260, 5), (33, 70, 30), (16, 256, 1024), (5, 3, 1), (40, 516, 36)])
def test_decay_projection(hip, dtype, tokens, channels, rank):
    """exp(-exp(tanh(a) w2 + w0)) against float64: sums of up to 1,024 float32 terms of size one, so that their error is at most a few
    times 2^-24 sqrt(rank) of the sum's size, which the two exponentials (slope at most 1 / e) do not enlarge."""
    a, w2t = _randn(tokens, rank, dtype=torch.float32, seed=196), _randn(rank, channels, dtype=dtype, seed=197, scale=0.3 * rank ** -0.5)
    w0 = _randn(channels, dtype=torch.float32, seed=198)
    want = torch.exp(-torch.exp(torch.tanh(a.double()) @ w2t.double() + w0.double()))
    assert (hip.decay_lora(a, w2t, w0).double() - want).abs().max() < 2e-6


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("heads,kv,dim,page", [(8, 2, 128, 16), (3, 3, 72, 5), (2, 1, 512, 8), (4, 2, 64, 16), (6, 1, 192, 8), (8, 2, 256, 16)])
@pytest.mark.parametrize("window", [0, 300, -128])
def test_decode_rows_a_wave_a_block_are_the_same_bits(hip, dtype, heads, kv, dim, page, window):
    """The general attention kernel's waves in blocks of their own against the whole block: rows of one key, of a tile and one more, of more
    tiles than waves, and a row of no keys."""
    lens = [1, 64, 65, 0, 513, 1100]
    n, per = len(lens), -(-max(lens) // page)
    pages = _randn(n * per, 2, kv, page * dim, dtype=dtype, seed=199)
    i32 = lambda v: torch.tensor(v, dtype=torch.int32, device="cuda")          # noqa: E731
    table, slots, at = torch.arange(n * per, dtype=torch.int32, device="cuda").view(n, per), i32(list(range(n))), i32(list(range(n + 1)))
    q, outs = _randn(n, heads, dim, dtype=dtype, seed=200), []
    parts = (torch.full((n, heads, 8, dim), float("nan"), dtype=torch.float64 if dtype == torch.float32 else torch.float32, device="cuda"),
             torch.full((n, heads, 8, 2), float("nan"), dtype=torch.float32, device="cuda"))
    for split in (False, True):
        out = torch.full_like(q, 7.0)
        args = (q.data_ptr(), out.data_ptr(), pages.data_ptr(), table.data_ptr(), per, slots.data_ptr(), i32(lens).data_ptr(), at.data_ptr(),
                n, n, heads, kv, dim, page, n * per, dim ** -0.5, window, max(lens), int(dtype == torch.bfloat16))
        if split:
            hip._call(hip.lib.holon_attention_generic_split, *args, *(p.data_ptr() for p in parts), hip._stream())
        else:
            hip._call(hip.lib.holon_attention_generic, *args, hip._stream())
        outs.append(out)
    assert torch.equal(*outs) and not outs[1][3].any() and outs[1].isfinite().all()


@pytest.mark.gpu
@pytest.mark.parametrize("heads,kv,dim", [(16, 4, 128), (4, 4, 64), (40, 2, 64)])
@pytest.mark.parametrize("window,sunk,cap", [(0, False, 0.0), (300, True, 3.0), (-128, True, 0.0)])
def test_float64_decode_rows_a_wave_a_block_are_the_same_bits(hip, heads, kv, dim, window, sunk, cap, monkeypatch):
    """The same of softmax attention on the float64 matrix cores, a row on the padding slot (position -1) among them."""
    from holon_amd.parts import softmax_attention as sa
    page, lens = 16, [1, 16, 17, 0, 129, 700]
    n, per = len(lens), 48
    pages = _randn(n * per, 2 * kv * page * dim, dtype=torch.float32, seed=201)
    i32 = lambda v: torch.tensor(v, dtype=torch.int32, device="cuda")          # noqa: E731
    table, order = torch.arange(n * per, dtype=torch.int32, device="cuda").view(n, per), i32(list(range(n)))
    rows = AttnRows(slots=order, lens=i32(lens), query_start=i32(list(range(n + 1))), decode_rows=order, chunk_rows=i32([]), n_decode=n,
                    n_chunk=0, max_decode_len=max(lens), max_chunk_query=0, max_chunk_len=0, in_order=True)
    q = _randn(n, heads, dim, dtype=torch.float32, seed=202)
    sink = _randn(heads, dtype=torch.float32, seed=203) if sunk else None
    outs = []
    for split in (False, True):
        monkeypatch.setattr(sa, "f64_split_pays", lambda *a, split=split: split)
        outs.append(hip.softmax_attention(q, pages, table, rows, order, i32([v - 1 for v in lens]), kv, dim, page, sink, dim ** -0.5, window,
                                          softcap=cap))
    assert torch.equal(*outs) and not outs[1][3].any() and outs[1].isfinite().all()


@pytest.mark.gpu
@pytest.mark.parametrize("rows", [1, 3, 16])
@pytest.mark.parametrize("experts,extra,groups,how", [(8, 0, 4, {"scale": 2.5}), (8, 1, 1, {}), (64, 0, 8, {"score": "sigmoid"}),
                                                      (5, 1, 1, {"score": "sigmoid_squared"})])
def test_a_router_beside_products_is_the_router(hip, rows, experts, extra, groups, how):
    """A mixture's routing in a launch of products, bit for bit the operation by itself, and the products what they are."""
    from holon_amd.parts.products import Product, Routing
    width = 640

    class Weights:
        folded, kernels = None, hip
        weight = _randn(528, width, dtype=torch.bfloat16, seed=204, scale=0.05)
        tiled = hip.tile_weight(weight)

        def __call__(self, x, dtype=None):
            return hip.linear(x, self.weight, dtype, self.tiled)
    x = _randn(rows, width, dtype=torch.bfloat16, seed=205)
    router = _randn(experts + extra, width, dtype=torch.float32, seed=206, scale=0.1)
    bias = _randn(experts, dtype=torch.float32, seed=207)
    routing = Routing(hip, x, router, bias, experts, 2, groups, max(1, groups // 2), **how)
    products = [Product(Weights(), x), routing, Product(Weights(), x, torch.float32)]
    for p, got in zip(products, hip.linear_group(products)):
        assert torch.equal(got, p.alone())
    assert torch.equal(hip.linear_group([routing])[0], routing.alone())


@pytest.mark.gpu
@pytest.mark.parametrize("m,n,k", [(129, 1024, 1024), (256, 1040, 1152), (272, 1264, 1024), (273, 2048, 1280), (1025, 1536, 1024), (3072, 1024, 1024)])
def test_products_of_many_rows_in_one_launch(hip, m, n, k):
    """Four products of one size among others, in one launch on 256 x 256 tiles: each within a rounding (2^-9) and float32 sums of k of
    its exact product, columns that end inside a tile, rows up to 16 beyond the last tile's 256 and more. What the group does not take
    (another size, a float32 result, the fifth) is what it is alone."""
    from holon_amd.parts.products import Product, block_group_pays

    class Weights:                                # what a projection holds
        folded, tiled, kernels = None, None, hip

        def __init__(self, i, out):
            self.weight = _randn(out, k, dtype=torch.bfloat16, seed=210 + i, scale=k ** -0.5)

        def __call__(self, x, dtype=None):
            return hip.linear(x, self.weight, dtype)
    linears = [Weights(i, out) for i, out in enumerate([n, n, 512, n, n, n, n])]
    xs = _randn(len(linears), m, k, dtype=torch.bfloat16, seed=209)
    products = [Product(lin, xs[i], torch.float32 if i == 5 else None) for i, lin in enumerate(linears)]
    assert block_group_pays(4, m, n, k)
    got = hip.linear_block_group(products)
    together = got[0].untyped_storage().data_ptr()
    assert [g.untyped_storage().data_ptr() == together for g in got] == [True, True, False, True, True, False, False]
    for i, (p, y) in enumerate(zip(products, got)):
        want = p.x.double() @ p.linear.weight.double().t()
        assert y.shape == want.shape and H.rel_rms(y, want) < 2.0 ** -9 + 2.0 ** -24 * k ** 0.5
        if i in (2, 5, 6):
            assert torch.equal(y, p.alone())
    with pytest.MonkeyPatch.context() as settled:
        settled.setattr(hip, "settled", True)
        assert all(torch.equal(y, p.alone()) for y, p in zip(hip.linear_block_group(products), products))


@pytest.mark.gpu
@pytest.mark.parametrize("softcap", [0.0, 20.0])
@pytest.mark.parametrize("geometry", [(8, 2, 64), (16, 4, 128), (16, 1, 256)])
def test_decode_rows_of_every_last_block(hip, geometry, softcap):
    """Decode rows of 1 to 64 keys, NaN in every cache slot behind them, in one wave and over four: each row within its
    budget of the plain form in float64, and bit for bit what it is with zeros there."""
    heads, kv_heads, d = geometry
    page, dtype, rows = 16, torch.bfloat16, [(n, 1) for n in range(64)]
    q, pages, table, attn = _paged_case(rows, heads, kv_heads, d, page, dtype, seed=31, max_seqs=64)
    held = torch.zeros(pages.shape[0], page, dtype=torch.bool)
    for slot, (s, n) in zip(attn.slots.tolist(), rows):
        pos = torch.arange(s + n)
        held[table[slot, pos // page].cpu().long(), pos % page] = True
    outs, free = [], (~held).cuda()
    for longest in (64, 256):
        attn.max_decode_len = longest
        for fill in (0.0, float("nan")):
            pages[:, 0].view(-1, kv_heads, page, d).masked_fill_(free[:, None, :, None], fill)
            pages[:, 1].view(-1, kv_heads, d, page).masked_fill_(free[:, None, None, :], fill)
            outs.append(hip.paged_attention(q, pages, table, attn, page, d ** -0.5, 0, softcap=softcap))
        assert torch.equal(outs[-1], outs[-2]) and torch.isfinite(outs[-1].float()).all()
        want = PLAIN.paged_attention(q.double(), pages.double(), table, attn, page, d ** -0.5, 0, softcap=softcap)
        assert H.op_budget_usage(outs[-1], want, dtype, d + 64) <= 1


@pytest.mark.gpu
@pytest.mark.parametrize("dim", [4, 1020, 1028, 2048, 2560, 3072, 3076, 4092, 4096, 4100])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
def test_stream_rows_of_one_type_are_those_of_several(hip, dtype, dim):
    """A pass over stream rows whose operands are asked for ahead gives the bits of the general one: of one type, or bfloat16 under float32
    weights that hold the same values (without filters; float32 rows under bfloat16 weights take the general form). The general one is
    taken by a term of the other type that holds the same values, and without terms by results in float32, rounded here: with and without
    terms, vector, second weight, filters."""
    import holon_amd.parts.parallel_block  # noqa: F401  (brings the operations)
    other = torch.float32 if dtype == torch.bfloat16 else torch.bfloat16
    rows = 3
    x, row = _randn(rows, dim, dtype=torch.float32, seed=220), _randn(dim, dtype=torch.float32, seed=221)
    t1, t2 = (_randn(rows, dim, dtype=torch.bfloat16, seed=s).to(dtype) for s in (222, 223))
    w1, w2 = (_randn(dim, dtype=torch.bfloat16, seed=s).to(dtype) for s in (224, 225))
    c1, c2 = (_randn(dim, 3, dtype=torch.bfloat16, seed=s).to(dtype) for s in (226, 227))
    held = _randn(2, rows, 2, dim, dtype=torch.bfloat16, seed=228).to(dtype)
    slots, starts = (torch.tensor(v, dtype=torch.int32, device="cuda") for v in ([2, 0, 1], [5, 0, 1]))
    for terms in ([], [t1], [t1, t2]):
        for added in (None, row):
            for second in (None, w2):
                got = []
                for to_terms, to_weights in ((dtype, dtype), (dtype, other)) + (((other, dtype),) if terms else ()):
                    xs, hs = x.clone(), held.clone()
                    args = (xs, [(t.to(to_terms), 1.0) for t in terms], added, w1.to(to_weights),
                            None if second is None else second.to(to_weights), 1e-6, dtype)
                    y = [*hip.stream_rms(*args), xs]
                    args[0].copy_(x)
                    y += [*hip.stream_rms_filter(*args, c1, c2 if second is not None else None, hs[0], hs[1] if second is not None else None,
                                                 slots, starts), xs.clone(), hs]
                    got.append([v for v in y if v is not None])
                if dtype == torch.bfloat16 and not terms:
                    y = [v.bfloat16() for v in hip.stream_rms(x.clone(), [], added, w1, second, 1e-6, torch.float32) if v is not None]
                    assert all(torch.equal(a, b) for a, b in zip(y, got[0])), (added is None, second is None)
                for one in got[1:]:
                    assert all(torch.equal(a, b) for a, b in zip(one, got[0], strict=True)), (len(terms), added is None, second is None)


@pytest.mark.gpu
@pytest.mark.parametrize("rows", [1024, 1025, 1792, 1793, 2048, 2049])
def test_many_stream_rows_under_float32_weights(hip, rows):
    """bfloat16 terms under float32 weights on both sides of the rows and widths from which they are not asked for ahead: bit for bit the
    general form (taken by results in float32 under bfloat16 weights, rounded here)."""
    import holon_amd.parts.parallel_block  # noqa: F401  (brings the operations)
    for dim in (1536, 1540, 2048, 2052, 2560, 2564, 3072, 3076, 4096):
        x, row = _randn(rows, dim, dtype=torch.float32, seed=229), _randn(dim, dtype=torch.float32, seed=230)
        t1, (w1, w2) = _randn(rows, dim, dtype=torch.bfloat16, seed=231), (_randn(dim, dtype=torch.bfloat16, seed=s) for s in (232, 233))
        for terms, added, second in (([], None, None), ([], row, w2), ([t1], None, w2), ([t1, t1], row, None)):
            a, b = x.clone(), x.clone()
            got = hip.stream_rms(a, [(t, 1.0) for t in terms], added, w1.float(), None if second is None else second.float(), 1e-6, torch.bfloat16)
            want = hip.stream_rms(b, [(t, 1.0) for t in terms], added, w1, second, 1e-6, torch.float32)
            assert torch.equal(a, b) and all(torch.equal(g, w.bfloat16()) for g, w in zip(got, want) if w is not None), (dim, len(terms))


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("heads,kv,dim,t,longest,split", [(16, 4, 128, 4, 128, False), (16, 4, 128, 4, 129, True), (16, 4, 128, 16, 384, False),
                                                          (16, 4, 128, 16, 385, True), (71, 1, 72, 2, 700, False), (71, 1, 72, 1, 385, True),
                                                          (12, 2, 96, 33, 700, False), (8, 2, 512, 16, 700, False), (8, 2, 512, 2, 385, True)])
def test_decode_rows_at_the_borders_of_a_wave_a_block(hip, dtype, heads, kv, dim, t, longest, split, monkeypatch):
    """`paged_attention` by the general kernel on both sides of the rule that gives every wave a block, by the blocks that a step really
    has: the form named, within its budget of the plain form, and no bigger a workspace than a few MB."""
    page = 5 if dtype == torch.bfloat16 else 16
    rows = [(longest - 1 - i * 7 % 60, 1) for i in range(t)]
    q, pages, table, attn = _paged_case(rows, heads, kv, dim, page, dtype, seed=230, max_seqs=t)
    called, made, empty = [], [], torch.empty
    call = hip._call
    with monkeypatch.context() as m:
        m.setattr(hip, "_call", lambda fn, *a: called.append(fn.__name__) or call(fn, *a))
        m.setattr(torch, "empty", lambda *a, **kw: made.append(empty(*a, **kw)) or made[-1])
        got = hip.paged_attention(q, pages, table, attn, page, dim ** -0.5, 0)
    assert called == ["holon_attention_generic_split" if split else "holon_attention_generic"]
    assert sum(x.numel() * x.element_size() for x in made) <= 5 << 20 and (split or not made)
    want = PLAIN.paged_attention(q.double(), pages.double(), table, attn, page, dim ** -0.5, 0)
    assert H.op_budget_usage(got, want, dtype, dim + longest) <= 1


@pytest.mark.gpu
@pytest.mark.parametrize("heads,kv,dim", [(4, 2, 128), (3, 3, 64), (34, 2, 64)])
@pytest.mark.parametrize("t,longest,window", [(1, 256, 0), (1, 257, 0), (3, 1100, 0), (50, 300, 1024), (129, 1023, 0), (129, 1024, 0), (140, 640, 129)])
def test_sigmoid_decode_rows_by_the_rules_of_blocks_and_waves(hip, heads, kv, dim, t, longest, window):
    """`sigmoid_attention` of decode rows on both sides of the lines that blocks and waves are chosen by (256, 257, 1,023 and 1,024 keys; up to 256
    (row, kv head) pairs and more): float32 sums of up to 1,100 bfloat16 products, rounded once (2^-9)."""
    from holon_amd.kernels.registry import kernel_op
    import holon_amd.parts  # noqa: F401  (brings the operations)
    page, lens = 16, [max(1, longest - 37 * i % longest) for i in range(t)]
    per = -(-longest // page)
    pages = _randn(t * per, kv * page * 2 * dim, dtype=torch.bfloat16, seed=240)
    table = torch.arange(t * per, dtype=torch.int32, device="cuda").view(t, per)
    i32 = lambda v: torch.tensor(v, dtype=torch.int32, device="cuda")          # noqa: E731
    order = i32(list(range(t)))
    q, gate = _randn(t, heads, dim, dtype=torch.bfloat16, seed=241), _randn(t, heads * dim, dtype=torch.bfloat16, seed=242)
    rows = AttnRows(slots=order, lens=i32(lens), query_start=i32(list(range(t + 1))), decode_rows=order, chunk_rows=i32([]), n_decode=t,
                    n_chunk=0, max_decode_len=longest, max_chunk_query=0, max_chunk_len=0, in_order=True)
    args = (q, pages, table, rows, order, i32([v - 1 for v in lens]), kv, dim, page, _randn(heads, dtype=torch.float32, seed=243), dim ** -0.5,
            window, gate)
    assert H.rel_rms(hip.sigmoid_attention(*args), kernel_op("sigmoid_attention").plain(*args)) < 2.0 ** -8


F64_BORDERS = [(16, 4, 128, 1, 256, False), (16, 4, 128, 1, 257, True), (16, 4, 128, 28, 300, True), (16, 4, 128, 29, 300, False),
               (32, 8, 128, 12, 300, True), (32, 8, 128, 13, 300, False), (16, 4, 64, 16, 257, True), (16, 4, 64, 17, 320, False),
               (16, 4, 64, 17, 321, True), (40, 2, 64, 31, 321, True), (40, 2, 64, 32, 700, False), (4, 4, 64, 32, 700, False),
               (4, 1, 128, 128, 300, True), (4, 1, 128, 133, 300, False), (4, 1, 64, 128, 700, False)]


def test_float64_decode_rows_are_split_where_their_blocks_fit():
    from holon_amd.parts.softmax_attention import f64_split_pays
    assert [f64_split_pays(t, h, kv, dim, longest, 0) for h, kv, dim, t, longest, _ in F64_BORDERS] == [b[-1] for b in F64_BORDERS]
    assert not f64_split_pays(1, 16, 4, 128, 700, 256) and f64_split_pays(1, 16, 4, 128, 700, -257)


@pytest.mark.gpu
@pytest.mark.parametrize("heads,kv,dim,t,longest,split", F64_BORDERS)
def test_float64_decode_rows_at_the_borders_of_a_wave_a_block(hip, heads, kv, dim, t, longest, split, monkeypatch):
    """`softmax_attention` of float32 decode rows on both sides of the rule that gives every wave a block: the form named, and its result that of
    the plain form in float64 within float32 exponentials and one rounding."""
    from holon_amd.kernels.registry import kernel_op
    import holon_amd.parts  # noqa: F401  (brings the operations)
    page, lens = 16, [longest - 7 * i % 60 for i in range(t)]
    per = -(-longest // page)
    pages = _randn(t * per, 2 * kv * page * dim, dtype=torch.float32, seed=250)
    i32 = lambda v: torch.tensor(v, dtype=torch.int32, device="cuda")          # noqa: E731
    table, order = torch.arange(t * per, dtype=torch.int32, device="cuda").view(t, per), i32(list(range(t)))
    rows = AttnRows(slots=order, lens=i32(lens), query_start=i32(list(range(t + 1))), decode_rows=order, chunk_rows=i32([]), n_decode=t,
                    n_chunk=0, max_decode_len=longest, max_chunk_query=0, max_chunk_len=0, in_order=True)
    q, positions, made, empty = _randn(t, heads, dim, dtype=torch.float32, seed=251), i32([v - 1 for v in lens]), [], torch.empty
    rest = (rows, order, positions, kv, dim, page, None, dim ** -0.5, 0)
    with monkeypatch.context() as m:
        m.setattr(torch, "empty", lambda *a, **kw: made.append(kw.get("dtype")) or empty(*a, **kw))
        got = hip.softmax_attention(q, pages, table, *rest)
    assert (torch.float64 in made) == split
    want = kernel_op("softmax_attention").plain(q.double(), pages.double(), table, *rest)
    assert H.rel_rms(got, want) < 1e-6


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("tokens,channels,rank", [(1, 1030, 30), (4, 255, 64), (5, 257, 9), (17, 7, 4), (33, 5, 16), (2, 4, 3), (20, 3, 5)])
def test_decay_projection_of_any_number_of_channels(hip, dtype, tokens, channels, rank):
    """Channels that do not come in fours: bit for bit those of a call whose channels do, and nothing behind them is written."""
    more = -(-channels // 4) * 4 + 4
    a, w2t = _randn(tokens, rank, dtype=torch.float32, seed=260), _randn(rank, more, dtype=dtype, seed=261, scale=0.3 * rank ** -0.5)
    w0, w = _randn(more, dtype=torch.float32, seed=262), w2t[:, :channels].contiguous()
    y = torch.full((tokens * channels + 4,), 7.0, dtype=torch.float32, device="cuda")
    hip._call(hip.lib.holon_decay_lora, a.data_ptr(), w.data_ptr(), w0.data_ptr(), y.data_ptr(), tokens, channels, rank,
              int(dtype == torch.bfloat16), hip._stream())
    assert torch.equal(y[:-4].view(tokens, channels), hip.decay_lora(a, w2t, w0)[:, :channels]) and (y[-4:] == 7.0).all()


@pytest.mark.parametrize("waves", [1, 16])
def test_moves_between_lanes_are_the_shuffles(waves):
    """Bit for bit what lane ^ o holds and what sums and maxima over steps by n / 2 .. 1 are; infinities, both zeros, tiny values."""
    import ctypes
    import pathlib
    from holon_amd.kernels import build
    source = pathlib.Path(__file__).parent / "kernels" / "lanes.hip"
    fn = ctypes.CDLL(str(build.source_library(source) or build.build_source(source))).test_lanes
    fn.argtypes, fn.restype = [ctypes.c_void_p, ctypes.c_void_p, ctypes.c_int, ctypes.c_void_p], ctypes.c_int
    rng = np.random.default_rng(waves)
    x = (rng.standard_normal((waves, 64)) * 10.0 ** rng.integers(-8, 8, (waves, 64))).astype(np.float32)
    x[:, 3], x[:, 17], x[:, 40], x[:, 55] = np.float32(np.inf), 0.0, -0.0, np.finfo(np.float32).min
    out = torch.full((waves, 7, 6, 64), torch.nan, device="cuda")
    given = torch.from_numpy(x).cuda()
    assert fn(given.data_ptr(), out.data_ptr(), waves, torch.cuda.current_stream().cuda_stream) == 0
    got, lane = out.cpu().numpy(), np.arange(64)
    for n, o in enumerate((1, 2, 4, 8, 16, 32)):
        other = x[:, lane ^ o]
        total, top = x, x
        for step in (s for s in (32, 16, 8, 4, 2, 1) if s <= o):
            total, top = total + total[:, lane ^ step], np.maximum(top, top[:, lane ^ step])
        want = (other, x + other, np.maximum(x, other), total, top, np.broadcast_to((lane ^ o).astype(np.float32), x.shape),
                np.broadcast_to(x[:, 2 * o - 1: 2 * o], x.shape))
        for k, w in enumerate(want):
            have, w = got[:, k, n], np.ascontiguousarray(w, np.float32)
            same = have == w if k in (2, 4) else have.view(np.uint32) == w.view(np.uint32)      # (a maximum: either zero)
            assert same.all(), (k, o)


def _moved(t, by=1):
    """The same values where no border of 16 bytes is: kernels that take pieces of eight values leave them to the general form."""
    return torch.empty(t.numel() + by, dtype=t.dtype, device=t.device)[by:].view(t.shape).copy_(t)


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("dim", [64, 128, 256])
def test_heads_in_pieces_are_the_heads_value_by_value(hip, dtype, dim):
    """q, k and v prepared, read-outs normed and gated, two maps combined: eight values a lane bit for bit as a value a lane; heads that do
    not fill a wave, every rotated width on and off the middle of a head, tokens without a place in the cache."""
    heads, kv, page_size, t, pages_n = 5, 2, 16, 19, 3
    positions = torch.arange(t, dtype=torch.int32).cuda() * 7 % 40
    write_page = (torch.arange(t, dtype=torch.int32) // page_size).cuda()
    write_off = (torch.arange(t, dtype=torch.int32) % page_size).cuda()
    write_page[3], write_off[5] = -1, page_size
    for rot in (0, 16, 48, dim // 2, dim):
        table = _randn(40, rot, dtype=torch.float32, seed=200) if rot else None
        for normed, biased, values, share, vdim in ((True, False, "own", 1, dim), (False, False, "own", 2, 24), (True, True, "own", 1, 40),
                                                    (False, True, "keys", 1, dim)):
            width = (heads + kv) * dim + (0 if values == "keys" else kv // share * vdim)
            qkv = _randn(t, width + 8, dtype=dtype, seed=201, scale=2.0)
            weights = [1 + 0.2 * _randn(dim, dtype=dtype, seed=202 + i) for i in range(2)] if normed else [None, None]
            bias = _randn(width, dtype=torch.float32, seed=204) if biased else None
            v_heads = kv if values == "keys" else kv // share
            made = []
            for rows in (qkv, _moved(qkv)):
                pages = torch.zeros(pages_n, kv * page_size * dim + v_heads * page_size * vdim, dtype=dtype, device="cuda")
                q = hip.head_prepare(rows, heads, kv, dim, vdim, *weights, 1e-5, table, positions, pages, write_page, write_off, page_size,
                                     bias=bias, values=values, value_share=share)
                made.append((q, pages))
            assert all(torch.equal(a, b) for a, b in zip(*made)), (rot, normed, biased, values, share)
    for cells in (1, 7, 33):
        o, gate = _randn(cells, heads, dim, dtype=torch.float32, seed=205), _randn(cells, heads * dim + 8, dtype=dtype, seed=206)
        den = _randn(cells, heads, dtype=torch.float32, seed=207).abs() + 0.1
        for per_head in (False, True):
            w = 1 + 0.2 * _randn(heads * dim if per_head else dim, dtype=dtype, seed=208)
            for act, under in (("silu", None), ("sigmoid", den)):
                got, want = (hip.gated_out(x, gate[:, : heads * dim], w, per_head, 1e-6, dtype, act=act, den=under) for x in (o, _moved(o)))
                assert torch.equal(got, want), (cells, per_head, act)
        y = _randn(cells, 2 * 4 * dim, dtype=dtype, seed=209)
        got, want = (hip.diff_combine(x, 4, 2, dim, 0.35, 1e-5, 0.65) for x in (y, _moved(y)))
        assert torch.equal(got, want), cells


@pytest.mark.parametrize("dtype", DTYPES)
def test_rows_in_pieces_are_the_rows_value_by_value(hip, dtype):
    """Token shifts and a latent's entries and queries: eight values a thread bit for bit as a value a thread."""
    for width in (8, 2040, 2048, 2056):
        counts = [1, 5, 17]
        starts, slots = torch.tensor([0, 3, 9], dtype=torch.int32).cuda(), torch.tensor([2, 0, 3], dtype=torch.int32).cuda()
        first = torch.tensor([0, 1, 6, 23], dtype=torch.int32).cuda()
        row = torch.repeat_interleave(torch.arange(3), torch.tensor(counts)).to(torch.int32).cuda()
        x, mu = _randn(23, width, dtype=dtype, seed=210), _randn(5, width, dtype=dtype, seed=211)
        made = []
        for rows in (x, _moved(x)):
            state = _randn(4, width, dtype=dtype, seed=212)
            y = hip.shift_mix(rows, mu, state, slots, starts, first, row, 3)
            step = hip.shift_mix(rows[:3].clone() if rows is x else _moved(rows[:3]), mu, state, slots, starts, first, row, 3, in_order=True)
            made.append((y, step, state))
        assert all(torch.equal(a, b) for a, b in zip(*made)), width
    t, page_size = 257, 16
    positions = (torch.arange(t, dtype=torch.int32) % 50).cuda()
    write_page = (torch.arange(t, dtype=torch.int32) // page_size).cuda()
    write_off = (torch.arange(t, dtype=torch.int32) % page_size).cuda()
    write_page[7] = 99
    for heads, dim, rot, rank, rd, copies in ((3, 128, 64, 192, 64, 1), (16, 8, 16, 24, 16, 2), (5, 72, 24, 512, 16, 2), (2, 64, 0, 64, 0, 1)):
        both = _randn(t, heads * (dim + rot) + rank + rot + 8, dtype=dtype, seed=213)
        table = _randn(50, rd, dtype=torch.float32, seed=214) if rd else None
        weight, made = 1 + 0.2 * _randn(rank, dtype=dtype, seed=215), []
        for rows in (both, _moved(both)):
            pages = torch.zeros(-(-t // page_size), copies * page_size * (rank + rot), dtype=dtype, device="cuda")
            q, full = hip.latent_rope_prepare(rows, heads, dim, rot, rank, weight, 1e-5, table, positions, pages, write_page, write_off, page_size,
                                              copies=copies)
            made.append((q, full[..., rank:].clone(), pages))
        assert all(torch.equal(a, b) for a, b in zip(*made)), (heads, dim, rot, rank, rd, copies)


@pytest.mark.parametrize("dtype", DTYPES)
def test_shifts_of_many_tokens_in_pieces_are_those_channel_by_channel(hip, dtype):
    """Steps on both sides of the size from which a thread takes 16 bytes of channels (196,608 values, 262,144 in float32), widths that do not fill
    a block or two, in pieces of float32 alone, rows of one token and of many, behind kept tokens and not, in order and not: bit for bit what operands off a border of
    16 bytes give, which go channel by channel; against the plain form a rounding or two of the result's type."""
    from holon_amd.kernels.registry import kernel_op
    i32 = lambda v: torch.tensor(v, dtype=torch.int32, device="cuda")                      # noqa: E731
    for tokens, width, mixes in ((95, 2048, 5), (96, 2048, 5), (127, 2048, 2), (128, 2048, 5), (200, 2056, 3), (203, 2060, 2), (96, 4096, 1), (24576, 16, 2), (50, 7872, 2),
                                 (260, 1032, 2)):
        counts = [1, 5, tokens - 6]
        first, row = i32([0, 1, 6, tokens]), torch.repeat_interleave(torch.arange(3), torch.tensor(counts)).to(torch.int32).cuda()
        x, mu, kept = _randn(tokens, width, dtype=dtype, seed=216), _randn(mixes, width, dtype=dtype, seed=217), _randn(4, width, dtype=dtype, seed=218)
        made = []
        for rows in (x, _moved(x)):
            state = kept.clone()
            made.append((hip.shift_mix(rows, mu, state, i32([2, 0, 3]), i32([0, 3, 9]), first, row, 3), state))
        state = kept.clone()
        want = kernel_op("shift_mix").plain(x, mu, state, i32([2, 0, 3]), i32([0, 3, 9]), first, row, 3), state
        assert all(torch.equal(a, b) for a, b in zip(*made)) and torch.equal(made[0][1], want[1]), (tokens, width)
        assert H.rel_rms(made[0][0], want[0]) < (2.0 ** -8 if dtype == torch.bfloat16 else 2.0 ** -22), (tokens, width)
        if tokens > 300:
            continue
        made, slots = [], torch.randperm(tokens, generator=torch.Generator().manual_seed(219)).to(torch.int32).cuda()
        starts, each = i32([n % 3 for n in range(tokens)]), i32(list(range(tokens + 1)))
        kept = _randn(tokens, width, dtype=dtype, seed=219)
        for rows in (x, _moved(x)):
            state = kept.clone()
            made.append((hip.shift_mix(rows, mu, state, slots, starts, each, each[:-1].contiguous(), tokens, in_order=True), state))
        assert all(torch.equal(a, b) for a, b in zip(*made)) and torch.equal(made[0][1][slots.long()], x), (tokens, width)


@pytest.mark.parametrize("dtype", DTYPES)
def test_routers_of_many_rows_are_those_of_few(hip, dtype):
    """Tokens that share what a wave reads of the router (one, two or four of them, by the rows) have bit for bit the weights of a token by
    itself: rows on both sides of the lines, experts that do not come in eights, widths that do not fill a wave's step."""
    for rows, width, experts, top, groups, keep in ((257, 2048, 8, 2, 1, 1), (1023, 260, 9, 3, 1, 1), (1024, 4, 1, 1, 1, 1), (2047, 1028, 17, 4, 1, 1),
                                                    (2048, 2044, 64, 6, 8, 3), (2061, 512, 12, 2, 4, 2)):
        x = _randn(rows, width, dtype=dtype, seed=220)
        router = _randn(experts + 1, width, dtype=torch.float32, seed=221, scale=width ** -0.5)
        bias = _randn(experts, dtype=torch.float32, seed=222, scale=0.2)
        calls = [(hip.moe_router, (router[:experts].contiguous(), bias, top, groups, keep, 1.5), {})]
        calls += [(hip.moe_router_top, (r, bias, experts, top, groups, keep), dict(score=how))
                  for r, how in ((router, "softmax"), (router[:experts].contiguous(), "sigmoid"), (router, "sigmoid_squared"))]
        for op, args, how in calls:
            want = torch.cat([op(x[at: at + 256].contiguous(), *args, **how) for at in range(0, rows, 256)])
            assert torch.equal(op(x, *args, **how), want), (rows, width, experts, how)


@pytest.mark.parametrize("rows", [1, 6, 16])
@pytest.mark.parametrize("hidden,experts,ff,shared", [(256, 8, 32, 0), (2048, 8, 256, 512), (512, 70, 544, 32), (288, 5, 96, 0)])
def test_experts_beside_a_product_are_both(hip, rows, hidden, experts, ff, shared, monkeypatch):
    """A mixture's second product and another one in one launch, bit for bit what either is by itself: tiles of 16, 8, 4, 2 and 1 waves
    that do and do not fill a block, every output form; a product that joins no launch, one beside which it does not pay, and none at all."""
    from holon_amd.kernels.registry import kernel_op
    from holon_amd.parts import products as pr
    from holon_amd.parts.products import ExpertsDown, Product
    bf, cols, gen = torch.bfloat16, experts * ff + shared, torch.Generator(device="cuda").manual_seed(rows)
    down_t = hip.tile_weight(_randn(hidden, cols, dtype=bf, seed=230, scale=ff ** -0.5))
    weights = (torch.rand(rows, experts, generator=gen, device="cuda") * (torch.rand(rows, experts, generator=gen, device="cuda") < 0.3)).contiguous()
    act = _randn(rows, cols, dtype=bf, seed=231)
    act[:, : experts * ff] *= (weights != 0).repeat_interleave(ff, 1)
    down = ExpertsDown(hip, act, weights, down_t, experts, ff, shared)
    whole = hip.linear(act, _randn(hidden, cols, dtype=bf, seed=230, scale=ff ** -0.5), tiled=down_t)
    assert torch.equal(down.alone(), whole) and torch.equal(hip.linear_group([down])[0], whole)
    plain = kernel_op("moe_down_few").plain(act, weights, down_t, experts, ff, shared)
    assert H.rel_rms(whole, plain) < 2.0 ** -8 if plain.any() else not whole.any()

    class Weights:                                # what a projection holds
        folded, kernels = None, hip

        def __init__(self, n, kk):
            self.weight = (0.05 * torch.randn(n, kk, generator=gen, device="cuda")).bfloat16()
            self.tiled = hip.tile_weight(self.weight)

        def __call__(self, x, dtype=None):
            return hip.linear(x, self.weight, dtype, self.tiled)
    for i, (n, kk) in enumerate(((2048, 2048), (16, 512), (5136, 512), (80, 1184), (80, 288), (528, 352), (48, 192))):
        p = Product(Weights(n, kk), torch.randn(rows, kk, generator=gen, device="cuda").bfloat16(), **({}, {"dtype": torch.float32}, {"relu2": True})[i % 3])
        for products in ([p, down], [down, p]):
            got = dict(zip(map(id, products), hip.linear_group(products)))
            want = p.alone()
            assert got[id(p)].dtype == want.dtype and torch.equal(got[id(p)], want) and torch.equal(got[id(down)], whole), (n, kk)
        with monkeypatch.context() as m:
            m.setattr(pr, "beside_pays", lambda *a: False)
            m.setattr(pr, "_beside", lambda *a: pytest.fail("a launch that does not pay"))
            apart = hip.linear_group([p, down])
        assert torch.equal(apart[0], want) and torch.equal(apart[1], whole), (n, kk)
