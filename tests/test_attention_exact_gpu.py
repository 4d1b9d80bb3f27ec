"""Attention of rows of several tokens with unrounded softmax weights: over the paged cache (``attention_exact``) with every
option it takes, and a latent attention's multiplied-out form, both against 64-bit sums over the same bfloat16 keys and values."""

from __future__ import annotations

import math

import pytest
import torch

from test_kernels_gpu import BF16, DEV, F32, close, make_batch, rand

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ops():
    from miniserve_amd.kernels import ops as o

    o.library()
    return o


def pages_for(totals, seed, windows=None):
    """A block table over scattered pages; entries wholly before ``windows[i]`` hold no page (given back)."""
    g = torch.Generator().manual_seed(seed)
    blocks = [-(-t // 16) for t in totals]
    order = torch.randperm(sum(blocks) + 3, generator=g).tolist()
    table = torch.full((len(totals), max(blocks) + 1), -1, dtype=torch.int32)  # (an odd width: the call pads it)
    for i, n in enumerate(blocks):
        for j in range(n):
            page = order.pop()
            keep = windows is None or (j + 1) * 16 > windows[i][1] or j * 16 < windows[i][0]
            table[i, j] = page if keep else -1
    return table.to(DEV), sum(blocks) + 3


def reference(q, k, v, positions, scale, window, keep_first, softcap, sink):
    """One head of one row: ``q [n, D]``, ``k [total, D]``, ``v [total, E]``, all float64."""
    j = torch.arange(k.shape[0], device=DEV)[None]
    p = positions[:, None]
    seen = j <= p
    if window:
        seen &= (j > p - window) | (j < keep_first)
    s = q @ k.T * scale
    if softcap:
        s = softcap * torch.tanh(s / softcap)
    s = s.masked_fill(~seen, -math.inf)
    top = s.amax(1, keepdim=True)
    if sink is not None:
        top = top.clamp(min=sink)
    e = torch.exp(s - top)
    den = e.sum(1, keepdim=True)
    return e @ v / (den if sink is None else den + torch.exp(sink - top))


# heads, key heads, key size, value size, new tokens, cached tokens, window, kept first keys, softcap, sinks, key heads per value head, float32 result
CASES = [
    (4, 2, 128, 128, [2, 65, 1, 130], [0, 3, 700, 61], 0, 0, 0.0, True, 1, False),
    (6, 2, 128, 128, [200], [0], 48, 5, 0.0, False, 1, False),
    (4, 4, 128, 256, [70, 33], [0, 129], 0, 0, 25.0, False, 2, True),
    (8, 1, 64, 64, [90, 5, 1], [10, 1000, 64], 100, 70, 0.0, False, 1, False),
    (16, 2, 64, 128, [64, 64], [0, 64], 64, 0, 8.0, True, 1, True),
    (48, 1, 128, 128, [3, 40], [500, 0], 0, 0, 0.0, True, 1, False),
    (32, 32, 128, 128, [700, 1300], [0, 0], 256, 4, 0.0, False, 1, False),  # enough blocks for 128-row tiles
    (32, 16, 64, 64, [1500], [100], 0, 0, 0.0, True, 1, False),
    # One query head per key head, so that a block's tokens spread widest: the window of a block's first token still covers the
    # kept first keys, that of its last tokens has left them behind.
    (4, 4, 128, 128, [80, 64], [0, 1], 16, 4, 0.0, False, 1, False),
    (2, 2, 64, 64, [130], [0], 65, 1, 0.0, False, 1, False),
    (3, 3, 128, 256, [330], [188], 456, 4, 0.0, True, 1, True),
    (2, 2, 64, 64, [64, 90, 64, 70], [500, 475, 511, 472], 512, 4, 0.0, False, 1, False),
    (2, 2, 128, 128, [100, 64], [40, 59], 60, 40, 0.0, False, 1, False),  # more kept keys than a wave's half of a tile
    (2, 2, 64, 64, [200], [30], 65, 100, 0.0, False, 1, False),  # more kept keys than the window holds
    (64, 64, 64, 64, [1280], [1000], 1024, 4, 0.0, False, 1, False),  # 128-row tiles
    (64, 64, 128, 128, [1280], [1010], 1024, 40, 0.0, False, 1, False),
    # Few keys, and many query heads per key head beside single tokens: the other kernel's, at both sides of the rules.
    (8, 1, 64, 64, [40, 1, 64], [0, 9, 0], 0, 0, 0.0, True, 1, False),
    (8, 1, 64, 64, [40, 1, 64], [0, 9, 1], 0, 0, 0.0, True, 1, False),
    (16, 16, 128, 256, [64, 2], [0, 60], 0, 0, 0.0, False, 2, True),
    (16, 1, 128, 128, [30, 1, 64, 3], [290, 400, 0, 7], 256, 0, 0.0, True, 1, False),
    (16, 1, 128, 128, [30, 1, 64, 3], [290, 400, 0, 7], 257, 0, 0.0, True, 1, False),
    (8, 1, 64, 64, [70, 1], [200, 300], 60, 30, 9.0, True, 1, False),
]


@pytest.mark.parametrize("case", CASES, ids=[str(i) for i in range(len(CASES))])
def test_exact_attention_over_the_cache(ops, case):
    hq, hkv, d, dv, new, cached, window, keep, cap, sinks, share, out32 = case
    totals = [a + b for a, b in zip(new, cached)]
    behind = [(keep if window else 0, max(0, c - window + 1) if window else 0) for c in cached]
    table, pages = pages_for(totals, 3, behind)
    kc, vc = rand((pages, hkv, 16, d), BF16, 1), rand((pages, hkv // share, dv, 16), BF16, 2)
    t = sum(new)
    q = rand((t, hq * d), BF16, 4, 2.0)
    sink = rand((hq,), F32, 5, 2.0) if sinks else None
    batch, scale = make_batch(new, cached), d ** -0.5
    batch.memo, batch.num_tokens = {}, t
    extra = dict(wide_heads=True, softcap=cap, sinks=sink, value_share=share) if (sinks or cap or share > 1) else dict(exact_weights=True)
    got = ops.paged_attention(q, kc, vc, table, batch, hq, hkv, d, scale, window, dv, keep_first=keep, out_dtype=F32 if out32 else None, **extra)
    assert got.dtype == (F32 if out32 else BF16)
    want, at = torch.empty((t, hq, dv), dtype=torch.float64, device=DEV), 0
    for i, (n, c) in enumerate(zip(new, cached)):
        pg = table[i, : -(-totals[i] // 16)].long().clamp(min=0)
        pos = torch.arange(c, c + n, device=DEV)
        for h in range(hq):
            kh = h * hkv // hq
            k = kc[pg, kh].reshape(-1, d)[: totals[i]].double()
            v = vc[pg, kh // share].transpose(1, 2).reshape(-1, dv)[: totals[i]].double()
            want[at : at + n, h] = reference(q[at : at + n, h * d : (h + 1) * d].double(), k, v, pos, scale, window, keep if window else 0, cap,
                                             None if sink is None else sink[h].double())
        at += n
    # float32 results: scores are float32 sums of exact products, exponentials and sums of weights a few units of 2^-24 each;
    # bfloat16 results are rounded once (2^-9 of the largest)
    close(got.view(t, hq, dv), want, 2e-5 if out32 else 6e-3, "attention")


SHORT, LONG = [1, 8, 9, 64, 65, 250, 257, 700, 1300], [1, 63, 65, 320, 1299, 2048, 2600, 3777, 4001]


@pytest.mark.parametrize("hq,hkv,d,dv,window,keep,cap,share,totals", [
    (4, 1, 128, 128, 0, 0, 0.0, 1, SHORT), (32, 2, 128, 256, 200, 0, 0.0, 2, SHORT), (6, 2, 128, 128, 130, 70, 9.0, 1, SHORT),
    (20, 1, 576, 512, 0, 0, 0.0, 1, SHORT), (3, 1, 576, 128, 300, 4, 0.0, 1, SHORT), (2, 1, 544, 128, 0, 0, 0.0, 1, SHORT),
    (64, 16, 128, 128, 0, 0, 0.0, 1, LONG), (32, 16, 128, 128, 2048, 0, 0.0, 2, LONG), (32, 32, 128, 128, 1500, 70, 9.0, 1, LONG),
    (16, 8, 576, 512, 0, 0, 0.0, 1, LONG), (16, 16, 576, 128, 2000, 4, 0.0, 1, LONG)])
def test_single_tokens_ask_for_a_tile_ahead(ops, hq, hkv, d, dv, window, keep, cap, share, totals):
    """Steps of single tokens whose keys have as many elements as the kernel holds (128, 576; 544 runs the form with a branch): the keys and
    values of a wave's next tile are under way while one is in work, and the page ids of the one after. Rows of one key, of a tile and
    one more, with no tile for some waves, with one or two, and (the long ones, with heads for most of the chip's blocks) with four to
    sixteen; keys and values that no token sees are no numbers, and pages wholly in front of the window are gone."""
    if totals is LONG:  # every block's four waves share the tiles of a split in turn: the page ids asked for two tiles ahead come to use
        tiles = -(-(min(max(totals), window) if window else max(totals)) // 64) + 1
        blocks = len(totals) * hkv * -(-(hq // hkv) // 16) * (dv // 128)
        assert tiles // max(1, min(tiles // 4, -(-ops.MFMA_SPLIT_BLOCKS // blocks))) // 4 >= 4
    table, pages = pages_for(totals, 3, [(keep if window else 0, max(0, n - window) if window else 0) for n in totals])
    kc, vc = rand((pages, hkv, 16, d), BF16, 1), rand((pages, hkv // share, dv, 16), BF16, 2)
    live = torch.zeros((pages, 16), dtype=torch.bool, device=DEV)
    for i, n in enumerate(totals):
        for j in range(n):
            if table[i, j // 16] >= 0 and (not window or j >= n - window or j < keep):
                live[table[i, j // 16], j % 16] = True
    kc.masked_fill_(~live[:, None, :, None], math.nan)
    runs = live.view(pages, 2, 8).any(2).repeat_interleave(8, 1)  # values come eight tokens at a time
    vc.masked_fill_(~runs[:, None, None, :], math.nan)
    q, sink, scale = rand((len(totals), hq * d), BF16, 4, 2.0), rand((hq,), F32, 5, 2.0), d ** -0.5
    batch = make_batch([1] * len(totals), [n - 1 for n in totals])
    batch.memo, batch.num_tokens = {}, len(totals)
    got = ops.paged_attention(q, kc, vc, table, batch, hq, hkv, d, scale, window, dv, keep_first=keep, out_dtype=F32, wide_heads=True, softcap=cap,
                              sinks=sink, value_share=share)
    want = torch.empty((len(totals), hq, dv), dtype=torch.float64, device=DEV)
    for i, n in enumerate(totals):
        pg = table[i, : -(-n // 16)].long().clamp(min=0)
        for h in range(hq):
            kh = h * hkv // hq
            k = kc[pg, kh].reshape(-1, d)[:n].double().nan_to_num()
            v = vc[pg, kh // share].transpose(1, 2).reshape(-1, dv)[:n].double().nan_to_num()
            want[i, h] = reference(q[i : i + 1, h * d : (h + 1) * d].double(), k, v, torch.tensor([n - 1], device=DEV), scale, window,
                                   keep if window else 0, cap, sink[h].double())[0]
    # scores are float32 sums of exact products, exponentials and sums of weights a few units of 2^-24 each
    close(got.view(len(totals), hq, dv), want, 2e-5, "attention")


@pytest.mark.parametrize("tokens", [1, 64])
@pytest.mark.parametrize("d,dv", [(128, 128), (576, 128), (64, 64)])
def test_keys_that_are_no_numbers(ops, d, dv, tokens):
    """A row that sees a key which is no number has no numbers for a result, also where all the scores of a wave so far are none (a whole
    tile of such keys, or the only key that a row sees); rows and heads that do not see one are as without it."""
    totals = [300, 150, 64 + tokens]
    table, pages = pages_for(totals, 6)
    kc, vc = rand((pages, 2, 16, d), BF16, 1), rand((pages, 2, dv, 16), BF16, 2)
    q = rand((len(totals) * tokens, 4 * d), BF16, 4, 2.0)
    batch = make_batch([tokens] * len(totals), [n - tokens for n in totals])
    batch.memo, batch.num_tokens = {}, len(totals) * tokens

    def run():
        got = ops.paged_attention(q, kc, vc, table, batch, 4, 2, d, d ** -0.5, 0, dv, out_dtype=F32, wide_heads=True, exact_weights=True)
        return got.view(len(totals), tokens, 2, 2, dv).clone()

    plain = run()
    assert plain.isfinite().all()
    kc[table[0, :4].long(), 0] = math.nan  # the first row's first 64 keys, of the first key head
    got = run()
    assert got[0, :, 0].isnan().all() and torch.equal(got[0, :, 1], plain[0, :, 1]) and torch.equal(got[1:], plain[1:])


def growing(growth, heads, tokens, cached, d=64):
    """Queries, and a cache of keys whose scores grow by ``growth`` (in units of log2, at a scale of ln 2) with every 64 keys."""
    total = cached + tokens
    table, pages = pages_for([total], 7)
    kc, vc = rand((pages, heads, 16, d), BF16, 1, 0.05), rand((pages, heads, d, 16), BF16, 2)
    at = torch.arange(total, device=DEV)
    kc[table[0].long()[at // 16], :, at % 16, 0] = (growth * at / 64).to(BF16)[:, None]
    q = rand((tokens, heads, d), BF16, 4)
    q[:, :, 0] = 1.0
    batch = make_batch([tokens], [cached])
    batch.memo, batch.num_tokens = {}, tokens
    return q, kc, vc, table, batch, total


@pytest.mark.parametrize("form", ["exact", "sinks"])
@pytest.mark.parametrize("growth", [6.0, 8.5, 40.0])
@pytest.mark.parametrize("heads,tokens", [(2, 150), (64, 1300)])  # 64-row tiles, 128-row tiles
def test_scores_that_grow_along_the_keys(ops, heads, tokens, growth, form):
    """The maximum that the exponents subtract may lag behind a row's own by up to 8: scores that rise by less in a tile of 64 keys, by
    little more, and by far more."""
    q, kc, vc, table, batch, total = growing(growth, heads, tokens, 500)
    d = q.shape[2]
    sink = rand((heads,), F32, 5, 2.0) + growth * total / 64 * math.log(2.0) if form == "sinks" else None
    extra = dict(exact_weights=True) if sink is None else dict(wide_heads=True, sinks=sink)
    got = ops.paged_attention(q.view(tokens, -1), kc, vc, table, batch, heads, heads, d, math.log(2.0), 0, d, out_dtype=F32, **extra).view(tokens, heads, d)
    pg, pos = table[0, : -(-total // 16)].long(), torch.arange(500, total, device=DEV)
    top = growth * total / 64  # the largest score: its float32 sum is off by 2^-24 of it, and a weight by as much of itself
    for h in range(0, heads, 7):
        k, v = kc[pg, h].reshape(-1, d)[:total].double(), vc[pg, h].transpose(1, 2).reshape(-1, d)[:total].double()
        want = reference(q[:, h].double(), k, v, pos, math.log(2.0), 0, 0, 0.0, None if sink is None else sink[h].double())
        close(got[:, h], want, 2e-5 + top * 2.0**-22, f"head {h}")


@pytest.mark.parametrize("heads,tokens", [(2, 150), (64, 1300)])
def test_a_row_does_not_depend_on_the_rows_beside_it(ops, heads, tokens):
    """Other scores in the rows between leave a row's bits as they are, also where theirs renew their maximum and the row's does not."""
    q, kc, vc, table, batch, _ = growing(6.0, heads, tokens, 500)
    d = q.shape[2]

    def run(q):
        return ops.paged_attention(q.view(tokens, -1), kc, vc, table, batch, heads, heads, d, math.log(2.0), 0, d, exact_weights=True, out_dtype=F32)

    other = q.clone()
    other[1::2] *= 4
    assert torch.equal(run(other)[::2], run(q)[::2])


def shifted(x, by):
    """The same values in a contiguous tensor that starts ``by`` bytes behind a 16-byte boundary."""
    n = by // x.element_size()
    flat = torch.empty(x.numel() + n, dtype=x.dtype, device=DEV)
    flat[n:] = x.flatten()
    return flat[n:].view(x.shape)


@pytest.mark.parametrize("which,by", [("q", 4), ("q", 8), ("k", 8), ("v", 4), ("table", 4)])
@pytest.mark.parametrize("form", ["exact", "sinks"])
def test_views_at_any_address(ops, which, by, form):
    """The kernel over LDS tiles takes bases at multiples of 16 bytes; others are served as they were without it."""
    hq, hkv, d, new, cached = 8, 2, 64, [150, 1, 70], [0, 90, 300]
    table, pages = pages_for([a + b for a, b in zip(new, cached)], 3)
    table = torch.nn.functional.pad(table, (0, -table.shape[1] % 4))  # rows of whole fours: not copied for their width
    args = {"q": rand((sum(new), hq * d), BF16, 4, 2.0), "k": rand((pages, hkv, 16, d), BF16, 1), "v": rand((pages, hkv, d, 16), BF16, 2), "table": table}
    extra = dict(exact_weights=True) if form == "exact" else dict(wide_heads=True, sinks=rand((hq,), F32, 5))

    def run(a):
        batch = make_batch(new, cached)
        batch.memo, batch.num_tokens = {}, sum(new)
        return ops.paged_attention(a["q"], a["k"], a["v"], a["table"], batch, hq, hkv, d, d ** -0.5, 0, d, **extra)

    close(run(dict(args, **{which: shifted(args[which], by)})), run(args).double(), 1.2e-2, "attention")  # both rounded to bfloat16


# heads, key heads, key size, value size, new tokens, cached tokens, window, kept first keys, key heads per value head
POISONED = [
    (4, 2, 128, 128, [70], [0], 0, 0, 1),
    (4, 4, 64, 64, [40, 3], [500, 1], 100, 20, 1),
    (4, 4, 128, 256, [33, 50, 1], [129, 7, 300], 0, 0, 2),
    (16, 2, 64, 128, [90], [410], 64, 0, 1),
    (64, 64, 64, 64, [1290], [1000], 256, 5, 1),  # 128-row tiles
]


@pytest.mark.parametrize("case", POISONED, ids=[str(i) for i in range(len(POISONED))])
def test_what_no_token_may_see_does_not_reach_a_result(ops, case):
    """Infinities and NaN in pages of other requests (page 0, which table entries without a page point at, among them) and behind a
    row's last key: the results are the bits of a cache that holds zeros there."""
    hq, hkv, d, dv, new, cached, window, keep, share = case
    totals = [a + b for a, b in zip(new, cached)]
    table, pages = pages_for(totals, 14, [(keep if window else 0, max(0, c - window + 1) if window else 0) for c in cached])
    table = torch.where(table >= 0, table + 1, table)  # page 0 belongs to no row
    clean = [rand((pages + 1, hkv, 16, d), BF16, 15), rand((pages + 1, hkv // share, dv, 16), BF16, 16)]
    owned = torch.zeros((pages + 1, 16), dtype=torch.bool, device=DEV)
    for i, n in enumerate(totals):
        first = max(0, cached[i] - window + 1) if window else 0
        for j in range(n):
            if (j >= first or j < keep) and int(table[i, j // 16]) > 0:
                owned[table[i, j // 16], j % 16] = True
    t = sum(new)
    q = rand((t, hq * d), BF16, 17, 2.0)
    batch = make_batch(new, cached)
    batch.memo, batch.num_tokens = {}, t
    extra = dict(wide_heads=True, value_share=share) if share > 1 else dict(exact_weights=True)
    got = []
    for bad in (0.0, math.nan, math.inf):
        kc, vc = (x.clone() for x in clean)
        kc.transpose(1, 2)[~owned] = bad
        vc.permute(0, 3, 1, 2)[~owned] = bad
        out = ops.paged_attention(q, kc, vc, table, batch, hq, hkv, d, d ** -0.5, window, dv, keep_first=keep, **extra)
        single = torch.tensor([n == 1 for n in new for _ in range(n)], device=DEV)
        got.append(out[~single])  # (tokens of rows that bring one run another kernel)
    assert got[0].isfinite().all()
    assert torch.equal(got[0], got[1]) and torch.equal(got[0], got[2])


# heads, new tokens, cached tokens, window, sinks, gate ("head", "element", None), latent size
EXPANDED = [
    (2, [130], [0], 0, False, None, 64),
    (3, [70, 1, 200, 2], [0, 300, 75, 500], 0, True, "head", 64),
    (2, [65, 64], [200, 64], 100, True, "element", 40),
    (8, [600, 1100], [0, 37], 0, False, "element", 64),  # 128-row tiles
    (16, [700], [1000], 512, False, None, 512),
]


@pytest.mark.parametrize("case", EXPANDED, ids=[str(i) for i in range(len(EXPANDED))])
def test_expanded_latent_attention(ops, case):
    heads, new, cached, window, sinks, gating, latent = case
    dn, r, dv = 128, 64, 128
    totals = [a + b for a, b in zip(new, cached)]
    table, pages = pages_for(totals, 6, [(0, max(0, c - window + 1) if window else 0) for c in cached])
    kc = rand((pages, 1, 16, latent + r), BF16, 7)
    uk, uv = rand((heads * dn, latent), BF16, 8, latent ** -0.5), rand((heads * dv, latent), BF16, 9, latent ** -0.5)
    t = sum(new)
    plain, full = rand((t, heads * dn), BF16, 10), rand((t, heads * (latent + r)), BF16, 11)
    sink = rand((heads,), F32, 12, 2.0) if sinks else None
    g = rand((t, 3 + heads * dv), F32, 13) if gating else None
    batch, scale = make_batch(new, cached), (dn + r) ** -0.5
    batch.memo, batch.num_tokens = {}, t
    plan = ops.latent_expansion(batch, kc, heads, dn, r, latent, dv, window)
    out = torch.full((t, heads * dv), 7.0, dtype=BF16, device=DEV)
    ops.expanded_attention(plain, full, kc, table, batch, plan, uk, uv, heads, dn, r, latent, dv, scale, window, sink,
                           (g, 3) if gating else None, gating == "element", out)
    at = 0
    for i, (n, c) in enumerate(zip(new, cached)):
        rows = slice(at, at + n)
        at += n
        if n == 1:  # left to the caller
            assert (out[rows] == 7.0).all()
            continue
        pg = table[i, : -(-totals[i] // 16)].long().clamp(min=0)
        both = kc[pg, 0].reshape(-1, latent + r)[: totals[i]]
        lat, turned = both[:, :latent].double(), both[:, latent:].double()
        pos = torch.arange(c, c + n, device=DEV)
        want = torch.empty((n, heads, dv), dtype=torch.float64, device=DEV)
        for h in range(heads):
            k = torch.cat(((lat @ uk[h * dn : (h + 1) * dn].double().T), turned), 1)
            q = torch.cat((plain[rows, h * dn : (h + 1) * dn], full[rows].view(n, heads, -1)[:, h, latent:]), 1).double()
            want[:, h] = reference(q, k, lat @ uv[h * dv : (h + 1) * dv].double().T, pos, scale, window, 0, 0.0, None if sink is None else sink[h].double())
        if gating:
            z = torch.sigmoid(g[rows, 3:].double())
            want = want * (z.view(n, heads, dv) if gating == "element" else z[:, :heads, None])
        # keys, values and the result are rounded to bfloat16 once each
        close(out[rows].view(n, heads, dv), want, 1.2e-2, f"row {i}")


def test_expansion_plan_covers_what_the_window_shows(ops):
    rows, at, left, base = ops.plan_latent_expansion([1, 5, 130], [9, 300, 0], 100)
    assert rows == [1, 1, 2, 2, 2] and at == [192, 256, 0, 64, 128] and left == [64, 49, 64, 64, 2]
    assert base == [0, -192, 128]
