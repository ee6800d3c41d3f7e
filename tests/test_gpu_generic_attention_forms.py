"""The generic attention kernel's forms give the same bits: float32 tiles on the matrix cores, tokens alone (a block or two a CU), heads
that share a block; at the edges of rounds, tiles, pages and windows, and against float64."""

import pytest
import torch

from tokamak_amd.kernels import ops
from tokamak_amd.kernels.build import load_library

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


def step(requests, nh, nkv, hd, vd, ps, dtype):
    """Requests of (cached, new) tokens: random queries, pages in no order, NaN in what no page holds; a table names the
    pages that a window has given back by a page of NaN."""
    gen = torch.Generator().manual_seed(sum(c + 7 * q for c, q in requests) + hd)
    pages = [-(-(c + q) // ps) for c, q in requests]
    order = (torch.randperm(sum(pages), generator=gen) + 1).tolist()
    keys = torch.full((sum(pages) + 1, nkv, hd // 8, ps, 8), float("nan"))
    values = torch.full((sum(pages) + 1, nkv, vd // 16, ps // 4, 16, 4), float("nan"))
    tables = torch.zeros((len(requests), max(pages)), dtype=torch.int32)
    rows, tiles, single, plain, row = [], [], [], [], 0
    for r, ((c, q), n) in enumerate(zip(requests, pages)):
        own, order = order[:n], order[n:]
        tables[r, :n] = torch.tensor(own, dtype=torch.int32)
        k, v = torch.randn(c + q, nkv, hd, generator=gen).to(dtype), torch.randn(c + q, nkv, vd, generator=gen).to(dtype)
        at = torch.arange(c + q)
        page = torch.tensor(own)[at // ps]
        keys[page, :, :, at % ps] = k.view(-1, nkv, hd // 8, 8).float()
        values[page, :, :, at % ps // 4, :, at % 4] = v.view(-1, nkv, vd // 16, 16).float()
        rows += [(c + t, r) for t in range(q)]
        tiles += [(row + t, min(16, q - t)) for t in range(0, q, 16)] if q > 1 else []
        single += [row] if q == 1 else []
        plain.append((k.double(), v.double()))
        row += q
    ints = lambda values: torch.tensor(values or [0], dtype=torch.int32, device=DEV)      # noqa: E731
    return {"q": torch.randn(row, nh * hd, generator=gen).to(dtype).to(DEV), "k": keys.to(dtype).to(DEV), "v": values.to(dtype).to(DEV), "tables": tables,
            "positions": ints([p for p, _ in rows]), "requests": ints([r for _, r in rows]), "plain": plain,
            "tiles": (ints([t for t, _ in tiles]), ints([n for _, n in tiles]), len(tiles), ints(single), len(single))}


def attend(s, nh, nkv, hd, vd, ps, tiled, share=None, **kw):
    out = torch.full((s["q"].shape[0], nh * vd), float("nan"), dtype=s["q"].dtype, device=DEV)
    ops.paged_attention_generic(s["q"], s["k"], s["v"], s["tables"].to(DEV), s["positions"], s["requests"], out, num_heads=nh, num_kv_heads=nkv,
                                head_dim=hd, page_size=ps, scale=hd ** -0.5, value_dim=vd, tiles=s["tiles"] if tiled else None, share_heads=share, **kw)
    return out


def seen(pos, keys, window=None, chunk=None, keep_first=0):
    at = torch.arange(keys)
    if window:
        return (at <= pos) & ((at > pos - window) | (at < keep_first))
    return (at <= pos) & (at >= (pos - pos % chunk if chunk else 0))


def exact(s, nh, nkv, hd, vd, sinks=None, softcap=None, **kw):
    out = []
    q, positions, of = s["q"].cpu().double().view(-1, nh, hd), s["positions"].tolist(), s["requests"].tolist()
    for n in range(q.shape[0]):
        k, v = s["plain"][of[n]]
        there = seen(positions[n], k.shape[0], **kw)
        for a in range(nh):
            score = k[there, a // (nh // nkv)] @ q[n, a] * hd ** -0.5
            score = score if softcap is None else softcap * torch.tanh(score / softcap)
            if sinks is not None:
                score = torch.cat([score, sinks[a:a + 1].cpu().double()])
            out.append(torch.softmax(score, 0)[:int(there.sum())] @ v[there, a // (nh // nkv)])
    return torch.stack(out).view(q.shape[0], nh * vd)


def give_back(s, ps, window, keep_first):
    """The pages that no query of the step sees belong to others: their places in the tables name a page of NaN."""
    first = {}
    for p, r in zip(s["positions"].tolist(), s["requests"].tolist()):
        first[r] = min(first.get(r, p), p)
    for r, pos in first.items():
        for page in range((pos - window + 1) // ps if pos >= window else 0):
            if page * ps >= keep_first:
                s["tables"][r, page] = 0


# tiles of one, 15, 16, 17 tokens, contexts at the edges of rounds of 64 and of pages; even and odd groups
FORMS = [(4, 2, 128, 128, 16, {}), (3, 1, 64, 64, 32, {"window": 64}), (4, 1, 128, 128, 48, {"window": 37, "keep_first": 5}), (2, 2, 64, 64, 16, {"chunk": 50}),
         (6, 3, 128, 128, 16, {"window": 100, "keep_first": 70, "softcap": 5.0}), (2, 1, 128, 128, 16, {"sinks": True}),
         (4, 2, 128, 128, 24, {}), (4, 2, 64, 32, 16, {"window": 65}), (2, 2, 192, 192, 8, {"chunk": 64})]


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("form", FORMS)
@pytest.mark.parametrize("requests", [[(0, 1), (63, 16), (64, 17), (0, 33)], [(200, 2), (447, 15), (575, 1), (128, 66)]])
def test_forms_agree(requests, form, dtype):
    nh, nkv, hd, vd, ps, kw = form
    kw = dict(kw, sinks=torch.linspace(-1.0, 1.0, nh, device=DEV)) if "sinks" in kw else kw
    s = step(requests, nh, nkv, hd, vd, ps, dtype)
    if "window" in kw:
        give_back(s, ps, kw["window"], kw.get("keep_first", 0))
    tiled, alone, shared = (attend(s, nh, nkv, hd, vd, ps, *how, **kw) for how in ((True,), (False, False), (False, True)))
    assert torch.equal(tiled, alone) and torch.equal(alone, shared)
    want = exact(s, nh, nkv, hd, vd, **kw)
    # float32 sums of hd and of the keys seen, and exponents of scores of magnitude up to 8: some 2^-24 (hd / 4 + 8 + 64) of values of up to 4;
    # bfloat16 results half a unit of theirs (2^-9) beside
    assert bool(((tiled.cpu().double() - want).abs() <= 4 * 2.0 ** -24 * (hd / 4 + 72) + (2.0 ** -8 * want.abs() if dtype == torch.bfloat16 else 0)).all())


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("hd, kw", [(128, {}), (64, {"window": 70, "keep_first": 3}), (192, {"window": 200})])
def test_more_tokens_alone_than_cus(dtype, hd, kw):
    nh, nkv, ps = 16, 8, 16
    s = step([(1 + 37 * i % 260, 1) for i in range(18)], nh, nkv, hd, hd, ps, dtype)
    many = attend(s, nh, nkv, hd, hd, ps, False, False, **kw)
    few = torch.empty_like(many)
    for at in range(0, 18, 6):      # the same tokens in blocks that have a CU each
        part = dict(s, q=s["q"][at:at + 6], positions=s["positions"][at:at + 6], requests=s["requests"][at:at + 6])
        few[at:at + 6] = attend(part, nh, nkv, hd, hd, ps, False, False, **kw)
    assert torch.equal(many, few) and torch.equal(many, attend(s, nh, nkv, hd, hd, ps, False, True, **kw)) and not bool(many.isnan().any())


# (the tiles' product takes all keys of a tile's tokens: a value of a later token must not meet an earlier one's weight of zero)
@pytest.mark.parametrize("number", [float("inf"), float("nan")])
@pytest.mark.parametrize("where", ["v", "k"])
@pytest.mark.parametrize("form", [f for f in FORMS if f[2] == f[3] and f[2] in (64, 128) and f[4] % 16 == 0])
def test_numbers_that_are_not_finite_show_where_they_are_seen(form, where, number):
    nh, nkv, hd, vd, ps, kw = form
    kw = dict(kw, sinks=torch.linspace(-1.0, 1.0, nh, device=DEV)) if "sinks" in kw else kw
    requests = [(63, 33), (0, 17), (130, 20), (64, 16)]
    s = step(requests, nh, nkv, hd, vd, ps, torch.float32)
    # the last token's key of a tile, one amid a tile, one that a window leaves behind within a tile, the first one's
    for r, key in enumerate([78, 9, 100, 64]):
        page = int(s["tables"][r, key // ps])
        if where == "v":
            s["v"][page, :, 1, key % ps // 4, 5, key % 4] = number
        else:
            s["k"][page, :, 1, key % ps, 3] = number
    tiled, alone = (attend(s, nh, nkv, hd, vd, ps, tiles, False, **kw) for tiles in (True, False))
    assert torch.equal(tiled.isnan(), alone.isnan()) and torch.equal(tiled.nan_to_num(nan=7.0), alone.nan_to_num(nan=7.0))
    row = 0
    for (cached, new), key in zip(requests, [78, 9, 100, 64]):
        for t in range(new):
            there = seen(cached + t, cached + new, **{n: v for n, v in kw.items() if n not in ("sinks", "softcap")})
            assert bool(there[key]) or bool(tiled[row + t].isfinite().all())
        row += new


@pytest.mark.parametrize("hd, kw", [(128, {}), (128, {"window": 70, "keep_first": 3}), (64, {}), (64, {"chunk": 90})])
def test_many_tiles_of_many_heads(hd, kw):
    """Enough tiles for blocks of two heads where the head size has them; infinities among the values, too."""
    nh, nkv, ps = 16, 4, 16
    s = step([(0, 170), (33, 140), (90, 16)], nh, nkv, hd, hd, ps, torch.float32)
    if "window" in kw:
        give_back(s, ps, kw["window"], kw.get("keep_first", 0))
    assert load_library("attention_generic").tk_attention_tile_heads(s["tiles"][2], nh, nkv, hd) == (2 if hd == 128 else 1)
    tiled, alone = (attend(s, nh, nkv, hd, hd, ps, tiles, False, **kw) for tiles in (True, False))
    assert torch.equal(tiled, alone) and bool(tiled.isfinite().all())
    page = int(s["tables"][0, 100 // ps])
    s["v"][page, :, 1, 100 % ps // 4, 5, 100 % 4] = float("inf")
    tiled, alone = (attend(s, nh, nkv, hd, hd, ps, tiles, False, **kw) for tiles in (True, False))
    assert torch.equal(tiled, alone) and bool(tiled[:100].isfinite().all()) and bool(tiled[100].isinf().any())
