"""The pooled-window attention on the matrix cores, against the
design's equations in 64 bits on the same bfloat16 operands; and against the general form's error."""

import math

import pytest
import torch

from kernel_util import make_batch

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


def reference(q, k, v, talk, i0, window, pool, scale):
    """q [t, H, d] at positions i0 ..., k / v [T, G, .] of all positions up to the last: float64 [t, H, e]."""
    t, heads = q.shape[:2]
    n, kv = k.shape[:2]
    nb = n // pool
    mean = lambda a: a[:nb * pool].reshape(nb, pool, *a.shape[1:]).mean(1)
    keys, values = torch.cat([k, mean(k)]), torch.cat([v, mean(v)])
    i = torch.arange(i0, i0 + t)[:, None]
    j, b = torch.arange(n)[None], torch.arange(nb)[None]
    seen = torch.cat([(j <= i) & (i - j < window), b * pool + pool - 1 <= i - window], dim=1)
    w = torch.stack([torch.softmax(((q[:, a] @ keys[:, a // (heads // kv)].T) * scale).masked_fill(~seen, -math.inf), dim=-1)
                     for a in range(heads)])
    w = (talk @ w.flatten(1)).view(heads, t, -1)
    return torch.stack([w[a] @ values[:, a // (heads // kv)] for a in range(heads)], dim=1)


CASES = {
    # H, G, dim, vdim, window, pool, page, (tokens, cached) of each request
    "wide": (32, 8, 128, 128, 64, 16, 16, [(17, 0), (1, 300), (40, 133), (16, 16)]),
    "long": (32, 8, 128, 128, 1024, 16, 16, [(70, 1500)]),
    "window of 1": (16, 4, 64, 64, 1, 3, 16, [(2, 0), (33, 50), (1, 0)]),
    "two heads a kv head": (16, 8, 128, 64, 37, 5, 48, [(15, 201), (31, 0), (1, 90), (3, 47)]),
    "a kv head a head": (16, 16, 64, 128, 100, 7, 32, [(48, 95), (5, 700)]),
    "single tokens": (32, 8, 128, 128, 256, 16, 16, [(1, 0), (1, 255), (1, 900), (1, 15), (1, 1200)]),
    "one kv head": (32, 1, 64, 64, 33, 1, 16, [(32, 31), (2, 255)]),
}


def step(name, opposite=False):
    """A case's step: what computes it, the result in 64 bits, the batch, the arrays on the GPU.  ``opposite``:
    every second head is the one before it but for a few of its numbers' last bits, and the mixing takes their difference."""
    from tokamak_amd.kernels import ops

    heads, kv, dim, vdim, window, pool, page, spans = CASES[name]
    g = torch.Generator().manual_seed(len(name))
    scale, ke, ve = dim ** -0.5, -(-kv * dim // pool), -(-kv * vdim // pool)
    talk = torch.eye(heads) + 0.3 * torch.randn(heads, heads, generator=g)
    if opposite:
        talk = torch.eye(heads).view(heads // 2, 2, heads).clone()
        talk = (talk - talk.flip(1)).view(heads, heads)
    total = sum(-(-(n + c) // page) for n, c in spans)
    order = torch.randperm(total + 3, generator=g).tolist()
    nan = float("nan")
    k_cache, v_cache = torch.full((total + 3, kv * dim * page), nan), torch.full((total + 3, kv * vdim * page), nan)
    k_pool, v_pool = torch.full((total + 3, ke * page), nan), torch.full((total + 3, ve * page), nan)
    rows, tables, queries, want = [], [], [], []
    for n, cached in spans:
        length = n + cached
        table, order = order[:-(-length // page)], order[-(-length // page):]
        tables.append(table)
        k = (1.5 * torch.randn(length, kv, dim, generator=g)).bfloat16().double()
        v = torch.randn(length, kv, vdim, generator=g).bfloat16().double()
        q = torch.randn(n, heads, dim, generator=g).bfloat16()
        if opposite:
            q = (0.25 * q).unflatten(1, (heads // 2, 2))
            q[:, :, 1] = q[:, :, 0]
            q[:, :, 1, :4] *= 1.0 + 2.0 ** -7
            q = q.flatten(1, 2)
        for p in range(length):
            at = p % page
            k_cache[table[p // page], at * kv * dim:(at + 1) * kv * dim] = k[p].flatten().float()
            v_cache[table[p // page], at * kv * vdim:(at + 1) * kv * vdim] = v[p].flatten().float()
        for b in range(length // pool):
            for array, x, e in ((k_pool, k, ke), (v_pool, v, ve)):
                mean = x[b * pool:(b + 1) * pool].mean(0).flatten().float()
                for c, value in zip(range(b * mean.numel(), (b + 1) * mean.numel()), mean.tolist()):
                    array[table[c // (page * e)], c % (page * e)] = value
        queries.append(q.flatten(1))
        want.append(reference(q.double(), k, v, talk.double(), cached, window, pool, scale).flatten(1))
        rows.append((n, cached, table))
    batch = make_batch(rows)
    arrays = [t.to(DEV) for t in (k_cache.bfloat16(), v_cache.bfloat16(), k_pool, v_pool)]
    q = torch.cat(queries).to(DEV)

    def run():
        out = torch.full((q.shape[0], heads * vdim), nan, dtype=torch.bfloat16, device=DEV)
        ops.pooled_window_attention(q, *arrays, batch.block_tables[0], batch, talk.to(DEV), out, num_heads=heads, num_kv_heads=kv,
                                    dim=dim, vdim=vdim, window=window, pool=pool, page_size=page, scale=scale)
        return out.cpu().double()

    assert ops.pooled_portions_pay(heads, kv, dim, vdim, page)
    return run, torch.cat(want), batch, arrays


@pytest.mark.parametrize("name", ["long", "window of 1", "two heads a kv head", "single tokens"])
def test_heads_mixed_with_opposite_signs(name):
    """What two nearly equal heads' weights differ by is a small part of them: it is there only if the weights, the mixing and
    the mixed weights keep float32's bits (of 16 of them, in two bfloat16 pieces, the result would be 2^-7 off)."""
    run, want, _, _ = step(name, opposite=True)
    # the final rounding, at most 2^-9 of a result, and half as much for the float32 scores
    off = float((run() - want).norm() / want.norm())
    assert off <= 2.0 ** -9 + 2.0 ** -10, off


@pytest.mark.parametrize("name", list(CASES))
def test_portions_on_the_matrix_cores(name, monkeypatch):
    from tokamak_amd.kernels import ops

    heads, kv, dim, vdim, window, pool, page, spans = CASES[name]
    run, want, batch, arrays = step(name)
    nan, tokens = float("nan"), want.shape[0]
    got = run()
    # rounded once to bfloat16 (2^-9 of the result), and 1e-4 of the largest sum of products where products cancel
    bound = 2.0 ** -8 * want.abs() + 1e-4 * float(want.abs().max())
    assert bool(((got - want).abs() <= bound).all()), float(((got - want).abs() - bound).max())
    monkeypatch.setattr(ops, "pooled_portions_pay", lambda *a: False)
    general = run()
    # no further from the 64-bit result than the form with float32 weights (both are the final rounding away)
    assert float((got - want).norm()) <= 1.02 * float((general - want).norm())
    # the step's own means: a mean of `pool` float32 sums in order, and nothing written beside the blocks it completes
    fresh = [torch.full_like(t, nan) for t in arrays[2:]]
    ops.pool_blocks(*arrays[:2], *fresh, batch.positions, batch.req_of_token, batch.block_tables[0], tokens,
                    k_width=kv * dim, v_width=kv * vdim, pool=pool, page_size=page)
    complete = sum((n + cached) // pool - cached // pool for n, cached in spans)
    for mean, known, width in zip(fresh, arrays[2:], (kv * dim, kv * vdim)):
        written = ~mean.isnan()
        assert int(written.sum()) == complete * width
        assert bool(((mean - known)[written].abs() <= pool * 2.0 ** -23 * 8.0).all())      # (no input is beyond 8)
