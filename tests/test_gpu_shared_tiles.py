"""Tiles whose heads share their keys and values through a ring of stages in LDS: walks shorter and longer than the ring, sizes
between whole chunks and blocks, the jump from the kept positions to the window, pages of several stages, groups of every block
width; what lies in the pages behind a request's last position is not a number and must not show."""

import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


def made(heads, kv, hd, vd, ps, portions, window, keep):
    """The operands of a step's portions (tokens, tokens before them), what it should give, and what its weights' rounding meets."""
    g = torch.Generator().manual_seed(hd + vd)
    rand = lambda *shape: torch.randn(*shape, generator=g).bfloat16()
    n = sum(t for t, _ in portions)
    pages = [-(-(t + ctx) // ps) for t, ctx in portions]
    numbers = torch.randperm(sum(pages), generator=g).tolist()
    table = torch.zeros((len(portions), max(pages)), dtype=torch.int32)
    k_cache = torch.full((sum(pages), kv, hd // 8, ps, 8), float("nan"), dtype=torch.bfloat16)
    v_cache = torch.full((sum(pages), kv, vd // 16, ps // 4, 16, 4), float("nan"), dtype=torch.bfloat16)
    q = rand(n, heads, hd)
    positions, request, first, count, want, bound = [], [], [], [], [], []
    for r, (tokens, ctx) in enumerate(portions):
        mine, numbers = numbers[:pages[r]], numbers[pages[r]:]
        table[r, :len(mine)] = torch.tensor(mine, dtype=torch.int32)
        k, v = rand(ctx + tokens, kv, hd), rand(ctx + tokens, kv, vd)
        for p in range(ctx + tokens):
            k_cache[mine[p // ps], :, :, p % ps] = k[p].view(kv, hd // 8, 8)
            v_cache[mine[p // ps], :, :, p % ps // 4, :, p % 4] = v[p].view(kv, vd // 16, 16)
        at = len(positions)
        positions += range(ctx, ctx + tokens)
        request += [r] * tokens
        first += range(at, at + tokens, 16)
        count += [min(16, tokens - i) for i in range(0, tokens, 16)]
        i, j = torch.arange(ctx, ctx + tokens)[:, None], torch.arange(ctx + tokens)[None]
        seen = (j <= i) & ((j > i - window) | (j < keep) if window else True)
        kk, vv = (x.float().repeat_interleave(heads // kv, 1).transpose(0, 1) for x in (k, v))
        scores = q[at:at + tokens].float().transpose(0, 1) @ kk.transpose(1, 2) * hd ** -0.5
        p = torch.softmax(scores.masked_fill(~seen, float("-inf")), -1)
        want.append((p @ vv).transpose(0, 1))
        bound.append((p @ vv.abs()).transpose(0, 1))
    ints = lambda x: torch.tensor(x, dtype=torch.int32, device=DEV)
    operands = [x.to(DEV) for x in (q, k_cache, v_cache, table)] + [ints(positions), ints(request)]
    sizes = dict(num_heads=heads, num_kv_heads=kv, head_dim=hd, value_dim=vd, page_size=ps, scale=hd ** -0.5, window=window, keep_first=keep)
    return operands, ints(first), ints(count), torch.full((n, heads, vd), float("nan"), dtype=torch.bfloat16, device=DEV), sizes, torch.cat(want), torch.cat(bound)


def near(out, want, bound):
    # weights rounded to bfloat16 (seven bits behind the leading one: 2^-8 each) and the result (2^-8), and a twentieth for float32
    # sums and exponentials
    off = (out.cpu().float() - want).abs() - 1.05 * 2.0 ** -7 * bound
    assert bool((off <= 0).all()), float(off.max())


@pytest.mark.parametrize("heads,kv,hd,vd,ps,portions,window,keep", [
    (4, 2, 64, 64, 16, [(1, 0), (16, 0), (17, 31)], None, 0),          # two waves a block; one to three stages
    (6, 2, 40, 48, 32, [(33, 15), (5, 200)], None, 0),                 # pieces and blocks behind the true sizes
    (4, 2, 80, 64, 16, [(1, 0), (16, 0), (17, 31)], None, 0),          # two heads a kv head share from 144 channels on
    (6, 2, 72, 80, 32, [(33, 15), (5, 200)], None, 0),
    (8, 2, 128, 128, 16, [(64, 0), (3, 333)], 50, 0),
    (5, 1, 8, 16, 48, [(20, 90)], 33, 20),                             # the smallest sizes; kept positions, then the window
    (9, 1, 136, 272, 16, [(40, 100)], 64, 4),                          # a second block of heads with one of its own
    (16, 2, 256, 256, 64, [(50, 0), (16, 112)], None, 0),
    (16, 1, 320, 256, 16, [(23, 41)], None, 0),
    (8, 1, 512, 448, 16, [(100, 60)], 96, 0),
    (4, 1, 512, 512, 32, [(18, 70)], None, 0)])
def test_shared_tiles(heads, kv, hd, vd, ps, portions, window, keep):
    from tokamak_amd.kernels import ops

    operands, first, count, out, sizes, want, bound = made(heads, kv, hd, vd, ps, portions, window, keep)
    assert ops.attention_tiles(*operands, first, count, first.numel(), out, **sizes)
    near(out, want, bound)


@pytest.mark.parametrize("heads,kv,hd,vd,contexts,window,keep,splits", [
    (8, 1, 32, 16, [0, 15, 16, 200], None, 0, 1),
    (8, 1, 64, 48, [63, 5], 20, 0, 5),                # most parts have no keys
    (17, 1, 136, 272, [300, 1], None, 0, 5),
    (16, 2, 128, 128, [700], 100, 4, 3),
    (32, 1, 512, 448, [1040, 90], 1024, 0, 2), (8, 1, 64, 272, [0, 400, 33], None, 0, 4), (24, 2, 40, 80, [130, 7], 50, 20, 1),      # 8, 16 and 4
    (32, 1, 512, 448, [1040], 1024, 0, 16)])          # 64 parts and one step more
def test_single_tokens_merged(heads, kv, hd, vd, contexts, window, keep, splits):
    """A token's keys dealt to parts, from one to as many as the merge takes, some of them without keys."""
    from tokamak_amd.kernels import ops

    operands, first, _, out, sizes, want, bound = made(heads, kv, hd, vd, 16, [(1, c) for c in contexts], window, keep)
    ops.attention_heads(*operands, first, first.numel(), out, num_splits=splits, **sizes)
    near(out, want, bound)
