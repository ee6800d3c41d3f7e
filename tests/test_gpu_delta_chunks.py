"""The delta rule's scan in chunks of 16 tokens, against the recurrence in 64 bits on the same operands and against the
walk a token at a time; state slots out of order, a foreign slot untouched."""

import pytest
import torch

from kernel_util import make_batch

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


def recurrence(q, k, v, a, beta, state):
    """[T, H, d] operands in float64, state [H, vdim, dim]."""
    out = []
    for t in range(q.shape[0]):
        state = state * a[t][:, None, :]
        u = beta[t][:, None] * (v[t] - (state * k[t][:, None, :]).sum(-1))
        state = state + u[:, :, None] * k[t][:, None, :]
        out.append((state * q[t][:, None, :]).sum(-1))
    return torch.stack(out), state


@pytest.mark.parametrize("heads,kv,dim,vdim,spans", [
    (2, 2, 128, 128, [129]), (4, 2, 64, 64, [16, 1, 47]), (8, 8, 16, 16, [32]), (3, 1, 48, 32, [100, 15, 17]),
    (4, 4, 80, 112, [64, 2]), (2, 1, 128, 16, [33, 400]),
    (2, 2, 16, 128, [31, 5]), (3, 1, 96, 128, [100, 15, 17]), (2, 2, 112, 112, [47, 400]), (8, 4, 80, 128, [64, 2, 33])])
@pytest.mark.parametrize("decays", ["slow", "fast", "none"])
def test_chunks(heads, kv, dim, vdim, spans, decays, monkeypatch):
    from tokamak_amd.kernels import ops

    monkeypatch.setattr(ops, "DELTA_CHUNKS_FROM_TOKENS", 16)
    g = torch.Generator().manual_seed(dim + len(spans))
    n = sum(spans)
    rand = lambda *shape: torch.randn(*shape, generator=g)
    unit = lambda x: x / x.norm(dim=-1, keepdim=True)
    # neighbours share much of their keys, so that a chunk's tokens correct one another
    q, k = unit(rand(n, kv, dim)) * dim ** -0.5, unit(rand(n, kv, dim) + rand(1, kv, dim))
    v, beta = rand(n, heads, vdim), torch.sigmoid(2.0 * rand(n, heads))
    # fast: decays of 1e-3 and far less within a chunk, down to those that are zero in float32 (nothing may be divided by one)
    z = rand(n, heads, dim)
    a = torch.exp(-torch.exp(z + {"slow": -3.0, "fast": 2.0, "none": -80.0}[decays]))
    row = torch.zeros((n, ops.delta_row(heads, kv, dim, vdim)))
    flat = torch.cat([x.flatten(1) for x in (q, k, v, a, beta)], 1)
    row[:, :flat.shape[1]] = flat
    slots = [len(spans) - 1 - i for i in range(len(spans))]
    state = rand(len(spans) + 1, heads, vdim, dim)
    batch = make_batch([(t, 50, [0] * 64) for t in spans])
    batch.state_slots.copy_(torch.tensor(slots, dtype=torch.int32))
    want, want_state, at = [], {}, 0
    for t, slot in zip(spans, slots):
        rows = slice(at, at + t)
        o, want_state[slot] = recurrence(*(x[rows].double().repeat_interleave(heads // kv, 1) for x in (q, k)), v[rows].double(),
                                         a[rows].double(), beta[rows].double(), state[slot].double())
        want.append(o)
        at += t
    want = torch.cat(want)

    def run(chunks):
        s, y = state.to(DEV), torch.empty((n, heads * vdim), device=DEV)
        ops.delta_scan(row.to(DEV), s, y, batch, heads=heads, kv_heads=kv, dim=dim, vdim=vdim, chunks=chunks)
        return y.cpu().double().view(n, heads, vdim), s.cpu()

    got, got_state = run(True)
    walked, walked_state = run(False)
    assert torch.equal(got_state[-1], state[-1]) and torch.equal(walked_state[-1], state[-1])
    # sums of float32 products: a few roundings of 2^-24 each.  No further from 64 bits than the walk, but for a quarter and
    # 2^-26 of chance: a walk of few tokens rounds little, and a chunk rounds its scaled rows, M and A once more
    def near(pair, exact):
        off = [float((x.double() - exact).norm() / exact.norm()) for x in pair]
        assert off[0] < 2.0 ** -21 and off[0] <= 1.25 * off[1] + 2.0 ** -26, off

    near((got, walked), want)
    for slot, s in want_state.items():
        near((got_state[slot], walked_state[slot]), s)


@pytest.mark.parametrize("where", ["q", "k", "v", "a", "beta", "state"])
@pytest.mark.parametrize("number", [float("inf"), float("-inf"), float("nan")])
def test_numbers_that_are_not_finite_look_ahead_alone(where, number, monkeypatch):
    """A token's number that is not finite shows from that token on, and, as the walk has it, only in what depends on it."""
    from tokamak_amd.kernels import ops

    monkeypatch.setattr(ops, "DELTA_CHUNKS_FROM_TOKENS", 16)
    heads, kv, dim, vdim, spans, bad = 4, 2, 96, 128, [100, 45], 100 + 23
    g = torch.Generator().manual_seed(5)
    n = sum(spans)
    rand = lambda *shape: torch.randn(*shape, generator=g)
    unit = lambda x: x / x.norm(dim=-1, keepdim=True)
    parts = {"q": unit(rand(n, kv, dim)) * dim ** -0.5, "k": unit(rand(n, kv, dim)), "v": rand(n, heads, vdim),
             "a": torch.exp(-torch.exp(rand(n, heads, dim) - 2.0)), "beta": torch.sigmoid(rand(n, heads))}
    state = rand(len(spans) + 1, heads, vdim, dim)
    if where == "state":
        state[1, 1, 9, 17] = number
    elif where == "beta":
        parts[where][bad, 1] = number
    else:
        parts[where][bad, 1, 17] = number
    row = torch.zeros((n, ops.delta_row(heads, kv, dim, vdim)))
    flat = torch.cat([parts[x].flatten(1) for x in ("q", "k", "v", "a", "beta")], 1)
    row[:, :flat.shape[1]] = flat
    batch = make_batch([(t, 50, [0] * 64) for t in spans])
    batch.state_slots.copy_(torch.tensor([0, 1], dtype=torch.int32))

    def run(chunks):
        s, y = state.to(DEV), torch.empty((n, heads * vdim), device=DEV)
        ops.delta_scan(row.to(DEV), s, y, batch, heads=heads, kv_heads=kv, dim=dim, vdim=vdim, chunks=chunks)
        return y.cpu(), s.cpu()

    for got, walked in zip(run(True), run(False)):
        assert torch.equal(got.isfinite(), walked.isfinite()) and not bool(got.isfinite().all()) or where == "q"
        if where == "q":      # (its own token's outputs of the two heads that share it, and nothing else)
            assert got.dim() > 2 or got.isfinite().logical_not().nonzero()[:, 0].unique().tolist() == [bad]
        there = walked.isfinite() & got.isfinite()
        assert bool(((got - walked)[there].abs() <= 2.0 ** -18 * walked[there].abs().max()).all())
