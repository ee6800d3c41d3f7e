"""The scans with a decay a key channel in chunks of 16 tokens, against the recurrences in 64 bits on the same
operands, and against the walk a token at a time; state slots out of order, a foreign slot untouched."""

import pytest
import torch

from kernel_util import make_batch

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


def recurrence(q, k, v, a, u, state):
    """[T, H, d] operands in float64, a the decays; u None: the newest token is in the state when it is read."""
    out = []
    for t in range(q.shape[0]):
        kv = k[t][:, :, None] * v[t][:, None, :]
        if u is None:
            state = a[t][:, :, None] * state + kv
            out.append((state * q[t][:, :, None]).sum(1))
        else:
            out.append(((state + u[:, :, None] * kv) * q[t][:, :, None]).sum(1))
            state = a[t][:, :, None] * state + kv
    return torch.stack(out), state


@pytest.mark.parametrize("form", ["gla", "wkv"])
@pytest.mark.parametrize("heads,dim,vdim,spans", [
    (2, 128, 128, [33]), (3, 64, 64, [16, 1, 47]), (8, 16, 16, [32]), (2, 48, 48, [100, 15, 17]), (4, 80, 112, [64, 2]),
    (2, 128, 16, [129])])
@pytest.mark.parametrize("decays", ["slow", "fast"])
def test_chunks(form, heads, dim, vdim, spans, decays, monkeypatch):
    from tokamak_amd.kernels import ops

    if form == "wkv":
        vdim = dim
    g = torch.Generator().manual_seed(dim + len(spans))
    n, hd, hv = sum(spans), heads * dim, heads * vdim
    rand = lambda *shape: torch.randn(*shape, generator=g)
    q, k, z = rand(n, hd).bfloat16(), rand(n, hd).bfloat16(), (2.0 * rand(n, hd)).bfloat16()
    v, gate = rand(n, hv).bfloat16(), rand(n, hv).bfloat16()
    # fast: decays of 1e-3 and far less within a chunk, down to those that are zero in float32 (nothing may be divided by one)
    bias = rand(hd) + ((2.0 if decays == "slow" else -60.0) if form == "gla" else (-3.0 if decays == "slow" else 2.0))
    u, gain = 0.5 * rand(hd), 1.0 + 0.2 * rand(hd if form == "wkv" else vdim)
    slots = [len(spans) - 1 - i for i in range(len(spans))]
    state = rand(len(spans) + 1, heads, dim, vdim)
    batch = make_batch([(t, 50, [0] * 64) for t in spans])
    batch.state_slots.copy_(torch.tensor(slots, dtype=torch.int32))
    x = z.double() + bias.double()
    decay = (torch.sigmoid(x) ** 0.125 if form == "gla" else torch.exp(-torch.exp(x))).view(n, heads, dim)
    want, want_state, at = [], {}, 0
    for t, slot in zip(spans, slots):
        rows = slice(at, at + t)
        o, s = recurrence(q[rows].double().view(t, heads, dim) * (dim ** -0.5 if form == "gla" else 1.0), k[rows].double().view(t, heads, dim),
                          v[rows].double().view(t, heads, vdim), decay[rows], None if form == "gla" else u.double().view(heads, dim),
                          state[slot].double())
        want.append(o)
        want_state[slot] = s
        at += t
    o = torch.cat(want)
    rms = o / torch.sqrt((o * o).mean(-1, keepdim=True) + 1e-5)
    want = (rms * (gain.double().view(heads, dim) if form == "wkv" else gain.double())).flatten(1) * (gate.double() * torch.sigmoid(gate.double()))

    def run():
        s, out = state.to(DEV), torch.empty((n, hv), dtype=torch.bfloat16, device=DEV)
        a = [t.to(DEV) for t in (q, k, v, gate, z)]
        if form == "gla":
            ops.gla_scan(*a, bias.to(DEV), gain.to(DEV), s, out, batch, heads=heads, dim=dim, vdim=vdim, q_scale=dim ** -0.5, tau=8.0, eps=1e-5)
        else:
            ops.wkv_scan(*a, bias.to(DEV), u.to(DEV), gain.to(DEV), s, out, batch, heads=heads, dim=dim, eps=1e-5)
        return out.cpu().double(), s.cpu()

    assert ops._scan_in_chunks(torch.bfloat16, dim, vdim, max(spans))
    got, got_state = run()
    assert torch.equal(got_state[-1], state[-1])
    for slot, s in want_state.items():
        assert float((got_state[slot].double() - s).norm() / s.norm()) < 1e-6      # sums of float32 products
    # the final rounding (2^-9), and 2^-20 of the head's outputs where terms cancel, behind a norm
    bound = 2.0 ** -8 * want.abs() + 2e-5 * want.abs().max()
    assert bool(((got - want).abs() <= bound).all()), float(((got - want).abs() - bound).max())
    monkeypatch.setattr(ops, "SCAN_CHUNKS_FROM_TOKENS", 1 << 30)
    walked, walked_state = run()
    assert float((got - want).norm()) <= 1.02 * float((walked - want).norm())
    for slot, s in want_state.items():
        off = [float((x[slot].double() - s).norm() / s.norm()) for x in (got_state, walked_state)]
        # no further from the 64-bit state than the walk (a fiftieth for chance); where decays leave nothing of the token before,
        # the walk rounds a number once and a chunk up to twice (2^-25 of it, and 2^-26 more)
        assert off[0] <= 1.02 * off[1] + (0.0 if decays == "slow" else 2.0 ** -26), off
