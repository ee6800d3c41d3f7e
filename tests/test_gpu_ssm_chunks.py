"""The state-space scan in chunks on the matrix cores, against a token-by-token walk in 64 bits, and its error against
that of the general form."""

import pytest
import torch

from kernel_util import make_batch

pytestmark = pytest.mark.gpu
DEV = "cuda:0"

CASES = {
    # heads, groups, state, vdim, tokens of each request
    "ragged": (8, 2, 128, 64, [200, 1, 64, 63, 65, 17]),
    "one group": (32, 1, 128, 64, [700, 33]),
    "small": (3, 3, 16, 16, [130, 16, 15]),
    "wide values": (4, 1, 64, 128, [128, 129, 2]),
    "odd tiles": (6, 3, 32, 48, [191, 32]),
    "partial sums": (16, 4, 128, 64, [150, 40]),
}


@pytest.mark.parametrize("name", list(CASES))
def test_state_space_scan_in_chunks(name, monkeypatch):
    from tokamak_amd.kernels import ops

    heads, groups, ns, vdim, lens = CASES[name]
    g = torch.Generator().manual_seed(len(name))
    n, inner = sum(lens), heads * vdim
    u = torch.randn(n, inner + 2 * groups * ns, generator=g).bfloat16()
    dt = torch.randn(n, heads, generator=g) * 2.0
    parts = torch.randn(3, n, heads, generator=g) if name == "partial sums" else None
    if parts is not None:
        dt = (parts[0] + parts[1]) + parts[2]
    dt = dt if parts is not None else dt.bfloat16()
    a_log, bias, skip = (torch.randn(heads, generator=g) for _ in range(3))
    start = torch.randn(len(lens) + 1, heads, vdim // 4, ns, 4, generator=g)
    batch = make_batch([(t, 50, [0] * 64) for t in lens])
    slots = [len(lens) - 1 - i for i in range(len(lens))]      # (out of order; the last slot is nobody's)
    batch.state_slots.copy_(torch.tensor(slots, dtype=torch.int32))

    want, state = torch.zeros(n, heads, vdim, dtype=torch.float64), start.double()
    x, b, c = (t.double() for t in u.split([inner, groups * ns, groups * ns], dim=1))
    per = heads // groups
    b, c = (t.view(n, groups, ns).repeat_interleave(per, 1) for t in (b, c))
    step = torch.nn.functional.softplus(dt.double() + bias.double())
    decay = torch.exp(-torch.exp(a_log.double()) * step)
    row = 0
    for slot, t in zip(slots, lens):
        s = state[slot].permute(0, 2, 1, 3).reshape(heads, ns, vdim)
        for i in range(row, row + t):
            xi = x[i].view(heads, 1, vdim)
            s = decay[i].view(-1, 1, 1) * s + step[i].view(-1, 1, 1) * b[i].unsqueeze(2) * xi
            want[i] = (s * c[i].unsqueeze(2)).sum(1) + skip.double().view(-1, 1) * xi[:, 0]
        state[slot] = s.view(heads, ns, vdim // 4, 4).permute(0, 2, 1, 3)
        row += t

    proj = (parts if parts is not None else dt).to(DEV)

    def run():
        y, kept = torch.full((n, inner), float("nan"), device=DEV), start.to(DEV)
        ops.ssd_scan(u.to(DEV), proj, 0, bias.to(DEV), a_log.to(DEV), skip.to(DEV), kept, y, batch, heads=heads, groups=groups,
                     state_size=ns, vdim=vdim)
        return y.view(n, heads, vdim).cpu().double(), kept.cpu().double()

    assert ops._ssm_in_chunks(u.to(DEV), ns, vdim, max(lens))
    got, kept = run()
    # sums of up to ns + 64 products of numbers up to 4.5 and a state that stays below 64: 2^-23 a term
    bound = 2.0 ** -23 * (ns + 64) * 64.0
    assert float((got - want).abs().max()) <= bound
    assert float((kept - state).abs().max()) <= bound
    monkeypatch.setattr(ops, "_ssm_in_chunks", lambda *a: False)
    monkeypatch.setattr(ops, "SSM_CHUNKS_FROM_TOKENS", 1 << 30)
    general, general_kept = run()
    # no further from the 64-bit result than the walk (a hundredth for so few numbers' chance)
    assert float((got - want).norm()) <= 1.01 * float((general - want).norm())
    assert float((kept - state).norm()) <= 1.01 * float((general_kept - state).norm())
