"""The experts' products of few tokens, an expert's weights read once, against float64 on the same operands: pairs
that share an expert and pairs that do not, more pairs than a pass takes, remainders of K and of the channels."""

import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


@pytest.mark.parametrize("n,top,experts,w,f,skew", [
    (1, 2, 16, 1024, 1024, 0), (1, 1, 1, 8, 8, 0), (8, 2, 16, 264, 248, 0), (17, 3, 5, 520, 40, 0), (32, 2, 64, 256, 1032, 0),
    (40, 2, 16, 1032, 264, 0), (64, 1, 3, 512, 72, 0), (100, 2, 4, 96, 24, 0), (70, 2, 8, 328, 88, 1), (130, 4, 33, 64, 16, 1)])
@pytest.mark.parametrize("on_output", [False, True])
def test_streamed_experts(n, top, experts, w, f, skew, on_output):
    from tokamak_amd.kernels import ops

    g = torch.Generator().manual_seed(n + w)
    h = torch.randn(n, w, generator=g).bfloat16()
    gate_up = (torch.randn(experts, 2 * f, w, generator=g) * 1.5 * w ** -0.5).bfloat16()
    down = (torch.randn(experts, w, f, generator=g) * f ** -0.5).bfloat16()
    score = torch.rand(n, experts, generator=g)
    if skew:
        score[:, 0] += 2.0      # one expert that every token takes
    chosen = score.topk(top, dim=-1).indices.int()
    weight = torch.rand(n, top, generator=g)
    assert ops.moe_stream_fits(h.to(DEV), gate_up.to(DEV), down.to(DEV), n * top) or n * top > 64
    args = [t.to(DEV) for t in (h, gate_up, chosen, weight)]
    act = torch.full((n * top, f), float("nan"), dtype=torch.bfloat16, device=DEV)
    out = torch.full((top, n, w), float("nan"), dtype=torch.float32, device=DEV)
    ops.moe_stream(*args, act, tokens=n, top=top, gated=True, weight_on_output=on_output)
    ops.moe_stream(act, down.to(DEV), args[2], None, out, tokens=n, top=top, gated=False)
    act, out = act.cpu(), out.cpu()
    for t in range(n):
        for k in range(top):
            e, x = int(chosen[t, k]), float(weight[t, k])
            both = gate_up[e].double() @ h[t].double()
            gate, up = both[:f], both[f:]
            want = torch.nn.functional.silu(gate) * up * x if on_output else torch.nn.functional.silu(x * gate) * (x * up)
            got = act[t * top + k].double()
            # one rounding to bfloat16 behind float32 sums of up to 1,032 products
            assert bool(((got - want).abs() <= 2.0 ** -8 * want.abs() + 1e-4).all())
            want = down[e].double() @ got
            assert float((out[k, t].double() - want).abs().max()) <= 2e-5 * (1.0 + float(want.abs().max()))
