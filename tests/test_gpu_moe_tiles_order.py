"""The experts' tiles of 128 pairs (csrc/moe_operands.hip, moe_tiles): channel blocks in groups with a last group that is
smaller, steps of K in pairs and one left over, tiles of 1 to 128 pairs, against float64."""

import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


# (tokens, width, features of an expert): even and odd numbers of steps of 64 in both products; 16, 17, 18 and 35 channel blocks
@pytest.mark.parametrize("n,w,f", [(97, 4160, 2240), (300, 4352, 2176), (33, 64, 2048), (129, 192, 4416)])
def test_tiles_in_groups_of_channel_blocks(n, w, f):
    from tokamak_amd.kernels import ops

    g = torch.Generator(device=DEV).manual_seed(n)
    experts = 3
    h = torch.randn(n, w, generator=g, device=DEV).bfloat16()
    gate_up = (torch.randn(experts, 2 * f, w, generator=g, device=DEV) * w ** -0.5).bfloat16()
    down = (torch.randn(experts, w, f, generator=g, device=DEV) * f ** -0.5).bfloat16()
    down[0, 5, -1] = float("inf")       # the last k of a channel: it meets that k alone
    chosen = torch.full((n, 1), 2, dtype=torch.int32, device=DEV)
    chosen[:n // 3] = 0
    chosen[0] = 1                       # a tile of one pair
    weight = torch.rand(n, 1, generator=g, device=DEV)
    lists = ops.moe_sort(chosen, experts, ops.MOE_WIDE_TILE_PAIRS)
    act = torch.full((n, f), float("nan"), dtype=torch.bfloat16, device=DEV)
    out = torch.full((1, n, w), float("nan"), dtype=torch.float32, device=DEV)
    ops.moe_tiles(h, ops.expert_operands(gate_up), lists, weight, act, tokens=n, top=1, gated=True)
    ops.moe_tiles(act, ops.expert_operands(down), lists, None, out, tokens=n, top=1, gated=False)
    for e in range(experts):
        token = (chosen[:, 0] == e).nonzero()[:, 0]
        x = weight[token].double()
        both = h[token].double() @ gate_up[e].double().T
        want = torch.nn.functional.silu(x * both[:, :f]) * (x * both[:, f:])
        # one rounding to bfloat16 behind float32 sums of up to 4,416 products
        assert bool(((act[token].double() - want).abs() <= 2.0 ** -8 * want.abs() + 1e-4).all())
        want = act[token].double() @ down[e].double().T
        got = out[0, token].double()
        finite = torch.isfinite(want)
        assert torch.equal(torch.isfinite(got), finite) and torch.equal(got[~finite].nan_to_num(), want[~finite].nan_to_num())
        size = act[token].double().abs() @ down[e].double().abs().T
        assert bool(((got - want).abs() <= f * 2.0 ** -23 * size)[finite].all())
