"""The experts' products with weights in operand order, against float64 on the same operands: an expert's weights read
once (few tokens) and tiles of 128 pairs (many); pairs that share an expert and pairs that do not, tiles and passes that
are nearly empty, remainders of K and of the channels."""

import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


@pytest.mark.parametrize("n,top,experts,w,f,skew", [
    (1, 2, 16, 1024, 1024, 0), (1, 1, 1, 64, 64, 0), (8, 2, 16, 320, 192, 0), (17, 3, 5, 576, 64, 0), (32, 2, 64, 256, 1088, 0),
    (40, 2, 16, 1088, 320, 0), (64, 1, 3, 512, 64, 0), (100, 2, 4, 128, 64, 0), (70, 2, 8, 320, 128, 1), (130, 4, 33, 64, 128, 1),
    (257, 2, 3, 192, 576, 1)])
@pytest.mark.parametrize("form", ["stream", "tiles"])
@pytest.mark.parametrize("on_output", [False, True])
def test_experts_in_operand_order(n, top, experts, w, f, skew, form, on_output):
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
    first, second = (ops.expert_operands(t.to(DEV)) for t in (gate_up, down))
    hd, cd, wd = (t.to(DEV) for t in (h, chosen, weight))
    act = torch.full((n * top, f), float("nan"), dtype=torch.bfloat16, device=DEV)
    out = torch.full((top, n, w), float("nan"), dtype=torch.float32, device=DEV)
    if form == "stream":
        ops.moe_stream(hd, first, cd, wd, act, tokens=n, top=top, gated=True, weight_on_output=on_output)
        ops.moe_stream(act, second, cd, None, out, tokens=n, top=top, gated=False)
    else:
        lists = ops.moe_sort(cd, experts, ops.MOE_WIDE_TILE_PAIRS)
        ops.moe_tiles(hd, first, lists, wd, act, tokens=n, top=top, gated=True, weight_on_output=on_output)
        ops.moe_tiles(act, second, lists, None, out, tokens=n, top=top, gated=False)
    act, out = act.cpu(), out.cpu()
    for e in range(experts):
        token, place = (chosen == e).nonzero(as_tuple=True)
        pair, x = token * top + place, weight[token, place].double()[:, None]
        both = h[token].double() @ gate_up[e].double().T
        gate, up = both[:, :f], both[:, f:]
        want = torch.nn.functional.silu(gate) * up * x if on_output else torch.nn.functional.silu(x * gate) * (x * up)
        got = act[pair].double()
        # one rounding to bfloat16 behind float32 sums of up to 1,088 products
        assert bool(((got - want).abs() <= 2.0 ** -8 * want.abs() + 1e-4).all())
        want = got @ down[e].double().T
        assert float((out[place, token].double() - want).abs().max().nan_to_num(0.0) if token.numel() else 0.0) <= 2e-5 * (1.0 + float(want.abs().max() if token.numel() else 0.0))
    assert bool(torch.isfinite(out).all())


@pytest.mark.parametrize("w,f,experts,top", [(4096, 320, 16, 2), (1280, 2560, 40, 3), (3072, 64, 5, 1)])
def test_a_pair_has_the_same_bits_whoever_stands_before_it(w, f, experts, top):
    """The form for few tokens: alone, in other orders of the step's tokens (and so of the experts it meets), among many."""
    from tokamak_amd.kernels import ops

    g = torch.Generator().manual_seed(w)
    n = 24
    h = torch.randn(n, w, generator=g).bfloat16().to(DEV)
    first, second = (ops.expert_operands((torch.randn(experts, r, k, generator=g) * k ** -0.5).bfloat16().to(DEV)) for r, k in ((2 * f, w), (w, f)))
    chosen, weight = torch.rand(n, experts, generator=g).topk(top, dim=-1).indices.int().to(DEV), torch.rand(n, top, generator=g).to(DEV)

    def run(tokens):
        index = torch.tensor(tokens, device=DEV)
        act = torch.empty((len(tokens) * top, f), dtype=torch.bfloat16, device=DEV)
        out = torch.empty((top, len(tokens), w), dtype=torch.float32, device=DEV)
        c = chosen[index].contiguous()
        ops.moe_stream(h[index].contiguous(), first, c, weight[index].contiguous(), act, tokens=len(tokens), top=top, gated=True)
        ops.moe_stream(act, second, c, None, out, tokens=len(tokens), top=top, gated=False)
        return act.view(len(tokens), top, f), out

    act, out = run(list(range(n)))
    for tokens in ([3], [0, 3], [3, 0], [2, 1, 3], [7, 5, 6, 4, 3, 2, 1, 0], list(range(n))[::-1]):
        a, o = run(tokens)
        for place, token in enumerate(tokens):
            assert torch.equal(a[place], act[token]) and torch.equal(o[:, place], out[:, token]), (tokens, token)


def test_more_experts_than_a_step_lists():
    """5,120 experts, the router's most: their pairs cannot be listed, so their weights stay in rows and many pairs run one
    by one."""
    from tokamak_amd.parts.routed_experts import RoutedExperts

    width, ff, experts, n = 64, 64, 5120, 100
    g = torch.Generator().manual_seed(3)
    part = RoutedExperts(hidden_size=width, intermediate_size=ff, num_experts=experts, top=1, dtype=torch.bfloat16, device=DEV)
    weights = {name: (torch.randn(spec.shape, generator=g) * width ** -0.5).to(torch.float32 if spec.held == "float32" else torch.bfloat16)
               for name, spec in part.expected_tensors("").items()}
    part.bind("", lambda name: weights[name].to(DEV))
    h = torch.randn(n, width, generator=g).bfloat16()
    got = part.forward(h.to(DEV), None).sum(0).cpu().double()
    scores = torch.sigmoid(h.double() @ weights["router"].double().T)
    for token, (score, expert) in enumerate(zip(*(t.tolist() for t in scores.max(1)))):
        x = score * h[token].double()
        gate, up, down = (weights[f"e{expert}.{name}"].double() for name in ("gate", "up", "down"))
        want = down @ (torch.nn.functional.silu(gate @ x) * (up @ x))
        assert float((got[token] - want).abs().max()) <= 2.0 ** -7 * float(want.abs().max())      # (activations rounded to bfloat16)


def test_binding_holds_one_matrix_twice_at_most():
    from tokamak_amd.parts.routed_experts import RoutedExperts

    width, ff, experts = 512, 1024, 16
    part = RoutedExperts(hidden_size=width, intermediate_size=ff, num_experts=experts, top=2, dtype=torch.bfloat16, device=DEV)
    expected = part.expected_tensors("")
    make = lambda name: torch.ones(expected[name].shape, dtype=torch.float32 if expected[name].held == "float32" else torch.bfloat16, device=DEV)
    torch.cuda.synchronize()
    before = torch.cuda.memory_allocated()
    torch.cuda.reset_peak_memory_stats()
    part.bind("", make)
    peak = torch.cuda.max_memory_allocated() - before
    # gate and up (two matrices an expert) as they are read and stacked; or they, laid out, beside down and its copy
    assert peak <= 4 * experts * width * ff * 2 + (1 << 20), peak
