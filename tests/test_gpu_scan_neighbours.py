"""A request's outputs and state have the same bits whoever shares its step: short spans walk, long ones run in chunks, each
by its own length, in one step."""

import pytest
import torch

from kernel_util import make_batch

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


@pytest.mark.parametrize("form,heads,dim,vdim", [("gla", 4, 64, 128), ("gla", 2, 128, 48), ("wkv", 4, 64, 64), ("ssd", 8, 128, 64),
                                                 ("ssd", 4, 32, 48)])
@pytest.mark.parametrize("spans", [[1, 200, 1], [31, 32, 63, 64, 65, 1], [1] * 70 + [130, 17]])
def test_a_request_has_the_same_bits_beside_any_other(form, heads, dim, vdim, spans):
    from tokamak_amd.kernels import ops

    g = torch.Generator(device=DEV).manual_seed(dim + len(spans))
    rand = lambda *shape: torch.randn(*shape, generator=g, device=DEV)
    n, groups = sum(spans), 2
    wide = heads * vdim
    x = [rand(n, heads * dim).bfloat16() for _ in range(3)] + [rand(n, wide).bfloat16() for _ in range(2)]
    conv = rand(n, wide + 2 * groups * dim).bfloat16()
    step, vectors = rand(n, heads).bfloat16(), [rand(heads) for _ in range(3)]
    bias, u, gain = rand(heads * dim), 0.5 * rand(heads * dim), 1.0 + 0.2 * rand(heads * dim if form == "wkv" else vdim)
    shape = (heads, vdim // 4, dim, 4) if form == "ssd" else (heads, dim, vdim)
    start = rand(len(spans), *shape)

    def run(which):
        at = [sum(spans[:i]) for i in which]
        rows = torch.cat([torch.arange(a, a + spans[i]) for a, i in zip(at, which)]).to(DEV)
        batch = make_batch([(spans[i], 50, [0] * 64) for i in which])
        state = start[torch.tensor(which, device=DEV)].clone()
        q, k, z, v, gate = (t[rows].contiguous() for t in x)
        if form == "ssd":
            out = torch.empty((len(rows), wide), device=DEV)
            ops.ssd_scan(conv[rows].contiguous(), step[rows].contiguous(), 0, *vectors, state, out, batch, heads=heads, groups=groups,
                         state_size=dim, vdim=vdim)
        else:
            out = torch.empty((len(rows), wide), dtype=torch.bfloat16, device=DEV)
            if form == "gla":
                ops.gla_scan(q, k, v, gate, z, bias, gain, state, out, batch, heads=heads, dim=dim, vdim=vdim, q_scale=dim ** -0.5,
                             tau=8.0, eps=1e-5)
            else:
                ops.wkv_scan(q, k, v, gate, z, bias - 3.0, u, gain, state, out, batch, heads=heads, dim=dim, eps=1e-5)
        return out.split([spans[i] for i in which]), state

    together, states = run(list(range(len(spans))))
    assert all(bool(torch.isfinite(t).all()) for t in together)
    for i in {0, 1, 2, len(spans) - 2, len(spans) - 1}:
        (alone,), (state,) = run([i])
        assert torch.equal(alone, together[i]) and torch.equal(state, states[i]), (i, spans[i])
