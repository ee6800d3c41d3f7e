"""Recorded steps whose layers hold two branches: every replay against the same step run kernel after kernel."""

import pytest
import torch

pytestmark = pytest.mark.gpu


def branching(block):
    """The part of a block that may run beside another, or None."""
    from tokamak_amd.parts.block import ParallelMixersBlock, ParallelSublayersBlock

    part = block.right if isinstance(block, ParallelMixersBlock) else block.feed_forward if isinstance(block, ParallelSublayersBlock) else None
    return part if part is not None and part.own_branch else None


@pytest.mark.parametrize("preset, layers", [("mepupel-0.6b", 6), ("supinex-0.6b", 4), ("dopirax-0.6b", 4), ("rorosun-0.6b", 4)])
@pytest.mark.parametrize("requests", [1, 5, 18])
@pytest.mark.parametrize("listed", [True, False])
def test_branches_give_the_bits_of_kernels_in_a_row(preset, layers, requests, listed, monkeypatch):
    """Steps of single tokens recorded with branches, and eager (no branches): equal bits of every logit, over many
    replays with other kernels between them, for contexts of unlike lengths; the layers launched from lists and
    one by one."""
    from replay_util import random_ids
    from tokamak_amd.config import find_preset
    from tokamak_amd.engine.runner import ModelRunner, StepEntry
    from tokamak_amd.kernels import ops
    from tokamak_amd.weights.random_init import expected_tensors_of
    from tokamak_amd.weights.sources import RandomSource

    arch, cfg = find_preset(preset)
    plan = arch.plan(arch.shorten(cfg, layers))
    source = RandomSource({n: s for n, s in expected_tensors_of(plan).items() if not s.ignored}, seed=3, matrix_std=0.02,
                          vector_jitter=0.1, dtype=torch.bfloat16, device="cuda:0")
    edges, order = [], ops.order_streams
    monkeypatch.setattr(ops, "order_streams", lambda first, then: edges.append((first, then)) or order(first, then))
    outs = []
    for use_graphs in (True, False):
        runner = ModelRunner(plan, source, dtype="bfloat16", page_size=16, kv_pool_tokens=160 * requests,
                             max_requests=requests, use_graphs=use_graphs)
        runner.model.replay_layers = listed
        forks = sum(branching(block).branch_pays(requests) for block in runner.model.blocks if branching(block) is not None)
        ids = [random_ids(plan.vocab_size, 20 + 5 * r + 12, r) for r in range(requests)]
        runner.step([StepEntry(r, ids[r][:20 + 5 * r], []) for r in range(requests)])
        got = []
        for i in range(12):
            got.append(runner.step([StepEntry(r, [ids[r][20 + 5 * r + i]], [0]) for r in range(requests)]).clone())
            torch.randn(1 << 20, device="cuda:0").sum()       # other work of the program's between replays
        torch.cuda.synchronize()
        assert bool(runner._graphs) == use_graphs and all(g.replays > 0 for g in runner._graphs.values())
        # a fork and a join for every layer with a branch and recorded shape, between two streams; with layers launched from lists
        # Python meets the first ones of a kind only
        if listed:
            assert bool(edges) == (use_graphs and forks > 0)
        else:
            assert len(edges) == 2 * forks * len(runner._graphs)
        for fork, join in zip(edges[::2], edges[1::2]):
            assert fork[0] != fork[1] and fork == join[::-1]
        edges.clear()
        outs.append(got)
    for i, (a, b) in enumerate(zip(*outs)):
        assert torch.isfinite(a).all() and torch.equal(a, b), f"step {i}"


def test_a_recording_asks_for_the_stream_a_few_times_only(monkeypatch):
    """A step of a new shape runs once and is recorded; its launches take the stream that was looked up once, not one
    each."""
    from tokamak_amd.config import find_preset
    from tokamak_amd.engine.runner import ModelRunner, StepEntry
    from tokamak_amd.weights.random_init import expected_tensors_of
    from tokamak_amd.weights.sources import RandomSource

    arch, cfg = find_preset("dopirax-0.6b")
    plan = arch.plan(arch.shorten(cfg, 8))
    source = RandomSource({n: s for n, s in expected_tensors_of(plan).items() if not s.ignored}, seed=3, matrix_std=0.02,
                          dtype=torch.bfloat16, device="cuda:0")
    runner = ModelRunner(plan, source, dtype="bfloat16", page_size=16, kv_pool_tokens=256, max_requests=4)
    runner.step([StepEntry(r, [5, 6, 7], []) for r in range(4)])
    asked, current = [], torch.cuda.current_stream
    monkeypatch.setattr(torch.cuda, "current_stream", lambda device=None: asked.append(device) or current(device))
    runner.step([StepEntry(r, [8], [0]) for r in range(4)])
    assert len(runner._graphs) == 1
    assert len(asked) <= 4 * 8        # (a fork, a switch and a pin for the layers that run in Python, and what torch's own recording asks: 16)
