"""Rows of logits walked in pieces of eight loads a thread (csrc/sampling.hip): rows on and off 16-byte borders, segments of one
piece and of several, rows shared between blocks and rows of one block alone choose the same tokens."""

import pytest
import torch

from tokamak_amd.sampling.params import SamplingParams
from tokamak_amd.sampling.sampler import greedy_tokens, sample_tokens

pytestmark = pytest.mark.gpu
DEV = "cuda:0"
KINDS = [SamplingParams(temperature=0.7, top_k=50, top_p=0.95), SamplingParams(temperature=0.9, top_p=0.8), SamplingParams(temperature=1.0),
         SamplingParams(temperature=0.0), SamplingParams(temperature=1.1, top_k=256), SamplingParams(temperature=3.0, top_p=0.99)]


# segments of less than a load a thread, of one piece of eight to its last quad and one more, of two pieces and a remainder
@pytest.mark.parametrize("vocab", [65536, 100003, 262144, 262148, 300001])
def test_the_same_tokens_by_every_walk(vocab):
    gen = torch.Generator(device=DEV).manual_seed(vocab)
    m = len(KINDS)
    rows = torch.randn(m, vocab, generator=gen, device=DEV) * 2.0
    rows.scatter_add_(1, torch.randint(0, vocab, (m, 40), generator=gen, device=DEV), 6.0 + torch.rand(m, 40, generator=gen, device=DEV))
    off = torch.full((m, vocab + 5), float("inf"), device=DEV)[:, 3:3 + vocab]       # (what is read beside a row would win)
    off.copy_(rows)
    seeds, draws = [17 * i + 3 for i in range(m)], list(range(m))
    want = sample_tokens(rows, KINDS, seeds, draws)
    assert torch.equal(sample_tokens(off, KINDS, seeds, draws), want)
    copies = (vocab // 1536) // m + 1                                                # more rows than are shared: a block each
    alone = sample_tokens(rows.repeat(copies, 1), KINDS * copies, seeds * copies, draws * copies)
    for at in range(0, m * copies, m):
        # (rows without thresholds draw from sums in float32 either way; those with, from whole numbers)
        assert torch.equal(alone[at:at + m], want)
    best = rows.double().argmax(1).int()
    assert torch.equal(greedy_tokens(rows), best) and torch.equal(greedy_tokens(off), best) and want[3] == best[3]
    for r, p in enumerate(KINDS):                                                    # what was drawn is what the thresholds keep
        if p.top_k > 0:
            assert (rows[r] > rows[r, want[r].long()]).sum() < p.top_k
