"""A step's rows with thresholds are shared between blocks where the vocabulary is large (65,536 and more) and the rows are
few; else a block takes a row.  Both must choose the same tokens: thresholds and the draws' masses are sums of integers."""

import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


@pytest.mark.parametrize("vocab,ld", [(5, 5), (33, 36), (127, 131), (4097, 4100), (20011, 20011), (70001, 70003), (151936, 151936)])
@pytest.mark.parametrize("spread", ["peaked", "normal", "alike", "holes"])
def test_shared_rows_choose_what_single_blocks_choose(vocab, ld, spread):
    from tokamak_amd.sampling.params import SamplingParams
    from tokamak_amd.sampling.sampler import sample_tokens

    g = torch.Generator().manual_seed(vocab)
    rows = 24
    x = torch.randn(rows, ld, generator=g)
    if spread == "peaked":
        x = 2.0 * x + 9.0 * (torch.rand(rows, ld, generator=g) > 0.999)
    elif spread == "alike":
        x = 1.0 + 1e-3 * x          # more values in the threshold's bin than a list holds
    elif spread == "holes":
        x[torch.rand(rows, ld, generator=g) < 0.5] = float("-inf")
        x[3] = float("nan")
        x[4, 1:] = float("-inf")
        x[5] = float("-inf")
    logits = x.to(DEV)[:, :vocab]
    kinds = [SamplingParams(temperature=t, top_k=k, top_p=p) for t, k, p in
             ((0.7, 20, 0.9), (1.0, 0, 0.8), (0.6, 1, 1.0), (1.3, 50, 1.0), (0.0, 0, 1.0), (1.0, 0, 1.0), (0.5, 7, 0.5), (1.0, 0, 1e-6),
              (0.9, 20000, 0.999), (1.0, 100000, 1.0), (0.2, 0, 0.99), (5.0, 0, 0.95))]
    params = [kinds[i % len(kinds)] for i in range(rows)]
    seeds, draws = [977 * i + 5 for i in range(rows)], list(range(rows))
    got = sample_tokens(logits, params, seeds, draws).tolist()
    copies = 11                     # 264 rows: a block a row
    wide = x.to(DEV).repeat(copies, 1)[:, :vocab]
    want = sample_tokens(wide, params * copies, seeds * copies, draws * copies).tolist()
    assert want[:rows] * copies == want
    assert sum(a != b for a, b in zip(got, want)) == 0, [(i, a, b) for i, (a, b) in enumerate(zip(got, want)) if a != b]
    assert all(0 <= t < vocab for t in got)


@pytest.mark.parametrize("vocab,ld", [(33, 36), (4097, 4100), (20011, 20011), (70001, 70003), (151936, 151936)])
@pytest.mark.parametrize("spread", ["peaked", "normal", "alike", "flat tail"])
def test_masses_do_not_depend_on_the_other_rows(vocab, ld, spread):
    """The distribution a row is drawn from has the same bits alone, beside others, and in a step of more rows than are
    shared; and its masses are float32's, also where a tail of tokens lies at 2^-31 of the best one."""
    from tokamak_amd.sampling.params import SamplingParams
    from tokamak_amd.sampling.sampler import sample_tokens

    g = torch.Generator().manual_seed(vocab)
    rows = 6
    x = torch.randn(rows, ld, generator=g)
    tail = min(10000, vocab - 1)
    if spread == "peaked":
        x = 2.0 * x + 9.0 * (torch.rand(rows, ld, generator=g) > 0.999)
    elif spread == "alike":
        x = 1.0 + 1e-3 * x
    elif spread == "flat tail":
        x = torch.full((rows, ld), float("-inf"))
        x[:, 0] = 0.0
        x[:, 1:1 + tail] = -21.4926      # 1.99 of the 2^-32 that the thresholds count in
    kinds = [SamplingParams(temperature=1.0, top_k=k, top_p=p) for k, p in
             ((tail, 1.0), (0, 0.9999999), (tail, 0.9999999), (0, 0.9), (7, 1.0), (0, 1.0))]
    params, seeds, draws = kinds, [31 * i + 5 for i in range(rows)], list(range(rows))
    logits = x.to(DEV)
    token, probs = sample_tokens(logits[:, :vocab], params, seeds, draws, return_probs=True)
    alone = [sample_tokens(logits[i:i + 1, :vocab], params[i:i + 1], seeds[i:i + 1], draws[i:i + 1], return_probs=True) for i in range(rows)]
    copies = 44                     # 264 rows: a block a row
    wide, wide_probs = sample_tokens(logits.repeat(copies, 1)[:, :vocab], params * copies, seeds * copies, draws * copies, return_probs=True)
    for i in range(rows):
        for t, p in ((alone[i][0][0], alone[i][1][0]), (wide[i], wide_probs[i]), (wide[i - rows], wide_probs[i - rows])):
            assert int(t) == int(token[i]) and torch.equal(p, probs[i])
    want = torch.where(probs > 0, logits[:, :vocab].double(), float("-inf")).softmax(-1)
    if spread == "flat tail":
        # the best token's share: the mass and the quotient rounded once each (the row without thresholds, the last,
        # adds its segments' masses in float32)
        assert float((probs.double() - want)[:-1, 0].abs().max()) <= 2.0 ** -22
    # e^x to some 2^-20 on the exponential unit
    assert float((probs.double() - want).norm() / want.norm()) <= 2.0 ** -19


def test_rows_without_thresholds_are_drawn_alone_as_beside_others():
    """No row with a threshold: the launches that share such rows are left out, and nothing else changes."""
    from tokamak_amd.sampling.params import SamplingParams
    from tokamak_amd.sampling.sampler import sample_tokens

    g = torch.Generator().manual_seed(2)
    rows, vocab = 9, 20011
    logits = (3.0 * torch.randn(rows + 1, vocab, generator=g)).to(DEV)
    params = [SamplingParams(temperature=t, top_k=k) for t, k in ((0.7, 0), (1.0, vocab), (0.0, 0), (2.0, vocab + 5), (0.0, 3), (1.0, 0), (0.1, 0), (5.0, 0), (1.0, 0))]
    seeds, draws = [13 * i + 1 for i in range(rows + 1)], list(range(rows + 1))
    alone, probs = sample_tokens(logits[:rows], params, seeds[:rows], draws[:rows], return_probs=True)
    beside, shared_probs = sample_tokens(logits, params + [SamplingParams(temperature=1.0, top_k=4)], seeds, draws, return_probs=True)
    assert torch.equal(alone, beside[:rows]) and torch.equal(probs, shared_probs[:rows])
