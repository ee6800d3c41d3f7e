"""A step's rows with thresholds are shared between blocks up to 256 rows; with more a block takes a row.  Both must choose the
same tokens: thresholds are found from integers, and the draws' numbers meet the same masses."""

import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


@pytest.mark.parametrize("vocab,ld", [(5, 5), (33, 36), (127, 131), (4097, 4100), (20011, 20011), (151936, 151936)])
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
    # one draw in some millions may lie between two summations of the same masses
    assert sum(a != b for a, b in zip(got, want)) == 0, [(i, a, b) for i, (a, b) in enumerate(zip(got, want)) if a != b]
    assert all(0 <= t < vocab for t in got)
