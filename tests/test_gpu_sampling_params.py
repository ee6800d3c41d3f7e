"""Sampling parameters that travel with the launch (up to 64 rows) and in device memory (more), and the rows that have a threshold."""

import numpy as np
import pytest
import torch

from tokamak_amd.kernels import ops
from tokamak_amd.sampling.params import SamplingParams
from tokamak_amd.sampling.sampler import sample_tokens

pytestmark = pytest.mark.gpu
DEV = "cuda:0"
KINDS = [SamplingParams(temperature=0.7, top_k=50, top_p=0.95), SamplingParams(temperature=0.9, top_p=0.9), SamplingParams(temperature=1.0),
         SamplingParams(temperature=0.0), SamplingParams(temperature=1.1, top_k=256), SamplingParams(temperature=0.0, top_k=5), SamplingParams(temperature=2.0, top_p=0.6)]


@pytest.mark.parametrize("vocab", [997, 70000])
@pytest.mark.parametrize("kinds", [KINDS, KINDS[2:4], KINDS[:1]])
def test_rows_choose_alike_by_either_way(vocab, kinds):
    gen = torch.Generator(device=DEV).manual_seed(vocab)
    rows = 65
    logits = torch.randn(rows, vocab, generator=gen, device=DEV) * 3.0
    params, seeds, draws = [kinds[i % len(kinds)] for i in range(rows)], [(1 << 62) + 977 * i for i in range(rows)], [i * i for i in range(rows)]
    assert ops.SAMPLE_INLINE_ROWS == 64
    whole = sample_tokens(logits, params, seeds, draws)                      # in device memory
    for m in (1, 63, 64):                                                    # with the launch
        at = rows - m
        out = torch.full((m + 3,), -7, dtype=torch.int32, device=DEV)
        got = sample_tokens(logits[at:], params[at:], seeds[at:], draws[at:], out=out)
        assert torch.equal(got, whole[at:]) and out[m:].tolist() == [-7] * 3
    greedy = [i for i, p in enumerate(params) if p.is_greedy]
    assert torch.equal(whole[greedy], logits[greedy].argmax(1).int())


def test_what_is_refused():
    logits, out = torch.zeros(2, 100, device=DEV), torch.zeros(2, dtype=torch.int32, device=DEV)
    params = np.zeros(16, dtype=np.int32)
    params[8:10] = np.array([1.0, 1.0], dtype=np.float32).view(np.int32)
    ops.sample(logits, params, out, None, 2)
    for rows in ([2, 0], [-1, 0]):
        params[14:] = rows
        with pytest.raises(ops.KernelError):
            ops.sample(logits, params, out, None, 2)
    with pytest.raises(ops.KernelError):
        ops.sample(logits, params[:14], out, None, 1)                        # no room for the row's number
    with pytest.raises(ops.KernelError):
        ops.sample(logits.repeat(33, 1), np.zeros(66 * 7, dtype=np.int32), torch.zeros(66, dtype=torch.int32, device=DEV))
