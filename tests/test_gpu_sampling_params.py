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


@pytest.mark.parametrize("rows", [65, 77])
def test_more_rows_than_travel_with_the_launch_are_shared(rows):
    """At 151,936 logits up to 77 rows with thresholds are shared between blocks: with their parameters in device memory as with the launch,
    and as a block a row chooses."""
    vocab = 151936
    gen = torch.Generator(device=DEV).manual_seed(rows)
    logits = torch.randn(rows, vocab, generator=gen, device=DEV) * 3.0
    logits[3] = logits[3].round()                                            # (many values in the threshold's bin)
    params, seeds, draws = [KINDS[i % len(KINDS)] for i in range(rows)], [977 * i for i in range(rows)], list(range(rows))
    whole = sample_tokens(logits, params, seeds, draws)
    for at in (0, rows - 64):
        part = slice(at, at + 64)
        assert torch.equal(sample_tokens(logits[part], params[part], seeds[part], draws[part]), whole[part])
    more = 78 - rows
    alone = sample_tokens(torch.cat([logits, logits[:more]]), params + params[:more], seeds + seeds[:more], draws + draws[:more])
    assert torch.equal(alone[:rows], whole)


@pytest.mark.parametrize("rows", [7, 66])
def test_rows_left_out_of_the_list_are_sampled_alone(rows):
    """The list of rows with thresholds is the caller's: what it leaves out, has out of order or out of range is not read unmade."""
    vocab = 151936
    gen = torch.Generator(device=DEV).manual_seed(rows)
    logits = torch.randn(rows, vocab, generator=gen, device=DEV) * 3.0
    host = np.zeros(8 * rows, dtype=np.int32)
    host[:4 * rows].view(np.int64)[:] = np.arange(2 * rows) * 31
    host[4 * rows:6 * rows].view(np.float32)[:] = [0.8] * rows + [0.9, 1.0] * (rows // 2) + [0.95] * (rows % 2)
    host[6 * rows:7 * rows] = [0, 40] * (rows // 2) + [300] * (rows % 2)

    def chosen(listed):
        given = host[:7 * rows + len(listed)].copy()
        given[7 * rows:] = listed
        out = torch.full((rows,), -1, dtype=torch.int32, device=DEV)
        ops.sample(logits, given if rows <= 64 else torch.from_numpy(given).to(DEV), out, None, len(listed))
        return out

    whole = chosen(list(range(rows)))
    for listed in ([], [0], [rows - 1], list(range(1, rows, 2)), list(range(rows - 1, -1, -1))):
        assert torch.equal(chosen(listed), whole)
    if rows > 64:      # (with the launch these are refused)
        assert torch.equal(chosen([2, 2, 5, 5, rows, 1 << 30]), whole) and torch.equal(chosen([-1, -7, 3]), whole)
