"""What the sampler's entry refuses before any launch: a list of rows with thresholds that names a row twice or none that is there."""

import ctypes

import numpy as np
import pytest
import torch

from tokamak_amd.kernels import ops
from tokamak_amd.kernels.build import load_library
from tokamak_amd.sampling.params import SamplingParams
from tokamak_amd.sampling.sampler import sample_tokens


@pytest.mark.parametrize("listed", [[1, 1], [0, 2, 0], [3], [-1], [0, 1, 2, 2]])
def test_lists_that_name_a_row_twice_are_refused(listed):
    rows, vocab = 3, 65536
    params = np.zeros(7 * rows + len(listed), dtype=np.int32)
    params[7 * rows:] = listed
    scratch = ctypes.create_string_buffer(64)      # (never written: the call ends before a launch)
    at = (ctypes.addressof(scratch) + 15) & ~15
    place = ctypes.c_void_p(at)
    sample = load_library("sampling").tk_sample
    sample.argtypes = ops._SIGS["sampling"]["tk_sample"]
    assert sample(place, vocab, rows, vocab, ctypes.c_void_p(params.ctypes.data), 1, len(listed), place, None, place, None) == -1


@pytest.mark.parametrize("rows, vocab, listed", [(3, 151936, [0, 2]), (77, 151936, None), (78, 151936, []), (3, 65535, []), (256, 32003, [])])
def test_rows_are_named_only_where_some_are_shared(rows, vocab, listed, monkeypatch):
    """The list of rows with thresholds is host work that a block a row has no use for."""
    given = {}
    monkeypatch.setattr(ops, "sample_shares_rows", lambda m, v: bool(load_library("sampling").tk_sample_shares_rows(m, v)))
    monkeypatch.setattr(ops, "sample", lambda logits, params, out, probs, shared: given.update(params=torch.as_tensor(params), shared=shared))
    monkeypatch.setattr(torch.Tensor, "pin_memory", lambda t: t)
    kinds = [SamplingParams(temperature=0.8, top_k=5), SamplingParams(temperature=1.0), SamplingParams(temperature=0.9, top_p=0.9)]
    params = [kinds[i % 3] for i in range(rows)]
    sample_tokens(torch.empty(rows, vocab, device="meta") if rows <= 64 else torch.empty(1).expand(rows, vocab), params, list(range(rows)), [0] * rows,
                  out=torch.empty(rows, dtype=torch.int32))
    want = [i for i in range(rows) if i % 3 != 1] if listed is None else listed
    assert given["shared"] == len(want) and given["params"][7 * rows:].tolist() == want
