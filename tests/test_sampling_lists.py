"""What the sampler's entry refuses before any launch: a list of rows with thresholds that names a row twice or none that is there."""

import ctypes

import numpy as np
import pytest

from tokamak_amd.kernels import ops
from tokamak_amd.kernels.build import load_library


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
