"""Which arguments of a recorded call are addresses inside the recorded layer's own tensors, on the CPU."""

from ctypes import c_int, c_void_p

import pytest
import torch

from tokamak_amd.engine.layer_replay import patched_calls


@pytest.mark.parametrize("where, own", [(-2, None), (0, 0), (2, 2), (62, 62), (64, None)])
def test_an_address_belongs_to_the_tensor_it_lies_in(where, own):
    """From a tensor's first byte to its last; a number that is no address, a null one and a tensor without elements are nobody's."""
    around = torch.zeros(3, 32, dtype=torch.bfloat16)      # (the bytes before and behind are no layer's)
    w, empty = around[1], torch.empty(0)
    tensors = {("part", "a", "w"): w, ("part", "a", "empty"): empty}
    at = w.data_ptr() + where
    calls = [("f", (c_void_p(at), 7, c_void_p(0), at, c_int(3)), 0), ("g", (), 1), ("f", (1.5, c_void_p(at)), 2)]
    key = ("part", "a", "w")
    got = patched_calls(calls, tensors)
    assert [(fn, status) for fn, _, _, status in got] == [("f", 0), ("g", 1), ("f", 2)]
    assert [args for _, args, _, _ in got] == [args for _, args, _ in calls]
    assert [p for _, _, p, _ in got] == ([(), (), ()] if own is None else [((0, key, own),), (), ((1, key, own),)])
    assert [p for _, _, p, _ in patched_calls(calls, {})] == [(), (), ()]


def test_neighbouring_tensors_keep_their_own_addresses():
    rows = torch.zeros(4, 16)
    tensors = {("cache", "", i): rows[i] for i in (2, 0, 3, 1)}
    calls = [("f", tuple(c_void_p(rows[i].data_ptr() + 4 * i) for i in range(4)), 0)]
    assert patched_calls(calls, tensors)[0][2] == tuple((i, ("cache", "", i), 4 * i) for i in range(4))
