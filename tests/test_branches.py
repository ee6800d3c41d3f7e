"""Which parts of a recorded step get a branch of their own, and what a branch may not do (without a GPU)."""

import pytest
import torch

from tokamak_amd.parts.attention import GQAAttention
from tokamak_amd.parts.base import Part
from tokamak_amd.parts.routed_experts import RoutedExperts


def experts(width, channels, shared=None, count=16, top=2):
    return RoutedExperts(hidden_size=width, intermediate_size=channels, num_experts=count, top=top, shared_size=shared,
                         dtype=torch.bfloat16, device="cpu")


# (width, channels of an expert, of the shared one, experts, top, requests, us a layer with the kernels in a row, with two branches)
MEASURED = [(1024, 1536, None, 16, 2, 1, 50.2, 55.2), (1024, 1536, None, 16, 2, 3, 54.8, 60.0), (1024, 1536, None, 16, 2, 4, 57.4, 59.1),
            (1024, 1536, None, 16, 2, 16, 64.5, 63.3), (1024, 1536, None, 16, 2, 40, 80.0, 72.9), (1024, 512, None, 16, 2, 32, 72.1, 74.1),
            (1024, 3072, None, 16, 2, 2, 62.9, 67.3), (1024, 3072, None, 16, 2, 4, 70.3, 65.3), (1024, 512, None, 64, 6, 8, 77.9, 66.3),
            (4096, 1024, None, 16, 2, 2, 130.5, 132.8), (4096, 1024, None, 16, 2, 4, 141.3, 138.1), (4096, 6144, None, 16, 2, 1, 172.2, 163.3),
            (1024, 1024, 1024, 16, 2, 1, 47.6, 45.5), (1024, 1024, 1024, 16, 2, 16, 61.5, 52.9)]


@pytest.mark.parametrize("width, channels, shared, count, top, requests, row, forked", MEASURED)
def test_experts_get_a_branch_where_it_was_faster(width, channels, shared, count, top, requests, row, forked):
    part = experts(width, channels, shared, count, top)
    assert part.own_branch and part.branch_pays(requests) == (forked < row)


def test_other_parts_have_none():
    assert not Part.own_branch and not GQAAttention.own_branch


def test_a_pinned_stream_is_the_threads_own(monkeypatch):
    """What one thread pins while it steps or records a model is not where another thread launches."""
    import threading
    from types import SimpleNamespace

    from tokamak_amd.kernels import ops

    current = threading.local()
    current.stream = 7
    monkeypatch.setattr(torch.cuda, "current_stream", lambda device=None: SimpleNamespace(cuda_stream=getattr(current, "stream", 9)))
    seen = []
    with ops.pinned_stream():
        current.stream = 8
        other = threading.Thread(target=lambda: seen.append(ops._stream().value))
        other.start()
        other.join()
        seen.append(ops._stream().value)
        with ops.pinned_stream():
            seen.append(ops._stream().value)
        seen.append(ops._stream().value)
    assert seen == [9, 7, 8, 7] and ops._stream().value == 8


def test_a_branch_runs_no_library_product(monkeypatch):
    """Those share one workspace a device, which the step's other branch may be using."""
    from types import SimpleNamespace

    from tokamak_amd.kernels import ops

    monkeypatch.setattr(torch.cuda, "current_stream", lambda device=None: SimpleNamespace(cuda_stream=7))
    a = torch.zeros(80, 64, dtype=torch.bfloat16)
    with ops.pinned_stream(), ops.branch_stream():
        with pytest.raises(ops.KernelError, match="share one workspace"):
            ops.gemm_library(a, a, torch.empty(80, 80, dtype=torch.bfloat16))
    with pytest.raises(ops.KernelError, match="GPU tensors"):        # (elsewhere as before)
        ops.gemm_library(a, a, torch.empty(80, 80, dtype=torch.bfloat16))
