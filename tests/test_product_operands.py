"""What reaches the flowing and the many-rows products, on the CPU: nothing that their entry points refuse."""

import pytest
import torch

from tokamak_amd.kernels import linear, ops


def rows(n, k, stride):
    return torch.zeros(n * max(stride, k) + k, dtype=torch.bfloat16).as_strided((n, k), (stride, 1))


@pytest.mark.parametrize("fits", [ops.gemm_flow_fits, lambda a, w: ops.gemm_many_fits(a, w, w.shape[0])])
@pytest.mark.parametrize("stride, taken", [(0, False), (8, False), (248, False), (256, True), (264, True), (260, False)])
def test_rows_that_overlap_go_elsewhere(fits, stride, taken):
    """Rows closer together than they are long (one row expanded, overlapping windows) are an error to both entry points; other
    forms of the product read them."""
    apart, them = rows(32, 256, 256), rows(32, 256, stride)
    assert fits(apart, apart)
    assert fits(them, apart) is taken and fits(apart, them) is taken


@pytest.mark.parametrize("m", [17, 64, 129, 300])
def test_a_limit_beside_the_silu_gate_is_not_looked_at(monkeypatch, m):
    """At any number of rows, by whichever kernel (which has a limit for the clamped gate alone)."""
    given = []
    for name in ("gemm_flow", "gemm_many"):
        monkeypatch.setattr(ops, name, lambda *args, gate, limit, **kwargs: given.append((gate, limit)))
    x, w = (torch.zeros(r, 256, dtype=torch.bfloat16) for r in (m, 2048))
    assert linear.gated_linear(x, w, "silu", 7.0).shape == (m, 1024)
    assert given == [("silu", None)]
