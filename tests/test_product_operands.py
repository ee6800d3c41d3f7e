"""Which operands the flowing and the many-rows products take, on the CPU: nothing that their entry points refuse."""

import pytest
import torch

from tokamak_amd.kernels import ops


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
