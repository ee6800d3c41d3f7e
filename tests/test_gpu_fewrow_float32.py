"""The float32 product of up to sixteen rows (csrc/gemm_tiled.hip): groups of 4, 8 and 16 weight rows, one and several
rounds of pieces, more groups than blocks, at their edges, against the tiled kernel, whose bits it gives."""

import pytest
import torch

from tokamak_amd.kernels import ops

DEV = "cuda:0"

# (m, n, k): every group size, a last group of one row, a last piece of four k, one and several rounds of 4, 6 and 8 waves, blocks with
# several groups, and the loads further ahead of a head
SHAPES = [(1, 1, 4), (4, 1021, 1024), (3, 1029, 5124), (4, 4100, 2560), (1, 1, 4104), (5, 2041, 2308), (8, 2056, 4348), (7, 4097, 516),
          (9, 33, 9000), (16, 4111, 1028), (13, 8200, 260), (16, 13000, 1536), (2, 65540, 260), (16, 65537, 1284)]


def test_every_form_is_met():
    forms = {ops.fewrows_form(m, n, k)[:3] for m, n, k in SHAPES}
    assert {g for g, _, _ in forms} == {4, 8, 16} and {w for _, w, _ in forms} == {4, 6, 8} and (16, 4, 4) in forms
    for m, n, k in SHAPES:
        group, _, _, blocks = ops.fewrows_form(m, n, k)
        assert group >= m and 1 <= blocks <= -(-n // group)


@pytest.mark.gpu
@pytest.mark.parametrize("m, n, k", SHAPES)
def test_the_tiled_kernels_bits(m, n, k):
    gen = torch.Generator(device=DEV).manual_seed(m + n + k)
    x = torch.randn(100, k + 4, generator=gen, device=DEV)[:, :k]
    w = torch.full((n + 2, k + 8), float("nan"), device=DEV)
    w[1:-1, 4:-4].normal_(generator=gen)                   # (what is read past a row or past the matrix shows)
    w = w[1:-1, 4:-4]
    w[n // 2, k // 2] = float("inf")                        # an infinity stays in its column
    x[1 % m] = 0.0                                          # and meets a row of zeros
    whole = torch.empty(100, n, device=DEV)
    ops.gemm_tiled(x, w, whole)
    wide = torch.full((m + 2, n + 8), float("nan"), device=DEV)
    ops.gemm_tiled(x[:m], w, wide[1:-1, 4:-4])
    assert torch.equal(wide[1:-1, 4:-4].view(torch.int32), whole[:m].view(torch.int32)) or torch.equal(
        wide[1:-1, 4:-4].nan_to_num(7.0), whole[:m].nan_to_num(7.0))
    assert bool(wide[0].isnan().all() and wide[-1].isnan().all() and wide[:, :4].isnan().all() and wide[:, -4:].isnan().all())
