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


# bundles of K dealt over the borders of groups: one piece, bundles fewer than, as many as and more than the waves, an odd last piece, blocks
# of one group and of two, a last group of one and of three rows
@pytest.mark.gpu
@pytest.mark.parametrize("m, n, k", [(1, 12000, 4), (4, 12001, 256), (3, 12007, 1028), (2, 17996, 2564), (16, 18000, 260), (5, 18001, 1284),
                                     (8, 20011, 2308), (1, 20480, 1540), (9, 18003, 772), (1, 65532, 516)])
def test_bundles_over_the_borders_of_groups(m, n, k):
    assert ops.fewrows_dealt(m, n)
    test_the_tiled_kernels_bits(m, n, k)


@pytest.mark.parametrize("m, n, k, dealt, rounds", [(1, 19456, 2560, 35.9, 39.7), (4, 19456, 2560, 37.0, 40.2), (1, 14000, 2560, 28.5, 31.5),
                                                    (1, 18624, 2176, 33.7, 37.2), (1, 38696, 2592, 70.2, 78.6), (1, 25216, 10624, 186, 209),
                                                    (1, 5120, 5120, 22.2, 21.6), (8, 13952, 3840, 47.0, 43.3)])
def test_bundles_are_dealt_where_that_was_faster(m, n, k, dealt, rounds):
    """Measured, us.  In rounds of a group 10 pieces of K keep six waves busy for ten twelfths of the time."""
    assert ops.fewrows_dealt(m, n) == (dealt < rounds)
    if dealt < rounds:
        group, waves, _, blocks = ops.fewrows_form(m, n, k)
        assert waves == 4 and group >= m and blocks <= -(-n // group)


@pytest.mark.parametrize("m, n, streamed, tiled", [(64, 12288, 90.0, 55.2), (48, 12288, 68.2, 55.0), (64, 6144, 84.6, 66.7), (56, 8200, 81.6, 43.6),
                                                   (64, 4096, 0.68, 1.0), (64, 2048, 0.67, 1.0), (32, 12288, 0.84, 1.0), (17, 1024, 0.27, 1.0)])
def test_rows_stream_the_weights_where_that_was_faster(m, n, streamed, tiled):
    """Measured times (us, or shares of the tiled kernel's)."""
    assert ops.fewrows_pays(m, n) == (streamed < tiled)
