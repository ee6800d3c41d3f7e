"""The float32 products at the edges of their tiles and stages: against float64, and the same bits whichever kernel
multiplies a row."""

import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


# tiles of 64 and of 128 outputs a side, stages of 64 and 32 k, pieces of 256: one short, whole, one more
@pytest.mark.parametrize("m,n,k", [(17, 63, 4), (65, 130, 60), (64, 64, 64), (129, 65, 68), (70, 200, 252), (66, 100, 260),
                                   (2050, 2051, 36), (2048, 2048, 292), (1, 151, 516), (16, 65, 1028), (130, 70, 1023)])
@pytest.mark.parametrize("aligned", [True, False])
def test_float32_product(m, n, k, aligned):
    from tokamak_amd.kernels import ops

    g = torch.Generator().manual_seed(m + n + k)
    pad = 0 if aligned else 1          # rows that do not begin on 16-byte borders
    x = torch.randn(m, k + pad, generator=g).to(DEV)[:, pad:]
    w = torch.randn(n, k + pad, generator=g).to(DEV)[:, pad:]
    out = torch.full((m, n), float("nan"), device=DEV)
    ops.gemm_tiled(x, w, out)
    want = x.cpu().double() @ w.cpu().double().T
    # two levels of sums: 2^-24 a step of a piece of 256 and of the pieces, times the sum of magnitudes
    bound = 2.0 ** -24 * (min(k, 256) + -(-k // 256)) * (x.cpu().double().abs() @ w.cpu().double().abs().T)
    assert bool(((out.cpu().double() - want).abs() <= bound).all())
    few = torch.full((min(m, 3), n), float("nan"), device=DEV)
    for split in (False, True):        # a few of the rows by themselves: the kernel for few rows where the operands allow it
        few.fill_(float("nan"))
        ops.gemm_tiled(x[:3], w, few, fewrows_split=split)
        assert torch.equal(few, out[:3])


# one operand's rows on 16-byte borders, the other's not; K whole pieces, and not
@pytest.mark.parametrize("m,n,k", [(17, 63, 4), (65, 130, 61), (129, 65, 68), (70, 200, 254), (2050, 2051, 35), (2048, 2048, 292), (66, 100, 3)])
@pytest.mark.parametrize("off", ["x", "w", "neither"])
def test_operands_on_and_off_their_borders(m, n, k, off):
    from tokamak_amd.kernels import ops

    g = torch.Generator().manual_seed(m + n + k)
    x, w = (torch.randn(rows, k, generator=g).to(DEV) for rows in (m, n))
    ld = (k + 7) // 4 * 4

    def placed(t, shift):
        there = torch.full((t.shape[0], ld), float("nan"), device=DEV)[:, shift:shift + k]
        return there.copy_(t)

    out, want = (torch.full((m, n), float("nan"), device=DEV) for _ in range(2))
    ops.gemm_tiled(placed(x, int(off == "x")), placed(w, int(off == "w")), out)
    ops.gemm_tiled(torch.nn.functional.pad(x, (1, 4 - (k + 1) % 4))[:, 1:1 + k], torch.nn.functional.pad(w, (1, 4 - (k + 1) % 4))[:, 1:1 + k], want)
    assert torch.equal(out, want)
    exact = x.cpu().double() @ w.cpu().double().T
    bound = 2.0 ** -24 * (min(k, 256) + -(-k // 256)) * (x.cpu().double().abs() @ w.cpu().double().abs().T)
    assert bool(((out.cpu().double() - exact).abs() <= bound).all())
