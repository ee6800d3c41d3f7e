"""The float32 product in tiles (csrc/gemm_float32.hip): every tile at its edges, stages of 32 k that K ends in, pieces of 256, against
float64 and against the kernel for operands off their borders, whose bits it gives."""

import pytest
import torch

from tokamak_amd.kernels import ops

DEV = "cuda:0"
# one tile less a row and a column, whole ones, one more; K of one step, of less than, exactly and more than a stage, two and three, and of
# pieces
SHAPES = [(0, 0, 4), (-1, -1, 28), (1, 3, 32), (0, 1, 36), (1, 1, 64), (-1, 2, 100), (2, 0, 256), (1, 1, 260), (3, -2, 516), (1, 1, 1024)]


def test_the_rule_meets_every_tile():
    met = {ops.float32_tile(m, n, k) for m, n, k in [(40, 512, 1024), (600, 12288, 2048), (300, 12288, 2048), (600, 4096, 2048),
                                                (1053, 2048, 6144)]}
    assert met == set(ops.FLOAT32_PRICES)
    assert ops.float32_tiles_pay(24, 151936, 1024) and ops.float32_tiles_pay(64, 1024, 1024)
    assert not ops.float32_tiles_pay(40, 4096, 2048) and not ops.float32_tiles_pay(64, 2048, 6144)
    assert not any(ops.float32_tiles_pay(m, 12288, k) for m in (17, 20, 24, 28, 32) for k in (1024, 2048))      # 43 us and 49


# us in tiles through LDS and through registers
@pytest.mark.parametrize("m, n, k, registers", [
    (2048, 4096, 64, True), (200, 4096, 64, True), (4096, 32768, 32, True), (4096, 8192, 96, True),      # 22.2 and 18.7, 5.9 and 5.2, 346 and 155, 82 and 77
    (100, 4096, 64, False), (1053, 2048, 32, False), (2048, 4096, 96, False), (4096, 16384, 128, False), (2048, 4096, 1024, False)])
def test_a_short_k_of_many_results_goes_through_registers(m, n, k, registers):
    assert ops.float32_through_registers(m, n, k) is registers


@pytest.mark.gpu
@pytest.mark.parametrize("m, n, k", [(130, 4100, 64), (2049, 2057, 32), (129, 4099, 36)])
def test_both_give_the_same_bits_there(m, n, k):
    gen = torch.Generator(device=DEV).manual_seed(m)
    x, w = (torch.randn(s, generator=gen, device=DEV) for s in ((m, k), (n, k)))
    out, tiles = torch.empty(m, n, device=DEV), torch.empty(m, n, device=DEV)
    assert ops.float32_through_registers(m, n, k)
    ops.gemm_tiled(x, w, out)
    ops._check(ops._fn("gemm_float32", "tk_gemm_float32")(ops._p(x), ops._p(w), ops._p(tiles), m, n, k, k, k, n, 96, 96, ops._stream()), "gemm_float32")
    assert torch.equal(out, tiles)


@pytest.mark.gpu
@pytest.mark.parametrize("more_m, more_n, k", SHAPES)
@pytest.mark.parametrize("tile", sorted(ops.FLOAT32_PRICES))
def test_every_tile(tile, more_m, more_n, k):
    m, n = 2 * tile[0] + more_m, 9 * tile[1] + more_n
    gen = torch.Generator(device=DEV).manual_seed(m + n + k)
    x = torch.full((m + 2, k + 8), float("nan"), device=DEV)[1:-1, 4:-4]      # (what is read past a row or past the matrix shows)
    w = torch.full((n + 2, k + 8), float("nan"), device=DEV)[1:-1, 4:-4]
    x.normal_(generator=gen)
    w.normal_(generator=gen)
    out = torch.full((m + 2, n + 5), float("nan"), device=DEV)
    inner = out[1:-1, 2:-3]
    ops._check(ops._fn("gemm_float32", "tk_gemm_float32")(ops._p(x), ops._p(w), ops._p(inner), m, n, k, x.stride(0), w.stride(0),
                                                          inner.stride(0), *tile, ops._stream()), "gemm_float32")
    want = x.double() @ w.double().T
    # 2^-24 a step of a piece of 256 and of the pieces, times the sum of magnitudes
    bound = 2.0 ** -24 * (min(k, 256) + -(-k // 256)) * (x.double().abs() @ w.double().abs().T)
    assert bool(((inner.double() - want).abs() <= bound).all())
    off = torch.empty((m, k + 1), device=DEV)[:, 1:].copy_(x)                  # rows off their borders: the other kernel
    other = torch.empty((m, n), device=DEV)
    ops.gemm_tiled(off, w, other)
    assert torch.equal(inner, other)
    edge = out.clone()
    edge[1:-1, 2:-3] = float("nan")
    assert bool(edge.isnan().all())


@pytest.mark.gpu
def test_what_it_refuses():
    x, w, out = (torch.zeros(64, 64, device=DEV) for _ in range(3))
    fn, tail = ops._fn("gemm_float32", "tk_gemm_float32"), (ops._stream(),)
    for k, lda, ldw, tile in [(62, 64, 64, (32, 32)), (0, 64, 64, (32, 32)), (64, 63, 64, (32, 32)), (64, 64, 66, (32, 32)), (64, 64, 64, (128, 128)),
                              (64, 1 << 24, 64, (32, 32))]:
        assert fn(ops._p(x), ops._p(w), ops._p(out), 64, 64, k, lda, ldw, 64, *tile, *tail) == -1
    assert fn(ops._p(x[:, 1:]), ops._p(w), ops._p(out), 64, 64, 60, 64, 64, 64, 32, 32, *tail) == -1
