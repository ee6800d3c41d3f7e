"""Products of many rows (csrc/gemm_many.hip): every tile at its edges, in one round of blocks and in several, in shares of K and
gated.  Operands are small whole numbers, whose sums are exact in float32 in any order, so the results are too."""

import pytest
import torch

from gated_reference import gated
from tokamak_amd.kernels import linear, ops

DEV = "cuda:0"
TILES = [(256, 256), (128, 256), (256, 128), (128, 128)]


def whole(rows, cols, most, seed):
    return torch.randint(-most, most + 1, (rows, cols), generator=torch.Generator().manual_seed(seed)).to(torch.bfloat16)


def inside(t, value=float("nan")):
    """The tensor as rows of a wider array of ``value``: what is read or written past a row's end shows."""
    wide = torch.full((t.shape[0] + 2, t.shape[1] + 16), value, dtype=t.dtype, device=DEV)
    wide[1:-1, 8:-8].copy_(t)
    return wide, wide[1:-1, 8:-8]


def outside_is_nan(wide):
    return bool(torch.isnan(wide[0]).all() and torch.isnan(wide[-1]).all() and torch.isnan(wide[:, :8]).all() and torch.isnan(wide[:, -8:]).all())


@pytest.mark.gpu
@pytest.mark.parametrize("tile", TILES)
@pytest.mark.parametrize("m, n, k", [(1, 8, 64), (127, 136, 128), (129, 256, 192), (257, 264, 64), (513, 520, 1088)])
def test_tiles_and_shares_of_k(tile, m, n, k):
    rows, columns = tile
    x, w = whole(m, k, 3, 1), whole(n, k, 3, 2)
    exact = x.double() @ w.double().T          # at most 9 k in size: whole numbers of float32
    xs, ws = inside(x)[1], inside(w)[1]
    for parts in {1, 2, 3, k // 64}:
        if parts <= k // 64:
            sums = torch.full((parts + 1, m, n), float("nan"), device=DEV)
            ops.gemm_many(xs, ws, sums[:parts], rows=rows, columns=columns)
            assert torch.equal(sums[:parts].double().sum(0).cpu(), exact) and torch.isnan(sums[parts]).all()


@pytest.mark.gpu
@pytest.mark.parametrize("tile, m, n", [((256, 256), 4200, 4360), ((128, 256), 2200, 4360), ((256, 128), 4200, 2312), ((128, 128), 3000, 3080)])
@pytest.mark.parametrize("k", [64, 192])
def test_more_tiles_than_blocks_run_at_once(tile, m, n, k):
    x, w = whole(m, k, 3, 3).to(DEV), whole(n, k, 3, 4).to(DEV)
    out = torch.full((1, m, n), float("nan"), device=DEV)
    ops.gemm_many(x, w, out, rows=tile[0], columns=tile[1])
    assert torch.equal(out[0], x.float() @ w.float().T)


@pytest.mark.gpu
@pytest.mark.parametrize("tile", TILES)
@pytest.mark.parametrize("m, n, k", [(1, 8, 64), (130, 72, 128), (255, 136, 192), (300, 1000, 64)])
def test_gates(tile, m, n, k):
    rows, columns = tile
    x, w = whole(m, k, 3, 5), whole(2 * n, k, 1, 6)
    sums = x.double() @ w.double().T
    g, u = sums[:, :n], sums[:, n:]
    xs, ws = inside(x)[1], inside(w)[1]
    for gate, limit, want in (("silu", None, g * torch.sigmoid(g) * u),
                              ("gelu_tanh", None, g * torch.sigmoid(2 * (2 / torch.pi) ** 0.5 * (g + 0.044715 * g ** 3)) * u),
                              ("clamped", 2.5, g.clamp(max=2.5) * torch.sigmoid(1.702 * g.clamp(max=2.5)) * (u.clamp(-2.5, 2.5) + 1))):
        wide, out = inside(torch.zeros(m, n, dtype=torch.bfloat16))
        ops.gemm_many(xs, ws, out, rows=rows, columns=columns, gate=gate, limit=limit)
        # half a unit of 2^-8 for the rounded result; the exponential's error is 2^-23 of its argument's size (up to 3 k), no more
        assert ((out.cpu().double() - want).abs() <= (2.0 ** -8 + 3 * k * 2.0 ** -22) * want.abs() + 1e-30).all() and outside_is_nan(wide)


SEVERAL = [((256, 256), 2100, 2568), ((128, 256), 1100, 2568), ((256, 128), 2100, 1288), ((128, 128), 2100, 1288)]


@pytest.mark.gpu
@pytest.mark.parametrize("tile, m, n", SEVERAL)
@pytest.mark.parametrize("parts, k", [(3, 320), (6, 704)])
def test_several_rounds_of_shares_of_unlike_length(tile, m, n, parts, k):
    """A block goes on to a unit of another share, longer or shorter than its own, while the loads of both are under way."""
    x, w = whole(m, k, 3, 9).to(DEV), whole(n, k, 3, 10).to(DEV)
    out = torch.full((parts + 1, m, n), float("nan"), device=DEV)
    ops.gemm_many(x, w, out[:parts], rows=tile[0], columns=tile[1])
    steps = k // 64
    for p in range(parts):
        cut = slice(p * steps // parts * 64, (p + 1) * steps // parts * 64)
        assert torch.equal(out[p], x[:, cut].float() @ w[:, cut].float().T), p
    assert torch.isnan(out[parts]).all()


@pytest.mark.gpu
@pytest.mark.parametrize("tile, m, n", [((256, 256), 2100, 3720), ((128, 256), 2100, 2056), ((256, 128), 4200, 1032), ((128, 128), 3000, 1480)])
@pytest.mark.parametrize("k", [64, 192])
def test_gates_in_several_rounds(tile, m, n, k):
    """Sums are exact, so the result is off by half a unit of 2^-8 and the exponential's error, 2^-23 of its argument's size."""
    x, w = whole(m, k, 1, 11).to(DEV), whole(2 * n, k, 1, 12).to(DEV)
    out = torch.full((m, n), float("nan"), dtype=torch.bfloat16, device=DEV)
    ops.gemm_many(x, w, out, rows=tile[0], columns=tile[1], gate="silu")
    sums = (x.float() @ w.float().T).double()
    want = torch.nn.functional.silu(sums[:, :n]) * sums[:, n:]
    assert ((out.double() - want).abs() <= (2.0 ** -8 + k * 2.0 ** -22) * want.abs() + 1e-30).all()


@pytest.mark.gpu
@pytest.mark.parametrize("tile", TILES)
@pytest.mark.parametrize("bad", [float("inf"), float("-inf"), float("nan")])
def test_what_is_not_finite_stays_in_its_row_and_channel(tile, bad):
    m, n, k = 300, 272, 192
    x, w = whole(m, k, 3, 13).to(DEV), whole(n, k, 3, 14).to(DEV)
    exact = x.float() @ w.float().T
    x[m - 1, k - 1] = w[n - 1, 0] = bad
    out = torch.empty(3, m, n, device=DEV)
    ops.gemm_many(x, w, out, rows=tile[0], columns=tile[1])
    assert torch.equal(out.sum(0)[:-1, :-1], exact[:-1, :-1])
    sums = x.float() @ w.float().T
    assert torch.equal(out.sum(0)[-1].nan_to_num(7.0), sums[-1].nan_to_num(7.0)) and torch.equal(out.sum(0)[:, -1].nan_to_num(7.0), sums[:, -1].nan_to_num(7.0))
    products = torch.empty(m, n // 2, dtype=torch.bfloat16, device=DEV)
    ops.gemm_many(x, w, products, rows=tile[0], columns=tile[1], gate="silu")
    assert torch.isfinite(products[:-1, :-1]).all() and not torch.isfinite(products[:-1, -1]).any()


@pytest.mark.gpu
@pytest.mark.parametrize("activation, limit", [("silu", None), ("clamped", 7.0), ("gelu_tanh", None)])
@pytest.mark.parametrize("m, n, k", [(128, 256, 256), (129, 256, 256), (300, 248, 320), (300, 252, 320), (300, 256, 328), (300, 504, 1024), (300, 512, 1024),
                                     (129, 128, 2048), (700, 2048, 2048)])
def test_gated_products_by_any_route(activation, limit, m, n, k):
    """On both sides of each condition of the route, the same numbers to bfloat16's rounding."""
    gen = torch.Generator().manual_seed(m + n + k)
    x = torch.randn(m, k, generator=gen).to(torch.bfloat16).to(DEV)
    w = (torch.randn(2 * n, k, generator=gen) * k ** -0.5).to(torch.bfloat16).to(DEV)
    got = linear.gated_linear(x, w, activation, limit).double()
    sums = x.double() @ w.double().T
    # a float32 sum of k products, then (some routes) rounded to bfloat16, whose eight bits are off by up to 2^-8
    off = 2.0 ** -8 * sums.abs() + k * 2.0 ** -24 * (x.double().abs() @ w.double().abs().T)
    want, slack = gated(sums, off, activation, limit)
    assert ((got - want).abs() <= slack).all()


@pytest.mark.gpu
@pytest.mark.parametrize("m, n, k, split", [(128, 264, 9216, True), (129, 264, 9216, True), (1100, 136, 9280, True), (1101, 136, 9280, False),
                                            (300, 264, 9152, False), (1700, 136, 16384, True), (1701, 136, 16384, False), (300, 260, 9216, False), (300, 20480, 9216, None)])
def test_long_products_leave_shares_of_k_to_a_reader_that_adds_them(m, n, k, split):
    """On both sides of each condition (below 129 rows other kernels split), and for a reader that takes only the product."""
    x, w = whole(m, k, 1, 7).to(DEV), whole(n, k, 1, 8).to(DEV)
    exact = x.float() @ w.float().T          # at most k in size
    got = linear.linear(x, w, allow_partials=True)
    assert split is None or (got.dim() == 3) == split or m <= 128
    if got.dim() == 3:
        assert got.dtype == torch.float32 and torch.equal(got.double().sum(0), exact.double())
    else:
        assert torch.equal(got, exact.to(torch.bfloat16))
    assert torch.equal(linear.linear(x, w), exact.to(torch.bfloat16))
