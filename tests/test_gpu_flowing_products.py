"""Products of up to 128 rows whose weights stream through LDS (csrc/gemm_flow.hip), at the edges of its tiles and shares.
Operands are small whole numbers, whose sums are exact in float32 in any order, so the results are too."""

import pytest
import torch

from gated_reference import gated, rounded
from tokamak_amd.kernels import linear, ops

DEV = "cuda:0"


def whole(rows, cols, most, seed):
    return torch.randint(-most, most + 1, (rows, cols), generator=torch.Generator().manual_seed(seed)).to(torch.bfloat16)


def inside(t):
    """The tensor as rows of a wider array of NaN: what is read or written past a row's end shows."""
    wide = torch.full((t.shape[0] + 2, t.shape[1] + 16), float("nan"), dtype=t.dtype, device=DEV)
    wide[1:-1, 8:-8].copy_(t)
    return wide, wide[1:-1, 8:-8]


def outside_is_nan(wide):
    return bool(torch.isnan(wide[0]).all() and torch.isnan(wide[-1]).all() and torch.isnan(wide[:, :8]).all() and torch.isnan(wide[:, -8:]).all())


ROWS = [1, 15, 16, 17, 33, 64, 65, 81, 97, 127, 128]


@pytest.mark.gpu
@pytest.mark.parametrize("m", ROWS)
@pytest.mark.parametrize("n, k", [(1, 128), (63, 256), (70, 384), (129, 1152), (260, 2048)])
def test_products_and_shares_of_k(m, n, k):
    x, w = whole(m, k, 3, 1), whole(n, k, 3, 2)
    exact = x.double() @ w.double().T          # at most 9 k in size: whole numbers of float32
    xs, ws = inside(x)[1], inside(w)[1]
    for dtype in (torch.bfloat16, torch.float32):
        wide, out = inside(torch.zeros(m, n, dtype=dtype))
        ops.gemm_flow(xs, ws, out)
        assert torch.equal(out.cpu(), exact.to(dtype)) and outside_is_nan(wide)
    wide, out = inside(torch.zeros(m, n, dtype=torch.bfloat16))
    ops.gemm_flow(xs, ws, out, activation="squared_relu")
    assert torch.equal(out.cpu(), (exact.clamp(min=0).float() ** 2).to(torch.bfloat16)) and outside_is_nan(wide)
    for parts in {1, 2, 3, k // 128}:
        if parts <= k // 128:
            sums = torch.full((parts + 1, m, n), float("nan"), device=DEV)
            ops.gemm_flow(xs, ws, sums[:parts])
            assert torch.equal(sums[:parts].double().sum(0).cpu(), exact) and torch.isnan(sums[parts]).all()


@pytest.mark.gpu
@pytest.mark.parametrize("m", [3, 17, 40, 96])
@pytest.mark.parametrize("parts", [2, 3, 4])
def test_shares_of_fewer_steps_than_there_are_tiles(m, parts):
    """Blocks of a share begin at each of its steps, and go round from its last to its first."""
    n, k = 700, 1408          # 11 tiles; 11 steps in shares of 2 to 6
    x, w = whole(m, k, 3, 15).to(DEV), whole(n, k, 3, 16).to(DEV)
    sums = torch.full((parts + 1, m, n), float("nan"), device=DEV)
    ops.gemm_flow(x, w, sums[:parts])
    for p in range(parts):
        cut = slice(p * 11 // parts * 128, (p + 1) * 11 // parts * 128)
        assert torch.equal(sums[p], x[:, cut].float() @ w[:, cut].float().T), p
    assert torch.isnan(sums[parts]).all()


@pytest.mark.gpu
@pytest.mark.parametrize("m", [3, 17, 40, 65, 96])
@pytest.mark.parametrize("bad", [float("inf"), float("-inf"), float("nan")])
def test_what_is_not_finite_stays_in_its_row_and_channel(m, bad):
    n, k = 136, 384
    x, w = whole(m, k, 3, 17).to(DEV), whole(n, k, 3, 18).to(DEV)
    exact = x.float() @ w.float().T
    x[m - 1, k - 1] = w[n - 1, 0] = bad
    out = torch.empty(2, m, n, device=DEV)
    ops.gemm_flow(x, w, out)
    assert torch.equal(out.sum(0)[:-1, :-1], exact[:-1, :-1])
    sums = x.float() @ w.float().T
    assert torch.equal(out.sum(0)[-1].nan_to_num(7.0), sums[-1].nan_to_num(7.0)) and torch.equal(out.sum(0)[:, -1].nan_to_num(7.0), sums[:, -1].nan_to_num(7.0))
    products = torch.empty(m, n // 2, dtype=torch.bfloat16, device=DEV)
    ops.gemm_flow(x, w, products, gate="silu")
    assert torch.isfinite(products[:-1, :-1]).all() and not torch.isfinite(products[:-1, -1]).any()


@pytest.mark.gpu
@pytest.mark.parametrize("m", ROWS)
@pytest.mark.parametrize("n, k", [(4, 128), (37, 256), (100, 512)])
def test_gates(m, n, k):
    x, w = whole(m, k, 3, 5), whole(2 * n, k, 1, 6)
    sums = x.double() @ w.double().T
    g, u = sums[:, :n], sums[:, n:]
    xs, ws = inside(x)[1], inside(w)[1]
    for gate, limit, want in (("silu", None, g * torch.sigmoid(g) * u),
                              ("gelu_tanh", None, torch.nn.functional.gelu(g, approximate="tanh") * u),
                              ("clamped", 2.5, g.clamp(max=2.5) * torch.sigmoid(1.702 * g.clamp(max=2.5)) * (u.clamp(-2.5, 2.5) + 1))):
        wide, out = inside(torch.zeros(m, n, dtype=torch.bfloat16))
        ops.gemm_flow(xs, ws, out, gate=gate, limit=limit)
        # half a unit of 2^-8 for the rounded result; the exponential's error is 2^-23 of its argument's size (up to 3 k);
        # 1 + tanh is off by 2^-22 of one where the tangent is near -1
        slack = 2.0 ** -22 * (g * u).abs() if gate == "gelu_tanh" else 0.0
        assert ((out.cpu().double() - want).abs() <= (2.0 ** -8 + 3 * k * 2.0 ** -22) * want.abs() + slack + 1e-30).all(), gate
        assert outside_is_nan(wide)


@pytest.mark.gpu
@pytest.mark.parametrize("m", [2, 3, 16, 17, 64, 65, 96, 97])
@pytest.mark.parametrize("n, k", [(1040, 256), (1040, 264), (1040, 2048)])
def test_every_route_gives_the_product(m, n, k):
    """On both sides of each condition of the routes, exactly."""
    x, w = whole(m, k, 2, 7).to(DEV), whole(n, k, 2, 8).to(DEV)
    exact = x.float() @ w.float().T
    assert torch.equal(linear.linear(x, w), exact.to(torch.bfloat16))
    assert torch.equal(linear.linear(x, w, torch.float32), exact)
    parts = linear.linear(x, w, allow_partials=True)
    assert torch.equal(parts.float().sum(0) if parts.dim() == 3 else parts, exact if parts.dim() == 3 else exact.to(torch.bfloat16))
    # (some routes round gate and up to bfloat16 first)
    want, slack = gated(exact.double(), rounded(exact.double()))
    assert ((linear.gated_linear(x, w).double() - want).abs() <= slack).all()


@pytest.mark.gpu
@pytest.mark.parametrize("m", [3, 16, 17, 64])
def test_rows_that_overlap_have_their_product(m):
    """One row of activations for all, and windows of one: rows closer together than they are long."""
    k, n = 256, 1040
    line, w = whole(1, k + 8 * m, 2, 9).to(DEV), whole(n, k, 2, 10).to(DEV)
    for x in (line[:, :k].expand(m, k), line.as_strided((m, k), (8, 1))):
        exact = x.float() @ w.float().T
        assert torch.equal(linear.linear(x, w), exact.to(torch.bfloat16))
        parts = linear.linear(x, w, allow_partials=True)
        assert torch.equal(parts.float().sum(0) if parts.dim() == 3 else parts, exact if parts.dim() == 3 else exact.to(torch.bfloat16))
        assert torch.equal(linear.activated_linear(x, w), (exact.clamp(min=0) ** 2).to(torch.bfloat16))
        want, slack = gated(exact.double(), rounded(exact.double()))
        assert ((linear.gated_linear(x, w).double() - want).abs() <= slack).all()


@pytest.mark.gpu
@pytest.mark.parametrize("m", [16, 17, 32, 33, 64, 65])
@pytest.mark.parametrize("n, k", [(40, 256), (1040, 256), (520, 4096), (16392, 128)])
def test_squared_relu_by_every_route(m, n, k):
    """In the epilogue of each product and behind shares of K.  Sums and their squares are exact in float32."""
    x, w = whole(m, k, 1, 11).to(DEV), whole(n, k, 1, 12).to(DEV)
    exact = (x.double() @ w.double().T).clamp(min=0) ** 2
    assert torch.equal(linear.activated_linear(x, w), exact.to(torch.bfloat16))


@pytest.mark.gpu
@pytest.mark.parametrize("activation, limit", [("silu", None), ("gelu_tanh", None), ("clamped", 2.5)])
@pytest.mark.parametrize("m", [17, 32, 33, 64, 65, 96])
@pytest.mark.parametrize("n, k", [(64, 4096), (1028, 2048), (1032, 2048), (16400, 128)])
def test_gates_behind_one_share_and_several(activation, limit, m, n, k):
    """Sums are exact, below 256 also in bfloat16, in which the library's route leaves them."""
    x, w = whole(m, k, 1, 13).to(DEV), whole(n, k, 1, 14).to(DEV)
    sums = x.double() @ w.double().T
    want, slack = gated(sums, torch.zeros_like(sums), activation, limit)
    assert sums.abs().max() <= 256
    assert ((linear.gated_linear(x, w, activation, limit).double() - want).abs() <= slack).all()
