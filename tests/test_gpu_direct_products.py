"""The products of up to sixteen rows whose weights go straight into matrix operands
(csrc/gemm_direct.hip): every form at the edges of its tiles, against 64-bit sums."""

import pytest
import torch

from tokamak_amd.kernels import ops

DEV = "cuda:0"

PLANS = {4: [(4, 1, 4), (4, 2, 8), (4, 4, 8)], 8: [(4, 1, 8), (8, 1, 4), (8, 2, 8)], 16: [(8, 1, 8), (8, 2, 4)]}
SHAPES = [(1, 4, 8), (2, 20, 72), (3, 1000, 264), (4, 96, 4104), (5, 36, 1032), (8, 1028, 520), (9, 20, 136), (16, 1000, 1800)]
CASES = [(m, n, k, plan) for m, n, k in SHAPES for plan in PLANS[4 if m <= 4 else 8 if m <= 8 else 16]]


def rand(*shape, seed=0, scale=1.0):
    return torch.randn(*shape, generator=torch.Generator().manual_seed(seed)) * scale


def operands(m, n, k):
    x, w = rand(m, k, seed=1).to(torch.bfloat16), rand(n, k, seed=2, scale=k ** -0.5).to(torch.bfloat16)
    exact, size = x.double() @ w.double().T, x.double().abs() @ w.double().abs().T
    return x, w, exact, size


def guarded(t):
    """The tensor as rows of a wider array of NaN: what is read or written past a row's end shows."""
    wide = torch.full((t.shape[0] + 2, t.shape[1] + 16), float("nan"), dtype=t.dtype, device=DEV)
    inner = wide[1:-1, 8:-8]
    inner.copy_(t)
    return wide, inner


def untouched(wide):
    return bool(torch.isnan(wide[0]).all() and torch.isnan(wide[-1]).all() and torch.isnan(wide[:, :8]).all()
                and torch.isnan(wide[:, -8:]).all())


# a sum of k products in float32, in any order, is within k 2^-24 of the sum of their magnitudes (2^-23: the matrix units may cut
# instead of rounding); a bfloat16 result adds half a unit of 2^-8
def bound(k, size, exact=None):
    return k * 2.0 ** -23 * size + (0.0 if exact is None else 2.0 ** -8 * exact.abs()) + 1e-30


@pytest.mark.gpu
@pytest.mark.parametrize("m, n, k, plan", CASES)
def test_plain_and_scaled(m, n, k, plan):
    x, w, exact, size = operands(m, n, k)
    xs, ws = guarded(x)[1], guarded(w)[1]
    for dtype in (torch.float32, torch.bfloat16):
        wide, out = guarded(torch.zeros(m, n, dtype=dtype))
        ops.gemm_direct(xs, ws, out, plan=plan)
        assert ((out.cpu().double() - exact).abs() <= bound(k, size, exact if dtype == torch.bfloat16 else None)).all()
        assert untouched(wide)
    relu = torch.empty(m, n, device=DEV)
    ops.gemm_direct(xs, ws, relu, activation="squared_relu", plan=plan)
    top = exact.abs() + bound(k, size)
    assert ((relu.cpu().double() - exact.clamp(min=0) ** 2).abs() <= 2 * top * bound(k, size) + 2.0 ** -23 * top ** 2).all()
    for slabs in (1, 37, 700):
        sumsq, eps = rand(slabs, m, seed=slabs).abs() * k / slabs, 1e-2
        scale = torch.rsqrt(sumsq.double().sum(0) / k + eps)[:, None]
        out = torch.empty(m, n, device=DEV)
        ops.gemm_direct(xs, ws, out, sumsq=sumsq.to(DEV), eps=eps, plan=plan)
        # the scale: a sum of `slabs` positive numbers, a division, a root of 1 ulp, a product
        assert ((out.cpu().double() - exact * scale).abs() <= scale * bound(k, size) + (slabs + 8) * 2.0 ** -24 * (exact * scale).abs()).all()


@pytest.mark.gpu
@pytest.mark.parametrize("m, n, k, plan", CASES)
def test_gated(m, n, k, plan):
    x, w, exact, size = operands(m, 2 * n, k)
    for activation, limit in (("silu", None), ("gelu_tanh", None), ("clamped", 0.7)):
        wide, out = guarded(torch.zeros(m, n, dtype=torch.bfloat16))
        ops.gemm_direct(x.to(DEV), w.to(DEV), out, gated=True, activation=activation, limit=limit, plan=plan)
        z, u = exact[:, :n], exact[:, n:]
        if activation == "silu":
            want = z * torch.sigmoid(z) * u
        elif activation == "gelu_tanh":
            want = torch.nn.functional.gelu(z, approximate="tanh") * u
        else:
            g = z.clamp(max=limit)
            want = g * torch.sigmoid(1.702 * g) * (u.clamp(-limit, limit) + 1)
        # |act'| <= 1.13 for each, |act(z)| <= |z|; the device's exponential and tanh are within 2^-18 of the value
        slack = 1.13 * bound(k, size[:, :n]) * (u.abs() + 2) + z.abs() * bound(k, size[:, n:]) + 2.0 ** -18 * z.abs() * (u.abs() + 2)
        assert ((out.cpu().double() - want).abs() <= slack + 2.0 ** -8 * want.abs() + 1e-30).all(), activation
        assert untouched(wide)


@pytest.mark.gpu
@pytest.mark.parametrize("m, n, k, plan", CASES)
def test_adds_into_the_stream(m, n, k, plan):
    x, w, exact, size = operands(m, n, k)
    stream, gamma = rand(m, n, seed=3), 1 + 0.3 * rand(n, seed=4)
    want = stream.double() + exact
    slack = bound(k, size) + 2.0 ** -24 * want.abs()
    wide, resid = guarded(stream)
    sumsq, scaled = ops.gemm_direct_add(x.to(DEV), w.to(DEV), resid, gamma.to(DEV), plan=plan)
    assert ((resid.cpu().double() - want).abs() <= slack).all() and untouched(wide)
    assert ((scaled.cpu().double() - want * gamma.double()).abs() <= 1.5 * slack + 2.0 ** -8 * (want * gamma.double()).abs()).all()
    columns = plan[0] * plan[1]
    assert sumsq.shape == (-(-n // columns), m)
    padded = torch.zeros(m, sumsq.shape[0] * columns, dtype=torch.float64)
    padded[:, :n] = resid.cpu().double()
    torch.testing.assert_close(sumsq.cpu().double(), (padded.view(m, -1, columns) ** 2).sum(2).T, rtol=columns * 2.0 ** -23, atol=1e-12)
    again = guarded(stream)[1]
    sums, none = ops.gemm_direct_add(x.to(DEV), w.to(DEV), again, None, plan=plan)
    assert none is None and torch.equal(sums, sumsq) and torch.equal(again, resid)


def test_every_size_has_a_form_of_the_kernel():
    """The plan names a form that is built, covers every column, and keeps the slabs within what the reader takes."""
    built = {(rows, tiles, groups) for m, plans in PLANS.items() for rows, groups, _ in plans for tiles in (-(-m // rows),)}
    for m in range(1, 17):
        for n in (4, 20, 64, 1000, 1024, 1028, 2560, 3072, 5120, 9728, 17408, 151936):
            for k in (8, 1024, 4096, 17408):
                for slabs in (0, 512):
                    rows, groups, waves = ops.direct_plan(m, n, k, most_slabs=slabs)
                    tiles = -(-m // rows)
                    assert (rows, tiles, groups) in built and waves in (4, 8) and rows * tiles >= m
                    blocks = -(-n // (rows * groups))
                    assert not slabs or blocks <= slabs or n > slabs * 16
    assert not ops.direct_pays("plain", 17, 64, 64) and not ops.direct_pays("add", 0, 64, 64)


# (what it competes with, rows, columns, K, us of the direct product, us of the other form)
MEASURED = [("activated", 16, 5120, 17408, 63.7, 33.7), ("activated", 8, 5120, 17408, 49.6, 32.9), ("activated", 3, 5120, 17408, 36.4, 32.2),
            ("activated", 16, 5120, 5120, 21.8, 14.7), ("activated", 16, 28672, 4096, 55.3, 38.2), ("activated", 16, 4432, 7048, 34.4, 18.3),
            ("activated", 16, 2048, 6144, 11.0, 15.5), ("activated", 16, 4096, 4096, 11.1, 12.2), ("activated", 8, 752, 9080, 9.2, 15.3),
            ("activated", 1, 5120, 5120, 10.7, 13.6),
            ("plain", 16, 24576, 4096, 48.1, 34.7), ("plain", 16, 28672, 4096, 55.1, 38.0), ("plain", 8, 24576, 4096, 37.2, 34.0),
            ("plain", 16, 13544, 760, 9.9, 8.0), ("plain", 9, 18792, 11184, 107, 94), ("plain", 4, 34816, 5120, 59.7, 71.7),
            ("plain", 16, 4096, 12288, 25.4, 64.0), ("plain", 6, 16384, 4096, 24.0, 28.6),
            ("add", 16, 368, 11144, 18.7, 10.2), ("add", 16, 824, 14256, 22.0, 14.6), ("add", 16, 3224, 3896, 12.3, 10.4),
            ("add", 3, 5120, 17408, 41.5, 34.5), ("add", 16, 6144, 5120, 22.0, 17.8),
            ("add", 16, 1024, 3072, 7.1, 7.7), ("add", 8, 4096, 12288, 21.1, 21.9), ("add", 6, 4096, 14336, 22.5, 24.4), ("add", 16, 4096, 4096, 11.4, 11.6),
            ("add", 9, 2560, 4096, 9.1, 8.3)]


@pytest.mark.parametrize("kind, m, n, k, direct, other", MEASURED)
def test_the_direct_product_is_taken_where_it_was_faster(kind, m, n, k, direct, other):
    assert ops.direct_pays(kind, m, n, k) == (direct < other)


@pytest.mark.gpu
@pytest.mark.parametrize("m, n, k, plan", [(1, 20, 72, (4, 1, 4)), (3, 96, 200, (4, 4, 8)), (4, 1000, 1160, (4, 2, 8)), (8, 40, 72, (8, 1, 8)), (5, 36, 136, (4, 1, 8)),
                                           (16, 100, 1096, (8, 2, 4)), (9, 20, 8, (8, 1, 8)), (2, 512, 264, None)])
def test_an_infinite_weight_stays_what_it_is(m, n, k, plan):
    """K is not whole steps: what the last step has no numbers for is zeros of both operands, so that a row whose last
    weights hold an infinity is infinite, not NaN."""
    x, w = rand(m, k, seed=1).abs().to(torch.bfloat16) + 0.125, rand(n, k, seed=2, scale=k ** -0.5).to(torch.bfloat16)
    row = n // 2
    w[row, k - 3] = float("inf")
    out = torch.empty(m, n, device=DEV)
    ops.gemm_direct(x.to(DEV), w.to(DEV), out, plan=plan)
    want = x.double() @ w.double().T
    assert torch.equal(out.cpu()[:, row], want[:, row].float()) and torch.isinf(want[:, row]).all()
    assert torch.isfinite(out).sum() == m * (n - 1)
