"""Several products of one shape in a launch (csrc/gemm_many.hip), and products of more than 128 rows into float32, at the edges of tiles and of
K's steps."""

import pytest
import torch

from tokamak_amd.kernels import gemm_bf16, linear, ops

DEV = "cuda:0"


def test_the_rule():
    assert ops.several_pay(4, 129, 4096, 4096) and ops.several_pay(4, 2048, 4096, 4096) and ops.several_pay(2, 300, 1024, 1024)
    assert not ops.several_pay(1, 2048, 4096, 4096) and not ops.several_pay(2, 129, 512, 8192)
    # a round and a bit of tiles of 256 x 256: four products, or two whose K is short, but not two or three that fill most of one each
    assert ops.several_pay(4, 2048, 2304, 6144) and ops.several_pay(2, 700, 12288, 1024) and ops.several_pay(2, 2048, 8192, 6144)
    assert not ops.several_pay(2, 700, 12288, 6144) and not ops.several_pay(3, 1500, 4096, 5120) and not ops.several_pay(4, 4096, 12288, 256)
    assert {ops.several_plan(4, m, n, k) for m, n, k in [(129, 4096, 4096), (512, 4096, 4096), (2048, 4096, 4096)]} >= {(128, 128), (256, 256)}


@pytest.mark.parametrize("m, n, k, several", [(129, 4096, 9216, False), (512, 12288, 12288, False), (1000, 4096, 16384, False), (129, 4096, 4096, True),
                                              (1101, 4096, 9216, True), (512, 2048, 8192, True)])
@pytest.mark.parametrize("shared", [False, True])
def test_products_in_shares_of_k_keep_their_sums(m, n, k, several, shared, monkeypatch):
    """What a product leaves for its reader to add in float32, several do, too."""
    went = []
    monkeypatch.setattr(ops, "gemm_several", lambda *a: went.append("several"))
    monkeypatch.setattr(gemm_bf16, "split_many", lambda x, w: went.append("shares"))
    x, w = (torch.empty(s, dtype=torch.bfloat16, device="meta") for s in ((m, k) if shared else (4, m, k), (4, n, k)))
    linear.several_linears(x, w)
    assert ops.several_pay(4, m, n, k) and went == (["several"] if several else ["shares"] * 4)


def test_more_than_a_launch_takes_or_off_its_borders_are_single_products(monkeypatch):
    went = []
    monkeypatch.setattr(linear, "linear", lambda x, w, allow_partials: went.append(tuple(x.shape)))
    made = lambda *s: torch.empty(s, dtype=torch.bfloat16, device="meta")      # noqa: E731
    linear.several_linears(made(200, 256), made(65, 256, 256))
    linear.several_linears(made(200, 256), made(3, 256 * 256 + 4)[:, :256 * 256].unflatten(1, (256, 256)))
    assert went == [(200, 256)] * 68


# integers, whose products and sums are exact in bfloat16's and float32's terms: every bit is known
@pytest.mark.gpu
@pytest.mark.parametrize("count, m, n, k", [(4, 129, 256, 64), (3, 300, 264, 128), (2, 257, 1016, 192), (4, 512, 1024, 1024), (4, 700, 4096, 320), (5, 1030, 520, 64)])
@pytest.mark.parametrize("shared", [False, True])
@pytest.mark.parametrize("tile", [None, *sorted(ops.MANY_PRICES)])
def test_several_products(count, m, n, k, shared, tile, monkeypatch):
    gen = torch.Generator().manual_seed(count * m + n + k)
    if tile is not None:
        monkeypatch.setattr(ops, "several_plan", lambda *a: tile)
    x = torch.full((1 if shared else count, m + 1, k + 8), float("nan"))
    w = torch.full((count, n + 1, k + 16), float("nan"))
    x[:, :m, :k] = torch.randint(-1, 2, (x.shape[0], m, k), generator=gen).float() * (torch.rand(x.shape[0], m, k, generator=gen) < 96 / k)
    w[:, :n, :k] = torch.randint(-1, 2, (count, n, k), generator=gen).float()
    a, b = (t.to(torch.bfloat16).to(DEV) for t in (x, w))
    a, b = a[:, :m, :k], b[:, :n, :k]
    out = torch.full((count, m + 1, n + 8), float("nan"), dtype=torch.bfloat16, device=DEV)
    ops.gemm_several(a[0] if shared else a, b, out[:, :m, :n])
    want = torch.matmul(x[:, :m, :k].double(), w[:, :n, :k].double().transpose(1, 2)).to(torch.bfloat16)
    assert torch.equal(out[:, :m, :n].cpu(), want)
    assert bool(out[:, m].isnan().all() and out[:, :, n:].isnan().all())


@pytest.mark.gpu
@pytest.mark.parametrize("m", [1, 64, 128, 129, 300])
@pytest.mark.parametrize("shared", [False, True])
def test_several_linears_are_the_linears(m, shared):
    gen = torch.Generator(device=DEV).manual_seed(m)
    x = torch.randn((m, 256) if shared else (4, m, 256), generator=gen, device=DEV).to(torch.bfloat16)
    w = torch.randn((4, 1024, 256), generator=gen, device=DEV).mul_(1 / 16).to(torch.bfloat16)
    for i, got in enumerate(linear.several_linears(x, w)):
        got = got.float().sum(0) if got.dim() == 3 else got.float()
        want = (x if shared else x[i]).double() @ w[i].double().T
        # sums of 256 products of 1 / 16 in float32, rounded to bfloat16: half a unit of 2^-8 of the value, and 256 times 2^-24 of some 4
        assert bool(((got.double() - want).abs() <= want.abs() * 2.0 ** -8 + 2.0 ** -14).all())


@pytest.mark.gpu
@pytest.mark.parametrize("m, n, k", [(129, 64, 64), (300, 1000, 128), (500, 4096, 64), (257, 264, 1024), (200, 100, 64), (140, 256, 72)])
def test_products_of_many_rows_into_float32(m, n, k):
    gen = torch.Generator().manual_seed(m + n + k)
    x, w = (torch.randint(-3, 4, s, generator=gen).to(torch.bfloat16).to(DEV) for s in ((m, k), (n, k)))
    got = linear.linear(x, w, out_dtype=torch.float32, allow_partials=True)
    assert torch.equal((got.sum(0) if got.dim() == 3 else got).cpu().double(), x.cpu().double() @ w.cpu().double().T)
