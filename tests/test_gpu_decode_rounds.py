"""Decode attention whose keys are dealt to blocks in rounds of 128: every number of splits at lengths around the rounds'
edges, tokens named by their requests or being them."""

import pytest
import torch
from kernel_util import pack_pages_whole, reference_attention

pytestmark = pytest.mark.gpu
DEV = "cuda:0"
LENGTHS = [1, 15, 16, 17, 127, 128, 129, 255, 257, 385, 1000, 1025]

@pytest.mark.parametrize("hd, nh, nkv, ps", [(128, 16, 8, 16), (64, 14, 2, 32), (128, 16, 1, 64)])
@pytest.mark.parametrize("splits", [1, 2, 3, 8, 9, 17])
def test_rounds(hd, nh, nkv, ps, splits):
    from tokamak_amd.kernels import ops

    n = len(LENGTHS)
    g = torch.Generator().manual_seed(hd + splits)
    pages = [-(-t // ps) for t in LENGTHS]
    k_cache = torch.full((sum(pages) + 1, nkv * hd * ps), float("nan"), dtype=torch.bfloat16)    # (slots that no token wrote)
    v_cache = k_cache.clone()
    order = (torch.randperm(sum(pages), generator=g) + 1).tolist()
    tables = torch.zeros(n, max(pages), dtype=torch.int32)
    q = torch.randn(n, nh, hd, generator=g).to(torch.bfloat16)
    want = torch.empty(n, nh, hd, dtype=torch.float64)
    for r, t in enumerate(LENGTHS):
        table = [order.pop() for _ in range(pages[r])]
        tables[r, :pages[r]] = torch.tensor(table)
        k, v = (torch.randn(t, nkv, hd, generator=g).to(torch.bfloat16) for _ in range(2))
        pack_pages_whole(k_cache, v_cache, k, v, table, ps)
        for off in range(t % ps or ps, ps):      # what lies behind the sequence's end in its last page must not count
            k_cache[table[-1]].view(nkv, hd // 8, ps, 8)[:, :, off] = float("nan")
            v_cache[table[-1]].view(nkv, hd // 16, ps // 4, 16, 4)[:, :, off // 4, :, off % 4] = float("nan")
        want[r] = reference_attention(q[r:r + 1], k, v, [t - 1], hd ** -0.5)[0]
    k_cache, v_cache, tables, q_dev = (t.to(DEV) for t in (k_cache, v_cache, tables, q))
    positions = torch.tensor([t - 1 for t in LENGTHS], dtype=torch.int32, device=DEV)
    items = torch.tensor(sorted(range(n), key=lambda r: -LENGTHS[r]), dtype=torch.int32, device=DEV)
    outs = []
    for requests in (torch.arange(n, dtype=torch.int32, device=DEV), None):
        out = torch.full((n, nh, hd), float("nan"), dtype=torch.bfloat16, device=DEV)
        assert ops.attention_mfma("heads", q_dev, k_cache, v_cache, tables, positions, requests, items, None, n, out,
                                  num_heads=nh, num_kv_heads=nkv, head_dim=hd, page_size=ps, scale=hd ** -0.5,
                                  split_keys=-(-1025 // splits // 128 + 1) * 128, num_splits=splits)
        outs.append(out)
    assert torch.equal(*outs)
    # probabilities and the result are rounded to bfloat16 (2^-9 each, of values of unit spread); the sums are float32
    torch.testing.assert_close(outs[0].cpu().double(), want, rtol=2.0 ** -8, atol=4 * 2.0 ** -8)
