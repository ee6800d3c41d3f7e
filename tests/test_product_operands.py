"""What reaches the flowing and the many-rows products, on the CPU: nothing that their entry points refuse."""

import pytest
import torch

from tokamak_amd.kernels import gemm_bf16, linear, ops


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


@pytest.mark.parametrize("m", [17, 64, 129, 300])
def test_a_limit_beside_the_silu_gate_is_not_looked_at(monkeypatch, m):
    """At any number of rows, by whichever kernel (which has a limit for the clamped gate alone)."""
    given = []
    for name in ("gemm_flow", "gemm_many"):
        monkeypatch.setattr(ops, name, lambda *args, gate, limit, **kwargs: given.append((gate, limit)))
    x, w = (torch.zeros(r, 256, dtype=torch.bfloat16) for r in (m, 2048))
    assert linear.gated_linear(x, w, "silu", 7.0).shape == (m, 1024)
    assert given == [("silu", None)]


# (rows, weight rows, k, us by the forms for few rows, us by the flowing one), plain products into bfloat16
WHOLE = [(17, 64, 4096, 11.1, 14.9), (32, 64, 4096, 14.1, 16.0), (33, 64, 4096, 21.8, 16.7), (64, 64, 4096, 27.7, 19.5),
         (17, 768, 2048, 7.2, 8.5), (33, 768, 2048, 13.9, 9.5), (17, 1024, 2048, 13.1, 8.5), (17, 12800, 4096, 30.9, 27.5),
         (64, 12800, 4096, 48.3, 31.4), (17, 16384, 5120, 39.5, 30.7), (32, 16384, 4096, 30.4, 34.7), (33, 16384, 4096, 40.3, 35.0),
         (64, 16384, 1024, 13.1, 9.7), (33, 16448, 2560, 26.1, 29.5), (64, 20480, 4096, 41.0, 55.0), (17, 20480, 5120, 48.9, 45.3),
         (32, 32768, 4096, 45.8, 62.3)]


@pytest.mark.parametrize("m, n, k, few, flow", WHOLE)
def test_a_product_in_one_share_flows_where_it_was_faster(m, n, k, few, flow):
    assert gemm_bf16.flows_whole(m, n, k) == (flow < few)


@pytest.mark.parametrize("m, n, taken", [(16, 1024, False), (17, 1016, False), (17, 1024, True), (32, 8, False), (33, 8, True), (64, 8, True), (65, 1024, False)])
def test_narrow_products_flow_from_33_rows(m, n, taken):
    x, w = (torch.zeros(r, 128, dtype=torch.bfloat16) for r in (m, n))
    assert gemm_bf16.flows(x, w, False) is taken and gemm_bf16.flows(x, w, True) is (m <= 96)


# (rows, weight rows, k, us of the flowing product with the activation in its epilogue, us in shares of K with the activation's kernel)
SHARES = [(24, 2048, 1024, 5.8, 6.4), (17, 1024, 1024, 5.6, 5.9), (64, 1024, 2048, 11.3, 8.8), (17, 8192, 1024, 6.4, 7.5), (64, 8192, 1024, 8.1, 11.0), (17, 4096, 2048, 9.0, 7.9),
          (64, 12800, 2048, 15.3, 19.3), (32, 4096, 4096, 17.7, 11.1), (33, 8192, 4096, 22.5, 17.9), (64, 12800, 4096, 31.5, 35.3),
          (17, 64, 8192, 29.4, 8.9), (48, 4096, 17408, 75.7, 30.6)]


@pytest.mark.parametrize("m, n, k, whole, shares", SHARES)
def test_k_is_shared_ahead_of_an_activation_where_that_was_faster(m, n, k, whole, shares):
    assert ops.flow_shares_pay(m, n, k) == (shares < whole)


@pytest.mark.parametrize("m, n, k, forms", [(17, 1024, 256, ["flow"]), (32, 8, 256, ["flow"]), (64, 8, 256, ["flow"]), (17, 512, 4096, ["shares", "relu"]),
                                            (33, 16384, 256, ["flow"]), (33, 16392, 256, ["stream"]), (65, 512, 4096, ["shares", "relu"])])
def test_squared_relus_form(monkeypatch, m, n, k, forms):
    """In the flowing product's epilogue, behind shares of K, or in the streaming product's, on both sides of each line."""
    seen = []
    monkeypatch.setattr(ops, "gemm_flow", lambda x, w, out, **kwargs: seen.append("shares" if out.dim() == 3 else "flow"))
    monkeypatch.setattr(ops, "gemm_stream", lambda *args, **kwargs: seen.append("stream"))
    monkeypatch.setattr(ops, "squared_relu", lambda *args: seen.append("relu"))
    linear.activated_linear(torch.zeros(m, k, dtype=torch.bfloat16), torch.zeros(n, k, dtype=torch.bfloat16))
    assert seen == forms


# rows, channels, k of a product whose reader adds shares of K, and the microseconds of both by the number of shares
PARTS = [(3, 5120, 8192, {1: 32.7, 2: 22.6, 3: 20.3, 4: 24.3, 5: 21.6, 6: 22.0, 8: 25.1, 10: 24.7, 12: 23.8, 16: 26.3}),
         (4, 3072, 4096, {1: 19.6, 2: 13.4, 3: 11.6, 4: 10.3, 5: 10.4, 6: 12.1, 8: 11.3, 10: 11.9, 12: 12.1, 16: 12.6}),
         (3, 6144, 2048, {1: 13.3, 2: 10.8, 3: 12.8, 4: 11.7, 5: 11.8, 6: 12.8, 8: 12.9}),
         (3, 12288, 1024, {1: 11.7, 2: 12.6, 3: 13.8, 4: 13.4}),
         (8, 4096, 4096, {1: 18.8, 2: 13.2, 3: 11.7, 4: 11.3, 5: 12.7, 6: 12.4, 8: 12.2, 10: 13.9, 12: 14.1, 16: 14.8}),
         (16, 1024, 3072, {1: 16.4, 2: 11.2, 3: 9.6, 4: 8.3, 5: 8.1, 6: 8.0, 8: 7.2, 10: 7.8, 12: 7.2}),
         (24, 2560, 9728, {1: 44.6, 2: 27.0, 3: 21.6, 4: 18.1, 5: 17.0, 6: 16.3, 8: 20.1, 10: 19.1, 12: 18.4, 16: 20.3}),
         (64, 4096, 12288, {1: 68.2, 2: 40.8, 3: 32.5, 4: 28.9, 5: 39.2, 6: 36.3, 8: 34.0, 10: 38.9, 12: 37.9, 16: 41.0}),
         (96, 5120, 17408, {1: 119.7, 2: 69.1, 3: 54.1, 4: 72.1, 5: 63.7, 6: 59.6, 8: 65.2, 10: 73.0, 12: 67.8, 16: 70.0})]


@pytest.mark.parametrize("m, n, k, took", PARTS)
def test_shares_of_k_are_near_the_best_measured(m, n, k, took):
    assert took[ops.flow_parts(m, n, k)] <= 1.09 * min(took.values())


@pytest.mark.parametrize("m, n, k, taken", [(3, 1024, 512, False), (4, 1024, 512, False), (5, 1024, 512, True), (2, 4096, 4096, False), (3, 4096, 4096, True)])
def test_small_matrices_of_three_and_four_rows_stay_with_the_direct_product(m, n, k, taken):
    x, w = (torch.zeros(r, k, dtype=torch.bfloat16) for r in (m, n))
    assert gemm_bf16.flows(x, w, True) is taken


@pytest.mark.parametrize("m, n, k, forms", [
    (16, 1024, 4096, []), (17, 1024, 4096, ["shares", "gate"]), (17, 1024, 128, ["flow"]), (64, 6144, 1024, ["flow"]), (17, 1028, 4096, ["flow"]),
    (65, 1028, 4096, []), (65, 1032, 4096, ["shares", "gate"]), (96, 1024, 4096, ["shares", "gate"]), (97, 1024, 4096, []),
    (32, 16400, 128, ["flow"]), (33, 16384, 128, ["flow"]), (33, 16400, 128, []), (64, 16400, 128, []), (65, 16400, 128, ["flow"])])
def test_gated_products_of_few_rows(monkeypatch, m, n, k, forms):
    """One share of K, several with the gate's kernel, or other forms, on both sides of each line."""
    seen = []
    monkeypatch.setattr(ops, "gemm_flow", lambda x, w, out, **kwargs: seen.append("shares" if out.dim() == 3 else "flow"))
    monkeypatch.setattr(ops, "silu_mul", lambda *args, **kwargs: seen.append("gate"))
    x, w = torch.zeros(m, k, dtype=torch.bfloat16), torch.zeros(n, k, dtype=torch.bfloat16)
    taken = linear._gated_flow(x, w, torch.empty(m, n // 2, dtype=torch.bfloat16), "clamped", 7.0)
    assert taken == bool(forms) and seen == forms


# rows, weight rows, k of a gated product, us by the library and the gate's kernel, us by the many-rows kernel
GATED = [(256, 256, 512, 19.4, 8.0), (129, 1024, 1024, 13.8, 12.6), (256, 512, 1024, 13.2, 14.8), (512, 4096, 2048, 21.3, 22.1),
         (700, 4096, 2048, 26.6, 22.0), (200, 16384, 2048, 32.4, 25.8), (256, 1024, 4096, 15.6, 38.3), (700, 4096, 4096, 36.5, 39.2),
         (1024, 4096, 4096, 46.4, 42.0), (200, 28672, 4096, 94.7, 71.9), (384, 8192, 5120, 53.1, 62.4), (2048, 28672, 5120, 514.8, 464.4),
         (512, 512, 8192, 22.6, 67.7), (512, 8192, 8192, 82.5, 80.2), (6000, 24576, 4096, 926.9, 912.1), (8192, 24576, 4096, 1219.3, 1259.9),
         (16384, 2048, 4096, 196.1, 210.4), (8192, 28672, 8192, 2593.1, 3565.3), (8192, 19456, 2560, 779.3, 695.2)]


@pytest.mark.parametrize("m, n, k, library, many", GATED)
def test_gated_products_of_many_rows_go_where_they_were_faster(m, n, k, library, many):
    assert ops.many_gate_pays(m, n // 2, k) == (many < library)


@pytest.mark.parametrize("n, k", [(4096, 12288), (5120, 17408), (1024, 9216), (1024, 8192), (1020, 9216), (8192, 28672)])
@pytest.mark.parametrize("most", [1, 128, 129, 1000, 1100, 1200, 2048, 8192])
def test_no_number_of_rows_holds_more_than_those_that_are_measured(n, k, most):
    """Whatever a row takes beside the product's operand and result."""
    def held(m):
        x, w = (torch.empty(rows, k, dtype=torch.bfloat16, device="meta") for rows in (m, n))
        parts = ops.many_split_plan(m, n, k)[2] if gemm_bf16.splits_many(x, w) else 1
        return 2 * m * k + (4 * parts if parts > 1 else 2) * m * n

    found = gemm_bf16.rows_of_most_shares(n, k, most)
    assert most in found and all(1 <= m <= most for m in found) and len(found) <= 8
    product = {m: held(m) for m in range(max(1, most - 2000), most + 1)}
    for row in (0, 20e3, 50e3, 100e3, 150e3, 200e3, 1e6):
        assert max(held(m) + row * m for m in found) >= max(took + row * m for m, took in product.items())


# rows, weight rows, k of a long product whose reader adds partial sums, us by the library, us in shares of K on the many-rows kernel
LONG = [(129, 64, 9216, 12.4, 11.6), (1024, 6144, 9216, 127.1, 125.8), (1700, 6144, 17408, 535.7, 326.6), (1024, 8192, 9216, 149.8, 145.1),
        (1100, 8192, 12288, 216.6, 230.2), (1100, 8192, 16384, 482.9, 290.1), (1536, 8192, 17408, 346.2, 386.6), (512, 12288, 12288, 168.9, 162.3),
        (768, 12288, 9216, 175.1, 186.3), (1024, 12288, 17408, 358.5, 386.4), (1700, 12288, 17408, 987.3, 656.9), (256, 16384, 9216, 122.8, 112.1),
        (300, 16384, 9216, 124.1, 137.3), (640, 16384, 10240, 197.0, 269.4), (1100, 16384, 12288, 625.8, 468.5), (160, 24576, 25600, 385.9, 610.8),
        (384, 24576, 9216, 264.2, 367.5)]


@pytest.mark.parametrize("m, n, k, library, shares", LONG)
def test_long_products_are_shared_where_that_was_faster(m, n, k, library, shares):
    assert gemm_bf16.many_shares_pay(m, n, k) == (shares < library)
    x, w = (torch.empty(rows, k, dtype=torch.bfloat16, device="meta") for rows in (m, n))
    assert gemm_bf16.splits_many(x, w) == (shares < library)


# rows, weight rows, k of a product whose reader adds partial sums, us by the forms before, us by the flowing one
PARTIAL = [(3, 8, 4096, 6.2, 5.8), (80, 8, 4096, 15.9, 7.1), (17, 1016, 16384, 13.5, 11.5), (32, 12800, 4096, 34.0, 31.5), (16, 14336, 8192, 53.2, 42.7),
           (8, 16384, 4096, 31.7, 40.0), (64, 13824, 4096, 35.0, 37.2), (65, 13824, 4096, 39.2, 38.0), (24, 20480, 2048, 121.1, 62.1),
           (16, 24576, 3072, 100.1, 78.0), (32, 17408, 8192, 142.6, 157.5), (33, 17408, 2048, 56.3, 75.1), (48, 20480, 8192, 109.5, 188.4),
           (64, 24576, 4096, 91.3, 129.7), (80, 20480, 2048, 83.6, 72.1), (80, 24576, 4096, 113.1, 134.8), (65, 28672, 8192, 209.1, 161.5)]


@pytest.mark.parametrize("m, n, k, before, flow", PARTIAL)
def test_products_into_partial_sums_flow_where_that_was_faster(m, n, k, before, flow):
    x, w = (torch.empty(rows, k, dtype=torch.bfloat16, device="meta") for rows in (m, n))
    assert gemm_bf16.flows(x, w, True) == (flow < before)


@pytest.mark.parametrize("m, n, k, forms", [(17, 20480, 2048, ["shares", "relu"]), (17, 20480, 8192, ["flow"])])
def test_squared_relu_of_wide_matrices_is_shared_only_where_shares_flow(monkeypatch, m, n, k, forms):
    seen = []
    monkeypatch.setattr(ops, "flow_shares_pay", lambda *shape: True)
    monkeypatch.setattr(ops, "gemm_flow", lambda x, w, out, **kwargs: seen.append("shares" if out.dim() == 3 else "flow"))
    monkeypatch.setattr(ops, "squared_relu", lambda *args: seen.append("relu"))
    monkeypatch.setattr(gemm_bf16, "flows_whole", lambda *shape: True)
    linear.activated_linear(*(torch.empty(rows, k, dtype=torch.bfloat16, device="meta") for rows in (m, n)))
    assert seen == forms
