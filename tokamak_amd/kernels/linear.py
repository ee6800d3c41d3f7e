"""y = x @ W^T for the projections of a step.

float32: hand-written kernels with true 32-bit multiply-add and one summation order
(tiled, or weight-streaming for up to 64 rows; row-wise deterministic, equal bits).  bfloat16: hand-written MFMA kernels for up to 64 rows; up
to 96 (large matrices 128) whose reader adds partial sums; gated products of 65 to 96 rows of small matrices, and of more than 128
that fill the GPU; long products of up to 1,100 or 1,700 rows whose reader adds partial sums.  Else the library product (as the
reference's nn.Linear does).

Decode steps of few rows (bfloat16, up to 16) can do without the kernels between the
products: a part's last product adds its result into the float32 residual stream itself
(``linear(..., add_into=StreamSink)`` -> ``Added``), leaving bf16(stream * gamma) for the
norm that reads the stream next and the rows' sums of squares; that norm then hands both on
as a ``DeferredNorm``, and the product after it applies the rows' scale to its own result
(an RMSNorm is a row scale times a column scale, and a product is linear in the row scale).
"""

from __future__ import annotations

from dataclasses import dataclass

import torch

from tokamak_amd.kernels import ops


# Where the direct product is not the faster form (ops.direct_pays) a product adds into the stream itself (one block
# walking the whole of K for 16 columns) only if K is short: up to one chunk of 256 for each of a block's sixteen
# waves.  With a longer K the split product and the norm kernel after it are as fast (measured: the o projection of
# an 8B-shaped layer gains 2 us, its down projection nothing).  The direct product adds at any K (down of an 8B-shaped
# layer at 8 rows: 20.3 us, split product and norm 21.3; at one row 16.7 against 20.6).
ADD_INTO_MAX_K = 16 * 256
GATED_SPLIT_UP_TO_BLOCKS = 160      # blocks of the gated streaming product up to which K is split instead, the gate behind it
GATED_WHOLEK_MAX_BYTES = 32 << 20   # gate and up together, up to which the whole-K form takes the gated product


@dataclass
class StreamSink:
    """Offered to a part whose last product may add its result into the residual stream
    itself: the float32 stream [M, H], and the weight [H] of the RMSNorm that reads the
    stream next (None if what follows is not one)."""

    resid: torch.Tensor
    gamma: torch.Tensor | None


@dataclass
class Added:
    """What ``linear(..., add_into=sink)`` returns in place of its result when the product
    has added it into the stream: ``sumsq`` [slabs, M], the sums of squares of every row of
    the new stream over slabs of columns, and, if the sink named a norm weight ``gamma``,
    ``scaled`` = bf16(stream * gamma)."""

    sumsq: torch.Tensor
    scaled: torch.Tensor | None
    gamma: torch.Tensor | None


@dataclass
class DeferredNorm:
    """An RMSNorm of the stream that is not finished: ``scaled`` = bf16(resid * weight) and
    the rows' sums of squares are at hand, the rows' scale rsqrt(mean(resid^2) + eps) is still
    to be applied.  ``linear`` and ``gated_linear`` take it in place of a tensor and apply the
    scale to their result; ``materialize()`` runs the norm kernel on the stream instead.  It
    must be used before the stream is written again."""

    resid: torch.Tensor
    weight: torch.Tensor
    eps: float
    dtype: torch.dtype
    scaled: torch.Tensor
    sumsq: torch.Tensor

    @property
    def shape(self):
        return self.resid.shape

    @property
    def device(self):
        return self.resid.device

    def materialize(self) -> torch.Tensor:
        out = torch.empty(self.resid.shape, dtype=self.dtype, device=self.resid.device)
        ops.add_rmsnorm(self.resid, None, self.weight, self.eps, out)
        return out


def _few_rows_fit(m: int, x: torch.Tensor, weight: torch.Tensor, rows: int) -> bool:
    """Whether the fused forms for few rows take these operands."""
    from tokamak_amd.kernels import gemm_bf16

    return (0 < m <= rows and x.dtype == torch.bfloat16 and weight.dtype == torch.bfloat16
            and x.dim() == 2 and x.stride(1) == 1 and weight.stride(1) == 1 and gemm_bf16.skinny_fits(x, weight))


def linear(x: torch.Tensor | DeferredNorm, weight: torch.Tensor, out_dtype: torch.dtype | None = None,
           allow_partials: bool = False, add_into: StreamSink | None = None) -> torch.Tensor | Added:
    """``x`` [M, K], ``weight`` [N, K] -> [M, N] in ``out_dtype`` (default: x's).

    With ``allow_partials`` the result may instead be float32 partial sums
    [P, M, N] that the consumer adds (the norm kernel and the q/k norm kernel do).
    With ``add_into`` the product may add its result into the sink's stream itself and
    return ``Added`` (bfloat16 steps of up to 16 rows do).
    """
    from tokamak_amd.kernels import gemm_bf16

    out_dtype = out_dtype or x.dtype
    m, n = x.shape[0], weight.shape[0]
    if isinstance(x, DeferredNorm):
        if _few_rows_fit(m, x.scaled, weight, ops.DIRECT_MAX_ROWS) and ops.direct_pays(
                "norm" if allow_partials else "plain", m, n, weight.shape[1]):
            return _direct(x.scaled, weight, out_dtype, allow_partials, x.sumsq, x.eps)
        if (_few_rows_fit(m, x.scaled, weight, ops.ROW_SCALE_MAX_ROWS) and n >= gemm_bf16.STREAM_MIN_ROWS_OUT
                and x.sumsq.shape[0] <= ops.ROW_SCALE_MAX_SLABS):
            splits = gemm_bf16.stream_splits(n, weight.shape[1], m) if allow_partials else 1
            if splits > 1:
                out = torch.empty((splits, m, n), dtype=torch.float32, device=x.device)
                return out[:ops.gemm_stream(x.scaled, weight, out, splits=splits, sumsq=x.sumsq, eps=x.eps)]
            out = torch.empty((m, n), dtype=out_dtype, device=x.device)
            ops.gemm_stream(x.scaled, weight, out, sumsq=x.sumsq, eps=x.eps)
            return out
        x = x.materialize()
    if m == 0:
        return torch.empty((0, n), dtype=out_dtype, device=x.device)
    if x.dtype == torch.float32:
        out = torch.empty((m, n), dtype=out_dtype, device=x.device)
        ops.gemm_tiled(x, weight, out)
        return out
    if add_into is not None and _few_rows_fit(m, x, weight, ops.WHOLEK_MAX_ROWS) and _sink_fits(add_into, m, n):
        if weight.shape[1] <= ADD_INTO_MAX_K:
            return Added(*ops.gemm_wholek_add(x, weight, add_into.resid, add_into.gamma), add_into.gamma)
        if ops.direct_pays("add", m, n, weight.shape[1]):
            return Added(*ops.gemm_direct_add(x, weight, add_into.resid, add_into.gamma), add_into.gamma)
    if (allow_partials or out_dtype == torch.bfloat16) and gemm_bf16.flows(x, weight, allow_partials):
        return gemm_bf16.flow(x, weight, allow_partials)
    if allow_partials and gemm_bf16.splits_many(x, weight):
        return gemm_bf16.split_many(x, weight)
    if _few_rows_fit(m, x, weight, ops.DIRECT_MAX_ROWS) and ops.direct_pays("parts" if allow_partials else "plain", m, n, weight.shape[1]):
        return _direct(x, weight, out_dtype, allow_partials)
    return gemm_bf16.gemm(x, weight, out_dtype, allow_partials)


def several_linears(x: torch.Tensor, weights: torch.Tensor) -> list[torch.Tensor]:
    """``linear(x_i, weights[i], allow_partials=True)`` for every i: ``weights`` [C, N, K], ``x`` [C, M, K], or [M, K] for all of them.  More than
    128 rows into bfloat16: one launch where that pays (``ops.several_pay``).  Long products whose reader adds float32 sums of shares of K
    (``gemm_bf16.splits_many``) stay such products: one launch would round each to bfloat16."""
    from tokamak_amd.kernels import gemm_bf16

    count, n, k = weights.shape
    m = x.shape[-2]
    first = x if x.dim() == 2 else x[0]
    if (m > ops.STREAM_MAX_ROWS and x.dtype == torch.bfloat16 and ops.gemm_several_fits(x, weights)
            and ops.several_pay(count, m, n, k) and not gemm_bf16.splits_many(first, weights[0])):
        out = torch.empty((count, m, n), dtype=x.dtype, device=x.device)
        ops.gemm_several(x, weights, out)
        return list(out)
    return [linear(x if x.dim() == 2 else x[i], weights[i], allow_partials=True) for i in range(count)]


def _direct(x: torch.Tensor, weight: torch.Tensor, out_dtype: torch.dtype, allow_partials: bool,
            sumsq: torch.Tensor | None = None, eps: float = 0.0) -> torch.Tensor:
    """The direct product; where the reader adds partial sums, one float32 sum [1, M, N] (what the split product
    would leave in several)."""
    m, n = x.shape[0], weight.shape[0]
    out = torch.empty((m, n), dtype=torch.float32 if allow_partials else out_dtype, device=x.device)
    ops.gemm_direct(x, weight, out, sumsq=sumsq, eps=eps)
    return out[None] if allow_partials else out


def _sink_fits(sink: StreamSink, m: int, n: int) -> bool:
    r, g = sink.resid, sink.gamma
    return (r.dtype == torch.float32 and r.shape == (m, n) and r.stride(1) == 1 and r.stride(0) % 4 == 0
            and r.data_ptr() % 16 == 0 and n % 4 == 0
            and (g is None or (g.dtype == torch.float32 and g.numel() == n and g.is_contiguous() and g.data_ptr() % 16 == 0)))


ACTIVATED_SPLIT_FROM = 3    # shares of K that the product would be cut in from which it is, and the activation runs behind it


def activated_linear(x: torch.Tensor, weight: torch.Tensor, activation: str = "squared_relu") -> torch.Tensor:
    """act(x @ weight^T) -> [M, N]; ``activation`` "squared_relu": max(z, 0)^2.

    bfloat16: in the epilogue of the direct product (up to 16 rows), of the flowing one (17 to 64 rows, K a multiple of
    128) or of the streaming one (up to 64 rows), where K need not be shared to fill the GPU.  Otherwise the product (in
    partial sums where that pays), then the activation's kernel, which adds partial sums before it."""
    from tokamak_amd.kernels import gemm_bf16

    if activation != "squared_relu":
        raise ValueError(f"unknown activation {activation!r}")
    m, (n, k) = x.shape[0], weight.shape
    out = torch.empty((m, n), dtype=x.dtype, device=x.device)
    if m == 0:
        return out
    # Beside the streaming forms, 284 sizes: 1.01 to 1.70 times as fast (4,096 x 4,096 at 32 rows 13.9 -> 11.1 us, 512 x 17,408 19.7 ->
    # 14.2; always in one share of K 0.21 to 1.70, those two 17.7 and 73).  Narrow ones too: here their other form is two kernels as well.
    flowing = (gemm_bf16.FLOW_ROWS[0] <= m <= gemm_bf16.FLOW_ROWS[1] and ops.gemm_flow_fits(x, weight)
               and gemm_bf16.flows_whole(m, max(n, gemm_bf16.STREAM_MIN_ROWS_OUT), weight.stride(0)))
    if _few_rows_fit(m, x, weight, ops.DIRECT_MAX_ROWS) and ops.direct_pays("activated", m, n, k):
        ops.gemm_direct(x, weight, out, activation=activation)
    elif flowing and not (ops.flow_shares_pay(m, n, k) and gemm_bf16.flows(x, weight, True)):
        ops.gemm_flow(x, weight, out, activation=activation)
    elif (not flowing and x.dtype == torch.bfloat16 and m <= gemm_bf16.SKINNY_MAX_ROWS and n >= gemm_bf16.STREAM_MIN_ROWS_OUT
            and gemm_bf16.skinny_fits(x, weight) and gemm_bf16.stream_splits(n, k, m) < ACTIVATED_SPLIT_FROM):
        ops.gemm_stream(x, weight, out, activation=activation)
    else:
        ops.squared_relu(linear(x, weight, allow_partials=True), out)
    return out


GATED_MANY_FROM = 129       # rows from which the gated product has its own kernel with the gate behind it in registers; up to 128
                            # the library's product and the gate's kernel are level with it (80 to 128 rows: 0.76 to 1.5 times)


FLOW_GATED_MOST = 36 << 20      # numbers of gate and up below which their product of 17 to 96 rows flows (a decode step of 24 rows of 2,048
                                # 895 -> 837 us); one of more is long enough for the forms below: in one share 0.71 to 1.6 times as fast
                                # (9,728 to 34,816 weight rows of 2,048 to 8,192; a decode step of 64 rows of 2,560 1,008 -> 1,044)


def _gated_flow(x: torch.Tensor, gate_up: torch.Tensor, out: torch.Tensor, activation: str, limit: float | None) -> bool:
    """The gated product of 17 to 96 rows of a small matrix with its weights streamed through LDS (csrc/gemm_flow.hip): the gate
    behind one share of K, or, where the blocks of one leave CUs idle, in a kernel that adds the shares of several.  Beside the
    streaming form (up to 64 rows) and the library's product with the gate's kernel, 51 sizes of 128 to 34,816 weight rows of
    1,024 to 8,192: 0.96 to 5.3 times as fast, in one share alone 0.28 to 1.75 (1,024 x 4,096 at 96 rows 14.8 -> 11.5 us, in one share
    26.7; 4,096 x 5,120 at 17 15.0 -> 12.2, 21.4).  From 33 to 64 rows more than 256 blocks stay with the streaming form: a CU
    holds one, and a second round that is not full was 0.87 to 1.12 times as fast (18,432 x 1,024 at 64 rows 14.5 us against 16.8)."""
    from tokamak_amd.kernels import gemm_bf16

    m, (n, k) = x.shape[0], gate_up.shape
    if (not gemm_bf16.FLOW_ROWS[0] <= m <= gemm_bf16.FLOW_SPLIT_ROWS[1] or gate_up.numel() >= FLOW_GATED_MOST
            or (32 < m <= gemm_bf16.SKINNY_MAX_ROWS and n > gemm_bf16.FLOW_WHOLE_MOST) or not ops.gemm_flow_fits(x, gate_up)):
        return False
    shares = ops.flow_shares_pay(m, n, k)
    if shares and n % 8 == 0:
        ops.silu_mul(gemm_bf16.flow(x, gate_up, True), out, activation, limit=limit)
        return True
    if shares and m > gemm_bf16.SKINNY_MAX_ROWS:      # (the gate's kernel takes whole groups of four channels; the library is ahead of one share)
        return False
    ops.gemm_flow(x, gate_up, out, gate=activation, limit=limit)
    return True


def _gated_many(x: torch.Tensor, gate_up: torch.Tensor, out: torch.Tensor, activation: str, limit: float | None) -> bool:
    """The gated product of many rows in one kernel, whose block has a channel's gate and up sums side by side, where its tiles fill
    enough of the GPU (``ops.many_gate_pays``): 1.25 times as fast on average as the library's first choice and the gate's kernel
    (24,576 x 4,096 at 2,048 rows 317 -> 288 us).  With the tanh form of gelu 1.00 to 1.23
    times at 24,576 x 4,096 and 19,456 x 2,560 (2,048 rows 329 -> 307 and 230 -> 187 us), 1.16 to 1.59 at 6,144 x 1,024."""
    if (x.shape[0] < GATED_MANY_FROM or activation not in ops.MANY_MODES or not ops.gemm_many_fits(x, gate_up, out.shape[1])
            or not ops.many_gate_pays(x.shape[0], out.shape[1], x.shape[1])):
        return False
    rows, columns = ops.many_plan(x.shape[0], out.shape[1], x.shape[1])
    ops.gemm_many(x, gate_up, out, rows=rows, columns=columns, gate=activation, limit=limit)
    return True


def _gated_split(x: torch.Tensor, gate_up: torch.Tensor, out: torch.Tensor, activation: str, limit: float | None) -> bool:
    """The gated product of few rows as a product split over K and a gate that adds the partial sums.  The gated
    streaming kernel cannot split K under the gate: a matrix of few rows (a shared expert: 8,192 of 4,096, 128 blocks) leaves
    half of the CUs idle and takes 24 us, split 19."""
    from tokamak_amd.kernels import gemm_bf16

    m, (n, k) = x.shape[0], gate_up.shape
    blocks = -(-n // (16 * ops.stream_waves(m, k, True, n // 2)))
    splits = gemm_bf16.stream_splits(n, k, m)
    if blocks > GATED_SPLIT_UP_TO_BLOCKS or splits < 3 or n % 8:
        return False
    parts = torch.empty((splits, m, n), dtype=torch.float32, device=x.device)
    ops.silu_mul(parts[:ops.gemm_stream(x, gate_up, parts, splits=splits)], out, activation, limit=limit)
    return True


def gated_linear(x: torch.Tensor | DeferredNorm, gate_up: torch.Tensor, activation: str = "silu",
                 limit: float | None = None) -> torch.Tensor:
    """act(x @ gate^T) * (x @ up^T) for ``gate_up`` = [gate; up] ([2I, K]) -> [M, I].

    ``activation``: "silu", "gelu_tanh", or "clamped" with its ``limit``: both halves clamped, see ``ops.silu_mul``.

    bfloat16 by rows: up to 16 the whole-K form (very small matrices, silu alone), the direct or the streaming one; 17 to 96, K
    a multiple of 128 and below ``FLOW_GATED_MOST`` numbers, the flowing one (``_gated_flow``); else up to 64 the streaming one,
    or it split over K and the gate's kernel; from 129, K a multiple of 64, I of 8 and enough tiles (``ops.many_gate_pays``), the
    many-rows one.  Otherwise, and in float32, the product, then the gate's kernel.
    """
    m = x.shape[0]
    if activation != "silu":
        if isinstance(x, DeferredNorm):
            x = x.materialize()
        out = torch.empty((m, gate_up.shape[0] // 2), dtype=x.dtype, device=x.device)
        if m == 0:
            return out
        from tokamak_amd.kernels import gemm_bf16

        if _gated_flow(x, gate_up, out, activation, limit):
            return out
        if x.dtype == torch.bfloat16 and m <= 64 and gemm_bf16.skinny_fits(x, gate_up):
            if ops.direct_pays("gated", m, out.shape[1], x.shape[1]) or not _gated_split(x, gate_up, out, activation, limit):
                ops.gemm_stream_swiglu(x, gate_up, out, activation=activation, limit=limit)
        elif not _gated_many(x, gate_up, out, activation, limit):
            ops.silu_mul(linear(x, gate_up), out, activation, limit=limit)
        return out
    inter = gate_up.shape[0] // 2
    # A small pair of matrices goes to the whole-K form, whose blocks of 16 columns let their waves split K, which
    # the streaming kernel cannot do under the gate; from 50 MB on the streaming kernel is ahead.  (Both
    # hand over to the direct product where it is the faster form, ops.direct_pays.)
    small = 2 * gate_up.numel() <= GATED_WHOLEK_MAX_BYTES
    if isinstance(x, DeferredNorm):
        if _few_rows_fit(m, x.scaled, gate_up, ops.ROW_SCALE_MAX_ROWS) and (
                x.sumsq.shape[0] <= ops.ROW_SCALE_MAX_SLABS or ops.direct_pays("gated", m, inter, gate_up.shape[1])):
            out = torch.empty((m, inter), dtype=x.dtype, device=x.device)
            if small and m <= ops.WHOLEK_MAX_ROWS:
                ops.gemm_wholek(x.scaled, gate_up, out, gated=True, sumsq=x.sumsq, eps=x.eps)
            else:
                ops.gemm_stream_swiglu(x.scaled, gate_up, out, sumsq=x.sumsq, eps=x.eps)
            return out
        x = x.materialize()
    out = torch.empty((m, inter), dtype=x.dtype, device=x.device)
    if m == 0 or _gated_flow(x, gate_up, out, activation, None):      # (silu has no limit, one that is given is not looked at)
        return out
    if x.dtype == torch.bfloat16 and m <= 64:
        from tokamak_amd.kernels import gemm_bf16

        if gemm_bf16.skinny_fits(x, gate_up):
            if small and _few_rows_fit(m, x, gate_up, ops.WHOLEK_MAX_ROWS):
                ops.gemm_wholek(x, gate_up, out, gated=True)
            elif small or ops.direct_pays("gated", m, inter, x.shape[1]) or not _gated_split(x, gate_up, out, activation, limit):
                ops.gemm_stream_swiglu(x, gate_up, out)
            return out
    if not _gated_many(x, gate_up, out, activation, None):
        ops.silu_mul(linear(x, gate_up), out)
    return out
