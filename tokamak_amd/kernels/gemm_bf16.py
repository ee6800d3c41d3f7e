"""bfloat16 matrix products with float32 accumulation."""

from __future__ import annotations

import functools

import torch

from tokamak_amd.kernels import ops

SKINNY_MAX_ROWS = 64
TARGET_WAVES = 4096     # waves wanted in flight for the direct-operand kernel
STREAM_MIN_ROWS_OUT = 1024    # weight rows from which the LDS-staged kernel (64 rows a block) is used
STREAM_TARGET_BLOCKS = 512


def skinny_fits(x: torch.Tensor, weight: torch.Tensor) -> bool:
    k = x.shape[1]
    return (k % 8 == 0 and x.stride(0) % 8 == 0 and weight.stride(0) % 8 == 0
            and x.data_ptr() % 16 == 0 and weight.data_ptr() % 16 == 0)


def skinny_plan(m: int, n: int, k: int) -> tuple[int, int]:
    """(tiles of 16 weight rows per block, waves of a block that split K) for the
    direct-operand kernel.  More row tiles per block let the activation fragments
    be reused; more waves put more loads in flight when the matrix has few rows.
    Chosen from measurements on the projection shapes of 0.6B to 32B models."""
    if m > 32:
        row_tiles = 4 if n >= 6144 else 2
    elif m <= 2 or n < 6144:
        row_tiles = 1
    else:
        row_tiles = 4 if n >= 65536 else 2
    blocks = -(-n // (16 * row_tiles))
    waves = 4
    while waves < 16 and blocks * waves < TARGET_WAVES:
        waves *= 2
    while waves > 1 and k // waves < 64:
        waves //= 2
    return row_tiles, waves


def _fill(total: int) -> float:
    """How well `total` blocks of four waves use the GPU: two a CU run at full rate, so up to 512
    count by their number; beyond, the CUs that get one block more than the others set the time, so
    a count just under the next multiple of 256 is good and one just over it is the worst (80 row
    blocks of a 14B-shaped down projection: 480 blocks 29 us, 560 blocks 35 us, 720 blocks 32 us);
    every further block a CU costs a little by itself (partial sums, shorter shares)."""
    room = max(STREAM_TARGET_BLOCKS, -(-total // 256) * 256)
    return total / room * 0.95 ** ((room - STREAM_TARGET_BLOCKS) // 256)


def stream_splits(n: int, k: int, m: int = 1) -> int:
    """Shares of K for the LDS-staged kernel so that enough blocks exist, and no more.

    Up to 32 rows (blocks of four waves): of the numbers of shares that K's chunks of 256 allow, the
    one whose blocks fill the CUs most evenly (``_fill``): 512 blocks or a little less, else a
    little less than 768.  17 to 32 rows of a large matrix: never fewer than two chunks a share,
    since every split also writes (and the next kernel reads) float32 partial sums of all rows.
    Small matrices (the projections of a 0.6B-shaped model) at any number of rows likewise, down
    to one chunk a share: such a product is read in one memory round trip then, and its time is
    round trips, not bytes.  More rows: a block holds more LDS and one block of six or eight waves
    runs on a CU, so a few blocks beyond the 256 CUs cost a whole further round (measured at
    32B-shaped sizes with 64 rows: 280 blocks of eight waves take 80 us where 240 take 57): at most
    256 blocks, never fewer than two chunks a share.  Against the best of every split measured on
    the projection shapes of 1.7B to 32B models at 4 to 32 rows this is within 1 % on average and
    10 % at worst (a small matrix with 32 rows)."""
    chunks = -(-k // 256)
    blocks = -(-n // (16 * ops.stream_waves(m, k, False, n)))
    small = 2 * n * k < ops.STREAM_SMALL_MATRIX_BYTES
    if m <= 32 or (small and m <= SKINNY_MAX_ROWS):
        if blocks >= STREAM_TARGET_BLOCKS:
            return 1
        least_share = 1 if m <= 16 or small else min(2, chunks)
        best, best_fill = 1, _fill(blocks)
        for share in range(chunks, least_share - 1, -1):        # chunks a share, fewest splits first
            splits = -(-chunks // share)
            if splits > 64:
                break
            fill = _fill(blocks * splits)
            if fill > best_fill:
                best, best_fill = splits, fill
        return best
    splits = max(1, STREAM_TARGET_BLOCKS // 2 // blocks)
    return max(1, min(splits, chunks // 2))


STREAM_PARTIALS_ROWS = 96           # rows up to which the split streaming product beats the library at every size
STREAM_PARTIALS_BIG = 64 << 20      # ... and the bytes of a matrix from which it does up to 128 rows


FLOW_SPLIT_ROWS = (3, 96)           # rows between which a product whose reader adds partial sums flows (csrc/gemm_flow.hip), if it is not very
                                    # wide (``flows_shared``): beside the forms below, 123 sizes of 1,024 to 12,288 channels, weights from memory, reader included: 1.09 times as fast at 3 to
                                    # 8 rows, 1.11 at 16, 1.15 at 24 to 64, 1.24 at 96, at worst 0.94 (12,288 x 4,096 at 48); 128 rows: level, 0.81 at worst.  With fewer rows it is
                                    # 1.06 times as fast alone, but beside an experts' branch its few large blocks wait for room (a
                                    # decode step of one request 623 -> 663 us, of two 731 -> 735)
FLOW_BEHIND_DIRECT_ROWS = 4         # rows up to which the direct product, where it pays (ops.direct_pays: K of up to 1,024), is ahead of it in
                                    # turn: 60 products 0.84 to 1.02 (1,024 x 512 at 4 rows, reader included, 5.2 us against 5.9); with 5 rows 1.01 to 1.09
FLOW_ROWS = (17, 64)                # ... and one into bfloat16, which nobody can add, in one share of K, where ``flows_whole`` says; with fewer rows
                                    # the direct form, with more the library is ahead of it.  (A logits head into float32, one share
                                    # of K: decode steps of 36 to 64 rows 7 to 53 us slower than with the streaming kernel.)
FLOW_WHOLE_MOST = 16384             # weight rows of a product in one share from 33 rows on: 256 blocks, of which a CU holds one


def flows_whole(m: int, n: int, stride: int) -> bool:
    """Whether a product of 17 to 64 rows in one share of K flows, by its weight rows and the numbers between them.  A block owns 64
    of them and walks all of K.  Beside the forms below (110 sizes of 64 to 65,536 rows of 1,024 to 17,408, weights from memory):

    - 33 to 64 rows: 1.15 to 2.07 times as fast up to 16,384 weight rows (64 x 4,096 at 64 rows 28 -> 20 us); beyond, where a second
      round of blocks begins, 0.71 to 1.05 (at 28,672, whose rounds are even, 1.13 to 1.52).
    - 17 to 32 rows: below 1,024 weight rows 0.67 to 1.00 but for one size (64 x 4,096 at 17 rows 11 -> 15 us): a few blocks, where
      gemm_skinny shares K among sixteen waves of four times as many.  From there on 1.00 to 1.63, beyond 16,384 0.94 to 1.15;
      but 0.73 to 0.93 from 16,384 weight rows on if they lie a multiple of 8 KB apart (16,384 x 4,096 reaches 3.8 TB/s, x 5,120 5.5)."""
    if m > 32:
        return n <= FLOW_WHOLE_MOST
    return n >= STREAM_MIN_ROWS_OUT and (n <= 14336 or stride % 4096 != 0)


def flows_shared(m: int, n: int, k: int, stride: int) -> bool:
    """Whether a product of 3 to 96 rows whose reader adds partial sums flows, by its weight rows and the numbers between them.
    Beside the forms below (2,900 products of 8 to 65,536 weight rows of 512 to 17,408, weights from memory, reader included):

    - up to 16,384 weight rows, a round of 256 blocks: 1.15 times as fast on average, 28 of 1,744 more than 5 % behind (8 x 4,096 at 80
      rows 15.9 -> 7.1 us); but 0.87, 0.79 to 1.07, beyond 12,800 if they lie 8 KB apart and up to 64 rows read them (16,384 x 4,096 at
      8 rows 31.7 us, here 40.0).
    - More, up to 32 rows: up to 80 M numbers 1.18, 0.87 to 2.1 (20,480 x 2,048 at 24 rows 121 -> 62); beyond, where shares fill several
      rounds badly, 0.98, 0.66 to 1.37, 86 of 324 (17,408 x 8,192 at 32 rows 143, here 158).
    - More, 33 to 64 rows: 0.86, 0.58 to 1.09 (20,480 x 8,192 at 48 rows 110, here 188), only 28,672, whose rounds are even, 0.99 to 1.38.
    - More, 65 to 96 rows: 1.08 at K of up to 2,048, 1.12 from 28,672 weight rows on, 3 of 147; else 0.91, 0.66 to 1.30, 78 of 126."""
    if n <= 16384:
        return m > SKINNY_MAX_ROWS or n <= 12800 or stride != 4096
    if m <= 32:
        return n * k <= 80 << 20
    return m > SKINNY_MAX_ROWS and (k <= 2048 or n >= 28672)


def flows(x: torch.Tensor, weight: torch.Tensor, allow_partials: bool) -> bool:
    """Whether a product goes to the flowing kernel: into partial sums, or into bfloat16."""
    m = x.shape[0]
    low, high = FLOW_SPLIT_ROWS if allow_partials else FLOW_ROWS
    if not low <= m <= high:
        return False
    (n, k), stride = weight.shape, weight.stride(0)
    if allow_partials:
        taken = flows_shared(m, n, k, stride) and not (m <= FLOW_BEHIND_DIRECT_ROWS and ops.direct_pays("parts", m, n, k))
    else:
        taken = flows_whole(m, n, stride)
    return taken and ops.gemm_flow_fits(x, weight)


def flow(x: torch.Tensor, weight: torch.Tensor, allow_partials: bool) -> torch.Tensor:
    """Partial sums [P, M, N], or the product in bfloat16, by the flowing kernel."""
    m, n, k = x.shape[0], *weight.shape
    out = (torch.empty((ops.flow_parts(m, n, k), m, n), dtype=torch.float32, device=x.device) if allow_partials
           else torch.empty((m, n), dtype=torch.bfloat16, device=x.device))
    ops.gemm_flow(x, weight, out)
    return out


# Rows up to which, from 129 on, a product whose reader adds partial sums is cut into shares of K (csrc/gemm_many.hip), by the K it
# has at least: tiles of a long K that are whole leave most CUs idle.  Beside the library's first choice, reader included: 2,560 x
# 9,728 1.07 to 1.30 times as fast, 4,096 x 12,288 1.04 to 1.98, 5,120 x 17,408 1.55 to 3.98; K of 9,728 and 12,288 at 1,300 to 2,048
# rows 0.99 to 1.18, K of 17,408 at 2,048 1.05; K of 8,192 0.92 to 1.55, of 6,144 0.83 to 1.31, of 5,120 and less mostly below 1.  One
# prompt of 512 / 1,000 tokens through twelve layers 4,096 wide 3.75 / 5.79 -> 3.42 / 5.44 ms, 1,000 through 2,560 wide 4.20 -> 3.91.
MANY_SPLIT_ROWS = ((16384, 1700), (9216, 1100))


def many_shares_pay(m: int, n: int, k: int) -> bool:
    """Whether a product of more than 128 rows whose reader adds partial sums may be cut into shares of K.  A wide one's whole tiles of
    256 x 256 fill most of the GPU by themselves, and the shares' sums are more to write and read; what the last round of such tiles
    leaves idle decides.  Beside the library's first choice, reader included, weights from memory, 1,442 products of 64 to 24,576
    weight rows of 9,216 to 28,672:

    - up to 6,144 weight rows: 1.72 times as fast on average, 0.94 to 4.6;
    - up to 16,384 with few of a round's 256 blocks left over (8,192 weight rows: 128, or 160 with K of 16,384 and more; beyond: 112):
      1.29, 0.89 to 2.7, three of 200 more than 5 % behind; with more left 1.04, 0.73 to 1.66, 33 of 75 (16,384 x 10,240 at 640 rows
      197 us, here 269 in three shares);
    - beyond: 0.96, 0.63 to 1.28, 44 of 87 (24,576 x 25,600 at 160 rows 386 us, here 611)."""
    if m <= 128 or k < MANY_SPLIT_ROWS[-1][0] or m > next(rows for least, rows in MANY_SPLIT_ROWS if k >= least):
        return False
    left = -(-m // 256) * -(-n // 256) % 256
    return n <= 6144 or (n <= 16384 and left <= (112 if n > 8192 else 160 if k >= 16384 else 128))


def splits_many(x: torch.Tensor, weight: torch.Tensor) -> bool:
    """Whether a product of many rows is cut into shares of K for its reader to add."""
    m, (n, k) = x.shape[0], weight.shape
    return many_shares_pay(m, n, k) and ops.gemm_many_fits(x, weight, n) and ops.many_split_plan(m, n, k)[2] > 1


def split_many(x: torch.Tensor, weight: torch.Tensor) -> torch.Tensor:
    """Partial sums [P, M, N] of a product of many rows."""
    m, n, k = x.shape[0], *weight.shape
    rows, columns, parts = ops.many_split_plan(m, n, k)
    out = torch.empty((parts, m, n), dtype=torch.float32, device=x.device)
    ops.gemm_many(x, weight, out, rows=rows, columns=columns)
    return out


@functools.lru_cache(maxsize=256)
def rows_of_most_shares(n: int, k: int, most: int) -> tuple[int, ...]:
    """The numbers of rows, up to ``most``, among which is the one at which a step holds most memory that a matrix [N, K] takes part in
    whose reader adds shares of K: those whose operand and result take more than those of any larger number (1,024 rows of 12,288 and
    four shares of 4,096 sums 92 MB, 1,100 and three 81, 2,048 and their product 67).  What else a step holds grows with its rows."""
    limit = min(most, MANY_SPLIT_ROWS[0][1]) if k % 64 == 0 and n % 8 == 0 else 0
    found, held_most = [], 0
    for m in (most, *range(min(limit, most - 1), 128, -1)):
        parts = ops.many_split_plan.__wrapped__(m, n, k)[2] if m <= limit and many_shares_pay(m, n, k) else 1
        held = 2 * m * k + (4 * parts if parts > 1 else 2) * m * n
        if held > held_most:
            found.append(m)
            held_most = held
    return tuple(found)


def stream_pays_beyond_64_rows(m: int, n: int, k: int) -> bool:
    """Whether a product of 65 to 128 rows whose reader adds partial sums goes to the streaming
    kernel (five to eight tiles of 16 rows, eight waves a block) rather than to the library.
    Against the library's fastest candidate, q/k/v, o and down of 1.7B- to 32B-shaped layers are
    10 to 40 % faster at 65 to 96 rows; at 128 rows the large matrices still are (down of a
    32B-shaped layer 82 against 119 us) and the small ones are level or behind, and the partial
    sums cost their reader a few microseconds more.  Whole decode steps: batch 80 at 1.7B / 8B /
    14B / 32B widths +1 / +4 / +13 / +7 %, batch 128 -4 / -3 / +4 / +5 % if every product
    took this path, hence the limit on small matrices."""
    if not SKINNY_MAX_ROWS < m <= ops.STREAM_MAX_ROWS or n < STREAM_MIN_ROWS_OUT:
        return False
    return m <= STREAM_PARTIALS_ROWS or 2 * n * k >= STREAM_PARTIALS_BIG


def gemm(x: torch.Tensor, weight: torch.Tensor, out_dtype: torch.dtype, allow_partials: bool = False) -> torch.Tensor:
    """x[M, K] @ weight[N, K]^T -> [M, N] in ``out_dtype``; or, if the caller can
    add them (``allow_partials``), float32 partial sums [P, M, N] of a split-K product.  (What
    ``flows`` or ``splits_many`` says is another kernel's does not come here.)

    Up to 64 rows (decode batches, wanted logits rows): hand-written
    weight-streaming MFMA kernels: the LDS-staged one, split over K into partial
    sums when the matrix has few rows and the caller adds them; the
    direct-operand one for very small matrices.  65 to 128 rows, if the caller adds partial
    sums: the same kernel with five to eight tiles of 16 rows where it was measured to pay
    (``stream_pays_beyond_64_rows``; up to 96 these are the products that do not flow: K not a
    multiple of 128, or a very wide matrix).  Else more than 64 rows
    with bfloat16 output: the library product (hipBLASLt, as the reference's
    nn.Linear ends in a library; csrc/blas_lt.hip); with float32 output: up to 128 rows the streaming kernel, more the many-rows one (where
    K is no multiple of 64 or N none of 8, the streaming one 128 rows at a time).
    """
    m = x.shape[0]
    n, k = weight.shape
    dev = x.device
    fits = skinny_fits(x, weight)
    if fits and allow_partials and (m <= SKINNY_MAX_ROWS or stream_pays_beyond_64_rows(m, n, k)):
        splits = stream_splits(n, k, m)
        if splits > 1:
            out = torch.empty((splits, m, n), dtype=torch.float32, device=dev)
            used = ops.gemm_stream(x, weight, out, splits=splits)
            return out[:used]
    if m > ops.STREAM_MAX_ROWS and out_dtype == torch.float32 and ops.gemm_many_fits(x, weight, n):
        # The many-rows kernel in one share of K, whatever the size: beside the streaming one, 64 or 128 rows at a time, 652 products of 129 to
        # 2,048 rows, 8 to 151,936 weight rows of 64 to 16,384, weights from memory, were all faster, also narrow ones of a long K in one
        # or two blocks, whose passes are as long a chain each: 1.15 to 35 times, 6 on average (129 rows: 4,096 x 64 12 -> 7 us, 64 x 4,096
        # 60 -> 26, 4,096 x 4,096 88 -> 38; 2,048 rows: 4,096 x 64, a decay's low rank, whose sums stay in float32, 133 -> 14)
        out = torch.empty((m, n), dtype=torch.float32, device=dev)
        rows, columns = ops.several_plan(1, m, n, k)
        ops.gemm_many(x, weight, out[None], rows=rows, columns=columns)
        return out
    if fits and (m <= SKINNY_MAX_ROWS or out_dtype == torch.float32):
        out = torch.empty((m, n), dtype=out_dtype, device=dev)
        # (a logits head over 65 to 128 rows at once: 320-365 us at 8B width, 490-530 in two passes)
        step = ops.STREAM_MAX_ROWS if n >= STREAM_MIN_ROWS_OUT else SKINNY_MAX_ROWS
        for at in range(0, m, step):
            xs, os_ = x[at:at + step], out[at:at + step]
            if n >= STREAM_MIN_ROWS_OUT:
                ops.gemm_stream(xs, weight, os_)
            else:
                row_tiles, waves = skinny_plan(xs.shape[0], n, k)
                ops.gemm_skinny(xs, weight, os_, row_tiles=row_tiles, waves=waves)
        return out
    out = torch.empty((m, n), dtype=out_dtype, device=dev)
    if out_dtype == torch.bfloat16:
        # hipBLASLt with kept plans and measured algorithms; shapes it has nothing for
        # (rows that are not 16-byte aligned, say) go through torch's binding of it
        if not (skinny_fits(x, weight) and ops.gemm_library(x, weight, out)):
            ops.not_replayable()
            torch.matmul(x, weight.t(), out=out)
    else:
        ops.gemm_tiled(x, weight, out)
    return out
