"""The lines between forms of attention kernels lie where both were measured; operands off the borders of a kernel's loads are refused."""

import pytest

from tokamak_amd.kernels import ops
from tokamak_amd.kernels.build import load_library


# us with a block a head and with heads that share one, over 600 keys
@pytest.mark.parametrize("float32, tokens, heads, kv_heads, shares", [
    (1, 8, 64, 8, False),       # 23 and 56: 64 blocks would leave most CUs idle
    (1, 16, 64, 8, False), (1, 24, 64, 8, True), (1, 96, 64, 8, True),      # 48 and 58, 103 and 57
    (1, 24, 16, 8, False), (1, 32, 16, 8, True),                            # 32 and 39, 45 and 41
    (1, 16, 32, 4, False), (1, 32, 16, 2, False), (1, 64, 8, 1, False),     # 23 and 56 each
    (0, 12, 64, 8, False), (0, 16, 64, 8, False), (0, 24, 64, 8, True),     # 35 and 56, 41 and 57, 66 and 58
    (0, 32, 16, 8, False), (0, 52, 16, 8, True), (0, 16, 32, 8, False), (0, 32, 32, 8, True),
    (0, 96, 16, 16, False), (1, 96, 32, 32, False), (0, 1, 64, 4, False)])
def test_heads_share_a_block_where_that_fills_the_gpu(float32, tokens, heads, kv_heads, shares):
    assert bool(load_library("attention_generic").tk_attention_heads_share(float32, tokens, heads, kv_heads)) is shares


# us with one head a block and with two
@pytest.mark.parametrize("tiles, heads, kv_heads, dim, a_block", [
    (2, 16, 8, 128, 1), (16, 16, 8, 128, 1), (17, 16, 8, 128, 2), (64, 32, 8, 128, 2),      # 17 tokens 16 and 24, 1,024 150 and 114
    (64, 12, 4, 128, 1), (64, 16, 16, 128, 1),                                              # (groups without pairs)
    (2, 16, 8, 64, 1), (64, 16, 8, 64, 1), (128, 32, 8, 64, 1)])                            # 12 and 17, 78 and 73
def test_two_heads_share_a_float32_tile_where_blocks_are_many(tiles, heads, kv_heads, dim, a_block):
    assert load_library("attention_generic").tk_attention_tile_heads(tiles, heads, kv_heads, dim) == a_block


# us apart and together, 16 heads over 8 kv heads, 1,024 tokens: 88 and 71 at 128 / 128, 67 and 75 at 64 / 64
@pytest.mark.parametrize("group, dim, value_dim, shares", [
    (1, 128, 128, False), (2, 128, 128, True), (3, 128, 64, True), (2, 96, 96, True), (2, 64, 64, False), (3, 64, 48, False),
    (2, 192, 128, False), (4, 64, 64, True), (4, 512, 448, True)])
def test_heads_share_a_bfloat16_tile(group, dim, value_dim, shares):
    assert bool(load_library("attention_tiles").tk_attention_tiles_share(group, dim, value_dim)) is shares


def test_parts_off_their_borders_are_refused():
    heads = load_library("attention_tiles").tk_attention_heads
    heads.argtypes = ops._SIGS["attention_tiles"]["tk_attention_heads"]
    for off in (4, 12, 2):      # (of the parts' maxima and sums, read in pairs; the call ends before a launch)
        at = [4096] * 4 + [16] + [4096] * 3 + [1, 4096, 4096, 4096 + off, 2, 8, 1, 64, 64, 16, 0.125, 0, 0, None, 0.0, None]
        assert heads(*at) == -2
