"""Which scans of the delta rule run in chunks: those of the sizes at which chunks were measured ahead of the walk."""

import pytest

from tokamak_amd.kernels import ops


@pytest.mark.parametrize("dim, vdim, tokens, chunks", [
    (128, 128, 320, True), (80, 112, 320, True), (96, 128, 2048, True), (112, 112, 400, True),
    (128, 128, 319, False), (128, 128, 160, False),
    # (walk over chunks, many requests: 0.98, 0.85, 0.69, 0.36, 0.92, 0.46)
    (96, 96, 320, False), (128, 64, 2048, False), (64, 64, 640, False), (128, 16, 2048, False), (64, 128, 320, False), (16, 16, 640, False),
    (144, 128, 2048, False), (128, 144, 2048, False), (100, 128, 2048, False), (128, 120, 2048, False)])
def test_the_line(dim, vdim, tokens, chunks):
    assert ops._delta_in_chunks(dim, vdim, tokens) is chunks
