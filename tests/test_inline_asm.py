"""Inline assembly names the registers that it writes beside its outputs."""

import re
from pathlib import Path

import pytest

import tokamak_amd

SOURCES = sorted((Path(tokamak_amd.__file__).parent / "csrc").glob("*.h*"))


@pytest.mark.parametrize("source", SOURCES, ids=lambda p: p.name)
def test_m0_and_scc_are_named_where_they_are_written(source):
    for statement in re.findall(r"asm volatile\((.*?)\);", source.read_text(), re.S):
        named = statement.rsplit(":", 1)[-1]
        if re.search(r"\bs_\w+ m0,", statement):
            assert '"m0"' in named, statement
        if re.search(r"\bs_(add|sub|and|or|xor|lshl|lshr|cmp)\w* ", statement):
            assert '"scc"' in named, statement
