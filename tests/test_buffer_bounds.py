"""CPU check of the kernels' bounds-checked loads: only the vector offset of a
raw buffer load is sure to be compared with the descriptor's size, so a load
that counts on reading zeros past the end carries its whole address there.
(What it does otherwise cannot be tried: it may read outside the buffer.)"""
from __future__ import annotations

import re
from pathlib import Path

import pytest

CSRC = Path(__file__).resolve().parent.parent / "bobcat_amd" / "csrc"


def buffer_loads(text: str) -> list[tuple[int, list[str]]]:
    """Position and arguments of every raw buffer load."""
    loads = []
    for m in re.finditer(r"raw_buffer_load_\w+\(", text):
        args, depth, start = [], 1, m.end()
        for i in range(m.end(), len(text)):
            depth += (text[i] in "([{") - (text[i] in ")]}")
            if depth == 0 or (depth == 1 and text[i] == ","):
                args.append(text[start:i].strip())
                start = i + 1
            if depth == 0:
                break
        loads.append((m.start(), args))
    return loads


@pytest.mark.parametrize("name", ["attn_prefill.hip", "attn_decode.hip"])
def test_attention_loads_have_no_scalar_offset(name):
    loads = buffer_loads((CSRC / name).read_text())
    assert loads
    for _, args in loads:
        assert len(args) == 4 and args[2] == "0", args


def test_gemm_loads_past_the_columns_have_no_scalar_offset():
    """The GEMM's stages past the columns exist for the formats whose rows need
    not be whole super-blocks of 256 columns: those take the checked form."""
    text = (CSRC / "gemm_tile.h").read_text()
    tail = re.search(r"constexpr bool TAIL = !GROUPED && \((.*?)\);", text).group(1)
    assert set(re.findall(r"BCH_\w+", tail)) == {"BCH_F32", "BCH_F16", "BCH_Q8_0", "BCH_Q4_0"}
    checked, plain = buffer_loads(text)
    assert re.search(r"if constexpr \(TAIL\)[^;]*$", text[:checked[0]]) and checked[1][2] == "0"
    assert re.search(r"else[^;]*$", text[checked[0]:plain[0]])
