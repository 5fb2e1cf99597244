"""CPU check of the drivers' prefill: where the norm may have left plain rows for
the library GEMM (pair_ok), the first launch that reads its outputs converts
them itself (split_ready is !pair_ok), whatever form of the SwiGLU follows.
(Mixed gate and up formats never have a library pair today, so no model can
show the difference.)"""
from __future__ import annotations

import re
from pathlib import Path

import pytest

CSRC = Path(__file__).resolve().parent.parent / "bobcat_amd" / "csrc"


@pytest.mark.parametrize("name", ["lfm2.hip", "qwen35.hip"])
def test_launches_after_a_pair_norm_convert_their_inputs(name):
    text = (CSRC / name).read_text()
    block = text[text.index("const bool blas_pair ="):]
    block = block[:block.index("L.down.format")]
    calls = [re.sub(r"\s+", " ", c) for c in re.findall(r"run_matmul\((.*?)\);", block, re.S)]
    gates = [c for c in calls if c.startswith(("s, L.gate", "st, L.gate"))]
    assert len(gates) == 2 and all(", !pair_ok" in c for c in gates), gates
