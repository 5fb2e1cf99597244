"""The prefill GEMM's tile at the sizes where it can go wrong: one token, a
partial block of 32 tokens, a token past a 128- or 256-token tile, a row past
a tile, one super-block of columns (every request of the pipeline past the
end), rows whose columns are no whole super-block, and every weight format.

Each product is compared with that of the half-rounded weights and inputs in
float64.  Bound: fp32 accumulation of n products, at most n·2^-24 of Σ|w·x|
and in practice ~√n·2^-24, so 1e-5 of the largest output holds with a wide
margin up to the 768 columns here.
"""
from __future__ import annotations

import numpy as np
import pytest

import oracle
from bobcat_amd.backend import Format, Store
from bobcat_amd.lfm2 import Lfm2Config, Lfm2Hip, Lfm2Weights, _matrix
from tests.test_gpu_ops import half_inputs

pytestmark = pytest.mark.gpu

FORMATS = [Format.Q4K, Format.Q5K, Format.Q6K, Format.Q8_0, Format.Q4_0, Format.F16, Format.F32]


@pytest.mark.parametrize("n_rows,n_cols,n_tokens", [(33, 256, 1), (64, 512, 31), (65, 512, 33), (130, 768, 129),
                                                    (96, 256, 257), (300, 512, 64)])
@pytest.mark.parametrize("fmt", FORMATS, ids=lambda f: f.name)
def test_matmul_tile_edges(hip, fmt, n_rows, n_cols, n_tokens):
    rng = np.random.default_rng(int(fmt) * 1000 + n_tokens)
    w = _matrix(fmt, n_rows, n_cols, rng)
    x = (rng.standard_normal((n_tokens, n_cols)) * 10.0 ** rng.integers(-3, 4, (n_tokens, 1))).astype(np.float32)
    prior = rng.standard_normal((n_tokens, n_rows)).astype(np.float32)
    dense = oracle.dequantize(int(fmt), w, n_rows * n_cols).reshape(n_rows, n_cols)
    want = half_inputs(x) @ dense.astype(np.float16).astype(np.float64).T
    wb, xb, yb = hip.buffer_from(w), hip.buffer_from(x), hip.buffer_from(prior)
    for store in (Store.ACCUMULATE, Store.OVERWRITE):
        hip.begin()
        hip.matmul(fmt, wb.at(0), n_rows, n_cols, xb.at(0), yb.at(0), n_tokens, store)
        hip.end()
        got = hip.read(yb.at(0), np.empty((n_tokens, n_rows), np.float32))
        ref = want + prior if store == Store.ACCUMULATE else want
        # Token by token: their scales differ by up to 1e7.
        assert (np.abs(got - ref).max(1) <= 1e-5 * np.abs(ref).max(1)).all(), store


@pytest.mark.parametrize("fmt", [Format.Q8_0, Format.F16], ids=lambda f: f.name)
def test_prefill_of_columns_without_whole_super_blocks(hip, fmt):
    """320 and 448 columns (five and seven stages): the last super-block's
    missing stages add nothing."""
    cfg = Lfm2Config("lfm2-tiny-320", n_embd=320, n_ff=448, n_heads=4, n_kv_heads=2, n_vocab=500,
                     attention_layers=[1], n_layers=3, embd_format=fmt, layer_format=fmt)
    weights = Lfm2Weights(cfg, seed=5)
    toks = np.random.default_rng(3).integers(0, cfg.n_vocab, 37).tolist()
    m = Lfm2Hip(hip, weights, n_ctx=64, kv_half=False)
    got = m.prefill(toks)
    m.close()
    cpu = oracle.Lfm2State(weights, n_ctx=64)
    for t in toks:
        want = cpu.step(t)
    # The prefill tolerance of the driver tests: weights and inputs rounded to half.
    assert np.abs(got - want).max() <= 1e-3 * np.abs(want).max()
