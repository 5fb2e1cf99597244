"""The prefill GEMM's tile at the sizes where it can go wrong: one token, a
partial block of 32 tokens, a token past a tile, a row past a tile, one
super-block of columns (every request of the pipeline past the end), rows whose
columns are no whole super-block, and every weight format.  The small shapes
all take the 64-row x 128-token tile; `gemm_shape` restates the launch's choice
on 256 CUs to name shapes, with rows and tokens left over, for the 64 x 256 and
(Q4_K) 128 x 256 tiles, alone and with their columns split, and the grouped
cases lie on both sides of the rule for their tiles.

Each product is compared with that of the half-rounded weights and inputs in
float64.  Bound: fp32 accumulation of n products, at most n·2^-24 of Σ|w·x|
and in practice ~√(n/16)·2^-24 of the largest output (16 products enter at
once), 1.3e-6 at 8,192 columns unsplit: 1e-5 of it holds with a wide margin.
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
    check_matmul(hip, fmt, n_rows, n_cols, n_tokens)


def check_matmul(hip, fmt, n_rows, n_cols, n_tokens):
    rng = np.random.default_rng(int(fmt) * 1000 + n_tokens)
    w = _matrix(fmt, n_rows, n_cols, rng)
    x = (rng.standard_normal((n_tokens, n_cols)) * 10.0 ** rng.integers(-3, 4, (n_tokens, 1))).astype(np.float32)
    prior = rng.standard_normal((n_tokens, n_rows)).astype(np.float32)
    want = half_inputs(x) @ half_weights(fmt, w, n_rows, n_cols).T
    wb, xb = hip.buffer_from(w), hip.buffer_from(x)
    for store in (Store.ACCUMULATE, Store.OVERWRITE, Store.SWIGLU):
        yb = hip.buffer_from(prior)
        hip.begin()
        hip.matmul(fmt, wb.at(0), n_rows, n_cols, xb.at(0), yb.at(0), n_tokens, store)
        hip.end()
        got = hip.read(yb.at(0), np.empty((n_tokens, n_rows), np.float32))
        ref = {Store.ACCUMULATE: lambda: want + prior, Store.OVERWRITE: lambda: want,
               Store.SWIGLU: lambda: silu(prior.astype(np.float64)) * want}[store]()
        # Token by token: their scales differ by up to 1e7.
        assert (np.abs(got - ref).max(1) <= 1e-5 * np.abs(ref).max(1)).all(), store


def silu(v):
    return v / (1 + np.exp(-v))


def half_weights(fmt, w, n_rows, n_cols):
    dense = oracle.dequantize(int(fmt), w, n_rows * n_cols).reshape(n_rows, n_cols)
    return dense.astype(np.float16).astype(np.float64)


def gemm_shape(fmt, n_rows, n_cols, n_tokens, cus=256):
    """(rows of the tile, its tokens, column splits): matmul.hip's choice."""
    up = lambda a, b: -(-a // b)
    tiles = lambda rows, tokens: up(n_rows, rows) * up(n_tokens, tokens)
    most, wide = 1, n_tokens > 128 and n_rows > 64
    if not (wide and tiles(128, 256) >= cus * 3 // 5):
        if wide and n_cols >= 8192:
            grow = lambda s: tiles(128, 256) * s < cus
        elif n_rows > 64 and tiles(128, 128) >= cus * 3 // 5:
            grow = lambda s: False
        else:
            grow = lambda s: tiles(64, 128) * s * 2 <= cus
        while grow(most) and most < 8 and n_cols // 64 // (2 * most) >= 8:
            most *= 2
    best, blocks = None, up(n_cols, 256)
    for rows, tokens, stage_us in [(64, 128, 0.36), (64, 256, 0.47)] + [(128, 256, 0.85)] * (fmt == Format.Q4K):
        for splits in [s for s in (1, 2, 4, 8) if s <= most and s <= blocks]:
            us = up(tiles(rows, tokens) * splits, cus) * (4 * up(blocks, splits) * stage_us + 4)
            us += (splits > 1) * (1 + 8e-6 / 4.5 * splits * n_tokens * n_rows)
            if best is None or us < best[0]:
                best = us, (rows, tokens, splits)
    return best[1]


TILES = [(65, 1024, 37, (64, 128, 2)), (8001, 256, 257, (64, 256, 1)), (8033, 768, 261, (64, 256, 1)),
         (200, 8192, 1030, (64, 256, 8))]
Q4K_TILES = [(4001, 256, 1030, (128, 256, 1)), (4033, 512, 1041, (128, 256, 1)), (5001, 8192, 130, (128, 256, 4))]


@pytest.mark.parametrize("fmt,n_rows,n_cols,n_tokens,shape", [(f, *c) for f in FORMATS for c in TILES] +
                         [(Format.Q4K, *c) for c in Q4K_TILES])
def test_matmul_every_tile(hip, fmt, n_rows, n_cols, n_tokens, shape):
    assert gemm_shape(fmt, n_rows, n_cols, n_tokens) == shape
    check_matmul(hip, fmt, n_rows, n_cols, n_tokens)


# Positions up to 40 per expert take tiles of 64, more of them 128 (Q4_K; F16
# and F32 always 128).  Expert 0 takes every token: more than one tile, whose
# last has waves without tokens.
@pytest.mark.parametrize("n_experts,n_used,n_tokens,n_rows,n_cols", [
    (3, 2, 190, 100, 512), (4, 3, 161, 257, 256), (2, 2, 41, 64, 768), (8, 2, 150, 72, 256), (1, 1, 33, 130, 256)])
@pytest.mark.parametrize("fmt", [Format.Q4K, Format.F16, Format.F32], ids=lambda f: f.name)
def test_grouped_tile_edges(hip, fmt, n_experts, n_used, n_tokens, n_rows, n_cols):
    rng = np.random.default_rng(int(fmt) + n_tokens)
    gate, up = (_matrix(fmt, n_experts * n_rows, n_cols, rng) for _ in range(2))
    G, U = (half_weights(fmt, w, n_experts * n_rows, n_cols).reshape(n_experts, n_rows, n_cols) for w in (gate, up))
    ids = np.stack([np.r_[0, 1 + rng.permutation(n_experts - 1)[:n_used - 1]] for _ in range(n_tokens)]).astype(np.uint32)
    route = hip.buffer_from(np.concatenate([ids, np.ones((n_tokens, n_used), np.float32).view(np.uint32)], 1))
    off, ent = hip.new_buffer((n_experts + 1) * 4), hip.new_buffer(ids.size * 4)
    gb, ub, yb = hip.buffer_from(gate), hip.buffer_from(up), hip.new_buffer(ids.size * n_rows * 4)
    e = ids.reshape(-1)
    for shared in (True, False):
        x = rng.standard_normal((n_tokens if shared else ids.size, n_cols)).astype(np.float32)
        rows = half_inputs(x)[np.arange(ids.size) // n_used if shared else np.arange(ids.size)]
        g, u = (np.stack([W[i] @ r for i, r in zip(e, rows)]) for W in (G, U))
        sg, su = (np.stack([np.abs(W[i]) @ np.abs(r) for i, r in zip(e, rows)]) for W in (G, U))
        xb = hip.buffer_from(x)
        for pair in (True, False):
            hip.begin()
            hip.moe_group(route.at(0), off.at(0), ent.at(0), n_experts, n_used, n_tokens)
            hip.matmul_experts(fmt, gb.at(0), ub.at(0) if pair else None, n_rows, n_cols, n_experts, xb.at(0), shared,
                               off.at(0), ent.at(0), n_used, yb.at(0), n_tokens)
            hip.end()
            got = hip.read(yb.at(0), np.empty((ids.size, n_rows), np.float32))
            # (1e-5 of the terms, as test_grouped_experts_match_oracle bounds them.)
            want, bound = (silu(g) * u, 1.1 * sg * np.abs(u) + np.abs(silu(g)) * su) if pair else (g, sg)
            assert (np.abs(got - want) <= 1e-5 * bound + 1e-30).all(), (shared, pair)


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
