"""The MFMA prefill attention for every group size (one to four query heads
per KV head: its waves are then four, two or one query tiles), at the edges
of its tiles (32, 64 and 128 queries) and key blocks (32), with and without
cached keys, against float64.

Bound: the queries and probabilities carry ~22 bits and the products are
exact, so an output is off by a few 2^-22 of the largest |v| plus the f32
sums' rounding: 4e-6 of the values' scale (3 standard deviations here).
"""
from __future__ import annotations

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("first,n_queries", [(0, 1), (0, 33), (31, 65), (100, 129), (1000, 40), (2100, 31)])
@pytest.mark.parametrize("group", [1, 2, 3, 4])
@pytest.mark.parametrize("hd", [64, 128, 256])
def test_attention_prefill_groups(hip, hd, group, first, n_queries):
    kv = 2
    heads, keys = kv * group, first + n_queries
    rng = np.random.default_rng(hd + 10 * group + first)
    q = (2 * rng.standard_normal((n_queries, heads, hd))).astype(np.float32)
    k, v = (rng.standard_normal((keys, kv, hd)).astype(np.float16) for _ in range(2))
    qb, kb, vb, ob = hip.buffer_from(q), hip.buffer_from(k), hip.buffer_from(v), hip.new_buffer(q.nbytes)
    hip.begin()
    hip.attention_prefill(qb.at(0), kb.at(0), vb.at(0), ob.at(0), heads, kv, hd, first, n_queries, keys)
    hip.end()
    got = hip.read(ob.at(0), np.empty_like(q))
    visible = np.arange(keys)[None] <= first + np.arange(n_queries)[:, None]
    for h in range(heads):
        s = q[:, h].astype(np.float64) @ k[:, h // group].astype(np.float64).T / np.sqrt(hd)
        s = np.where(visible, s, -np.inf)
        p = np.exp(s - s.max(1, keepdims=True))
        want = p / p.sum(1, keepdims=True) @ v[:, h // group].astype(np.float64)
        assert np.abs(got[:, h] - want).max() < 4e-6 * 3, h


@pytest.mark.parametrize("group", [1, 2, 3, 4])
@pytest.mark.parametrize("hd", [64, 128, 256])
def test_later_tiles_values_stay_out(hip, hd, group):
    """An infinite value of a token leaves the query tiles before the token's
    own (32 queries each) as they are without it, though the tile's last key
    block of 32 holds the token: the batch starts inside a block."""
    kv, first, n_queries, tile = 1, 20, 128, 32
    heads, keys = kv * group, first + n_queries
    rng = np.random.default_rng(hd + group)
    q = rng.standard_normal((n_queries, heads, hd)).astype(np.float32)
    k, v = (rng.standard_normal((keys, kv, hd)).astype(np.float16) for _ in range(2))
    bad = v.copy()
    bad[first + 2 * tile + 1, 0, 3] = np.inf
    got = []
    for values in (v, bad):
        qb, kb, vb, ob = hip.buffer_from(q), hip.buffer_from(k), hip.buffer_from(values), hip.new_buffer(q.nbytes)
        hip.begin()
        hip.attention_prefill(qb.at(0), kb.at(0), vb.at(0), ob.at(0), heads, kv, hd, first, n_queries, keys)
        hip.end()
        got.append(hip.read(ob.at(0), np.empty_like(q)))
    assert (got[0][:2 * tile] == got[1][:2 * tile]).all()
