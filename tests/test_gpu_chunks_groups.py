"""The chunked DeltaNet form on its tile edges and on values that are not
finite, against the sequential rule in float64; the grouping of expert entries."""
from __future__ import annotations

import ctypes as C

import numpy as np
import pytest

from bobcat_amd._lib import DeltaShape, lib
from bobcat_amd.backend import _view
from test_gpu_qwen35 import delta_rule_f64

pytestmark = pytest.mark.gpu


def chunked(hip, y, beta, decay, state, n_k, n_v, dk, dv, q_scale):
    shape, n = DeltaShape(n_k, n_v, dk, dv), len(y)
    yb, bb, db, sb = (hip.buffer_from(v) for v in (y, beta, decay, state))
    ob = hip.new_buffer(n * n_v * dv * 4)
    wb = hip.new_buffer(lib().bch_gdn_chunk_scratch_floats(C.byref(shape), n) * 4)
    hip.begin()
    assert lib().bch_gdn_recurrence_chunked(hip.handle, _view(yb.at(0)), _view(bb.at(0)), _view(db.at(0)),
                                            _view(sb.at(0)), _view(ob.at(0)), C.byref(shape), n, C.c_float(q_scale),
                                            _view(wb.at(0))) == 0, lib().bch_last_error()
    hip.end()
    return hip.read(ob.at(0), np.empty((n, n_v * dv), np.float32)), hip.read(sb.at(0), np.empty_like(state))


# Blocks of 16 tokens in chunks of 64; tiles of 16 value columns, the last of 8
# where the head's columns are an odd number of eights; one, or two, or three
# tiles per wave.
@pytest.mark.parametrize("n_k,n_v,dk,dv,n_tokens", [(1, 1, 64, 8, 1), (1, 2, 64, 24, 15), (2, 2, 128, 136, 17),
                                                    (1, 1, 128, 256, 79), (2, 4, 64, 64, 129), (1, 3, 128, 16, 192)])
@pytest.mark.parametrize("bad", [None, "value", "key", "query"])
def test_chunked_rule_on_edges_and_nonfinite_tokens(hip, n_k, n_v, dk, dv, n_tokens, bad):
    """Finite results within 1e-5 of the largest (the bound of the other
    DeltaNet tests).  A token with an infinite value in one column, or a NaN
    in its key or query, leaves every earlier token as it is, and what it
    spoils is what it spoils in the sequential rule."""
    rng = np.random.default_rng(dk + dv + n_tokens)
    key_dim = n_k * dk
    y = rng.standard_normal((n_tokens, 2 * key_dim + n_v * dv)).astype(np.float32)
    beta = rng.uniform(0.1, 1.0, (n_tokens, n_v)).astype(np.float32)
    decay = np.exp(-rng.uniform(0.0, 2.5, (n_tokens, n_v))).astype(np.float32)
    state = (rng.standard_normal((n_v, dk, dv)) * 0.1).astype(np.float32)
    t = n_tokens * 2 // 3
    if bad == "value":
        y[t, 2 * key_dim + dv // 2] = np.inf
    elif bad:
        y[t, (0 if bad == "query" else key_dim) + dk // 2] = np.nan
    q_scale = 1 / np.sqrt(dk)
    got, got_state = chunked(hip, y, beta, decay, state, n_k, n_v, dk, dv, q_scale)
    with np.errstate(all="ignore"):
        want, want_state = delta_rule_f64(y, beta, decay, state, n_k, n_v, dk, dv, q_scale)
    for g, w in ((got, want), (got_state, want_state)):
        finite = np.isfinite(w)
        assert bad or finite.all()
        assert (np.isfinite(g) == finite).all()
        if finite.any():
            assert np.abs(g - w)[finite].max() < 1e-5 * np.abs(w[finite]).max()


@pytest.mark.parametrize("n_experts,n_used,n_tokens", [(1, 1, 70), (3, 2, 1), (64, 4, 300), (65, 3, 341), (128, 8, 2049)])
def test_group_entries_by_expert(hip, n_experts, n_used, n_tokens):
    """Entries by expert, in token order within: runs of fewer and more than
    64 entries per wave, ids of 0 to 7 bits, one and two waves' width of
    experts, ids read from LDS and (above 16,384 entries) from the route."""
    rng = np.random.default_rng(n_experts)
    ids = np.stack([rng.choice(n_experts, n_used, replace=False) for _ in range(n_tokens)]).astype(np.uint32)
    route = hip.buffer_from(np.concatenate([ids, np.zeros_like(ids)], axis=1).reshape(-1))
    offsets, entries = hip.new_buffer((n_experts + 1) * 4), hip.new_buffer(ids.size * 4)
    hip.begin()
    hip.moe_group(route.at(0), offsets.at(0), entries.at(0), n_experts, n_used, n_tokens)
    hip.end()
    flat = ids.reshape(-1)
    assert (hip.read(entries.at(0), np.empty(ids.size, np.uint32)) == np.argsort(flat, kind="stable")).all()
    counts = np.bincount(flat, minlength=n_experts)
    assert (hip.read(offsets.at(0), np.empty(n_experts + 1, np.uint32)) == np.concatenate([[0], np.cumsum(counts)])).all()
