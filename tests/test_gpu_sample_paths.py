"""The sampler's candidate searches at the sizes and distributions where they
can go wrong: k around the 768 up to which a bound of the threads' maxima is
used, fewer logits than threads, ties everywhere, the largest logits all with
one thread (a list of little more than k) or with fewer threads than k (more
than the list holds: the radix select), most of them masked or all equal (the
radix select again, whole waves in one bin), and cuts whose bin holds more than
the list (top_k = 0 on equal logits).

The oracle ranks by logit, then id, as the GPU does, and both take the draw
`u`: kept away from candidate boundaries (draws of a uniform grid's
midpoints), the token must be the same, whole numbers exactly.
"""
from __future__ import annotations

import numpy as np
import pytest

from bobcat_amd._lib import Sampling

pytestmark = pytest.mark.gpu


def draw(hip, logits, st, u):
    lb, rb, ob = hip.buffer_from(logits), hip.buffer_from(np.zeros(1, np.uint32)), hip.new_buffer(4)
    hip.begin()
    hip.sample_draw(lb.at(0), len(logits), rb.at(0), 0, st, u, ob.at(0))
    hip.end()
    return int(hip.read(ob.at(0), np.empty(1, np.uint32))[0])


def logits_of(kind, n, rng):
    if kind == "normal":
        return (3 * rng.standard_normal(n)).astype(np.float32)
    if kind == "ties":
        return rng.integers(0, 3, n).astype(np.float32)
    if kind == "one_thread":  # every 1,024th logit is far above the rest
        x = rng.standard_normal(n).astype(np.float32) * 0.1
        x[5::1024] += 8
        return x
    if kind == "few_threads":  # those of 70 threads, at 65,536 logits 4,480 of them
        x = rng.standard_normal(n).astype(np.float32) * 0.1
        x[np.arange(n) % 1024 < 70] += 8
        return x
    if kind == "equal":
        return np.full(n, 2.5, np.float32)
    return np.where(np.arange(n) % 7 == 0, np.float32(0), -np.inf).astype(np.float32)  # "masked"


@pytest.mark.parametrize("kind", ["normal", "ties", "one_thread", "few_threads", "masked", "equal"])
@pytest.mark.parametrize("n,top_k", [(100, 20), (1000, 999), (5000, 768), (5000, 769), (65536, 40), (65536, 768),
                                     (65536, 4000)])
def test_top_k_set(hip, kind, n, top_k):
    """With equal weights for all candidates (a huge temperature) the token
    drawn at u = (i + 0.5) / k is the candidate of rank i."""
    rng = np.random.default_rng(n + top_k)
    x = logits_of(kind, n, rng)
    order = np.lexsort((np.arange(n), -x.astype(np.float64)))[:top_k]
    order = order[np.isfinite(x[order])]  # (a masked candidate weighs nothing)
    st = Sampling(1e6, top_k, 1.0, 0.0, 1.0)
    for i in (0, len(order) // 3, len(order) - 1):
        assert draw(hip, x, st, (i + 0.5) / len(order)) == order[i], i


@pytest.mark.parametrize("kind,n", [("normal", 65536), ("normal", 300), ("ties", 30000), ("one_thread", 20000),
                                    ("equal", 30001)])
@pytest.mark.parametrize("top_k,top_p,min_p", [(0, 0.9, 0.0), (0, 1.0, 0.05), (5000, 0.5, 0.0)])
def test_large_candidate_sets(hip, kind, n, top_k, top_p, min_p):
    rng = np.random.default_rng(n)
    x = logits_of(kind, n, rng)
    wrong = 0
    for u in np.linspace(0.03, 0.97, 9):
        st = Sampling(0.8, top_k, top_p, min_p, 1.0)
        want = exact(x, top_k, top_p, min_p, 0.8, u)
        got = draw(hip, x, st, float(np.float32(u)))
        wrong += got not in want
    assert wrong == 0


def exact(x, top_k, top_p, min_p, temperature, u):
    """The tokens within 1e-4 of the draw in float64: the f32 weights of up
    to 65,536 candidates round to 2^-24 each, so a cumulative sum is off by
    less than 1e-5 and the top-p cut by a few candidates at most."""
    x = x.astype(np.float64)
    order = np.lexsort((np.arange(len(x)), -x))
    if top_k:
        order = order[:top_k]
    p = np.exp(x[order] - x[order[0]])
    p /= p.sum()
    found = set()
    for slack in (-1e-5, 0, 1e-5):
        keep = order[:int(np.searchsorted(np.cumsum(p), min(top_p + slack, 1.0))) + 1]
        q = p[:len(keep)]
        keep, q = keep[q >= q[0] * min_p * (1 - 1e-5)], q[q >= q[0] * min_p * (1 - 1e-5)]
        w = np.exp(np.log(q / q[0]) / temperature)
        c = np.cumsum(w / w.sum())
        lo, hi = np.searchsorted(c, u - 1e-4), np.searchsorted(c, u + 1e-4)
        found.update(keep[lo:hi + 1].tolist())
    return found


@pytest.mark.parametrize("bits", [0x7fc00000, 0xffc00000, 0xffffffff], ids=hex)
@pytest.mark.parametrize("n,top_k", [(100, 0), (100, 40), (5000, 40), (5000, 700), (5000, 1000), (5000, 0)])
def test_nan_logits_draw_a_token(hip, n, top_k, bits):
    """What a NaN makes of the weights is open, but the token is one of the
    vocabulary: the next step reads its embedding row."""
    rng = np.random.default_rng(n + top_k)
    x = rng.standard_normal(n).astype(np.float32)
    x.view(np.uint32)[rng.integers(0, n, 7)] = bits
    for u in (0.0, 0.4, 0.999):
        assert draw(hip, x, Sampling(0.8, top_k, 0.95, 0.05, 1.0), u) < n
