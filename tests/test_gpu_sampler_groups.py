"""The sampler's group maxima, candidate lists and streamed sums at their
edges, against the oracle's restatement of generation/sampler.rs (the same
token)."""
import numpy as np
import pytest

import oracle as O
from synapse_amd import hip

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module", autouse=True)
def gpu():
    hip.init(0)


def _check(x, hist=(), draws=4, seed=1, **kw):
    for u in O.stdrng_f32(seed, draws):
        want = O.sample_combined(x, np.asarray(hist, np.uint32), u=float(u), **kw)
        got = hip.sample(x, hist, u=float(u), **kw)
        assert got == want, (x.size, kw, float(u), got, want)


# one group, a part of one, whole groups, the 1024 logits of a prep workgroup
# and one more, 4096 groups (all in registers) and one more (general route)
@pytest.mark.parametrize("n", [1, 2, 63, 64, 65, 1024, 1025, 262144, 262145])
def test_vocabulary_edges(n):
    x = (np.random.default_rng(n).standard_normal(n) * 3).astype(np.float32)
    hist = np.random.default_rng(n + 1).integers(0, n, 30)
    for kw in (dict(temperature=0.0), dict(temperature=0.9, top_k=3),
               dict(temperature=0.8, top_k=40, top_p=0.9, repetition_penalty=1.2)):
        _check(x, hist, **kw)


def test_more_candidates_than_groups_and_ties():
    rng = np.random.default_rng(3)
    x = rng.standard_normal(5000).astype(np.float32)
    _check(x, temperature=1.0, top_k=100, top_p=0.7)   # k above the 79 groups
    x = np.round(rng.standard_normal(20000) * 2).astype(np.float32)  # few distinct values
    _check(x, temperature=1.0, top_k=50)
    x = np.zeros(9000, np.float32)                     # every value at the threshold
    x[7] = -0.0
    _check(x, temperature=1.0, top_k=20, top_p=0.5)
    _check(x, temperature=0.0)


def test_masked_logits():
    x = np.full(30000, -np.inf, np.float32)
    live = np.random.default_rng(5).integers(0, 30000, 60)
    x[live] = np.random.default_rng(6).standard_normal(60).astype(np.float32)
    for kw in (dict(temperature=0.0), dict(temperature=0.7, top_k=20, top_p=0.9),
               dict(temperature=0.7, top_k=100), dict(temperature=1.0)):
        _check(x, live[:5], **kw)


def test_history_counts():
    # a token penalised once per occurrence, more entries than threads, ids
    # outside the vocabulary ignored
    x = (np.random.default_rng(8).standard_normal(4000) * 4).astype(np.float32)
    top = np.argsort(x)[-40:]
    hist = np.concatenate([np.repeat(top[-5:], 7), np.random.default_rng(9).integers(0, 6000, 1500)])
    for kw in (dict(temperature=0.0, repetition_penalty=1.1),
               dict(temperature=0.8, top_k=30, repetition_penalty=1.05)):
        _check(x, hist, **kw)


# the streamed sums: one block of 4096, one more, several; flat and peaked
@pytest.mark.parametrize("n", [4095, 4096, 4097, 20000])
@pytest.mark.parametrize("scale", [0.2, 6.0])
def test_full_softmax_stream(n, scale):
    x = (np.random.default_rng(n).standard_normal(n) * scale).astype(np.float32)
    _check(x, draws=6, temperature=1.0)
    _check(x, draws=3, temperature=1.0, top_p=0.6)


# NaN logits leave the group maxima for the general route; infinite ones do not
@pytest.mark.parametrize("n", [5, 64, 700, 5000, 30000])
def test_nan_and_infinite_logits(n):
    rng = np.random.default_rng(n)
    base = (rng.standard_normal(n) * 3).astype(np.float32)
    both = base.copy()
    both[0], both[n // 2] = np.nan, np.inf
    for x in (both, np.full(n, np.nan, np.float32)):
        for kw in (dict(temperature=0.9, top_k=3),
                   dict(temperature=0.8, top_k=40, top_p=0.9, repetition_penalty=1.2)):
            _check(x, (1, 2, 1), **kw)
    ends = base.copy()
    ends[[0, n - 1]] = np.inf
    half = base.copy()
    half[:n // 2] = -np.inf
    for x in (ends, half):
        for kw in (dict(temperature=0.0), dict(temperature=0.9), dict(temperature=0.9, top_k=3),
                   dict(temperature=0.7, top_p=0.6)):
            _check(x, (1, 2, 1), **kw)
