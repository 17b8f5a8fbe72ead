"""The top-k selection's candidate bound (top_k <= 64): an entry can be among
the first k only if it reaches the k-th largest of the 128 slices' largest
entries (rounded down to a bf16).  Cases on both sides of each rule: a slice
that passes more than 64 entries or none, up to and past 256 candidates over
all slices, fewer than k slices with entries, slices of more than one round of
loads, and a softmax denominator whose bound leaves float(1 / sum) open.  All
against the oracle, bit for bit."""

import numpy as np
import pytest

import llmi_hip as H
import oracle as O

pytestmark = pytest.mark.gpu

SLICES = 128


def check(lg: np.ndarray, k: int, top_p: float = 0.9):
    o = O.oracle()
    want = o.sampling_probabilities(lg, 1.0, k, top_p)
    got = H.sampling_probabilities(lg, H.Sampling(1.0, k, top_p))
    assert np.array_equal(got.view(np.uint32), np.asarray(want, np.float32).view(np.uint32))
    assert H.sampling_last_paths() & 16
    for t in o.draw_uniform(k, 3):
        assert H.sample(lg, H.Sampling(1.0, k, top_p), t) == o.sample_target(lg, 1.0, k, top_p, t)


@pytest.mark.parametrize("ties", [True, False])
@pytest.mark.parametrize("slices,each", [(1, 64), (1, 65), (1, 300), (4, 64), (4, 65), (5, 51), (5, 52), (64, 4), (64, 5)])
def test_candidates_per_slice_and_in_all(slices, each, ties):
    """`each` entries of `slices` slices stand above all others."""
    n, rng = 49152, np.random.default_rng(100 * slices + each)
    per = n // SLICES
    lg = np.minimum(rng.normal(-3.0, 1.0, n), 0.0).astype(np.float32)
    for b in rng.permutation(SLICES)[:slices]:
        at = b * per + rng.permutation(per)[:each]
        lg[at] = 2.0 if ties else 2.0 + rng.random(each).astype(np.float32)
    for k in sorted({1, slices, min(64, slices + 1), 64}):
        check(lg, k)


@pytest.mark.parametrize("n,k", [(65, 64), (100, 40), (129, 2), (3 * 384, 40), (262144, 64), (262145, 40), (300001, 3)])
def test_slice_sizes(n, k):
    rng = np.random.default_rng(n)
    lg = rng.normal(0.0, 3.0, n).astype(np.float32)
    check(lg, k)
    lg[rng.random(n) < 0.999] = -np.inf  # most slices hold nothing
    lg[n - 1] = 0.5
    check(lg, k, 1.0)


@pytest.mark.parametrize("spread", [True, False])
def test_open_reciprocal_takes_the_sequential_sum(spread):
    """`ones` logits of 0 and the rest so low that their e is 0: the
    denominator is exactly `ones`, chosen where the bound around it straddles a
    rounding boundary of the float reciprocal."""
    n = 60000
    c = np.arange(100, 59000, dtype=np.float64)
    slack = 4.0 * (n + 65536.0) * 2.0**-53 * c
    ones = int(c[np.flatnonzero((1.0 / (c - slack)).astype(np.float32) != (1.0 / (c + slack)).astype(np.float32))[0]])
    lg = np.full(n, -300.0, np.float32)
    at = np.random.default_rng(1).permutation(n)[:ones] if spread else np.arange(ones) + 17
    lg[at] = 0.0
    for k in (40, 64):
        check(lg, k)
        assert H.sampling_last_paths() & 1
