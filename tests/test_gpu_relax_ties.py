"""Prefix sets of maps whose bracket is one tied value, holds a large tie, or
is equal in the top words alone, against the oracle."""
import numpy as np
import pytest

import iqhip
import iqref

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [65536, 70001, 216225])  # word and wavefront remainders
@pytest.mark.parametrize("kind", ["levels3", "levels40", "runs", "constant", "top", "holes"])
def test_tied_prefix_sets_match_oracle(ctx, n, kind):
    rng = np.random.default_rng(n)
    D, A = rng.random(n), rng.random(n)
    if kind == "levels3":  # a bracket inside one tie
        D, A = np.floor(D * 3), np.floor(A * 3)
    elif kind == "levels40":  # a bracket over a few ties of more than 512 values
        D, A = np.floor(D * 40) / 7, np.floor(A * 40)
    elif kind == "runs":  # ties in consecutive places
        D, A = np.arange(n) // 1500 * 0.3, np.sort(np.floor(A * 25))[::-1].copy()
    elif kind == "constant":
        D[:], A[:] = 2.5, 0.0
        D[n // 2] = 3.0
    elif kind == "top":  # equal in their top 32 bits, apart from ties below
        D, A = 1.0 + D * 2.0 ** -22, 1.0 + np.floor(A * 5) * 2.0 ** -40
    elif kind == "holes":
        D, A = np.floor(D * 9), np.floor(A * 5)
        D[rng.random(n) < 0.5] = np.inf
        A[np.isinf(D)] = np.inf
    for tol in (1e-4, 0.1, 0.34, 0.999, 1.0):
        print(n, kind, tol, flush=True)
        got = iqhip.relaxation(D, [A], tol, ctx=ctx)
        assert np.array_equal(got, iqref.relaxation(D, [A], tol)), tol


@pytest.mark.parametrize("n", [57343, 57344, 57377])  # below, at and above the smallest sampled map
@pytest.mark.parametrize("kind", ["continuous", "levels"])
def test_smallest_sampled_map_matches_oracle(ctx, n, kind):
    rng = np.random.default_rng(n)
    D, A = rng.random(n), rng.random(n)
    if kind == "levels":
        D, A = np.floor(D * 30), np.floor(A * 4)
    for tol in (1e-4, 0.1, 0.999):
        print(n, kind, tol, flush=True)
        assert np.array_equal(iqhip.relaxation(D, [A], tol, ctx=ctx), iqref.relaxation(D, [A], tol)), tol
