"""Prefix sets of the relaxation whose order statistic is bracketed by a sample."""
import numpy as np
import pytest

import iqhip
import iqref

pytestmark = pytest.mark.gpu


# below, at and above the smallest sampled map; word and wavefront remainders
@pytest.mark.parametrize("n", [32767, 32768, 32800, 65599])
@pytest.mark.parametrize("kind", ["continuous", "sorted", "steps", "inf", "subnormal"])
def test_sampled_prefix_sets_match_oracle(ctx, n, kind):
    """Sets are exact whatever the sample says: values in order, tied in
    blocks of 1 to 700, a third disabled, or equal in their top 32 bits."""
    rng = np.random.default_rng(n)
    D, A = rng.random(n) * 1e3, rng.random(n)
    if kind == "sorted":
        D.sort()
    elif kind == "steps":
        D, A = np.floor(D * n / 4e5) / 7, np.floor(A * n / 40)
    elif kind == "inf":
        D[rng.random(n) < 0.33] = np.inf
        A[np.isinf(D)] = np.inf
    elif kind == "subnormal":
        D, A = D * 5e-324 * 1e6, np.floor(A * 1e6) * 5e-324
    for tol in (1e-4, 0.1, 0.5, 0.999, 1.0):
        print(n, kind, tol, flush=True)
        got = iqhip.relaxation(D, [A], tol, ctx=ctx)
        assert np.array_equal(got, iqref.relaxation(D, [A], tol)), tol
