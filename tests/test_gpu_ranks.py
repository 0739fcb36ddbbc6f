"""Dense ranks of whole numbers by presence bits, at the edges of their range."""
import numpy as np
import pytest

import iqhip
import iqref

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [256, 257, 1025, 4096, 4097, 9000])  # fewest ranked so, the workgroup, the LDS sort's most
@pytest.mark.parametrize("span", [1, 31, 32, 32767, 32768, 200000])
@pytest.mark.parametrize("kind", ["codes", "signed", "large", "fraction"])
def test_whole_number_ranks_bitwise(ctx, n, span, kind):
    rng = np.random.default_rng(n + span)
    D = rng.integers(0, span + 1, n).astype(np.float64)
    D[rng.choice(n, 2, replace=False)] = [0.0, span]  # the span is met exactly
    if kind == "signed":
        D -= span // 2
        D[rng.choice(n, n // 8, replace=False)] = -0.0
        D[rng.choice(n, 2, replace=False)] = [-(span // 2), span - span // 2]
    elif kind == "large":
        D += 2.0**52
    elif kind == "fraction":
        D[n // 3] += 0.5 if D[n // 3] < span else -0.5
    ev = np.arange(n)
    got = iqhip.taumodel(ev, D, [D[::-1].copy()], ctx=ctx)
    ref = iqref.taumodel(ev, D, [D[::-1].copy()])
    assert np.array_equal(got.view(np.uint64), ref.view(np.uint64))
