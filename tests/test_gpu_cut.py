"""Register-resident min cut against the oracle at the edges of its forms: one
wavefront, one node a lane, two and three nodes a lane, global scratch; both
element types, every cut axis, ties and infinite values."""
import numpy as np
import pytest

import iqhip
import iqref

pytestmark = pytest.mark.gpu


def _slabs(rng, shape, dtype, ties=False):
    A, B = rng.standard_normal(shape), rng.standard_normal(shape)
    if ties:  # categorical codes: zero gradients, capacities from 0 to 2^53
        A, B = np.digitize(A, [0.3, 1.0]), np.digitize(B, [0.3, 1.0])
    return A.astype(dtype), B.astype(dtype)


# interior nodes: 1, 63, 64, 65, 128, 1,023, 1,024, 1,025, 2,048, 2,049, 3,072, 3,080
@pytest.mark.parametrize("shape,dim", [((3, 1, 1), 0), ((3, 9, 7), 0), ((6, 16, 1), 0), ((15, 5, 1), 0), ((8, 6, 4), 2),
                                       ((5, 31, 11), 0), ((32, 6, 8), 1), ((43, 25, 1), 0), ((16, 16, 10), 2),
                                       ((3, 683, 3), 0), ((32, 5, 32), 1), ((9, 55, 8), 0)])
@pytest.mark.parametrize("dtype", [np.float32, np.float64])
def test_cut_sizes_match_oracle(shape, dim, dtype):
    rng = np.random.default_rng(51)
    for ties in (False, True):
        A, B = _slabs(rng, shape, dtype, ties)
        print("cut", shape, dim, dtype.__name__, "ties" if ties else "", flush=True)
        assert np.array_equal(iqhip.graphcut(A, B, dim), iqref.graphcut(A, B, dim))


@pytest.mark.parametrize("dtype", [np.float32, np.float64])
def test_cut_infinite_values_match_oracle(dtype):
    rng = np.random.default_rng(52)
    for k in range(4):
        A, B = _slabs(rng, (6, 13, 4), dtype)
        for X, n in ((A, k), (B, 3 - k)):
            X[tuple(rng.integers(0, s, 2 * n) for s in X.shape)] = np.inf
        print("cut with infinite values", k, flush=True)
        assert np.array_equal(iqhip.graphcut(A, B, 0), iqref.graphcut(A, B, 0))
