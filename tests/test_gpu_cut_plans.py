"""Plans whose slabs lie on both sides of the register-resident cut's 3,072
nodes, against the oracle: every slab takes the form of its own size; and
single cuts that fill their wavefronts."""
import numpy as np
import pytest

import iqhip
import iqref
from test_gpu_simulate import _compare, _smooth

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("overlap", [(0.2, 0.075, 0.1), (0.2, 0.1, 0.15), (0.25, 0.15, 0.05)],
                         ids=["4800-800", "4800-1600-1600", "6400-3200"])  # interior nodes by axis
@pytest.mark.parametrize("dtype", [np.float32, np.float64])
def test_slabs_of_both_forms_match_oracle(overlap, dtype):
    T = _smooth(np.random.default_rng(53), (58, 55, 27), 5, dtype)
    kw = dict(overlap=overlap, path="random")
    plan, _ = iqhip.make_plan(T, (40, 40, 20), (70, 72, 36), rng=np.random.default_rng(1), **kw)
    plan.run(np.random.default_rng(2).random((1, plan.npath)))
    _, relabels, cuts = plan.cut_stats()
    plan.close()
    # only the register-resident form counts its relabel passes
    assert cuts > 0 and (relabels > 0) == (overlap[1] < 0.15)
    print("slabs", overlap, dtype.__name__, flush=True)
    _compare(T, (40, 40, 20), (70, 72, 36), **kw)


@pytest.mark.parametrize("shape,dim", [((10, 16, 1), 0), ((16, 4, 4), 1), ((4, 64, 1), 0), ((6, 16, 8), 0)],
                         ids=["128", "128-y", "128-long", "512"])
@pytest.mark.parametrize("dtype", [np.float32, np.float64])
def test_full_wavefronts_match_oracle(shape, dim, dtype):
    """Teams whose lanes all hold a node."""
    rng = np.random.default_rng(54)
    A, B = (rng.standard_normal(shape).astype(dtype) for _ in range(2))
    print("cut", shape, dim, flush=True)
    assert np.array_equal(iqhip.graphcut(A, B, dim), iqref.graphcut(A, B, dim))
