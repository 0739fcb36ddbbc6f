"""Learned shortlist over integer codes, whose full scan takes its distances
as exact and follows with no recheck: whole shortlists, checked batches and
sampled checks equal the plain full scan."""
import numpy as np
import pytest

import iqhip
from iqhip import synth

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("check", [dict(K=10 ** 9, check_every=0), dict(K=64, check_every=1, min_recall=1.0),
                                   dict(K=10 ** 9, check_every=2, min_recall=0.5, check_queries=3)],
                         ids=["whole", "checked", "sampled"])
def test_codes_equal_the_full_scan(check):
    T = synth.channels((72, 70, 12), np.random.default_rng(92)).astype(np.float64)
    plan, _ = iqhip.make_plan(T, (12, 12, 4), (72, 60, 12), overlap=(0.25, 0.25, 0.25), tol=0.1, nreal=4,
                              rng=np.random.default_rng(1))
    u = np.random.default_rng(5).random((4, plan.npath))
    plan.run(u)
    ref = plan.results(grids=True, chosen=True)
    plan.learn(nsamples=2048, iters=6, seed=1)
    plan.set_proposal(True, **check)
    print("codes", check, flush=True)
    plan.run(u)
    got = plan.results(grids=True, chosen=True)
    assert np.array_equal(got["chosen"], ref["chosen"])
    for a, b in zip(got["grids"], ref["grids"]):
        assert np.array_equal(a, b)
    plan.close()
