"""The group size of the MFMA scan is timed on launches like a run's."""
import numpy as np
import pytest

import iqhip

pytestmark = pytest.mark.gpu


def test_timed_launches_list_what_a_run_lists():
    """An image of ties lists every window of every query.  Most of the run's
    waves are four tiles of eight realizations: 32 queries, as a timed launch."""
    rng = np.random.default_rng(63)
    T = (rng.random((100, 100, 20)) < 1e-4).astype(np.float32)
    plan, _ = iqhip.make_plan(T, (8, 8, 4), (240, 8, 4), overlap=(0.25, 0.25, 0.25), nreal=8,
                              rng=np.random.default_rng(1))
    _, timed = plan.scan_tuning()
    u = np.random.default_rng(2).random((8, plan.npath))
    plan.run(u)
    plan.profile(True)
    plan.run(u)
    launches, seconds, _, _ = plan.scan_stats()
    print("timed", timed, "run", seconds / launches * 1e6, flush=True)
    assert launches > 30 and max(timed.values()) > 0.75 * seconds / launches * 1e6
    plan.close()
