"""MFMA scan with every group size (IQHIP_SCAN_NW; the default is timed per
plan) against the oracle: stored and listed bounds, split, bf16-exact and
rounded data."""
import numpy as np
import pytest

import iqhip
from test_gpu_simulate import _compare, _smooth

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nw", [2, 3, 4])
@pytest.mark.parametrize("kind", ["split", "codes", "rounded"])
@pytest.mark.parametrize("ti,tile,sim,nreal", [
    ((41, 50), (10, 9), (40, 37), 3),            # one tile of queries, stored: rows not a multiple of 8, 12 or 16
    ((71, 57, 20), (8, 8, 4), (14, 14, 8), 40),  # two tiles and more, listed
], ids=["stored", "listed"])
def test_group_sizes_match_oracle(monkeypatch, ti, tile, sim, nreal, kind, nw):
    monkeypatch.setenv("IQHIP_SCAN_NW", str(nw))
    rng = np.random.default_rng(62)
    T = _smooth(rng, ti, 5, np.float64 if kind == "rounded" else np.float32)
    if kind == "codes":
        T = np.digitize(T, np.quantile(T, [0.5, 0.8])).astype(np.float64)
    kw = dict(overlap=(0.25,) * len(ti), nreal=nreal)
    plan, _ = iqhip.make_plan(T, tile, sim, rng=np.random.default_rng(1), **kw)
    assert plan.scan_tuning()[0] == (nw, nw)  # the scan ran, with that size
    plan.close()
    print("groups of", nw, ti, kind, flush=True)
    _compare(T, tile, sim, **kw)
