"""MFMA scans on both sides of the 256 wavefronts from which they list their
candidates: 252, 256 and 260, with four to a group."""
import numpy as np
import pytest

import iqhip
from test_gpu_simulate import _compare, _smooth

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dist", [(31, 109, 9), (32, 127, 8), (30, 77, 13)], ids=["252", "256", "260"])  # 7x9, 8x8, 5x13 groups
@pytest.mark.parametrize("kind", ["split", "codes", "rounded", "holes", "flat"])
def test_both_forms_match_oracle(monkeypatch, dist, kind):
    monkeypatch.setenv("IQHIP_SCAN_NW", "4")
    rng = np.random.default_rng(64)
    tile = (8, 7, 4)
    ti = tuple(d + t - 1 for d, t in zip(dist, tile))
    T = _smooth(rng, ti, 5, np.float64 if kind == "rounded" else np.float32)
    if kind == "codes":
        T = np.digitize(T, np.quantile(T, [0.5, 0.8])).astype(np.float64)
    elif kind == "holes":
        T[10:13, 40:60, 3:5] = np.nan
    elif kind == "flat":
        T = (rng.random(ti) < 1e-3).astype(np.float32)
    kw = dict(overlap=(0.25, 0.3, 0.25), nreal=2)
    plan, _ = iqhip.make_plan(T, tile, (20, 17, 10), rng=np.random.default_rng(1), **kw)
    assert plan.scan_tuning()[0] == (4, 4)
    plan.close()
    print("candidates", dist, kind, flush=True)
    _compare(T, tile, (20, 17, 10), **kw)
