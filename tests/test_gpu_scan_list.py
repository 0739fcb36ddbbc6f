"""MFMA scans of several rounds of workgroups, which list the candidates near
their bound: ragged blocks, disabled windows, codes, and ties up to every window."""
import numpy as np
import pytest

from test_gpu_simulate import _compare, _smooth

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("kind", ["split", "holes", "codes", "flat"])
@pytest.mark.parametrize("ti", [(71, 57, 20), (46, 90, 27)], ids=["whole", "ragged"])  # 64 and 39 candidates along x
def test_listed_scan_matches_oracle(ti, kind):
    """320 queries of one overlap: 10 query tiles, 4,760 wavefronts and more."""
    rng = np.random.default_rng(17)
    T = _smooth(rng, ti, 5, np.float32)
    if kind == "holes":
        T[10:14, 20:24, 5] = np.nan
    elif kind == "codes":
        T = np.digitize(T, np.quantile(T, [0.5, 0.8])).astype(np.float64)
    elif kind == "flat":
        T = (rng.random(ti) < 1e-4).astype(np.float32)
    print("listed scan", ti, kind, flush=True)
    _compare(T, (8, 8, 4), (14, 8, 4), overlap=(0.25, 0.25, 0.25), nreal=320)
