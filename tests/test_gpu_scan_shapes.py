"""MFMA scan against the oracle through whole simulations: chunk shapes of 8, 4
and 2 voxels along y (overlaps of 2 to 9 voxels), candidate grids around the
32-wide and 8- to 16-row blocks, odd k-step counts, split and bf16-exact data."""
import numpy as np
import pytest

from test_gpu_simulate import _compare, _smooth

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("ti,tile,sim,overlap", [
    ((41, 40), (10, 9), (40, 37), (0.2, 0.2)),            # 32 x 32 candidates, overlap 2
    ((42, 43), (10, 10), (38, 41), (0.3, 0.3)),           # 33 x 34, overlap 3
    ((60, 38), (16, 17), (52, 50), (0.25, 0.29)),         # overlaps 4 and 5
    ((50, 61), (18, 27), (60, 66), (1 / 3, 1 / 3)),       # overlaps 6 and 9
    ((25, 26, 12), (9, 10, 4), (24, 26, 10), (0.45, 0.4, 0.5)),
    ((40, 30, 20), (24, 8, 16), (50, 20, 24), (0.34, 0.25, 0.25)),  # regions cut along z
], ids=["ov2", "ov3", "ov4-5", "ov6-9", "volume", "deep"])
@pytest.mark.parametrize("kind", ["split", "codes"])
def test_scan_shapes_match_oracle(ti, tile, sim, overlap, kind):
    rng = np.random.default_rng(61)
    T = _smooth(rng, ti, 5, np.float32)
    if kind == "codes":
        T = np.digitize(T, np.quantile(T, [0.5, 0.8])).astype(np.float64)
    print("scan", ti, tile, kind, flush=True)
    _compare(T, tile, sim, overlap=overlap, path="random", nreal=3)
