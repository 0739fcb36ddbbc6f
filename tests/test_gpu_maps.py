"""Exact FP64 maps on the matrix cores (k_maps_mfma) through whole
simulations against the oracle: tiles whose window region is staged whole, by
planes, by rows and by parts of rows; query counts around the tile of
sixteen; hard data from one point to many in a tile; several realizations
sharing their hard and soft maps; infinite training-image values."""
import numpy as np
import pytest

import iqhip
from test_gpu_simulate import _compare, _smooth

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("ti,tile,sim,dtype", [
    ((41, 37), (9, 7), (60, 44), np.float32),          # region staged whole, odd extents
    ((41, 41, 13), (32, 32, 8), (50, 40, 13), np.float32),  # planes
    ((40, 36, 20), (12, 10, 4), (30, 30, 12), np.float64),
    ((150, 140), (120, 118), (200, 150), np.float32),  # rows of one plane
    ((640, 9), (615, 4), (700, 9), np.float64),        # parts of a row
], ids=["whole", "planes", "volume64", "rows", "parts"])
def test_soft_and_hard_match_oracle(ti, tile, sim, dtype):
    rng = np.random.default_rng(41)
    T = _smooth(rng, ti, 5, dtype)
    aux_ti = _smooth(rng, ti, 3, dtype)
    aux = _smooth(rng, sim, 3, dtype)
    hard = {tuple(int(rng.integers(n)) for n in sim): float(rng.standard_normal()) for _ in range(7)}
    print("maps", ti, tile, flush=True)
    _compare(T, tile, sim, soft=[(aux, aux_ti)], hard=hard, nreal=2, overlap=tuple(0.25 for _ in ti), tol=0.2)


@pytest.mark.parametrize("nreal", [1, 3, 4, 17])
def test_query_counts_match_oracle(nreal):
    rng = np.random.default_rng(42)
    T = _smooth(rng, (36, 33), 5, np.float32)
    aux_ti = _smooth(rng, (36, 33), 3, np.float32)
    aux = _smooth(rng, (34, 30), 3, np.float32)
    print("maps, realizations", nreal, flush=True)
    _compare(T, (8, 9), (34, 30), soft=[(aux, aux_ti), (aux + 1, aux_ti)], nreal=nreal, overlap=(0.25, 0.25))


@pytest.mark.parametrize("npoints", [40, 700])
def test_dense_hard_data_match_oracle(npoints):
    # up to all 100 voxels of a tile: the tiled form of the hard maps
    rng = np.random.default_rng(43)
    T = _smooth(rng, (37, 40), 5, np.float64)
    hard = {(int(i % 34), int(i // 34)): float(rng.standard_normal()) for i in rng.choice(34 * 31, npoints, replace=False)}
    print("hard points", npoints, flush=True)
    _compare(T, (10, 10), (34, 31), hard=hard, nreal=2, overlap=(0.25, 0.25))


def test_infinite_image_values_match_oracle():
    # windows that hold an infinite value have a distance of NaN or infinity;
    # the padding of a voxel list must not spread them to other windows
    rng = np.random.default_rng(44)
    T = _smooth(rng, (40, 38), 5, np.float64)
    T[0, 0] = np.inf
    print("infinite value", flush=True)
    plan, _ = iqhip.make_plan(T, (9, 9), (34, 34), overlap=(0.25, 0.25), rng=np.random.default_rng(1), hard={(3, 3): 0.5})
    u = np.random.default_rng(2).random(plan.npath)
    plan.run(u)
    res = plan.results()
    assert (res["chosen"][0] != 0).all() and np.isfinite(res["grids"][0]).all()
