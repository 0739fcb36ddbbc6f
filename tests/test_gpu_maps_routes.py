"""Exact maps gathered and on the matrix cores (IQHIP_MAPS; the default goes by
the work of a batch), each through whole simulations against the oracle."""
import numpy as np
import pytest

from test_gpu_simulate import _compare, _smooth

pytestmark = pytest.mark.gpu


@pytest.fixture(params=["gather", "matrix"])
def route(request, monkeypatch):
    monkeypatch.setenv("IQHIP_MAPS", request.param)
    return request.param


@pytest.mark.parametrize("ti,tile,sim,dtype", [
    ((41, 37), (9, 7), (60, 44), np.float32),               # region staged whole, odd extents, 63 voxels
    ((30, 31), (8, 8), (34, 30), np.float64),               # 64 voxels
    ((41, 41, 13), (32, 32, 8), (50, 40, 13), np.float32),  # planes; lists of several thousand voxels
    ((40, 36, 20), (12, 10, 4), (30, 30, 12), np.float64),
    ((150, 140), (120, 118), (200, 150), np.float32),       # rows of one plane
    ((640, 9), (615, 4), (700, 9), np.float64),             # parts of a row
], ids=["whole", "full", "planes", "volume64", "rows", "parts"])
def test_soft_and_hard_match_oracle(route, ti, tile, sim, dtype):
    rng = np.random.default_rng(47)
    T = _smooth(rng, ti, 5, dtype)
    aux_ti, aux = _smooth(rng, ti, 3, dtype), _smooth(rng, sim, 3, dtype)
    hard = {tuple(int(rng.integers(n)) for n in sim): float(rng.standard_normal()) for _ in range(7)}
    print("maps", route, ti, tile, flush=True)
    _compare(T, tile, sim, soft=[(aux, aux_ti)], hard=hard, nreal=2, overlap=tuple(0.25 for _ in ti), tol=0.2)


@pytest.mark.parametrize("nreal", [1, 3, 4, 17])
@pytest.mark.parametrize("dtype", [np.float32, np.float64])
def test_query_counts_match_oracle(route, nreal, dtype):
    rng = np.random.default_rng(48)
    T = _smooth(rng, (36, 33), 5, dtype)
    aux_ti, aux = _smooth(rng, (36, 33), 3, dtype), _smooth(rng, (34, 30), 3, dtype)
    print("maps", route, "realizations", nreal, flush=True)
    _compare(T, (8, 9), (34, 30), soft=[(aux, aux_ti), (aux + 1, aux_ti)], nreal=nreal, overlap=(0.25, 0.25))


@pytest.mark.parametrize("ti,tile,sim", [((43, 41), (9, 10), (50, 47)), ((24, 22, 11), (7, 8, 4), (25, 24, 10))],
                         ids=["plane", "volume"])
@pytest.mark.parametrize("kind", ["cancelling", "subnormal"])
@pytest.mark.parametrize("conditioned", [False, True], ids=["plain", "hard"])
def test_chain_order_decides_picks(route, ti, tile, sim, kind, conditioned):
    """Distances that are nothing but the rounding of the FP64 chains, and
    subnormal products."""
    rng = np.random.default_rng(84)
    scale, off = (1e-6, 1e4) if kind == "cancelling" else (1e-158, 0.0)
    T = off + scale * rng.standard_normal(ti)
    hard = {tuple(int(rng.integers(s)) for s in sim): off + scale * float(rng.standard_normal()) for _ in range(9)}
    print(route, kind, ti, conditioned, flush=True)
    _compare(T, tile, sim, overlap=(0.25,) * len(ti), tol=1e-3, nreal=3, path="random",
             **(dict(hard=hard) if conditioned else {}))


def test_infinite_and_inactive_values_match_oracle(route):
    rng = np.random.default_rng(85)
    T = _smooth(rng, (40, 38), 5, np.float64)
    T[0, 0] = np.inf
    T[20:23, 17:19] = np.nan
    print(route, "infinite and inactive values", flush=True)
    _compare(T, (9, 9), (34, 34), overlap=(0.25, 0.25), nreal=2, hard={(3, 3): 0.5})
