"""Exact maps on the matrix cores, bit for bit: images whose distances are
nothing but the rounding of the FP64 chains, subnormal products, infinite
values; and the plans of Float32 images that no scan takes."""
import numpy as np
import pytest

import iqhip
from test_gpu_simulate import _compare, _smooth

pytestmark = pytest.mark.gpu


def _hard(rng, sim, n):
    return {tuple(int(rng.integers(s)) for s in sim): float(rng.standard_normal()) for _ in range(n)}


@pytest.mark.parametrize("ti,tile,sim", [((43, 41), (9, 10), (50, 47)), ((24, 22, 11), (7, 8, 4), (25, 24, 10))],
                         ids=["plane", "volume"])
@pytest.mark.parametrize("kind", ["cancelling", "subnormal"])
@pytest.mark.parametrize("conditioned", [False, True], ids=["plain", "hard"])
def test_chain_order_decides_picks(ti, tile, sim, kind, conditioned):
    """cancelling: values of 1e4 + 1e-6 x, whose true distances (1e-12 a voxel)
    lie far below the rounding of A2 - 2 AB + B2 (1e-8 a voxel): the picks are
    the rounding of the chains.  subnormal: squares of about 1e-316, where a
    flushed product or partial sum changes the distance."""
    rng = np.random.default_rng(81)
    T = rng.standard_normal(ti)
    T = 1e4 + 1e-6 * T if kind == "cancelling" else 1e-158 * T
    hard = {k: float(v * 1e-158 if kind == "subnormal" else 1e4 + 1e-6 * v) for k, v in _hard(rng, sim, 9).items()}
    print(kind, ti, conditioned, flush=True)
    _compare(T, tile, sim, overlap=(0.25,) * len(ti), tol=1e-3, nreal=3, path="random",
             **(dict(hard=hard) if conditioned else {}))


@pytest.mark.parametrize("conditioned", [False, True], ids=["plain", "hard"])
@pytest.mark.parametrize("dtype", [np.float32, np.float64])
def test_infinite_value_matches_oracle(dtype, conditioned):
    """Windows that hold the infinite value have a distance of NaN or infinity;
    no other window's changes."""
    rng = np.random.default_rng(82)
    T = _smooth(rng, (40, 38), 5, dtype)
    T[0, 0] = np.inf
    print("infinite value", dtype.__name__, conditioned, flush=True)
    _compare(T, (9, 9), (34, 34), overlap=(0.25, 0.25), nreal=2, **(dict(hard={(3, 3): 0.5}) if conditioned else {}))


def test_float32_image_without_a_scan():
    """Boxes of 64 x 64 voxels do not fit the scans' LDS: the exhaustive map
    reads the image in its own type."""
    T = _smooth(np.random.default_rng(83), (71, 68, 6), 5, np.float32)
    kw = dict(overlap=(0.1, 0.05, 0.5), tol=0.2)
    plan, _ = iqhip.make_plan(T, (64, 64, 4), (120, 100, 6), rng=np.random.default_rng(1), **kw)
    assert plan.scan_tuning()[0] == (0, 0)
    plan.close()
    print("float32, exhaustive", flush=True)
    _compare(T, (64, 64, 4), (120, 100, 6), **kw)
