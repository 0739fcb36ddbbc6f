"""Float64 images that the MFMA scan takes rounded to FP32: the superset its
interval leaves to the FP64 recheck, at scales far below one."""
import numpy as np
import pytest

import iqhip
from test_gpu_simulate import _compare, _smooth

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("power", [0, -1, -40, -60, -80])
def test_superset_stays_near_the_band(power):
    """The interval is a share of about 2^-12 of the distances at every scale;
    where it exceeds them every window is a member.  (Picks differ between
    scales: the cut's weights hold an absolute 2^-52.)"""
    T = _smooth(np.random.default_rng(71), (61, 57), 5, np.float64)
    T *= 1.5 / np.abs(T).max()
    T[np.abs(T) < 2.0 ** -18] = 0.0  # stays in the scan's range at every scale
    print("scale 2 **", power, flush=True)
    plan, _ = iqhip.make_plan(np.ldexp(T, power), (13, 11), (70, 64), overlap=(0.2, 0.3), rng=np.random.default_rng(1))
    plan.run(np.random.default_rng(2).random((1, plan.npath)))
    queries, members, band = plan.select_stats()
    plan.close()
    assert queries > 0 and members < 2 * band + queries


@pytest.mark.parametrize("scale", [1e-9, 1e-18, 1e-24])
def test_small_values_match_oracle(scale):
    T = _smooth(np.random.default_rng(72), (33, 29, 13), 5, np.float64) * scale
    print("scale", scale, flush=True)
    _compare(T, (9, 10, 5), (30, 37, 14), overlap=(0.25, 0.25, 0.25))


@pytest.mark.parametrize("nreal", [1, 70])  # a wavefront per 16 candidates, and fewer
def test_wide_superset_matches_oracle(nreal):
    T = np.random.default_rng(73).standard_normal((60, 57))
    print("white noise, realizations", nreal, flush=True)
    _compare(T, (8, 8), (20, 22), overlap=(0.25, 0.25), tol=1.0, nreal=nreal)


@pytest.mark.parametrize("offset,scanned", [(2000.0, False), (0.0, True), (0.2, True)], ids=["depth", "centred", "porosity"])
def test_inactive_voxels_do_not_hide_an_offset(offset, scanned):
    """The zeros in place of inactive voxels make the variance of a far-off
    image look large; no window that counts holds one."""
    T = _smooth(np.random.default_rng(74), (64, 61), 5, np.float64)
    T = offset + (50.0 if offset > 1 else 0.05) * T / T.std()
    T[:14, :20] = np.nan
    kw = dict(overlap=(0.2, 0.25))
    plan, _ = iqhip.make_plan(T, (13, 12), (70, 64), rng=np.random.default_rng(1), **kw)
    plan.run(np.random.default_rng(2).random((1, plan.npath)))
    queries, members, band = plan.select_stats()
    plan.close()
    assert queries > 0 and band > 0 and (members > 0) == scanned  # the exhaustive map counts no superset
    print("offset", offset, flush=True)
    _compare(T, (13, 12), (70, 64), **kw)
