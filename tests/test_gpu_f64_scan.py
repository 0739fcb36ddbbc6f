"""Float64 training images that are not FP32-exact: the MFMA scan runs on
their FP32 rounding with a widened interval and the FP64 recheck decides, or
the exhaustive FP64 map runs; picks, cuts and grids equal the oracle's."""
import numpy as np
import pytest

import iqhip
import iqref
from test_gpu_simulate import _compare, _smooth

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("shape,tile,sim,kw", [
    ((61, 57), (13, 11), (70, 64), dict(overlap=(0.2, 0.3), path="random")),
    ((33, 29, 13), (9, 10, 5), (30, 37, 14), dict(overlap=(0.25, 0.25, 0.25), tol=0.2)),
    ((40, 40), (8, 8), (33, 41), dict(tol=1.0, path="dilation")),
], ids=["2d", "3d", "wide-band"])
def test_rounded_scan_matches_oracle(shape, tile, sim, kw):
    rng = np.random.default_rng(31)
    T = _smooth(rng, shape, 5, np.float64)
    print("float64", shape, flush=True)
    _compare(T, tile, sim, **kw)


@pytest.mark.parametrize("offset,scale", [(3.0, 1.0), (1e4, 1.0), (0.0, 1e-40), (0.0, 1e20)],
                         ids=["small-offset", "large-offset", "tiny", "huge"])
def test_offset_and_scaled_values_match_oracle(offset, scale):
    # small offset: still scanned; large offset and out-of-range values: the
    # exhaustive map
    rng = np.random.default_rng(32)
    T = (_smooth(rng, (50, 46), 5, np.float64) + offset) * scale
    print("float64 offset", offset, "scale", scale, flush=True)
    _compare(T, (11, 12), (48, 50), overlap=(0.25, 0.25))


def test_learned_proposal_still_needs_fp32_exact_values():
    rng = np.random.default_rng(33)
    plan, _ = iqhip.make_plan(_smooth(rng, (40, 40, 10), 5, np.float64), (10, 10, 4), (40, 40, 10),
                              overlap=(0.25, 0.25, 0.25))
    with pytest.raises(iqhip._lib.IQError):
        plan.learn(nsamples=256, iters=2)
