"""Integer training images against the oracle: codes whose FP32 distances are
exact (no FP64 recheck), codes just past that limit, codes beyond bf16 and
half-integers (interval and recheck), with wide and tied bands."""
import numpy as np
import pytest

from test_gpu_simulate import _compare, _smooth

pytestmark = pytest.mark.gpu


# tile 12 x 10, overlap 1/4: masks of up to 57 voxels (one side), 120 at most;
# 4 V m^2 reaches 2^24 at m = 200 to 290
@pytest.mark.parametrize("top", [1, 2, 100, 180, 255, 256, 300])
@pytest.mark.parametrize("dtype", [np.float32, np.float64])
def test_integer_codes_match_oracle(top, dtype):
    rng = np.random.default_rng(71)
    x = _smooth(rng, (48, 44), 5, np.float64)
    T = np.round((x - x.min()) / (x.max() - x.min()) * top).astype(dtype)
    print("codes to", top, dtype.__name__, flush=True)
    _compare(T, (12, 10), (50, 46), overlap=(0.25, 0.25), path="random", tol=0.3)


@pytest.mark.parametrize("scale", [-1.0, 0.5, 1024.0])
def test_scaled_codes_match_oracle(scale):
    rng = np.random.default_rng(72)
    T = (scale * np.digitize(_smooth(rng, (30, 28, 9), 3, np.float32), [0.0, 0.2])).astype(np.float32)
    print("scaled codes", scale, flush=True)
    _compare(T, (9, 8, 4), (30, 26, 9), overlap=(0.3, 0.3, 0.5), nreal=2, tol=1.0)
