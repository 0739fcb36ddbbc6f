"""Hard-data maps of plans whose tiles hold few points and many: each tile's
map is made by the kernel for its number of points."""
import numpy as np
import pytest

from test_gpu_simulate import _compare, _smooth

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [3, 4, 6, 10])  # blocks of 9 to 100 points; the line is at 11 for this tile
def test_sparse_and_dense_tiles_match_oracle(n):
    rng = np.random.default_rng(45)
    T = _smooth(rng, (37, 40), 5, np.float32)
    hard = {tuple(int(rng.integers(n)) for n in (50, 44)): float(rng.standard_normal()) for _ in range(9)}
    hard.update({(21 + i, 12 + j): float(rng.standard_normal()) for i in range(n) for j in range(n)})
    print("dense block of", n * n, "points", flush=True)
    _compare(T, (10, 10), (50, 44), hard=hard, nreal=2, overlap=(0.25, 0.25))


def test_sparse_and_dense_volume_match_oracle():
    rng = np.random.default_rng(46)
    T = _smooth(rng, (30, 28, 14), 5, np.float64)
    hard = {tuple(int(rng.integers(n)) for n in (30, 30, 12)): float(rng.standard_normal()) for _ in range(12)}
    hard.update({(12 + i, 13 + j, 2 + k): float(rng.standard_normal()) for i in range(7) for j in range(7) for k in range(3)})
    print("dense block in a volume", flush=True)
    _compare(T, (9, 8, 5), (30, 30, 12), hard=hard, nreal=3, overlap=(0.25, 0.25, 0.25))
