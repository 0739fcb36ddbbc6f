"""Distance maps at the edges of the voxel groups and of the 32-bit byte offsets."""
import numpy as np
import pytest

import iqhip
import iqref

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", [np.float32, np.float64])
@pytest.mark.parametrize("nv", [0, 1, 15, 16, 17, 32, 47])  # groups of 16 voxels and their remainders
@pytest.mark.parametrize("tail", [0, 1, 255])            # candidates in the last workgroup, of 256
def test_voxel_groups_match_oracle(ctx, dtype, nv, tail):
    rng = np.random.default_rng(nv)
    kern = rng.standard_normal((6, 4, 2))
    img = rng.standard_normal((512 + tail + 5, 4, 2)).astype(dtype)
    w = np.zeros(kern.size, dtype=np.uint8)
    w[rng.choice(kern.size, nv, replace=False)] = 1
    w = w.reshape(kern.shape, order="F")
    got = iqhip.fastdistance(img, kern, w, ctx=ctx)
    assert np.array_equal(got, iqref.fastdistance(img.astype(np.float64), kern, w))


@pytest.mark.parametrize("dtype", [np.float32, np.float64])
@pytest.mark.parametrize("past", [0, 1])  # the last image below 4 GiB, the first of 4 GiB and more
def test_image_beyond_32_bit_byte_offsets(ctx, dtype, past):
    """Integer values: the sums are exact in any order."""
    nz = (1 << 32) // (128 * 128 * np.dtype(dtype).itemsize) - 1 + past
    img = np.zeros((128, 128, nz), dtype=dtype, order="F")
    rng = np.random.default_rng(past)
    for z in (0, 1, nz // 2 - 1, nz // 2, nz - 2, nz - 1):
        img[:, :, z] = rng.integers(-9, 10, (128, 128))
    kern = rng.integers(-9, 10, (127, 128, 2)).astype(np.float64)
    w = rng.random(kern.shape) < 0.01
    w[-1, -1, -1] = True
    print(img.shape, img.dtype, int(w.sum()), flush=True)
    got = iqhip.fastdistance(img, kern, w, ctx=ctx)
    for z in (0, nz // 2 - 1, nz // 2, nz // 2 + 1, nz - 2):
        for x in (0, 1):
            ref = (((img[x : x + 127, :, z : z + 2].astype(np.float64) - kern) ** 2) * w).sum()
            assert got[x, 0, z] == ref
