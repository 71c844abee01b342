"""GPU check of a tiled gather with more tiles than one launch takes."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

gtn = pytest.importorskip("grassmanntn_amd")


def test_tiles_beyond_one_launch():
    """(17, r, 17) transposed: four tiles a pair of the outer legs, 2^23 + 64 of them, 2^23 a launch; moved
    values are bitwise equal."""
    from grassmanntn_amd._device import DeviceArray
    from test_gather_grids import _transpose
    shape = (17, (1 << 21) + 16, 17)
    n = int(np.prod(shape))
    src = (np.arange(n, dtype=np.uint32) * np.uint32(2654435761) >> np.uint32(9)).astype(np.float32).reshape(shape)
    got = _transpose(shape, (2, 1, 0)).run(DeviceArray.from_numpy(src)).numpy()
    assert got.shape == shape[::-1]
    for i in range(shape[2]):
        assert np.array_equal(got[i], src[:, :, i].T), i
