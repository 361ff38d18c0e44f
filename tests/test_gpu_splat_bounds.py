"""Block-culled splat frames (vp_gpu_splat_blocks) long enough for the tile
bounds to do their work: lists of tens of thousands of blocks behind a wall, so
that every wave of the raster takes many blocks, refreshes its bounds several
times, and drops blocks and splats against bounds that are filled.

ids equal the oracle's and depths bit for bit: dropping changes no result, and
both sides evaluate the same IEEE operations in the same order (tolerance 0)."""
import numpy as np
import pytest

from tests.test_gpu_splat_occlusion import _same
from voxplat_amd import workload as W

pytestmark = pytest.mark.gpu


def _box(x, y, z, keep=lambda x, y, z: x >= 0):
    z, y, x = np.meshgrid(np.arange(*z), np.arange(*y), np.arange(*x), indexing="ij")
    k = keep(x, y, z)
    return np.stack([x[k], y[k], z[k], (x[k] + y[k] + z[k]) & 63], -1).astype(np.int16)


@pytest.fixture(scope="module")
def wall():
    """4.2 M splats behind a wall with a lattice of holes and an open end: the
    hidden ones first in the list, then the wall, then a few before it."""
    hidden = _box((0, 320), (0, 160), (0, 82))
    front = _box((0, 280), (0, 160), (100, 101), lambda x, y, z: (x % 11 != 3) | (y % 13 != 5))
    near = _box((60, 260), (40, 130), (140, 141), lambda x, y, z: (x * 7 + y * 5) % 97 == 0)
    return np.concatenate([hidden, front, near])


# wider than 2^18 pixels; sides that leave remainders in the 8x8 tiles and in the
# groups of eight, and (the largest) more groups per wave than one refresh takes
@pytest.mark.parametrize("size,far", [((640, 480), 4096.0), ((1001, 517), 333.3),
                                      ((523, 1031), 1000.0), ((2049, 161), 4096.0),
                                      ((4099, 2053), 777.7)])
@pytest.mark.parametrize("pose", [
    ((150.3, 80.2, 260.7), 0.0, 0.0),        # before the wall
    ((300.6, 140.1, 190.2), -35.0, 20.0),    # from the side, past its open end
    ((40.4, 60.3, 90.0), 150.0, 5.0),        # between the wall and what it hides
])
def test_hidden_lists(gpu, wall, size, far, pose):
    assert _same(gpu, wall, W.make_camera(*pose, *size, far=far)) > 0.05


@pytest.mark.parametrize("pose", [
    ((160.0, 80.0, 250.0), 0.0, 0.0),        # along an axis from a lattice point
    ((160.0, 300.0, 60.0), 0.0, 90.0),       # straight down
])
def test_axis_rays(gpu, wall, pose):
    # odd sizes put a pixel centre on the view axis: rays with zero components
    assert _same(gpu, wall, W.make_camera(*pose, 701, 399)) > 0.05


def test_levels(gpu, wall):
    """Levels per splat, the coarse ones hidden and in front."""
    lod = (np.arange(len(wall)) // 1000 % 5).astype(np.uint8)
    cam = W.make_camera((150.3, 80.2, 260.7), 5.0, 3.0, 1001, 517)
    assert _same(gpu, wall, cam, lod) > 0.05
