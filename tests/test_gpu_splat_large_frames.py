"""Block-culled splat frames past the size up to which the tile bounds are left
out (2^18 pixels), where near blocks are handed out in quarters: frame sizes
around that limit and around the 8x8 tiles, near and far cameras, short lists,
mixed levels.

Both paths evaluate the same IEEE operations per fragment as the oracle, so ids
and depths are equal bit for bit (tolerance 0)."""
import numpy as np
import pytest

from tests.test_gpu_splat_occlusion import _same, lists  # noqa: F401
from voxplat_amd import workload as W

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("size", [(512, 512), (513, 512), (2101, 129), (131, 2049), (640, 481)])
@pytest.mark.parametrize("mixed", [False, True])
def test_frame_sizes(gpu, lists, size, mixed):  # noqa: F811
    recs, lod = lists
    pick = np.ones(len(lod), bool) if mixed else lod == 0
    cam = W.make_camera((120.3, 95.7, 150.2), 10.0, 35.0, *size)
    assert _same(gpu, recs[pick], cam, lod[pick] if mixed else None) > 0.0


@pytest.mark.parametrize("far", [4096.0, 333.3, 50.0])
@pytest.mark.parametrize("pose", [
    ((128.0, 20.0, 64.0), 90.0, 0.0),        # inside the terrain: every block is near
    ((-900.0, 300.0, 64.0), 90.0, 15.0),     # far outside: no block is near
    ((30.5, 70.0, 110.0), 135.0, 12.0),      # just above the surface, grazing
])
def test_near_and_far_blocks(gpu, lists, far, pose):  # noqa: F811
    recs, lod = lists
    _same(gpu, recs[lod == 0], W.make_camera(*pose, 521, 507, far=far))


@pytest.mark.parametrize("n", [1, 64, 65, 255, 257, 1000])
def test_short_lists(gpu, lists, n):  # noqa: F811
    recs, lod = lists
    l0 = recs[lod == 0]
    cam = W.make_camera((120.3, 95.7, 150.2), 10.0, 35.0, 700, 400)
    _same(gpu, l0[len(l0) // 2:len(l0) // 2 + n], cam)
