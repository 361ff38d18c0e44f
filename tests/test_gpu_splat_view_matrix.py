"""Block-culled splat frames (vp_gpu_splat_blocks) of cameras whose view
translation is not a plain translation: far from the origin its rounding is
many times that of a translation, so a splat near the eye at the edge of the
view volume must not be judged by margins made for a translation.

ids equal the oracle's and depths bit for bit: both sides evaluate the same
IEEE operations in the same order (tolerance 0)."""
import math

import numpy as np
import pytest

from tests.test_gpu_splat_occlusion import _same
from voxplat_amd import workload as W

pytestmark = pytest.mark.gpu


def _camera(loc, yaw, pitch, width, height):
    """make_camera's pose with the rotation in the view translation."""
    cam = W.make_camera(loc, yaw, pitch, width, height)
    P = W._perspective(math.radians(70.0), width / height, 0.1, 4096.0)
    turn = W._rotation(math.radians(pitch), (1, 0, 0)) @ W._rotation(math.radians(yaw), (0, 1, 0))
    for m, to in ((turn @ W._translation([-v for v in loc]), cam.view_translation),
                  (P, cam.proj_view_rot), (np.linalg.inv(P), cam.inv_proj_view_rot)):
        for i, v in enumerate(W._colmajor(m)):
            to[i] = v
    return cam


# splats inside the volume by the stated operation order, outside it by more
# than 1e-4 w + 1e-3 where the sums are fused
@pytest.mark.parametrize("loc,yaw,pitch,at", [
    ((32515.3, 201.2, 32476.2), 144.0, 23.0, (32519, 186, 32484)),
    ((32551.2, 140.1, 32224.0), 342.0, -20.0, (32541, 145, 32221)),
    ((32173.4, 176.9, 32092.4), 285.0, 57.0, (32164, 172, 32083)),
    ((32424.1, 346.8, 32003.8), 328.0, -22.0, (32387, 340, 31994)),
    ((32050.5, 369.3, 32439.4), 211.0, 42.0, (32050, 361, 32441)),
])
def test_a_splat_at_the_edge_of_the_view_is_drawn(gpu, loc, yaw, pitch, at):
    cam = _camera(loc, yaw, pitch, 700, 400)
    assert _same(gpu, np.array([[*at, 5]], np.int16), cam) > 0.0


@pytest.mark.parametrize("size", [(700, 400), (90, 70)])
def test_a_scene_through_a_rotated_view(gpu, size):
    z, y, x = np.mgrid[-24:24, -4:4, -24:24]
    keep = (x * 7 + y * 3 + z * 5) % 4 != 0
    lst = np.stack([x[keep] + 32500, y[keep] + 100, z[keep] + 32500, (x[keep] & 63)], -1)
    cam = _camera((32500.3, 121.7, 32497.1), 30.0, 40.0, *size)
    assert _same(gpu, lst.astype(np.int16), cam) > 0.1
