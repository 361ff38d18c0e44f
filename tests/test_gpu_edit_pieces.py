"""Sphere edits (vp_gpu_edit_spheres) over the 16-byte pieces of a row: radii
from none to more than a chunk, spheres across chunk and world borders, at the
kept bottom rows and overlapping in list order, every chunk edge, against the
edit's definition voxel by voxel."""
import numpy as np
import pytest

from tests.gpuutil import dev, host
from voxplat_amd import abi

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("rb,mb", [(2, (3, 2, 2)), (3, (2, 2, 2)), (4, (2, 1, 2)), (5, (1, 1, 1)),
                                   (6, (1, 0, 1))])
def test_spheres_of_all_sizes(gpu, rb, mb):
    import torch

    w = abi.WorldDesc.make(rb, mb)
    R = w.R
    rng = np.random.default_rng(rb)
    X, Y, Z = ((1 << b) * R for b in mb)
    world = rng.integers(0, 5, (Z, Y, X)).astype(np.uint8)
    spheres = [abi.Sphere(int(rng.integers(-8, X + 8)), int(rng.integers(-8, Y + 8)),
                          int(rng.integers(-8, Z + 8)), int(r), int(rng.integers(0, 60)))
               for r in (0, 1, 2, 3, 4, 7, 8, 9, 15, 16, 17, 31, 32, 33, 70)[::-1]]
    spheres += [abi.Sphere(8, 3, 8, 5, 9), abi.Sphere(16, 16, 16, 8, 0), abi.Sphere(15, 2, 17, 8, 7)]

    def chunks(v):
        mx, my, mz = (1 << b for b in mb)
        return np.ascontiguousarray(v.reshape(mz, R, my, R, mx, R).transpose(0, 2, 4, 1, 3, 5)).reshape(-1)
    vd = dev(chunks(world))
    gpu.edit_spheres(w, vd, spheres)
    torch.cuda.synchronize()
    z, y, x = np.mgrid[0:Z, 0:Y, 0:X].astype(np.int64)
    for s in spheres:
        inside = (x - s.cx) ** 2 + (y - s.cy) ** 2 + (z - s.cz) ** 2 < s.radius ** 2
        world[inside & (y >= 2)] = s.voxel
    assert np.array_equal(host(vd), chunks(world))
