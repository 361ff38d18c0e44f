"""Lists of 64^3 chunks by the shape that runs where none is set (one
1024-thread workgroup per CU) and by 512 threads, two per CU: records with and
without face flags, at the list lengths where a chunk's share changes.

Records equal the oracle's, and the face flags their definition, bit for bit
(integers: tolerance 0)."""
import numpy as np
import pytest

from oracle import oracle as O
from tests import refimpl as RI
from tests.gpuutil import dev, gpu_remesh
from voxplat_amd import abi

pytestmark = pytest.mark.gpu

R, N = 64, 65


@pytest.fixture(scope="module", params=["unset", "512x2"])
def ctx(request):
    """A context of its own: others on the session's may have set a shape."""
    from voxplat_amd import GPU

    g = GPU(0)
    if request.param == "512x2":
        g.set_remesh_shape(None, 512, 2, 4)
    yield g
    g.close()


@pytest.fixture(scope="module")
def scene():
    """2x2x2 chunks; a chunk's records and, per chunk, its records' flags."""
    w = abi.WorldDesc.make(6, (1, 1, 1))
    rng = np.random.default_rng(17)
    vox = RI.random_world(w, rng, 0.6, colours=(1, 64))
    smap = O.shadow_build(w, vox)
    world = RI.world_array(w, vox)
    return w, vox, smap, [_flags(w, world, c) for c in range(w.chunks)]


def _flags(w, world, chunk):
    """Face bits of a chunk's records: bit 2a = +a open, 2a + 1 = -a open (for
    coordinates >= 1); cells at coordinate R show the face towards the chunk;
    coarser records those of the level-0 cell their colour comes from, the
    non-zero child with the greatest (z, y, x) at each level."""
    mask = RI.closed_form_mask(w, world, chunk).reshape(N, N, N)
    ox, oy, oz = (R * v for v in RI.chunk_coords(w, chunk))
    air = np.pad(world, 1)[oz:oz + R + 2, oy:oy + R + 2, ox:ox + R + 2] == 0
    bits = np.zeros((N, N, N), np.int16)
    core = bits[:R, :R, :R]
    i = slice(1, R + 1)
    for a, (up, down) in enumerate([((i, i, slice(2, None)), (i, i, slice(0, R))),
                                    ((i, slice(2, None), i), (i, slice(0, R), i)),
                                    ((slice(2, None), i, i), (slice(0, R), i, i))]):
        low = air[down].copy()
        low[(slice(None),) * (2 - a) + (0,)] = False
        core |= (air[up] << (2 * a)).astype(np.int16) | (low << (2 * a + 1)).astype(np.int16)
    bits[:R, :R, R], bits[:R, R, :R], bits[R, :R, :R] = 2, 8, 32
    src = np.where(mask != 0, np.arange(N ** 3).reshape(N, N, N) + 1, 0)
    out = [bits.reshape(-1)[src[src != 0] - 1]]
    for l in range(1, 5):
        n = (R >> l) + 1
        pad = np.zeros((2 * n,) * 3, src.dtype)
        pad[:src.shape[0], :src.shape[1], :src.shape[2]] = src
        src = np.zeros((n,) * 3, src.dtype)
        for k in range(8):                   # ascending (dz, dy, dx): the last one stays
            child = pad[k >> 2::2, k >> 1 & 1::2, k & 1::2]
            src = np.where(child != 0, child, src)
        out.append(bits.reshape(-1)[src[src != 0] - 1])
    return np.concatenate(out)


# shares of a list: 256 (one workgroup per CU) or 512 (two) over its length, at
# most 16; 300 is past both
@pytest.mark.parametrize("n", [1, 2, 16, 17, 33, 65, 129, 257, 300])
def test_lists(ctx, scene, n):
    w, vox, smap, flags = scene
    ids = np.random.default_rng(n).integers(0, w.chunks, n).astype(np.uint32)
    vd, sd = dev(vox), dev(smap)
    recs, offs, counts = O.remesh_list(w, vox, ids, smap, threads=8)
    got = gpu_remesh(ctx, w, vd, ids, sd)
    assert got[3] == 0 and np.array_equal(got[1], offs) and np.array_equal(got[2], counts)
    assert np.array_equal(got[0], recs)
    got = gpu_remesh(ctx, w, vd, ids, sd, v2=True)
    assert got[3] == 0 and np.array_equal(got[1], offs) and np.array_equal(got[2], counts)
    raw = np.ascontiguousarray(got[0]).view(np.uint8).reshape(-1, 8)
    attr = recs[:, 3].astype(np.uint16)
    want = np.concatenate([flags[c] for c in ids])
    assert np.array_equal(got[0][:, :3], recs[:, :3])
    assert np.array_equal(raw[:, 6], (attr & 0x3F).astype(np.uint8))
    assert np.array_equal(raw[:, 7], (want | (attr & 0x40).astype(np.int16)).astype(np.uint8))
