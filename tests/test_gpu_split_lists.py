"""Short chunk lists, whose chunks are shared out to several workgroups: the
remesh (vp_gpu_cull_mesh) and the quad mesh (vp_gpu_mesh) at the list lengths
where the share changes, against the oracle, bit-exact."""
import numpy as np
import pytest

from oracle import oracle as O
from tests import refimpl as RI
from tests.gpuutil import dev, gpu_remesh, host, ids_dev
from voxplat_amd import abi

pytestmark = pytest.mark.gpu


def _world(rb, seed=11, density=0.6):
    w = abi.WorldDesc.make(rb, (1, 1, 1))
    vox = RI.random_world(w, np.random.default_rng(seed), density)
    return w, vox, O.shadow_build(w, vox)


def _ids(w, n):
    return np.random.default_rng(n).integers(0, w.chunks, n).astype(np.uint32)


# 2 workgroups per CU: the share drops where n passes 512 / 16, 512 / 4, 512 / 2
# on 256 CUs; a chunk of edge R has at most R / 4 shares
@pytest.mark.parametrize("rb,n", [(6, 1), (6, 2), (6, 31), (6, 33), (6, 129), (6, 257), (5, 1),
                                  (5, 65), (4, 1), (4, 127), (4, 256), (4, 257), (4, 513), (3, 5),
                                  (2, 1), (2, 7)])
def test_short_lists(gpu, rb, n):
    import torch

    w, vox, smap = _world(rb)
    ids = _ids(w, n)
    recs, offs, counts = O.remesh_list(w, vox, ids, smap, threads=8)
    got = gpu_remesh(gpu, w, vox, ids, smap)
    assert got[3] == 0
    for a, b in zip(got, (recs, offs, counts)):
        assert np.array_equal(a, b)
    g, ix, fo = gpu.mesh(w, dev(vox), ids_dev(ids), dev(smap))
    torch.cuda.synchronize()
    assert gpu.status() == 0
    eg, eix, efo = O.mesh_list(w, vox, ids, smap, threads=8)
    f = int(efo[-1])
    assert np.array_equal(host(fo, np.uint64), efo)
    assert np.array_equal(host(g)[:f], eg) and np.array_equal(host(ix, np.uint32)[:f], eix)


@pytest.mark.parametrize("n", [1, 3])
def test_a_chunk_past_the_capacity_is_left_out_whole(gpu, n):
    """One record (face) too few for the last chunk: none of its parts writes."""
    import torch

    w, vox, smap = _world(6)
    ids = _ids(w, n)
    vd, sd, idd = dev(vox), dev(smap), ids_dev(ids)
    recs, offs, counts = O.remesh_list(w, vox, ids, smap, threads=8)
    total, kept = int(offs[-1]) // 4, int(offs[-2]) // 4
    out = torch.full((total, 4), -7, dtype=torch.int16, device="cuda")
    _, o, c = gpu.cull_mesh(w, vd, idd, shadow_map=sd, capacity=total - 1, records=out)
    torch.cuda.synchronize()
    assert gpu.status() == abi.VP_STATUS_OVERFLOW
    assert np.array_equal(host(o, np.uint64), offs) and np.array_equal(host(c, np.uint32), counts)
    assert np.array_equal(host(out)[:kept], recs[:kept]) and (host(out)[kept:] == -7).all()
    eg, eix, efo = O.mesh_list(w, vox, ids, smap, threads=8)
    total, kept = int(efo[-1]), int(efo[-2])
    geom = torch.full((total, 4, 4), -7, dtype=torch.int16, device="cuda")
    index = torch.full((total, 6), -7, dtype=torch.int32, device="cuda")
    fo = torch.empty(n + 1, dtype=torch.int64, device="cuda")
    gpu.mesh(w, vd, idd, sd, capacity=total - 1, out=(geom, index, fo))
    torch.cuda.synchronize()
    assert gpu.status() == abi.VP_STATUS_OVERFLOW
    assert np.array_equal(host(fo, np.uint64), efo)
    assert np.array_equal(host(geom)[:kept], eg[:kept]) and (host(geom)[kept:] == -7).all()
    assert np.array_equal(host(index, np.uint32)[:kept], eix[:kept])
    assert (host(index)[kept:] == -7).all()


def test_share_follows_the_device_count(gpu):
    """A list whose length is in device memory: each length shares as it fits."""
    import torch

    w, vox, smap = _world(6)
    ids = _ids(w, 300)
    vd, sd, idd = dev(vox), dev(smap), ids_dev(ids)
    recs, offs, counts = O.remesh_list(w, vox, ids, smap, threads=8)
    for m in (0, 1, 40, 300):
        k = int(offs[m]) // 4
        r, o, c = gpu.cull_mesh(w, vd, idd, shadow_map=sd, d_n=dev(np.array([m], np.uint32)),
                                capacity=max(k, 1))
        torch.cuda.synchronize()
        assert gpu.status() == 0
        assert np.array_equal(host(o, np.uint64)[:m + 1], offs[:m + 1])
        assert np.array_equal(host(c, np.uint32)[:m], counts[:m])
        assert np.array_equal(host(r)[:k], recs[:k])
