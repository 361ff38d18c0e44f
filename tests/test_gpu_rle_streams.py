"""RLE decode (vp_gpu_rle) where its pieces, batches and shares can go wrong:
runs around 16-byte pieces with few and many starts, streams longer than the
run values kept in LDS, words behind the terminator, streams at odd word
offsets, and list lengths around the shares of a chunk; every byte against the
runs written out."""
import numpy as np
import pytest

from tests.gpuutil import dev, host, ids_dev
from voxplat_amd import abi

pytestmark = pytest.mark.gpu


def _stream(chunk):
    """Maximal runs of a flat chunk, and the terminator."""
    at = np.concatenate([[0], np.nonzero(np.diff(chunk))[0] + 1])
    end = np.concatenate([at[1:], [len(chunk)]])
    return np.concatenate([chunk[at].astype(np.uint32) << 24 | (end - at).astype(np.uint32),
                           np.zeros(1, np.uint32)])


def _chunk(n, kind, rng):
    if kind == "fill":
        return np.full(n, 9, np.uint8)
    if kind == "alternate":               # every byte a run: past the LDS values at R = 64
        return (np.arange(n) % 2 + 3).astype(np.uint8)
    if kind == "holes":                   # 5% single-voxel holes
        return np.where(rng.random(n) < 0.05, 0, 7).astype(np.uint8)
    if kind == "mixed":                   # long runs, then 6, 7, 8, 9 starts per 16 bytes
        out = np.zeros(n, np.uint8)
        for p in range(n // 2, n - 15, 16):
            c = rng.integers(5, 10)
            cut = np.sort(rng.choice(16, c, replace=False))
            out[p:p + 16] = np.searchsorted(cut, np.arange(16), "right") + rng.integers(0, 3)
        return out
    return np.concatenate([[5], np.zeros(n - 2), [6]]).astype(np.uint8)      # the ends differ


KINDS = ["holes", "fill", "mixed", "alternate", "ends"]


@pytest.mark.parametrize("rb,n", [(6, 1), (6, 2), (6, 5), (6, 65), (6, 129), (6, 257), (6, 600),
                                  (5, 7), (4, 600), (3, 5), (2, 9)])
def test_decode_lists(gpu, rb, n):
    import torch

    b = max(n - 1, 1).bit_length()
    w = abi.WorldDesc.make(rb, (b // 3, b - 2 * (b // 3), b // 3))
    R3 = w.R ** 3
    rng = np.random.default_rng(rb * 1000 + n)
    kinds = [_chunk(R3, k, rng) for k in KINDS]
    ids = rng.permutation(w.chunks)[:n].astype(np.uint32)
    pick = [kinds[i % len(KINDS)] for i in range(n)]
    streams = [_stream(k) for k in kinds]
    # a gap of i % 3 words after stream i: odd word addresses, words never read
    parts = [np.concatenate([streams[i % len(KINDS)], np.full(i % 3, 0x01000005, np.uint32)])
             for i in range(n)]
    offs = np.concatenate([[0], np.cumsum([len(p) for p in parts])]).astype(np.uint64)
    out = torch.full((w.chunks * R3,), 0xAB, dtype=torch.uint8, device="cuda")
    gpu.rle_decode(w, dev(np.concatenate(parts)), dev(offs), ids_dev(ids), out)
    torch.cuda.synchronize()
    assert gpu.status() == 0
    got = out.view(w.chunks, R3)[torch.from_numpy(ids.astype(np.int64)).cuda()].cpu().numpy()
    for i in range(n):
        assert np.array_equal(got[i], pick[i]), f"entry {i}"
    rest = np.setdiff1d(np.arange(w.chunks), ids)
    if len(rest):
        left = out.view(w.chunks, R3)[torch.from_numpy(rest.astype(np.int64)).cuda()]
        assert bool((left == 0xAB).all())


def test_early_terminator_and_short_streams(gpu):
    """A 0 word in the middle ends a stream, in the first batch and in a later
    one; bytes past the runs read 0 and the status says so."""
    import torch

    w = abi.WorldDesc.make(6, (2, 0, 0))
    R3 = w.R ** 3
    out = dev(np.full(w.chunks * R3, 0xAB, np.uint8))
    full = _stream(_chunk(R3, "holes", np.random.default_rng(2)))
    parts = []
    for cut in (3, 5000, 4096, 8191):
        s = full.copy()
        s[cut] = 0
        parts.append(s)
    offs = np.concatenate([[0], np.cumsum([len(p) for p in parts])]).astype(np.uint64)
    gpu.rle_decode(w, dev(np.concatenate(parts)), dev(offs), ids_dev([0, 1, 2, 3]), out)
    torch.cuda.synchronize()
    assert gpu.status() == abi.VP_STATUS_BAD_RLE
    got = host(out).reshape(w.chunks, R3)
    for i, cut in enumerate((3, 5000, 4096, 8191)):
        exp = np.repeat((full[:cut] >> 24).astype(np.uint8), full[:cut] & 0xFFFFFF)
        assert np.array_equal(got[i, :len(exp)], exp) and not got[i, len(exp):].any()
