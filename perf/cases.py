"""Performance cases of the voxel pipeline: what a program built on it has it do.

A case names a kind of call, a world and the call's sizes.  `prepare` makes the
world and what such a program keeps (buffers, node lists, a captured frame),
`run` is one pass through the public entry points, `work` the bytes that pass
cannot do without, `exact` the computed (floating) outputs in 64 bits.

Worlds are the generator's seeded terrain with 5% caves; a world is given by
its chunk edge (root), chunk counts per axis (bx, by, bz, as powers of two) and
the highest column (hmax).

    python -c "from perf import cases; print(cases.listed())"
"""
from __future__ import annotations

import math

import numpy as np
import torch

from voxplat_amd import GPU, RemeshGraph, abi, frustum_planes
from voxplat_amd import splat_fit as SF
from voxplat_amd import workload as W
from voxplat_amd.world_frame import Frame, ResidentWorld, locality_order

DEV = "cuda"


def _world(root, bx, by, bz, hmin=0, hmax=255, period=256):
    return {"root": root, "bx": bx, "by": by, "bz": bz, "hmin": hmin, "hmax": hmax,
            "period": period}


# one 64^3 chunk; 1024x256x1024; 2048x256x2048; 4096x512x4096 voxels
_ONE = _world(6, 0, 0, 0, 8, 56, 64)
_W1K = _world(6, 4, 2, 4)
_W2K = _world(6, 5, 2, 5)
_W4K = _world(6, 6, 3, 6)


def listed():
    return [
        # one edited chunk remeshed by itself: the drop-in per-chunk call, where latency counts
        dict(name="remesh_chunk", kind="remesh", edits=0, v2=False, order="index", tuned=False,
             **_ONE),
        # a player's few edits: the dozen or so chunks they touch, in index order
        dict(name="remesh_edit", kind="remesh", edits=4, v2=False, order="index", tuned=False,
             **_W2K),
        # a whole small world with the records that carry face flags
        dict(name="remesh_v2", kind="remesh", edits=0, v2=True, order="index", tuned=False,
             **_W1K),
        # a whole large world, scheduled and tuned as the benchmark does it, replayed as a graph
        dict(name="remesh_world", kind="remesh", edits=0, v2=False, order="locality", tuned=True,
             **_W4K),
        # the quad mesh of the chunks around a camera
        dict(name="mesh_near", kind="mesh", reach=2, **_W2K),
        # the quad mesh of every chunk
        dict(name="mesh_world", kind="mesh", reach=0, **_W1K),
        # reopening every chunk of a compressed world
        dict(name="decode_world", kind="decode", part=1.0, **_W2K),
        # a frame of chunk management: a burst of edits, then the dirty chunks
        # remeshed and all others compressed (the 10,000 edits per 524,288
        # chunks of the full-size world, at this world's size)
        dict(name="edit_frame", kind="frame", edits=80, **_W2K),
        # the octree's node buffers of all levels after a full remesh
        dict(name="nodes_world", kind="nodes", **_W2K),
        # one frame of the whole level-0 list at 1080p, shaded
        dict(name="splat_1080p", kind="splat", width=1920, height=1080, rgb=True, **_W2K),
        # one frame with the level of detail selected per node, at 1080p
        dict(name="lod_frame_1080p", kind="lod", width=1920, height=1080, **_W2K),
        # a colour-fit step: 16 views forward and backward
        dict(name="fit_16x512", kind="fit", views=16, size=512, **_W1K),
    ]


def draw(rng):
    def log_int(lo, hi):
        return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))

    def world(most):
        """A world of up to 2^most chunks of 64^3, or, one time in four, of as
        many chunks or more of 16^3 or 32^3."""
        bits = rng.randint(0, most)
        by = min(rng.randint(max(0, bits - 12), 3), bits)
        bx = rng.randint(max(0, bits - by - 6), min(6, bits - by))
        bz = bits - by - bx
        root = 6
        if rng.random() < 0.25:
            root = rng.choice([4, 5])
            bx, bz = min(bx + 6 - root, 7), min(bz + 6 - root, 7)
        return terrain(root, bx, by, bz)

    def scene():
        """A world wide enough to look at: 512 to 2048 voxels across."""
        root = rng.choice([5, 6, 6, 6])
        side = [rng.randint(9, 11) - root for _ in range(2)]
        return terrain(root, side[0], rng.randint(0, 2) + 6 - root, side[1])

    def terrain(root, bx, by, bz):
        top = (1 << by) << root
        return _world(root, bx, by, bz, 0, rng.randint(max(4, top // 2), min(top, 512) - 1),
                      rng.choice([64, 128, 256]))

    kind = rng.choice(["remesh", "remesh", "remesh", "mesh", "decode", "encode", "frame", "nodes",
                       "splat", "lod", "fit"])
    c = {"kind": kind}
    if kind == "remesh":
        c.update(edits=rng.choice([0, log_int(1, 200)]), v2=rng.random() < 0.25,
                 order=rng.choice(["index", "locality"]), tuned=False, **world(13))
    elif kind == "mesh":
        c.update(reach=rng.choice([0, rng.randint(1, 4)]), **world(11))
    elif kind in ("decode", "encode"):
        c.update(part=round(math.exp(rng.uniform(math.log(0.02), 0.0)), 3), **world(13))
    elif kind == "frame":
        c.update(edits=log_int(1, 300), **world(12))
    elif kind == "nodes":
        c.update(**world(12))
    elif kind in ("splat", "lod"):
        w = log_int(160, 2600)
        c.update(width=w, height=max(90, int(w * rng.uniform(0.5, 1.1)) | 1), **scene())
        if kind == "splat":
            c["rgb"] = rng.random() < 0.5
    else:
        c.update(views=rng.randint(1, 24), size=rng.randint(64, 512), **scene())
    return c


# ---- inputs ------------------------------------------------------------------
def _resident(gpu, c, seed):
    if c["kind"] == "fit":                # one scene; the seed draws colours, targets and views
        seed = 4
    cfg = W.WorldConfig("case", c["root"], (c["bx"], c["by"], c["bz"]), W.SEED_BASE + seed,
                        c["period"], c["hmin"], c["hmax"])
    world = ResidentWorld(gpu, cfg, DEV)
    world.generate()
    return world


def _top(world):
    """The height of a column of the world, for the camera poses."""
    w = world.w
    cols = world.voxels.view(1 << w.max_bitw[2], 1 << w.max_bitw[1], 1 << w.max_bitw[0], w.R, w.R,
                             w.R)

    def top(x, z):
        col = cols[z // w.R, :, x // w.R, z % w.R, :, x % w.R].reshape(-1)
        nz = torch.nonzero(col).reshape(-1)
        return int(nz.max().item()) + 1 if nz.numel() else 0
    return top


def _poses(world, n, seed):
    """Seeded poses over the terrain (location, yaw, pitch), as the benchmark's
    but turned towards the world's middle, so that small worlds are in view."""
    X, _, Z = world.w.size
    rng, top = np.random.default_rng(seed), _top(world)
    out = []
    for _ in range(n):
        x, z = float(rng.uniform(0.125, 0.875) * X), float(rng.uniform(0.125, 0.875) * Z)
        y = top(int(x), int(z)) + rng.uniform(64.0, min(512.0, 0.25 * (X + Z)))
        yaw = math.degrees(math.atan2(X / 2 - x, z - Z / 2)) + rng.uniform(-40.0, 40.0)
        out.append(((x, float(y), z), float(yaw), float(rng.uniform(10.0, 60.0))))
    return out


def _all_ids(w):
    return torch.arange(w.chunks, dtype=torch.int32, device=DEV)


def _columns(c, floor=0.65):
    """Voxels under the terrain, at most: columns times the highest column, or
    `floor` of it where the world is wide enough for its mean to hold."""
    X, Z = (1 << c["bx"]) << c["root"], (1 << c["bz"]) << c["root"]
    wide = X * Z >= 16 * c["period"] ** 2
    return X * Z, X * Z * (c["hmax"] + 1) * (floor if wide else 1.0)


def _room(c, least, per_voxel, per_column):
    """Rows of an output buffer a program sets aside: a bound from the world's
    sizes, so that it does not depend on the seed, or `least` if that is more.
    Small chunks hold more seam cells."""
    cols, vox = _columns(c)
    seams = 1.0 + 6.0 / (1 << c["root"])
    edits = 18000 * c.get("edits", 0)      # the shells of a burst's spheres
    return max(int(seams * (per_voxel * vox + per_column * cols)) + edits + 4096, least)


# with 5% caves about a quarter of the solid voxels are exposed and the coarser
# levels add half as many; a cave is six faces and two runs
_RECORDS, _FACES, _WORDS = (0.42, 6.0), (0.31, 6.0), (0.125, 6.0)


def _level0(world):
    recs, offs, _ = world.gpu.cull_mesh(world.w, world.voxels, _all_ids(world.w),
                                        shadow_map=world.smap, uniform=world.uniform, lod=False)
    return recs[:int(offs[-1].item()) // 4].contiguous()


def prepare(case, seed):
    gpu = GPU(0)
    world = _resident(gpu, case, seed)
    w, vox, uni, smap = world.w, world.voxels, world.uniform, world.smap
    st = {"case": case, "gpu": gpu, "world": world}
    kind = case["kind"]
    if kind == "remesh":
        ids = _all_ids(w)
        if case["edits"]:
            world.edit(W.edit_burst(w, n=case["edits"], seed=seed))
            ids = world.lists()[0]
        if case["order"] == "locality":
            ids, _, _ = locality_order(gpu, w, vox, ids, smap, uni)
        _, offs, counts = gpu.cull_mesh(w, vox, ids, shadow_map=smap, uniform=uni, v2=case["v2"],
                                        count_only=True)
        n = int(offs[-1].item()) // 4
        recs = torch.zeros((_room(case, n, *_RECORDS), 4), dtype=torch.int16, device=DEV)
        # buffers for a list of any length
        offs = torch.zeros(w.chunks + 1, dtype=torch.int64, device=DEV)
        counts = torch.zeros((w.chunks, 5), dtype=torch.int32, device=DEV)
        st.update(ids=ids, offs=offs, counts=counts, recs=recs, n=n, graph=None)
        if case["tuned"]:
            gpu.autotune_remesh(w, vox, ids, smap, recs, n, offs, counts, uniform=uni, reps=2)
            st["graph"] = RemeshGraph(gpu, w, vox, ids, smap, offs, counts, recs, n, uniform=uni)
    elif kind == "mesh":
        ids = _all_ids(w)
        if case["reach"]:
            rng = np.random.default_rng(seed)
            at = [int(rng.integers(0, 1 << b)) for b in w.max_bitw]
            near = torch.ones(w.chunks, dtype=torch.bool, device=DEV)
            shift = {0: 0, 2: w.max_bitw[0] + w.max_bitw[1]}
            for a in (0, 2):
                pos = (ids >> shift[a]) & ((1 << w.max_bitw[a]) - 1)
                near &= (pos - at[a]).abs() <= case["reach"]
            ids = ids[near].contiguous()
        _, _, offs = gpu.mesh(w, vox, ids, smap, uniform=uni, count_only=True)
        n = int(offs[-1].item())
        box = dict(case)                  # the columns the list can reach
        for a in ("bx", "bz"):
            if case["reach"]:
                box[a] = min(case[a], (2 * case["reach"]).bit_length())
        room = _room(box, n, *_FACES)
        st.update(ids=ids, n=n, out=(torch.zeros((room, 4, 4), dtype=torch.int16, device=DEV),
                                     torch.zeros((room, 6), dtype=torch.int32, device=DEV),
                                     torch.zeros(w.chunks + 1, dtype=torch.int64, device=DEV)))
    elif kind in ("decode", "encode"):
        g = torch.Generator().manual_seed(seed)
        n = max(1, int(w.chunks * case["part"]))
        ids = torch.randperm(w.chunks, generator=g)[:n].sort().values.to(torch.int32).to(DEV)
        words, offs, idle = gpu.rle_encode(w, vox, ids)
        if kind == "encode":
            words = torch.zeros(_room(case, int(words.numel()), *_WORDS), dtype=torch.int32,
                                device=DEV)
        st.update(ids=ids, words=words, offs=offs, idle=idle)
        if kind == "decode":
            vox.view(w.chunks, -1).index_fill_(0, ids.long(), 0)
    elif kind == "frame":
        _, offs, _ = gpu.cull_mesh(w, vox, _all_ids(w), shadow_map=smap, uniform=uni,
                                   count_only=True)
        _, woffs, _ = gpu.rle_encode(w, vox, _all_ids(w), count_only=True)
        fr = Frame(world, _room(case, int(offs[-1].item()) // 4, *_RECORDS),
                   _room(case, int(woffs[-1].item()), *_WORDS))
        g = fr.graph
        for t in (g.dirty_ids, g.idle_ids, g.splats, g.words, g.idle_uniform):
            t.zero_()
        st.update(frame=fr, spheres=W.edit_burst(w, n=case["edits"], seed=seed))
    elif kind in ("nodes", "lod"):
        recs, offs, counts = gpu.cull_mesh(w, vox, _all_ids(w), shadow_map=smap, uniform=uni)
        nodes = gpu.svl_nodes_all(w, recs, _all_ids(w), offs, counts)
        room = [_room(case, 0, *_RECORDS) // k for k in (1, 2, 8, 32, 64)]
        nodes = [(torch.zeros((max(room[l], int(o[-1].item())), 4), dtype=torch.int16, device=DEV),
                  o) for l, (_, o) in enumerate(nodes)]
        gpu.svl_nodes_all(w, recs, _all_ids(w), offs, counts, out=nodes)
        st.update(ids=_all_ids(w), recs=recs, offs=offs, counts=counts, nodes=nodes)
        if kind == "lod":
            loc, yaw, pitch = _poses(world, 1, seed)[0]
            size = (case["width"], case["height"])
            caps = [int(o[-1].item()) for _, o in nodes]
            st.update(loc=loc, cam=W.make_camera(loc, yaw, pitch, *size),
                      planes=frustum_planes(W.make_view_projection(loc, yaw, pitch, *size)),
                      cap=max(sum(caps[:2]), 1), draws=sum(abi.node_count(w, l) for l in range(5)))
            st.update(recs=None, offs=None, counts=None)
    elif kind == "splat":
        loc, yaw, pitch = _poses(world, 1, seed)[0]
        H, Wd = case["height"], case["width"]
        lst = _level0(world)
        rgb = torch.empty((H, Wd, 3), dtype=torch.float32, device=DEV) if case["rgb"] else None
        st.update(list=lst, bounds=gpu.splat_bounds(lst), cam=W.make_camera(loc, yaw, pitch, Wd, H),
                  out=(torch.empty((H, Wd), dtype=torch.float32, device=DEV),
                       torch.empty((H, Wd), dtype=torch.int32, device=DEV), rgb, None))
        gpu.reserve(0, Wd * H)
    else:
        lst = _level0(world)
        n, V, S = int(lst.shape[0]), case["views"], case["size"]
        g = torch.Generator(device=DEV).manual_seed(seed)
        st.update(list=lst, bounds=gpu.splat_bounds(lst),
                  cams=[W.make_camera(*p, S, S) for p in _poses(world, V, seed)],
                  target=torch.rand((V, S, S, 3), generator=g, device=DEV),
                  rgb=torch.rand((n, 3), generator=g, device=DEV).requires_grad_(True))
    return st


# ---- one pass ----------------------------------------------------------------
def run(st):
    case, gpu, world = st["case"], st["gpu"], st["world"]
    w, kind = world.w, case["kind"]
    if kind == "remesh":
        if st["graph"] is not None:
            st["graph"].launch()
        else:
            gpu.cull_mesh(w, world.voxels, st["ids"], shadow_map=world.smap, uniform=world.uniform,
                          v2=case["v2"], capacity=st["n"], out=(st["offs"], st["counts"]),
                          records=st["recs"])
        return {"records": st["recs"], "offsets": st["offs"], "counts": st["counts"]}
    if kind == "mesh":
        geom, index, offs = gpu.mesh(w, world.voxels, st["ids"], world.smap, uniform=world.uniform,
                                     capacity=st["n"], out=st["out"])
        return {"geometry": geom, "index": index, "offsets": offs}
    if kind == "decode":
        world.open(st["ids"], st["words"], st["offs"], st["idle"])
        return {"voxels": world.voxels, "uniform": world.uniform}
    if kind == "encode":
        words, offs, idle = gpu.rle_encode(w, world.voxels, st["ids"],
                                           out=(st["words"], st["offs"], st["idle"]))
        return {"words": words, "offsets": offs, "uniform": idle}
    if kind == "frame":
        fr = st["frame"]
        world.edit(st["spheres"])
        fr.run()
        g = fr.graph
        return {"records": g.splats, "offsets": g.offsets, "level_counts": g.level_counts,
                "dirty": g.dirty_ids, "idle": g.idle_ids, "counts": g.counts, "words": g.words,
                "word_offsets": g.word_offsets, "idle_uniform": g.idle_uniform,
                "voxels": world.voxels, "uniform": world.uniform, "map": world.smap}
    if kind == "nodes":
        out = gpu.svl_nodes_all(w, st["recs"], st["ids"], st["offs"], st["counts"], out=st["nodes"])
        return {"records": [r for r, _ in out], "offsets": [o for _, o in out]}
    if kind == "lod":
        depth, ids, drawn = gpu.draw_frame(w, [r for r, _ in st["nodes"]],
                                           [o for _, o in st["nodes"]], st["planes"], st["loc"],
                                           st["cam"], st["draws"], st["cap"])
        return {"depth": depth, "ids": ids, "drawn": drawn}
    if kind == "splat":
        depth, ids, rgb, _ = gpu.splat(st["list"], st["cam"], rgb=case["rgb"], out=st["out"],
                                       bounds=st["bounds"])
        return {"depth": depth, "ids": ids, "rgb": rgb}
    rgb = st["rgb"]
    rgb.grad = None
    img = SF.render_views(gpu, rgb, st["list"], st["cams"], bounds=st["bounds"])
    ((img - st["target"]) ** 2).mean().backward()
    return {"image": img.detach(), "grad": rgb.grad}


# ---- the bytes of a pass -------------------------------------------------------
def _map_bytes(w):
    sx, sz = w.shadow_dims()
    return 2 * sx * sz


def work(case):
    st = prepare(case, 1)
    w, kind, world = st["world"].w, case["kind"], st["world"]
    R = w.R
    uni = world.uniform
    if kind == "remesh":
        # mixed chunks and three halo planes, the map rows over the chunks, the records
        n = int(st["ids"].numel())
        mixed = int((uni[st["ids"].long()] < 0).sum())
        share = min(1.0, n / w.chunks)
        b = mixed * (R ** 3 + 3 * R * R) + share * _map_bytes(w) + 8 * st["n"] + 28 * n
    elif kind == "mesh":
        n = int(st["ids"].numel())
        mixed = int((uni[st["ids"].long()] < 0).sum())
        b = mixed * (R + 2) ** 3 + min(1.0, n / w.chunks) * _map_bytes(w) + 56 * st["n"] + 8 * n
    elif kind in ("decode", "encode"):
        n = int(st["ids"].numel())
        b = n * R ** 3 + 4 * int(st["offs"][-1].item()) + 10 * n
    elif kind == "frame":
        run(st)
        fr = st["frame"]
        fr.sync()
        nd, ni = int(fr.dirty.numel()), int(fr.idle.numel())
        mixed = int((world.uniform[fr.dirty.long()] < 0).sum())
        mixed_idle = int((world.uniform[fr.idle.long()] < 0).sum())
        b = mixed * (R ** 3 + 3 * R * R) + 8 * fr.records + 28 * nd + mixed_idle * R ** 3 + \
            4 * fr.words_n + 10 * ni
        # the edits write the voxels inside their spheres and mark chunks
        b += sum(int(4.19 * s.radius ** 3) for s in st["spheres"]) + 3 * w.chunks
    elif kind == "nodes":
        n = sum(int(o[-1].item()) for _, o in st["nodes"])
        b = 16 * n + 28 * w.chunks + 8 * sum(abi.node_count(w, l) + 1 for l in range(5))
    elif kind == "lod":
        b = 8 * run(st)["drawn"] + 8 * case["width"] * case["height"] + \
            8 * sum(abi.node_count(w, l) + 1 for l in range(5))
    elif kind == "splat":
        px = case["width"] * case["height"]
        b = 8 * _in_view(st["list"], st["cam"]) + 32 * (int(st["list"].shape[0]) // 256 + 1) + \
            (20 if case["rgb"] else 8) * px
    else:
        px, n = case["views"] * case["size"] ** 2, int(st["list"].shape[0])
        # per view the splats in view; image, target and weights once; the gradient
        b = sum(8 * _in_view(st["list"], cam) + 32 * (n // 256 + 1) for cam in st["cams"]) + \
            (12 + 12 + 8) * px + 12 * n
    return {"bytes": float(b), "flops": 0.0}


# ---- the resolve in 64 bits ------------------------------------------------------
def _mat(m):
    return torch.tensor([float(v) for v in m], dtype=torch.float64, device=DEV).view(4, 4).T


def _vertex(recs, size, cam):
    """View-space centres, clip coordinates and the in-volume test of splats of
    edge `size` (a number or a column)."""
    c = recs[:, :3].to(torch.float64) + 0.5 * size
    T, P = _mat(cam.view_translation), _mat(cam.proj_view_rot)
    v = c @ T[:3, :3].T + T[:3, 3]
    clip = v @ P[:, :3].T + P[:, 3]
    cw = clip[:, 3:4]
    return v, clip, ((clip[:, :3] >= -cw) & (clip[:, :3] <= cw)).all(1)


def _in_view(recs, cam, step=1 << 23):
    return sum(int(_vertex(recs[a:a + step], 1.0, cam)[2].sum())
               for a in range(0, int(recs.shape[0]), step))


def _rays(cam):
    Wd, H = cam.width, cam.height
    x = (torch.arange(Wd, dtype=torch.float64, device=DEV) + 0.5) / Wd * 2 - 1
    y = (torch.arange(H, dtype=torch.float64, device=DEV) + 0.5) / H * 2 - 1
    p = torch.stack([x.repeat(H), y.repeat_interleave(Wd), -torch.ones(H * Wd, device=DEV).double(),
                     torch.ones(H * Wd, device=DEV).double()], 1)
    r = p @ _mat(cam.inv_proj_view_rot).T
    r = r[:, :3] / r[:, 3:4]
    return r / r.norm(dim=1, keepdim=True)


def _slabs(v, half, ray):
    a, b = (v - half) / ray, (v + half) / ray
    return torch.minimum(a, b).max(1).values, torch.maximum(a, b).min(1).values


def _resolve(recs, lod, cam, step=1 << 23, most=1 << 25):
    """Depth (1 where nothing is hit) and the splat of each pixel (-1: none):
    every splat's point sprite, every covered pixel's ray against its cube."""
    Wd, H = cam.width, cam.height
    rays = _rays(cam)
    pix, dep, idx = [], [], []
    for a in range(0, int(recs.shape[0]), step):
        size = (2.0 ** lod[a:a + step].double()).unsqueeze(1) if lod is not None else \
            torch.ones((min(step, int(recs.shape[0]) - a), 1), dtype=torch.float64, device=DEV)
        v, clip, ok = _vertex(recs[a:a + step], size, cam)
        at = torch.nonzero(ok).reshape(-1)
        v, clip, size = v[at], clip[at], size[at].reshape(-1)
        cw = clip[:, 3]
        nx, ny = clip[:, 0] / cw, clip[:, 1] / cw
        reduce = torch.maximum((nx * Wd / H).abs(), ny.abs()) + 0.03
        edge = (H * 1.1 / clip[:, 2] * reduce.clamp(min=1.0) * size).clamp(1.0, 2048.0)
        wx, wy = (nx + 1) * (0.5 * Wd), (ny + 1) * (0.5 * H)
        x0 = torch.ceil(wx - edge / 2 - 0.5).clamp(min=0).long()
        x1 = (torch.ceil(wx + edge / 2 - 0.5) - 1).clamp(max=Wd - 1).long()
        y0 = torch.ceil(wy - edge / 2 - 0.5).clamp(min=0).long()
        y1 = (torch.ceil(wy + edge / 2 - 0.5) - 1).clamp(max=H - 1).long()
        cx = (x1 - x0 + 1).clamp(min=0)
        cnt = cx * (y1 - y0 + 1).clamp(min=0)
        ends = cnt.cumsum(0)
        done, first = 0, 0
        while first < int(cnt.numel()):
            last = max(first + 1, int(torch.searchsorted(ends, done + most, right=True)))
            s = torch.repeat_interleave(torch.arange(first, last, device=DEV), cnt[first:last])
            j = torch.arange(int(s.numel()), device=DEV) - (ends[s] - cnt[s] - done)
            p = (y0[s] + j // cx[s]) * Wd + x0[s] + j % cx[s]
            t0, t1 = _slabs(v[s], 0.5 * size[s].unsqueeze(1), rays[p])
            d = t0 / cam.far_plane
            hit = (t0 <= t1) & (d < 1.0)
            pix.append(p[hit])
            dep.append(d[hit].clamp(min=0.0))
            idx.append(at[s[hit]] + a)
            done, first = int(ends[last - 1]), last
    none = torch.iinfo(torch.int64).max
    depth = torch.ones(Wd * H, dtype=torch.float64, device=DEV)
    best = torch.full((Wd * H,), none, dtype=torch.int64, device=DEV)
    for p, d in zip(pix, dep):
        depth.scatter_reduce_(0, p, d, "amin")
    for p, d, i in zip(pix, dep, idx):
        m = d == depth[p]
        best.scatter_reduce_(0, p[m], i[m], "amin")
    return depth, torch.where(best == none, -1, best), rays


def _shade(recs, lod, cam, depth, ids, rays, colour=None):
    """Image [H W, 3] and the weight of the splat's colour in it."""
    back = torch.tensor([0.5, 0.5, 0.7], dtype=torch.float64, device=DEV)
    hit = torch.nonzero(ids >= 0).reshape(-1)
    i, ray = ids[hit], rays[hit]
    size = (2.0 ** lod[i].double()).unsqueeze(1) if lod is not None else \
        torch.ones((int(i.numel()), 1), dtype=torch.float64, device=DEV)
    v = _vertex(recs[i], size, cam)[0]
    t0, _ = _slabs(v, 0.5 * size, ray)
    h = v - ray * t0.unsqueeze(1)
    m = h.abs()
    normal = (m == m.max(1, keepdim=True).values).double() * torch.sign(h)
    lit = (normal[:, 0] - normal[:, 1]) * math.sqrt(0.5)
    attr = recs[i, 3].long()
    sh = ((attr >> 6) & 1).double()
    scale = (1.0 - sh).clamp(min=0.7) * torch.maximum(sh.clamp(min=0.7), torch.sign(lit))
    if colour is None:
        base = torch.stack([((attr >> k) & 3).double() / 3.0 for k in (4, 2, 0)], 1)
    else:
        base = colour[i].double()
    fog = (depth[hit] - 256.0 / cam.far_plane).clamp(min=0.0001).sqrt()
    weight = torch.zeros(ids.numel(), dtype=torch.float64, device=DEV)
    weight[hit] = scale * (1.0 - fog)
    img = back.repeat(int(ids.numel()), 1)
    img[hit] = base * weight[hit].unsqueeze(1) + back * fog.unsqueeze(1)
    return img, weight


def _drawn_list(st):
    """The records and levels of the nodes a frame draws: from the level-4
    nodes down, a node in view is drawn once it is farther than 1024 voxels
    per level."""
    w = st["world"].w
    mx = [1 << b for b in w.max_bitw]
    offs = [o.cpu().numpy() for _, o in st["nodes"]]
    planes = np.asarray(st["planes"], np.float64).reshape(6, 4)
    recs, lods = [], []

    def walk(l, at):
        if any((at[a] << l) >= mx[a] for a in range(3)):
            return
        edge = w.R << l
        c = np.array([p * edge + edge // 2 for p in at], np.float64)
        if (planes[:, :3] @ c + planes[:, 3] < -0.85 * edge).any():
            return
        if l == 0 or np.linalg.norm(np.asarray(st["loc"]) - c) > 1024 * l:
            b = [abi.node_bits(w, l, a) for a in range(3)]
            k = ((at[2] << b[1] | at[1]) << b[0]) | at[0]
            lo, hi = int(offs[l][k]), int(offs[l][k + 1])
            if hi > lo:
                recs.append(st["nodes"][l][0][lo:hi])
                lods.append(torch.full((hi - lo,), l, dtype=torch.uint8, device=DEV))
            return
        for k in range(8):
            walk(l - 1, (2 * at[0] + (k >> 2), 2 * at[1] + (k >> 1 & 1), 2 * at[2] + (k & 1)))

    for x in range((mx[0] >> 4) + 1):
        for y in range((mx[1] >> 4) + 1):
            for z in range((mx[2] >> 4) + 1):
                walk(4, (x, y, z))
    if not recs:
        return torch.zeros((0, 4), dtype=torch.int16, device=DEV), \
            torch.zeros(0, dtype=torch.uint8, device=DEV)
    return torch.cat(recs), torch.cat(lods)


def exact(case, seed):
    kind = case["kind"]
    if kind not in ("splat", "lod", "fit"):
        return None                       # whole numbers and bytes only
    st = prepare(case, seed)
    if kind == "fit":
        lst, V, S = st["list"], case["views"], case["size"]
        img = torch.empty((V, S * S, 3), dtype=torch.float64, device=DEV)
        grad = torch.zeros((int(lst.shape[0]), 3), dtype=torch.float64, device=DEV)
        rgb = st["rgb"].detach()
        for k, cam in enumerate(st["cams"]):
            depth, ids, rays = _resolve(lst, None, cam)
            img[k], weight = _shade(lst, None, cam, depth, ids, rays, rgb)
            d = (img[k] - st["target"][k].double().view(-1, 3)) * (2.0 / img.numel())
            hit = ids >= 0
            grad.index_add_(0, ids[hit], d[hit] * weight[hit].unsqueeze(1))
        return {"image": img.view(V, S, S, 3), "grad": grad}
    cam = st["cam"]
    shape = (cam.height, cam.width)
    lst, lod = _drawn_list(st) if kind == "lod" else (st["list"], None)
    depth, ids, rays = _resolve(lst, lod, cam)
    if kind == "lod":
        return {"depth": depth.view(shape), "ids": None, "drawn": None}
    img = _shade(lst, None, cam, depth, ids, rays)[0].view(*shape, 3) if case["rgb"] else None
    return {"depth": depth.view(shape), "ids": None, "rgb": img}
