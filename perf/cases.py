"""The calls whose time matters to a program that keeps a voxel world on the GPU.

A case names one public path of the framework and its sizes:

apply    one Batch per tree applied to a resident forest (VoxTree::apply_batch, batched),
         then the changed trees read back densely at the level of detail that is drawn, and
         (worlds of single scattered voxels) by the point reads of the tick.
         Two batches of the same voxels alternate (values v and v + 1), as the reference's
         benchmark harness applies them, so every pass rebuilds every tree and frees what
         it replaced.
edits    sphere edits as edit lists (sorted by tree and Morton path on the device), applied,
         and the touched world read back at a level of detail.
set      VoxOpsWrite::set of one voxel in each tree (a quarter of them removals).
get      VoxOpsRead::get of many voxels, in arrival order or grouped by tree.
dense    to_vec of every tree at full resolution or a level of detail: what a mesher reads.
export   the data section of a .vtm save of the resident world.
train    one step of the node-growth predictor: gradient and Adam.

Worlds are resident before the call (built in prepare), as in a program that edits and
reads them.  Everything is made from the seed on the GPU; launch shapes are the library's
defaults.
"""
import math

import numpy as np
import torch

from voxelis_amd import api, lib
from voxelis_amd._lib import check
from voxelis_amd.predictor import GrowthMLP

MIB = 1 << 20
TORCH_INT = {1: torch.uint8, 2: torch.int16, 4: torch.int32}


def listed():
    return [
        # one 32^3 chunk edited and drawn again: the smallest call, launches and latency
        {"name": "apply_one_tree", "path": "apply", "content": "checker", "trees": 1, "depth": 5, "width": 1, "lod": 0, "reads": 0},
        # a 64 x 64 terrain of 32^3 chunks rebuilt (ids change everywhere), drawn far away
        {"name": "apply_terrain", "path": "apply", "content": "terrain", "trees": 4096, "depth": 5, "width": 1, "lod": 2, "reads": 0},
        # the headline's world: depths 5 to 7, dense fills and sparse random voxels, u16 ids
        {"name": "apply_uneven", "path": "apply", "content": "uneven", "trees": 2048, "depth": 7, "width": 2, "lod": 3, "reads": 2_000_000},
        # scattered 32-bit voxels of many colours (i32, the reference's test type), odd count
        {"name": "apply_scatter_i32", "path": "apply", "content": "scatter", "trees": 333, "depth": 6, "width": 4, "lod": 2, "reads": 500_000},
        # a brush stroke: one small sphere in a 2 x 2 x 2 neighbourhood of chunks
        {"name": "edits_brush", "path": "edits", "side": 2, "height": 2, "spheres": 1, "radius": 9.0, "depth": 5, "width": 2, "lod": 0},
        # the served stream's cycle: 64 spheres of radius 2 to 40 over 16384 chunks
        {"name": "edits_spheres", "path": "edits", "side": 32, "height": 16, "spheres": 64, "radius": 40.0, "depth": 5, "width": 2, "lod": 3},
        # one voxel set or removed in every chunk of the terrain
        {"name": "set_voxels", "path": "set", "trees": 4096, "depth": 5, "width": 1, "lod": 3},
        # 4 M single reads in arrival order (ray casts, physics) over the terrain
        {"name": "get_any", "path": "get", "content": "terrain", "trees": 4096, "depth": 5, "width": 1, "queries": 1 << 22, "grouped": False},
        # reads grouped by tree, ragged groups, deep u16 trees
        {"name": "get_grouped", "path": "get", "content": "uneven", "trees": 777, "depth": 7, "width": 2, "queries": 9_000_001, "grouped": True},
        # every chunk of a 16-bit world extracted for meshing
        {"name": "dense_u16", "path": "dense", "content": "uneven", "trees": 300, "depth": 6, "width": 2, "lod": 0},
        # a save of a world of 300 k patterns
        {"name": "export_u16", "path": "export", "branches": 300_000, "chunks": 1024, "width": 2},
        # the admission predictor's training step at its default batch
        {"name": "train_step", "path": "train", "rows": 8192},
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    path = rng.choice(["apply", "apply", "apply", "edits", "set", "get", "get", "dense", "export", "train"])
    if path == "apply":
        content = rng.choice(["checker", "terrain", "uneven", "scatter"])
        width = 1 if content == "checker" else rng.choice([2, 4]) if content == "scatter" else rng.choice([1, 2])
        if content == "uneven":
            return {"path": path, "content": content, "trees": _log(rng, 3, 1200), "depth": rng.choice([6, 7]), "width": 2,
                    "lod": 3, "reads": _log(rng, 10_000, 1_000_000)}
        depth = rng.choice([4, 5, 6])
        most = {4: 8000, 5: 4096, 6: 500}[depth]
        return {"path": path, "content": content, "trees": _log(rng, 1, most), "depth": depth, "width": width,
                "lod": rng.choice([1, 2]), "reads": _log(rng, 10_000, 500_000) if content == "scatter" else 0}
    if path == "edits":
        side = _log(rng, 2, 32)
        return {"path": path, "side": side, "height": rng.randint(1, 16), "spheres": _log(rng, 1, 64),
                "radius": round(rng.uniform(4.0, 40.0), 2), "depth": rng.choice([4, 5]), "width": rng.choice([1, 2]), "lod": 2}
    if path == "set":
        return {"path": path, "trees": _log(rng, 1, 8000), "depth": rng.choice([4, 5]), "width": rng.choice([1, 2]), "lod": 2}
    if path == "get":
        deep = rng.random() < 0.4
        return {"path": path, "content": "uneven" if deep else "terrain", "trees": _log(rng, 1, 700 if deep else 4096),
                "depth": rng.choice([6, 7]) if deep else 5, "width": 2 if deep else rng.choice([1, 2]),
                "queries": _log(rng, 400_000, 16_000_000), "grouped": rng.random() < 0.5}
    if path == "dense":
        deep = rng.random() < 0.5
        lod = rng.choice([0, 0, 1])
        return {"path": path, "content": "uneven" if deep else "terrain", "trees": _log(rng, 20, 300) if deep else _log(rng, 100 * 8 ** lod, 4096),
                "depth": 6 if deep else 5, "width": 2 if deep else rng.choice([1, 2]), "lod": lod}
    if path == "export":
        return {"path": path, "branches": _log(rng, 3000, 600_000), "chunks": _log(rng, 1, 4096), "width": rng.choice([1, 2, 4])}
    return {"path": path, "rows": _log(rng, 200, 20000)}


# ---------------------------------------------------------------- inputs

def _morton_xyz(depth, dev):
    """x, y, z of every voxel of a tree of `depth` in Morton order."""
    m = torch.arange(8 ** depth, dtype=torch.int64, device=dev)
    out = []
    for axis in range(3):
        c = torch.zeros_like(m)
        for b in range(depth):
            c |= ((m >> (3 * b + axis)) & 1) << b
        out.append(c)
    return out


def _heights(grid, chunk, gen, dev):
    """Dune heights [grid * chunk, grid * chunk] in 8 .. 23 of a 32-voxel column (scaled with
    the chunk): four octaves of smooth noise."""
    size = grid * chunk
    h = torch.zeros(size, size, device=dev)
    amp, norm = 1.0, 0.0
    for period in (128, 64, 32, 16):
        k = size // period + 4
        lattice = torch.rand(1, 1, k, k, generator=gen, device=dev)
        up = torch.nn.functional.interpolate(lattice, size=(k * period, k * period), mode="bicubic", align_corners=False)
        h += amp * up[0, 0, period:period + size, period:period + size].clamp(0.0, 1.0)
        norm += amp
        amp *= 0.5
    h = (h / norm).clamp(0.0, 0.9999)
    return ((8 + torch.floor(16 * h)) * chunk / 32).to(torch.int64)


def _depths(case, seed):
    if case["content"] != "uneven":
        return [case["depth"]] * case["trees"]
    r = np.random.default_rng(seed)
    return [int(d) for d in r.integers(5, case["depth"] + 1, case["trees"])]


def _content(case, seed, dev):
    """Per tree its depth, and the voxels of all trees, one after the other in Morton order
    (0: empty), as int32."""
    gen = torch.Generator(device=dev).manual_seed(seed)
    depths = _depths(case, seed)
    total = sum(8 ** d for d in depths)
    kind, n, d = case["content"], case["trees"], case["depth"]
    if kind == "checker":  # v = ((x + y + z + t) & 1) + 1, the phase of each tree from the seed
        x, y, z = _morton_xyz(d, dev)
        t = torch.randint(0, 97, (n, 1), generator=gen, device=dev)
        return depths, (((x + y + z)[None] + t) % 2 + 1 + t % 5).reshape(-1).to(torch.int32)
    if kind == "terrain":
        chunk, grid = 1 << d, max(1, math.isqrt(n - 1) + 1)
        x, y, z = _morton_xyz(d, dev)
        h = _heights(grid, chunk, gen, dev)
        out = torch.empty(n, 8 ** d, dtype=torch.int32, device=dev)
        for t in range(n):
            cz, cx = divmod(t, grid)
            hh = h[cz * chunk:(cz + 1) * chunk, cx * chunk:(cx + 1) * chunk][z, x]
            out[t] = (y < hh).to(torch.int32) + 2 * (y == hh).to(torch.int32)
        return depths, out.reshape(-1)
    # uneven: a dense fill or sparse voxels of 0.1, 1 or 10 %; scatter: sparse voxels of 1 %
    r = np.random.default_rng(seed + 1)
    top = 65535 if case["width"] == 2 else (1 << 24) - 1  # 32 bits: 24-bit colours
    off = int(r.integers(0, 60000))
    out = torch.zeros(total, dtype=torch.int32, device=dev)
    base, fills = 0, {}
    for dd in depths:
        dense = kind == "uneven" and r.random() < 0.5
        density = float(r.choice([0.001, 0.01, 0.1])) if kind == "uneven" else 0.01
        cells = out[base:base + 8 ** dd]
        if dense:
            if dd not in fills:
                x, y, z = _morton_xyz(dd, dev)
                fills[dd] = ((x + y + z + off) % 65535 + 1).to(torch.int32)
            cells.copy_(fills[dd])
        else:
            at = torch.randint(0, 8 ** dd, (max(1, round(density * 8 ** dd)),), generator=gen, device=dev)
            # a voxel's id follows from its place, so that a place drawn twice has one id
            v = ((at + base) * 0x9E3779B1 + seed * 0x85EBCA6B) % ((1 << 61) - 1)
            cells[at] = (((v >> 13) ^ v) % top + 1).to(torch.int32)
        base += 8 ** dd
    return depths, out


def _narrow(v, width):
    return v.to(TORCH_INT[width])


def _batch(depths, v, width):
    """Dense Batch buffers of every tree: (masks [P, 2], values [P, 8]) per tree."""
    bits = (v.view(-1, 8) != 0).to(torch.uint8)
    weight = torch.tensor([1, 2, 4, 8, 16, 32, 64, 128], dtype=torch.uint8, device=v.device)
    masks = torch.zeros(bits.shape[0], 2, dtype=torch.uint8, device=v.device)
    masks[:, 0] = (bits * weight).sum(dim=1, dtype=torch.uint8)
    cuts = [8 ** (d - 1) for d in depths]
    return list(torch.split(masks, cuts)), list(torch.split(_narrow(v, width).view(-1, 8), cuts))


def _next(v, width):
    """The other batch's ids: v + 1 where a voxel is set, never 0."""
    top = {1: 255, 2: 65535, 4: (1 << 31) - 1}[width]
    return torch.where(v == 0, v, torch.where(v == top, 1, v + 1))


def _budget(case, seed):
    """Room for the world's nodes twice over (an apply frees what it replaced at its end)."""
    if case["content"] == "uneven":
        share = 0.06 if case["trees"] >= 64 else 0.2  # nodes per voxel; a few trees may all be dense ones
    else:
        share = {"checker": 0.01, "terrain": 0.02, "scatter": 0.08}[case["content"]]
    return max(64 * MIB, int(share * sum(8 ** d for d in _depths(case, seed)) * (78 + case["width"])))


def _world(case, seed):
    """A resident forest with the case's content applied, and its two batches' views."""
    dev = torch.device("cuda", torch.cuda.current_device())
    it = api.VoxInterner(case["width"], _budget(case, seed))
    depths, v = _content(case, seed, dev)
    f = api.Forest(it, depths)
    masks, a = _batch(depths, v, case["width"])
    status = f.apply(masks, a)
    assert (status == 1).all(), "the world was not built"
    return it, f, masks, a, v


def _dense_reader(it, f, lod):
    """A buffer for every tree at `lod`, and the call that fills it."""
    n = int(8 ** max(0, int(f.depths_host.max()) - lod))
    out = torch.zeros(f.n, n, dtype=TORCH_INT[it.value_size], device=it.device)
    args = (it.h, f.n, f.roots.data_ptr(), f.depths.data_ptr(), lod, n, out.data_ptr())
    return out, lambda: check(lib().vx_trees_to_vec(*args), "to_vec")


def _reads(case, seed, f, v):
    """Point reads: half of them anywhere, half at voxels that are set."""
    dev, n = v.device, case["reads"]
    gen = torch.Generator(device=dev).manual_seed(seed + 3)
    first = torch.tensor(np.concatenate([[0], np.cumsum(8 ** f.depths_host.astype(np.int64))]), device=dev)
    at = torch.randint(0, v.numel(), (n,), generator=gen, device=dev)
    if v.numel() < 1 << 30:
        hit = torch.nonzero(v)[:, 0]
    else:  # the set voxels of an evenly spread part
        hit = torch.nonzero(v[: v.numel() // 64 * 64].view(-1, 64)[:, 0])[:, 0] * 64
    at[::2] = hit[torch.randint(0, len(hit), (len(at[::2]),), generator=gen, device=dev)]
    tree = torch.searchsorted(first, at, right=True) - 1
    m = at - first[tree]
    xyz = torch.zeros(n, 3, dtype=torch.int64, device=dev)
    for axis in range(3):
        for b in range(7):
            xyz[:, axis] |= ((m >> (3 * b + axis)) & 1) << b
    return {"tree": tree.to(torch.int32), "xyz": xyz.to(torch.int32).contiguous(),
            "val": torch.zeros(n, dtype=TORCH_INT[case["width"]], device=dev), "pres": torch.zeros(n, dtype=torch.uint8, device=dev)}


def _sphere_lists(case, seed, dev):
    """Two edit lists of the same spheres (ids v and v + 1; a quarter carves), as (offsets,
    xyz, values) grouped by tree in submission order."""
    r = np.random.default_rng(seed)
    side, height, chunk = case["side"], case["height"], 1 << case["depth"]
    size = np.array([side, height, side]) * chunk
    top = 255 if case["width"] == 1 else 65535
    tree, local, val = [], [], []
    for _ in range(case["spheres"]):
        c = [int(q) for q in r.integers(0, size)]
        radius = float(r.uniform(min(2.0, case["radius"] / 2), case["radius"]))
        v = 0 if case["spheres"] > 1 and r.random() < 0.25 else int(r.integers(1, top + 1))
        k = int(radius)
        ax = [torch.arange(max(0, c[i] - k), min(int(size[i]), c[i] + k + 1), device=dev) for i in range(3)]
        p = torch.stack(torch.meshgrid(*ax, indexing="ij"), dim=-1).reshape(-1, 3)
        p = p[((p - torch.tensor(c, device=dev)) ** 2).sum(dim=1) <= radius * radius]
        t = p // chunk
        tree.append((t[:, 2] * height + t[:, 1]) * side + t[:, 0])
        local.append((p % chunk).to(torch.int32))
        val.append(torch.full((len(p),), v, dtype=torch.int32, device=dev))
    tree, order = torch.sort(torch.cat(tree), stable=True)
    local, val = torch.cat(local)[order].contiguous(), torch.cat(val)[order]
    n = side * side * height
    offs = torch.searchsorted(tree, torch.arange(n + 1, device=dev)).cpu().numpy().astype(np.uint64)
    return [(offs, local, _narrow(v, case["width"])) for v in (val, _next(val, case["width"]))]


def _section(case, seed):
    """A .vtm data section of about the case's number of branches: leaves, then four levels
    of branches over shuffled nodes of the level below (all of them used, each about as
    often), then the chunks.  A loaded world keeps the file's numbering."""
    r = np.random.default_rng(seed)
    width, want, chunks = case["width"], case["branches"], case["chunks"]
    nleaf = 255 if width == 1 else min(65535, max(512, want // 4))
    many = np.array([m for m in range(256) if bin(m).count("1") >= 4])  # four to eight children
    kids, masks, below, first = [], [], (1, nleaf), 1 + nleaf
    for n in [max(1, int(want * q)) for q in (0.6, 0.25, 0.1, 0.05)]:
        n = max(n, below[1] // 4 + 1)  # every node below has a parent
        m = r.permutation(np.resize(many, n))
        on = ((m[:, None] >> np.arange(8)) & 1).astype(bool)
        k = np.zeros((n, 8), dtype=np.int64)
        k[on] = below[0] + r.permutation(np.resize(np.arange(below[1]), int(on.sum())))
        kids.append(k)
        masks.append(m)
        below = (first, n)
        first += n
    kids, masks = np.concatenate(kids), np.concatenate(masks)

    def varint(v):  # [n] -> bytes [n, 5] and which of them are written
        v = v.astype(np.int64)
        parts = np.stack([(v >> (7 * i)) & 0x7F for i in range(5)], axis=-1)
        last = np.stack([(v >> (7 * (i + 1))) == 0 for i in range(5)], axis=-1)
        used = np.concatenate([np.ones(v.shape + (1,), bool), np.cumsum(last, axis=-1)[..., :-1] == 0], axis=-1)
        return np.where(last, parts, parts | 0x80).astype(np.uint8), used

    def big(v):  # big-endian value bytes
        return np.stack([(v >> (8 * (width - 1 - i))) & 0xFF for i in range(width)], axis=-1).astype(np.uint8)

    def join(cols):  # rows of (bytes, used) pieces, written one after the other
        b = np.concatenate([c[0] for c in cols], axis=1)
        return b[np.concatenate([c[1] for c in cols], axis=1)].tobytes()

    def full(b):
        return b, np.ones(b.shape, bool)

    values = np.arange(1, nleaf + 1) if width < 4 else np.unique(r.integers(1, 1 << 31, 2 * nleaf))[:nleaf]
    leaves = join([varint(np.arange(1, nleaf + 1)), full(big(values))])
    kb, ku = varint(kids)
    ku &= kids[:, :, None] != 0
    ids = np.arange(1 + nleaf, 1 + nleaf + len(kids))
    branches = join([varint(ids), full(masks[:, None].astype(np.uint8)), (kb.reshape(len(kids), -1), ku.reshape(len(kids), -1)),
                     full(big(r.permutation(np.resize(values, len(kids)))))])
    roots = below[0] + r.permutation(np.resize(np.arange(below[1]), max(chunks, below[1])))
    chunks = len(roots)
    pos = np.stack([np.arange(chunks) % 64, np.zeros(chunks, int), np.arange(chunks) // 64], axis=1)
    pb = np.ascontiguousarray(pos.astype(">i4")).view(np.uint8).reshape(-1, 12)
    magic = np.tile(np.frombuffer(b"VoxTreeChunk", dtype=np.uint8), (chunks, 1))
    tail = join([full(magic), full(pb), varint(roots)])
    u32 = lambda n: int(n).to_bytes(4, "big")  # noqa: E731
    return u32(nleaf) + leaves + u32(len(kids)) + branches + u32(chunks) + tail


# ---------------------------------------------------------------- the program

def prepare(case, seed):
    dev = torch.device("cuda", torch.cuda.current_device())
    path = case["path"]
    s = {"path": path, "at": 0}
    if path == "apply":
        it, f, masks, a, v = _world(case, seed)
        _, b = _batch(f.depths_host.tolist(), _next(v, case["width"]), case["width"])
        out, dense = _dense_reader(it, f, case["lod"])
        if case["reads"]:
            s["reads"] = _reads(case, seed, f, v)
        s.update(it=it, f=f, keep=(masks, a, b), views=[f.make_views(masks, b), f.make_views(masks, a)], out=out, dense=dense)
    elif path == "edits":
        it = api.VoxInterner(case["width"], 1024 * MIB)
        n = case["side"] ** 2 * case["height"]
        f = api.Forest(it, [case["depth"]] * n)
        lists = _sphere_lists(case, seed, dev)
        # dunes in the bottom layer, air above
        g = {"content": "terrain", "trees": case["side"] ** 2, "depth": case["depth"], "width": case["width"]}
        depths, v = _content(g, seed, dev)
        masks, a = _batch(depths, v, case["width"])
        low = api.Forest(it, depths)
        assert (low.apply(masks, a) == 1).all(), "the world was not built"
        ground = torch.arange(n, device=dev).view(case["side"], case["height"], case["side"])[:, 0, :].reshape(-1)
        f.roots[ground] = low.roots
        out, dense = _dense_reader(it, f, case["lod"])
        f.apply_edits(*lists[1])  # the spheres exist; passes change their ids
        s.update(it=it, f=f, lists=lists, out=out, dense=dense)
    elif path == "set":
        it, f, masks, a, v = _world({**case, "content": "terrain"}, seed)
        gen = torch.Generator(device=dev).manual_seed(seed + 1)
        top = 200 if case["width"] == 1 else 60000
        sets = []
        for k in range(4):  # four places in every tree; each is visited with one id, then another (a quarter removes)
            xyz = torch.randint(0, 1 << case["depth"], (f.n, 3), generator=gen, device=dev, dtype=torch.int32)
            v1 = torch.randint(4, top, (f.n,), generator=gen, device=dev, dtype=torch.int32)
            v2 = torch.where(torch.rand(f.n, generator=gen, device=dev) < 0.5, 0, v1 + 1)
            sets += [(k, xyz, _narrow(v1, case["width"])), (k + 4, xyz, _narrow(v2, case["width"]))]
        sets = [(xyz, val) for _, xyz, val in sorted(sets, key=lambda e: e[0])]
        out, dense = _dense_reader(it, f, case["lod"])
        f.set_voxels(*sets[-1])
        s.update(it=it, f=f, sets=sets, out=out, dense=dense)
    elif path == "get":
        it, f, _, _, _ = _world(case, seed)
        gen = torch.Generator(device=dev).manual_seed(seed + 2)
        q = case["queries"]
        tree = torch.randint(0, f.n, (q,), generator=gen, device=dev)
        xyz = torch.randint(0, 1 << 7, (q, 3), generator=gen, device=dev, dtype=torch.int32)
        val = torch.zeros(q, dtype=TORCH_INT[case["width"]], device=dev)
        pres = torch.zeros(q, dtype=torch.uint8, device=dev)
        if case["grouped"]:
            tree = torch.sort(tree)[0]
            s["offsets"] = torch.searchsorted(tree, torch.arange(f.n + 1, device=dev))
        xyz = xyz & ((1 << f.depths[tree].to(torch.int32)) - 1)[:, None]
        s.update(it=it, f=f, tree=tree.to(torch.int32), xyz=xyz.contiguous(), val=val, pres=pres)
    elif path == "dense":
        it, f, _, _, _ = _world(case, seed)
        out, dense = _dense_reader(it, f, case["lod"])
        s.update(it=it, f=f, out=out, dense=dense)
    elif path == "export":
        it = api.VoxInterner(case["width"], max(64 * MIB, case["branches"] * 400))
        f, pos = api.Forest.deserialize(it, _section(case, seed), 4)
        s.update(it=it, f=f, pos=pos)
    else:
        gen = torch.Generator(device=dev).manual_seed(seed)
        x = torch.randn(case["rows"], 16, generator=gen, device=dev)
        t = (2.0 + x[:, :5].sum(dim=1) + 0.3 * torch.randn(case["rows"], generator=gen, device=dev)).clamp(0.0, 9.0)
        s.update(model=GrowthMLP(device=dev, seed=seed % (1 << 31)), x=x, t=t)
    return s


def run(s):
    path = s["path"]
    if path == "apply":
        s["f"].apply_views(s["views"][s["at"]])
        s["at"] ^= 1
        s["dense"]()
        r = s.get("reads")
        if r is None:
            return {"status": s["f"].status, "voxels": s["out"]}
        s["f"].get_device(r["tree"], r["xyz"], r["val"], r["pres"])
        return {"status": s["f"].status, "voxels": s["out"], "read": r["val"], "present": r["pres"]}
    if path == "edits":
        s["f"].apply_edits(*s["lists"][s["at"]], sync=False)
        s["at"] ^= 1
        s["dense"]()
        return {"status": s["f"].status, "voxels": s["out"]}
    if path == "set":
        s["f"].set_voxels(*s["sets"][s["at"]], sync=False)
        s["at"] = (s["at"] + 1) % len(s["sets"])
        s["dense"]()
        return {"status": s["f"].status, "voxels": s["out"]}
    if path == "get":
        if "offsets" in s:
            s["f"].get_grouped_device(s["offsets"], s["xyz"], s["val"], s["pres"])
        else:
            s["f"].get_device(s["tree"], s["xyz"], s["val"], s["pres"])
        return {"values": s["val"], "present": s["pres"]}
    if path == "dense":
        s["dense"]()
        return {"voxels": s["out"]}
    if path == "export":
        return {"section": np.frombuffer(s["f"].serialize(s["pos"]), dtype=np.uint8)}
    m = s["model"]
    g, y, loss = m.gradient(s["x"], s["t"])
    m.adam_step(g, 3e-3)
    return {"grad": g, "y": y, "loss": loss, "params": m.p, "m": m.m, "v": m.v}


# ---------------------------------------------------------------- what a pass cannot do without

def work(case):
    path, w = case["path"], case.get("width", 4)
    if path in ("apply", "dense", "set"):
        depths = _depths({"content": "terrain", **case}, 0)
        out = len(depths) * 8 ** max(0, max(depths) - case["lod"]) * w
    if path == "apply":
        # masks of every brick, the values of written bricks, the dense result, the reads
        voxels = sum(8 ** d for d in depths)
        share = {"checker": 1.0, "terrain": 0.55, "uneven": 0.6, "scatter": 0.08}[case["content"]]
        return {"bytes": voxels / 8 * 2 + share * voxels * w + out + case["reads"] * (17 + w), "flops": 0}
    if path == "edits":
        # coordinates and value of every edit, the dense result
        mean = (case["radius"] ** 4 - 2.0 ** 4) / 4 / max(1.0, case["radius"] - 2.0) * 4.19
        return {"bytes": case["spheres"] * mean * (12 + w) + case["side"] ** 2 * case["height"] * 8 ** (case["depth"] - case["lod"]) * w, "flops": 0}
    if path == "set":
        # per tree: coordinates, value, status, the path read and its new nodes written
        return {"bytes": case["trees"] * (12 + w + 4 + 2 * 64 * case["depth"]) + out, "flops": 0}
    if path == "get":
        return {"bytes": case["queries"] * (12 + (0 if case["grouped"] else 4) + w + 1), "flops": 0}
    if path == "dense":
        return {"bytes": out, "flops": 0}
    if path == "export":
        # a node's columns read, its record written
        return {"bytes": case["branches"] * (64 + 4 + w + 4 + 1 + 20) + max(case["chunks"], case["branches"] // 20) * 36, "flops": 0}
    n, params = case["rows"], 5313
    return {"bytes": n * (16 + 1 + 1) * 4 + params * 4 * 7, "flops": 6 * n * (16 * 64 + 64 * 64 + 64)}


def exact(case, seed):
    """The training step in 64 bits; every other path returns whole numbers."""
    if case["path"] != "train":
        return None
    dev = torch.device("cuda", torch.cuda.current_device())
    gen = torch.Generator(device=dev).manual_seed(seed)
    n = case["rows"]
    x = torch.randn(n, 16, generator=gen, device=dev)
    t = (2.0 + x[:, :5].sum(dim=1) + 0.3 * torch.randn(n, generator=gen, device=dev)).clamp(0.0, 9.0)
    r = np.random.default_rng(seed % (1 << 31))  # He-uniform weights, as the model draws them
    w1 = r.uniform(-1, 1, (64, 16)) * math.sqrt(6.0 / 16)
    w2 = r.uniform(-1, 1, (64, 64)) * math.sqrt(6.0 / 64)
    w3 = r.uniform(-1, 1, 64) * math.sqrt(3.0 / 64)
    z = np.zeros(64)
    p = np.concatenate([w1.ravel(), z, w2.ravel(), z, w3, z[:1]]).astype(np.float32).astype(np.float64)
    x, t = x.cpu().double().numpy(), t.cpu().double().numpy()
    w1, b1, w2, b2, w3, b3 = p[:1024].reshape(64, 16), p[1024:1088], p[1088:5184].reshape(64, 64), p[5184:5248], p[5248:5312], p[5312]
    a1 = x @ w1.T + b1
    h1 = np.maximum(a1, 0)
    a2 = h1 @ w2.T + b2
    h2 = np.maximum(a2, 0)
    y = h2 @ w3 + b3
    dy = 2 * (y - t) / n
    d2 = (a2 > 0) * dy[:, None] * w3
    d1 = (a1 > 0) * (d2 @ w2)
    g = np.concatenate([(d1.T @ x).ravel(), d1.sum(axis=0), (d2.T @ h1).ravel(), d2.sum(axis=0), dy @ h2, [dy.sum()]])
    m, v = 0.1 * g, 0.001 * g * g
    p = p - 3e-3 * (m / 0.1) / (np.sqrt(v / 0.001) + 1e-8)
    return {"grad": g, "y": y, "loss": np.array([((y - t) ** 2).mean()]), "params": p, "m": m, "v": v}
