"""The free stack put in index order between calls: worlds large enough for it (2^18 frees) that
replace, empty and shrink, an apply rolled back on such a stack, and nodes of every kind
allocated from it; no index is handed out twice and none is lost."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

MB = 1024 * 1024


def _voxels(rng, trees, depth, share, torch, top):
    n = 8 ** (depth - 1)
    v = rng.integers(1, top, (trees, n, 8)).astype(np.uint32 if top > 65535 else np.uint16)
    v[rng.random(v.shape) >= share] = 0
    v[:, 0, 0] = 1
    m = np.zeros((trees, n, 2), dtype=np.uint8)
    m[:, :, 0] = np.packbits(v != 0, axis=2, bitorder="little")[:, :, 0]
    return m, v


@pytest.mark.parametrize("width", [2, 4])
def test_replaced_worlds_keep_every_node(width):
    import torch
    if not torch.cuda.is_available():
        pytest.skip("needs a GPU")
    from voxelis_amd import api
    rng = np.random.default_rng(width)
    trees, depth = 48, 6
    top = 60000 if width == 2 else 1 << 24
    it = api.VoxInterner(width, 512 * MB)
    f = api.Forest(it, [depth] * trees)
    check = api.VoxInterner(width, 512 * MB)  # the same world built in a fresh interner
    freed = 0
    for step in range(6):
        if step == 3:  # empty, then a smaller world
            f.fill([0] * trees)
            assert it.counts() == (0, 1) and it.alive_nodes() == 1
        m, v = _voxels(rng, trees, depth, 0.02 if step == 3 else 0.1, torch, top)
        if step and step != 3:  # every written voxel gets another value, the rest is cleared first
            f.fill([0] * trees)
        dev = [[api.to_device(a[t]) for t in range(trees)] for a in (m, v)]
        if step == 4:  # rolled back on a sorted stack, then again
            before = (it.counts(), it.alive_nodes(), f.canonical_hashes())
            st = f.apply(*dev, node_limit=1000)
            assert (st == -8).all()
            assert (it.counts(), it.alive_nodes(), f.canonical_hashes()) == before
        st = f.apply(*dev)
        assert (st == 1).all()
        v2 = np.where(v == 0, 0, v % (top - 1) + 1).astype(v.dtype)  # every tree replaced in one apply
        dev2 = [api.to_device(v2[t]) for t in range(trees)]
        r0 = it.stats()["recycled"]
        st = f.apply(dev[0], dev2)
        assert (st == 1).all()
        freed = max(freed, it.stats()["recycled"] - r0)
        g = api.Forest(check, [depth] * trees)
        assert (g.apply(dev[0], dev2) == 1).all()
        assert f.canonical_hashes() == g.canonical_hashes()
        assert it.counts() == check.counts()
        assert it.alive_nodes() == check.alive_nodes()
        g.fill([0] * trees)
    assert freed >= 1 << 18, freed
    f.fill([0] * trees)
    assert it.counts() == (0, 1) and it.alive_nodes() == 1
