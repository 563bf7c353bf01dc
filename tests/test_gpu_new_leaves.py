"""Leaves created while the bricks that use them are built: an id that is new in every brick
of many trees, as many new ids as voxels, the same new id twice in a brick, a reservation
that holds exactly the new nodes and one that is a node short, and a tree that fails in the
brick pass beside trees that use the same new ids."""
import numpy as np
import pytest

import oracle_lib as O
from gpu_helpers import assert_same, oracle_apply_dense

pytestmark = pytest.mark.gpu

MB = 1024 * 1024
NP = {1: np.uint8, 2: np.uint16, 4: np.uint32}


@pytest.fixture(scope="module")
def vx():
    import torch
    if not torch.cuda.is_available():
        pytest.skip("needs a GPU")
    from voxelis_amd import api, workloads
    return api, workloads


def _worlds(api, width, depths):
    it, it_o = api.VoxInterner(width, 64 * MB), O.Interner(width, 64 * MB)
    return it, it_o, api.Forest(it, depths), [O.Tree(d) for d in depths]


def _ids(width, k):
    """The k-th id of a run that spreads over the width's range and is never 0."""
    return (1 + (np.asarray(k, dtype=np.uint64) * 2654435761) % ((1 << (8 * width)) - 1)).astype(NP[width])


@pytest.mark.parametrize("brick_rounds", [1, 4])
@pytest.mark.parametrize("width", [1, 2, 4])
@pytest.mark.parametrize("kind", ["one", "two", "distinct", "mixed"])
def test_new_ids_everywhere(vx, width, kind, brick_rounds):
    api, W = vx
    rng = np.random.default_rng(width)
    depths = [4, 5, 2, 3, 4, 4, 5, 3]
    it, it_o, f, trees = _worlds(api, width, depths)
    it.set_tuning(brick_rounds=brick_rounds)
    for step in range(4):
        ms, vs = [], []
        for t, d in enumerate(depths):
            n = 1 << d
            y, z, x = np.meshgrid(np.arange(n), np.arange(n), np.arange(n), indexing="ij")
            if kind == "one":  # every brick all the same (the tree becomes one leaf)
                dense = np.full((n, n, n), _ids(width, 1000 * step + 1))
            elif kind == "two":  # every brick mixed, each new id twice and more in it
                dense = _ids(width, 1000 * step + (x + y + z) % 2)
            elif kind == "distinct":  # a new id per voxel (u8: every id)
                dense = _ids(width, 100000 * (step + 1) + (n * n * y + n * z + x) + 40000 * (t % 2))
            else:  # sparse and dense parts, old ids and new ones
                dense = np.where(rng.random((n, n, n)) < 0.3, _ids(width, rng.integers(0, 60 + 40 * step, (n, n, n))), 0)
                dense[0, 0, 0] = _ids(width, 777 + step)
            m, v = W.dense_to_batch(dense.astype(NP[width]), d)
            ms.append(m)
            vs.append(v)
        want = []
        for t, m, v in zip(trees, ms, vs):
            before = t.root
            try:
                snap = O.lib().vxo_snapshot_take(it_o.h)
                want.append(1 if oracle_apply_dense(it_o, t, m, v)[0] else 0)
            except O.OraclePanic:
                O.lib().vxo_snapshot_restore(it_o.h, snap)
                t.root = before
                want.append(-1)
            finally:
                O.lib().vxo_snapshot_free(snap)
        st = f.apply([api.to_device(m) for m in ms], [api.to_device(v) for v in vs])
        assert [min(int(s), 1) if s >= 0 else -1 for s in st] == want, (step, st, want)
        assert_same(it, f, it_o, trees, full_reads=step == 3, what=f"{kind} step {step}")


@pytest.mark.parametrize("width", [1, 2, 4])
def test_reservation_of_new_leaves(vx, width):
    api, W = vx
    depths = [4, 4, 3]
    it, it_o, f, trees = _worlds(api, width, depths)
    for step in range(3):
        bat = []
        for d in depths:
            n = 1 << d
            y, z, x = np.meshgrid(np.arange(n), np.arange(n), np.arange(n), indexing="ij")
            bat.append(W.dense_to_batch(_ids(width, 50 * step + (x + 2 * y + 3 * z) % 40), d))
        dev = [[api.to_device(b[k]) for b in bat] for k in (0, 1)]
        before = (it.counts(), f.canonical_hashes())
        assert (f.apply(*dev, dry_run=True, counts=True) == 1).all()
        branches, leaves, _ = f.counts_host()
        assert leaves == 40 if step == 0 else leaves > 0
        for short in (1, branches, branches + leaves - 1, branches + leaves):
            if branches + leaves - short >= 1:
                st = f.apply(*dev, node_limit=branches + leaves - short, counts=True)
                assert (st == -8).all(), (short, st)
                assert f.counts_host()[0] is None
                assert (it.counts(), f.canonical_hashes()) == before, (step, short)
        st = f.apply(*dev, node_limit=branches + leaves, counts=True)
        assert (st == 1).all()
        assert f.counts_host()[:2] == (branches, leaves)
        for t, (m, v) in zip(trees, bat):
            assert oracle_apply_dense(it_o, t, m, v)[0]
        assert_same(it, f, it_o, trees, what=f"step {step}")


@pytest.mark.parametrize("width", [1, 2, 4])
@pytest.mark.parametrize("brick_rounds", [1, 4])
def test_failed_tree_beside_new_ids(vx, width, brick_rounds):
    """Tree 0 (and tree 5) partly write a collapsed brick: they fail and leave nothing, while
    the other trees build equal bricks of the same new ids; a call in which every tree fails
    takes no node, whatever its reservation."""
    api, W = vx
    depth, n = 3, 9
    it, it_o, f, trees = _worlds(api, width, [depth] * n)
    it.set_tuning(brick_rounds=brick_rounds)
    first = np.zeros((8, 8, 8), dtype=NP[width])
    first[:2, :2, :2] = _ids(width, 1)  # one collapsed brick
    first[4, 4, 4] = _ids(width, 2)
    m, v = W.dense_to_batch(first, depth)
    assert (f.apply([api.to_device(m)] * n, [api.to_device(v)] * n) == 1).all()
    for t in trees:
        assert oracle_apply_dense(it_o, t, m, v)[0]
    good = np.zeros((8, 8, 8), dtype=NP[width])
    good[4:, 4:, 4:] = _ids(width, 10 + np.arange(64).reshape(4, 4, 4) % 7)
    bad = good.copy()
    bad[0, 0, 0] = _ids(width, 99)
    pick = [k in (0, 5) for k in range(n)]
    bat = [W.dense_to_batch(bad if p else good, depth) for p in pick]
    st = f.apply([api.to_device(b[0]) for b in bat], [api.to_device(b[1]) for b in bat])
    assert [int(s) for s in st] == [-5 if p else 1 for p in pick]
    for t, b, p in zip(trees, bat, pick):
        if not p:
            assert oracle_apply_dense(it_o, t, *b)[0]
    assert_same(it, f, it_o, trees, what="two failed trees")
    bad2 = bad.copy()
    bad2[bad2 != 0] += 20
    m2, v2 = W.dense_to_batch(bad2, depth)
    before = it.counts()
    st = f.apply([api.to_device(m2)] * n, [api.to_device(v2)] * n, node_limit=64)
    assert (st == -5).all()
    assert it.counts() == before
    assert_same(it, f, it_o, trees, what="every tree failed")


@pytest.mark.parametrize("width", [2, 4])
def test_applies_out_of_nodes_leave_no_request_behind(vx, width):
    """Many new ids at once, in a used table, with a reservation that runs out at once: again and
    again nothing is left of it, and then the same ids are created."""
    api, W = vx
    rng = np.random.default_rng(width)
    trees, depth = 48, 5
    n = 8 ** (depth - 1)
    it = api.VoxInterner(width, 64 * MB)
    f = api.Forest(it, [depth] * trees)
    top = (1 << 16) - 1 if width == 2 else 1 << 24
    for step in range(3):
        v = rng.integers(1, top, (trees, n, 8)).astype(NP[width])
        v[rng.random(v.shape) >= 0.1] = 0
        m = np.zeros((trees, n, 2), dtype=np.uint8)
        m[:, :, 0] = np.packbits(v != 0, axis=2, bitorder="little")[:, :, 0]
        f.fill([0] * trees)  # (their leaves' places in the table are free again)
        dev = [[api.to_device(a[t]) for t in range(trees)] for a in (m, v)]
        before = (it.counts(), it.alive_nodes())
        for k in range(12):
            assert (f.apply(*dev, node_limit=1 + 40 * k) == -8).all()
            assert (it.counts(), it.alive_nodes()) == before, (step, k)
        assert (f.apply(*dev) == 1).all()
        assert it.counts()[0] == len(np.unique(v[v != 0]))
