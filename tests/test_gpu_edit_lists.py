"""Edit lists by the winner of each voxel: lists around the sizes of a block's run, many writes
to few voxels, runs that cross trees, trees without edits between edited ones, rejected and
failing trees among them, and calls whose edited trees differ from the last call's (the
winners' array is zero again whatever came before)."""
import numpy as np
import pytest

import oracle_lib as O
from gpu_helpers import assert_same

pytestmark = pytest.mark.gpu

MB = 1024 * 1024
NP = {1: np.uint8, 2: np.uint16, 4: np.uint32}


@pytest.fixture(scope="module")
def vx():
    import torch
    if not torch.cuda.is_available():
        pytest.skip("needs a GPU")
    from voxelis_amd import api
    return api


@pytest.mark.parametrize("width", [1, 2, 4])
@pytest.mark.parametrize("sizes", [[1], [255], [256], [257], [3000], [0, 5, 0, 0, 300, 1, 0], [1] * 70, [0, 0, 0]])
def test_lists_of_every_shape(vx, width, sizes):
    api = vx
    rng = np.random.default_rng(len(sizes) + sizes[0])
    depths = [2 + (k * 3) % 4 for k in range(len(sizes))]
    it, it_o = api.VoxInterner(width, 64 * MB), O.Interner(width, 64 * MB)
    f, trees = api.Forest(it, depths), [O.Tree(d) for d in depths]
    for step in range(4):
        # each step edits other trees; values of few ids (0 among them) and voxels repeat
        sz = sizes if step % 2 == 0 else sizes[::-1]
        offs = np.concatenate([[0], np.cumsum(sz)]).astype(np.uint64)
        xyz = [rng.integers(0, 1 << d, (k, 3)).astype(np.int32) for d, k in zip(depths, sz)]
        val = [rng.integers(0, 4 + 9 * step, k).astype(NP[width]) for k in sz]
        all_xyz, all_val = np.concatenate(xyz), np.concatenate(val)
        st = f.apply_edits(offs, api.to_device(all_xyz) if len(all_xyz) else None,
                           api.to_device(all_val) if len(all_val) else None, counts=step == 2)
        for t, x, v, s in zip(trees, xyz, val, st):
            if len(x) == 0:
                assert s == 0
                continue
            b = t.create_batch()
            b.set_many(x, v.astype(np.uint64))
            before = t.root
            try:
                snap = O.lib().vxo_snapshot_take(it_o.h)
                assert s == (1 if t.apply_batch(it_o, b) else 0)
            except O.OraclePanic:
                O.lib().vxo_snapshot_restore(it_o.h, snap)
                t.root = before
                assert s < 0
            finally:
                O.lib().vxo_snapshot_free(snap)
        assert_same(it, f, it_o, trees, full_reads=step == 3, what=f"step {step}")
    if sum(sizes) == 0:
        assert it.counts() == (0, 1)


def test_rejected_and_failing_trees(vx):
    """A tree too shallow, one with a coordinate outside, one untouched, beside good ones; the
    next call on the same trees finds nothing of the failed lists."""
    api = vx
    depths = [1, 4, 3, 5, 2]
    it, it_o = api.VoxInterner(2, 64 * MB), O.Interner(2, 64 * MB)
    f, trees = api.Forest(it, depths), [O.Tree(d) for d in depths]
    xyz = np.array([[0, 0, 0], [3, 2, 1], [16, 0, 0], [7, 7, 7], [31, 31, 31], [0, -1, 0], [1, 1, 1]], dtype=np.int32)
    val = np.arange(1, 8, dtype=np.uint16)
    offs = np.array([0, 1, 3, 4, 5, 7], dtype=np.uint64)
    st = f.apply_edits(offs, api.to_device(xyz), api.to_device(val))
    assert [int(s) for s in st] == [-3, -4, 1, 1, -4]
    for k, e in ((2, 3), (3, 4)):
        b = trees[k].create_batch()
        b.set_many(xyz[e:e + 1], val[e:e + 1].astype(np.uint64))
        assert trees[k].apply_batch(it_o, b)
    assert_same(it, f, it_o, trees, what="failing lists")
    offs = np.array([0, 0, 1, 1, 1, 2], dtype=np.uint64)
    st = f.apply_edits(offs, api.to_device(np.array([[5, 5, 5], [0, 1, 0]], dtype=np.int32)),
                       api.to_device(np.array([9, 10], dtype=np.uint16)))
    assert [int(s) for s in st] == [0, 1, 0, 0, 1]
    for k, x, v in ((1, [5, 5, 5], 9), (4, [0, 1, 0], 10)):
        b = trees[k].create_batch()
        b.set_many(np.array([x], dtype=np.int32), np.array([v], dtype=np.uint64))
        assert trees[k].apply_batch(it_o, b)
    assert_same(it, f, it_o, trees, what="the call after")
