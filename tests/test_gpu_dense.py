"""vx_trees_to_vec by cells of 8^3 voxels: mixed depths in one call, levels of detail, strides
that are not a tree's size, buffers that are not aligned to whole rows, trees of a few voxels
beside deep ones; what lies outside the trees stays as it was."""
import numpy as np
import pytest

import oracle_lib as O
from gpu_helpers import oracle_apply_dense

pytestmark = pytest.mark.gpu

MB = 1024 * 1024
NP = {1: np.uint8, 2: np.uint16, 4: np.uint32}


@pytest.fixture(scope="module", params=[1, 2, 4])
def world(request):
    """Trees of depth 1 to 7: sparse, dense, uniform below some level, a filled and an empty one."""
    import torch
    if not torch.cuda.is_available():
        pytest.skip("needs a GPU")
    from voxelis_amd import api, workloads as W
    w = request.param
    rng = np.random.default_rng(w)
    depths = [2, 5, 3, 6, 4, 7, 5, 5, 3, 2, 4]
    it, it_o = api.VoxInterner(w, 64 * MB), O.Interner(w, 64 * MB)
    f, trees = api.Forest(it, depths), [O.Tree(d) for d in depths]
    ms, vs = [], []
    for k, d in enumerate(depths):
        n = 1 << d
        if k % 3 == 0:
            dense = np.where(rng.random((n, n, n)) < 0.05, rng.integers(1, 200, (n, n, n)), 0)
            dense[0, 0, 0] = 3
        elif k % 3 == 1:
            dense = rng.integers(1, 4, (n, n, n))
        else:
            dense = np.zeros((n, n, n), dtype=np.int64)
            dense[: n // 2] = 7
            dense[-1, -1, -1] = 9
        m, v = W.dense_to_batch(dense.astype(NP[w]), d)
        ms.append(api.to_device(m))
        vs.append(api.to_device(v))
        if d == 7:  # past the reference's depths (and the oracle's): its own voxels are the check
            trees[k].to_vec = lambda it, lod=0, dense=dense: dense if lod == 0 else None
        elif k < 9:
            oracle_apply_dense(it_o, trees[k], m, v)
    hp = [k < 9 for k in range(len(depths))]
    st = f.apply(ms, vs, has_patches=hp, fills=[None] * 9 + [5, None])
    assert (st[:9] == 1).all()
    trees[9].fill(it_o, 5)
    return torch, it, f, it_o, trees, w


@pytest.mark.parametrize("lod", [0, 1, 2, 3])
@pytest.mark.parametrize("extra,shift", [(0, 0), (3, 0), (0, 1), (512, 5)])
def test_to_vec_strided(world, lod, extra, shift):
    from voxelis_amd import lib
    torch, it, f, it_o, trees, w = world
    size = [8 ** max(0, t.depth - lod) for t in trees]
    stride = max(size) + extra
    buf = torch.full(((f.n * stride + 64) * w,), 0xEE, dtype=torch.uint8, device="cuda")
    assert lib().vx_trees_to_vec(it.h, f.n, f.roots.data_ptr(), f.depths.data_ptr(), lod, stride,
                                 buf.data_ptr() + shift * w) == 0
    torch.cuda.synchronize()
    got = buf.cpu().numpy().view(NP[w])
    canary = np.frombuffer(b"\xee" * w, dtype=NP[w])[0]
    assert (got[:shift] == canary).all()
    for k, t in enumerate(trees):
        row = got[shift + k * stride: shift + (k + 1) * stride]
        want = t.to_vec(it_o, lod)
        if want is not None:
            assert np.array_equal(row[:size[k]], np.asarray(want).reshape(-1).astype(NP[w])), (k, t.depth)
        assert (row[size[k]:] == canary).all(), k


def test_to_vec_small_stride_skips_large_trees(world):
    """Trees that do not fit the stride are skipped and reported; the others are written."""
    from voxelis_amd import lib
    torch, it, f, it_o, trees, w = world
    for stride in (64, 512, 4100):
        buf = torch.full((f.n * stride * w,), 0xEE, dtype=torch.uint8, device="cuda")
        assert lib().vx_trees_to_vec(it.h, f.n, f.roots.data_ptr(), f.depths.data_ptr(), 0, stride, buf.data_ptr()) == 0
        torch.cuda.synchronize()
        got = buf.cpu().numpy().view(NP[w]).reshape(f.n, stride)
        for k, t in enumerate(trees):
            if 8 ** t.depth <= stride:
                assert np.array_equal(got[k, :8 ** t.depth], np.asarray(t.to_vec(it_o)).reshape(-1).astype(NP[w])), (stride, k)
            else:
                assert (got[k].view(np.uint8) == 0xEE).all(), (stride, k)
