"""The GC's last round follows whole subtrees inside a block: trees with more nodes under a
share of the front than a pass takes (children wait in the block's runs), every height of
tree, fills and clears of such trees, and nodes shared between trees that go one after the
other.  Afterwards only what the oracle holds is left."""
import numpy as np
import pytest

import oracle_lib as O
from gpu_helpers import assert_same, oracle_apply_dense

pytestmark = pytest.mark.gpu

MB = 1024 * 1024


@pytest.fixture(scope="module")
def vx():
    import torch
    if not torch.cuda.is_available():
        pytest.skip("needs a GPU")
    from voxelis_amd import api, workloads
    return api, workloads


def _random(W, rng, depth, share, np_dtype):
    n = 1 << depth
    dense = np.where(rng.random((n, n, n)) < share, rng.integers(1, 60000 if np_dtype == np.uint16 else 250, (n, n, n)), 0)
    dense[0, 0, 0] = 1
    return W.dense_to_batch(dense.astype(np_dtype), depth)


@pytest.mark.parametrize("gc_grid", [1, 3, 1024])
@pytest.mark.parametrize("depths", [[2], [3], [5], [6], [6, 6, 2, 5, 3, 6], [5] * 40])
def test_replaced_filled_and_cleared(vx, depths, gc_grid):
    api, W = vx
    rng = np.random.default_rng(len(depths) + depths[0])
    it, it_o = api.VoxInterner(2, 256 * MB), O.Interner(2, 256 * MB)
    it.set_tuning(gc_grid=gc_grid)
    f, trees = api.Forest(it, depths), [O.Tree(d) for d in depths]
    for step in range(3):
        # half of the trees are equal, so that their nodes are shared
        bat, same = [], {}
        for k, d in enumerate(depths):
            if k % 2 and d in same:
                bat.append(same[d])
            else:
                bat.append(_random(W, rng, d, 0.5 if step != 1 else 0.05, np.uint16))
                same[d] = bat[-1]
        want = []
        for t, b in zip(trees, bat):
            t.clear(it_o)  # (a partly written brick of the next step would meet a leaf brick)
            want.append(oracle_apply_dense(it_o, t, *b)[0])
        f.fill([0] * len(depths))
        st = f.apply([api.to_device(b[0]) for b in bat], [api.to_device(b[1]) for b in bat])
        assert all(want) and (st == 1).all()
        assert_same(it, f, it_o, trees, full_reads=False, what=f"step {step}")
        # whole trees replaced by one apply: every voxel written, few ids
        n = [1 << d for d in depths]
        full = [W.dense_to_batch(((np.arange(m ** 3) % (7 + step)) + 1).reshape(m, m, m).astype(np.uint16), d)
                for m, d in zip(n, depths)]
        st = f.apply([api.to_device(b[0]) for b in full], [api.to_device(b[1]) for b in full])
        assert (st == 1).all()
        for t, b in zip(trees, full):
            assert oracle_apply_dense(it_o, t, *b)[0]
        assert_same(it, f, it_o, trees, full_reads=False, what=f"step {step}, replaced")
    f.fill([0] * len(depths))
    for t in trees:
        t.clear(it_o)
    assert it.counts() == it_o.counts() == (0, 1)
    assert it.alive_nodes() == 1  # the empty branch
